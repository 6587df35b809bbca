// Pieces shared by the kernels whose rows stream through LDS.
#pragma once

#include <type_traits>

#include "bwd_common.h"

namespace evo {

typedef short s16x4s __attribute__((ext_vector_type(4)));

template <int D>
struct StreamGeo {
    static constexpr int C = D / 8, ROW = D * 2;   // 16-byte chunks, bytes per row
    // the low bits of the row reversed (head dim 64: of every second row, two rows share the 64 banks)
    static __device__ __forceinline__ int x(int r) {
        return D == 32 ? (r >> 2) & 3 : D == 64 ? ((r >> 1) & 1) << 2 | ((r >> 2) & 1) << 1 | ((r >> 3) & 1)
                       : (r & 1) << 3 | ((r >> 1) & 1) << 2 | ((r >> 2) & 1) << 1 | ((r >> 3) & 1);
    }
    static __device__ __forceinline__ int at(int r, int c) { return r * ROW + ((c ^ x(r)) << 4); }
};

__device__ __forceinline__ void wait_loads() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
// all but the youngest N of the wave's loads and stores (they end in the order they were issued)
template <int N>
__device__ __forceinline__ void wait_loads_but() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }
__device__ __forceinline__ void wait_loads_and_lds() { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory"); }
__device__ __forceinline__ void wait_lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
// 16 bytes per lane from memory into LDS, lane after lane from `dst` (uniform) on.  As an instruction the compiler does not know:
// it takes every read of LDS after one that it knows as depending on it and waits for all loads of the wave first, also where
// the read is of the other buffer, so that no stage was ever on its way while another was computed on.  The kernels wait
// themselves (`wait_loads`), before the barrier that opens the buffer.  What the compiler counts without these loads only
// makes its own waits longer: where a wave waits for a bias tile, nothing younger than that tile should be under way.
// (With the caller's fp32 rows kept unscaled until they are used, and dBias stored without a wait: B = 4, S = 1, N = 1024, H = 32, D = 64, step 691 ->
// 611 us; three waves per SIMD had hidden most of it elsewhere: S = N = 768, H = 4, D = 32 2311 -> 2284; S = 200, N = 640, H = 5, D = 64 1006 -> 987.)
// (s_nop: five states between a vector instruction's write of a scalar register and its use as an address.  Clobbers: the address register m0, which
// the compiler may want to keep something in, and memory, so that no read or write of the buffer that is filled moves across, with the waits' own.)
__device__ __forceinline__ void dma16(__amdgpu_buffer_rsrc_t rs, unsigned char *dst, int off) {
    const unsigned base = (unsigned)(uintptr_t)(__attribute__((address_space(3))) void *)dst;
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 4\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" : : "s"(base), "v"(off), "s"(rs) : "m0", "memory");
}

// The first N of `x`, loaded above, are wanted from here on: all are under way by now.  A load written where a condition decides about its use
// (`dead ? zeros : scaled(load)`) is put into that branch, asked for there and waited for at once: KSD round trips to memory one after the other
// ahead of a workgroup's first stage.  Training step, S = 64, N = 512, H = 4, D = 128 303 -> 294 us; S = 200, N = 640, H = 5, D = 64, fp32 bias 925 -> 921.
template <int N, typename V, int M>
__device__ __forceinline__ void asked_together(V (&x)[M]) {
    static_assert(N <= M, "");
#ifdef __HIP_DEVICE_COMPILE__
#pragma unroll
    for (int i = 0; i < N; ++i) asm volatile("" : "+v"(x[i]));
#endif
}

// Rows r0 .. r0 + ROWS - 1 of two arrays that share their strides, into LDS at `dst` and `dst` + ROWS rows: this wave's share
// of the 1 KB pieces.  Rows at or beyond N repeat the last one (their keys carry the mask floor, their queries
// probability zero).
template <int D, int ROWS, int NW>
__device__ __forceinline__ void dma_rows(__amdgpu_buffer_rsrc_t a, __amdgpu_buffer_rsrc_t b, unsigned char *dst, int r0, int N, int sn2,
                                         int wave, int lane) {
    typedef StreamGeo<D> G;
    constexpr int PIECES = ROWS * G::ROW / 1024, RPP = 1024 / G::ROW;   // rows per piece
#pragma unroll
    for (int i = 0; i < (PIECES + NW - 1) / NW; ++i) {
        const int m = wave + i * NW;
        if (PIECES % NW != 0 && m >= PIECES) break;   // (uniform over the wave)
        const int r = m * RPP + lane / G::C, c = (lane % G::C) ^ G::x(r);
        const int off = min(r0 + r, N - 1) * sn2 + c * 16;
        dma16(a, dst + m * 1024, off);
        dma16(b, dst + ROWS * G::ROW + m * 1024, off);
    }
}

// A operand of a product that contracts over 32 staged rows (kb .. kb + 31): row 32 dt + li of the transpose, the eight rows
// that step `ts` of an accumulator tile holds.
template <typename T, int D>
__device__ __forceinline__ typename Mfma<T>::v8 transposed(const unsigned char *tile, int kb, int ts, int dt, int lane) {
    typedef StreamGeo<D> G;
    const int g = lane >> 5, col = dt * 32 + 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
    typename Mfma<T>::v8 r;
#pragma unroll
    for (int h2 = 0; h2 < 2; ++h2) {
        const int row = kb + 16 * ts + 8 * h2 + 4 * g + ((lane & 15) >> 2);
        const s16x4s w = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (s16x4s __attribute__((address_space(3))) *)(tile + G::at(row, col >> 3) + (col & 7) * 2));
        const typename Mfma<T>::v4 v = __builtin_bit_cast(typename Mfma<T>::v4, w);
#pragma unroll
        for (int i = 0; i < 4; ++i) r[4 * h2 + i] = v[i];
    }
    return r;
}

// The bias tiles of one wave: its 32 rows (or, COLS, its 32 columns) against the tiles of the other side.
// BT: 1 prepared fp32 tiles (times log2 e), 2 prepared 16-bit tiles as given; the caller's rows (few S rows), 3 in fp32, 4 in the
// dtype of q, 5 in fp32 where rows start anywhere and end within a group of four.  A tile is kept as it comes from memory: whatever is done to it (`value`) would wait for it.
typedef f32x4 f32x4_at4 __attribute__((aligned(4)));   // (the load path takes 16 bytes at any multiple of four)
struct Rows16 {   // entry r, the 16 bits as given, in the low half of w[r] (columns) or two to a register (rows)
    unsigned w[16];
};
template <typename T, int BT, bool COLS>
struct BiasStream {
    typedef typename std::conditional<BT == 2, Tile16, typename std::conditional<BT == 4, Rows16, f32x16>::type>::type Tile;
    const float *t32;
    const unsigned short *t16;
    const char *mat;
    int64_t step;
    unsigned col, row_stride;
    float mul;
    int NT, N, g;
    __device__ __forceinline__ BiasStream(const EvoAttnParams &p, const Extra &e, const Prob &pr, int own_tile, int own_row, bool dead, int lane) {
        NT = (p.N + 31) / 32;
        N = p.N;
        g = lane >> 5;
        mul = dead ? 0.0f : kLog2e;
        const int bb = e.bias_batches > 1 ? pr.b : 0;
        if (BT >= 3) {
            row_stride = dead ? 0u : (unsigned)p.bias_stride_row;
            col = (unsigned)own_row;
            mat = dead ? dead_bias(p, e, pr.b, pr.s) : (const char *)p.bias + ((int64_t)bb * p.bias_stride_b + (int64_t)pr.h * p.bias_stride_h + (COLS ? 0 : (int64_t)own_row * p.bias_stride_row)) * (BT == 4 ? 2 : 4);
        } else {
            const int64_t first = (((int64_t)bb * p.H + pr.h) * NT * NT + (COLS ? own_tile : own_tile * NT)) * 1024;
            step = dead ? 0 : COLS ? (int64_t)NT * 1024 : 1024;
            if (BT == 1) t32 = (COLS ? e.bk : e.bq) + (dead ? e.zero_tile : first) + lane * 4;
            if (BT == 2) t16 = (COLS ? e.bk16 : e.bq16) + (dead ? e.zero_tile : first) + lane * 8;
        }
    }
    // tile t of the other side on its way; past the last one that one again (not used)
    __device__ __forceinline__ void load(int t, Tile &dst) const {
        t = min(t, NT - 1);
        if constexpr (BT == 1) load_tile32(t32 + t * step, dst);
        if constexpr (BT == 2) load_tile16(t16 + t * step, dst);
        // (rows: groups past column n repeat the last whole group, columns: rows past n - 1 the last one; as bias_tile_rows and _cols)
        if constexpr (BT >= 3 && COLS) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const unsigned o = (unsigned)min(t * 32 + crow(r, g), N - 1) * row_stride + col;
                if constexpr (BT != 4) dst[r] = ((const float *)mat)[o];
                else dst.w[r] = ((const unsigned short *)mat)[o];
            }
        }
        if (BT == 5 && !COLS && t * 32 + 32 > N) {   // (uniform: the last tile, entry by entry)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                if constexpr (BT == 5) dst[r] = ((const float *)mat)[min(t * 32 + crow(r, g), N - 1)];
            }
            return;
        }
        if constexpr (BT >= 3 && !COLS) {
#pragma unroll
            for (int rr = 0; rr < 4; ++rr) {
                const int c = min(t * 32 + 8 * rr + 4 * g, N - 4);
                if constexpr (BT != 4) {
                    const f32x4 v = BT == 5 ? *reinterpret_cast<const f32x4_at4 *>((const float *)mat + c) : *reinterpret_cast<const f32x4 *>((const float *)mat + c);
#pragma unroll
                    for (int i = 0; i < 4; ++i) dst[4 * rr + i] = v[i];
                } else {
                    const uint2 v = *reinterpret_cast<const uint2 *>((const unsigned short *)mat + c);
                    dst.w[2 * rr] = v.x;
                    dst.w[2 * rr + 1] = v.y;
                }
            }
        }
    }
    // as the C operand of the score product, log2 units
    __device__ __forceinline__ f32x16 value(const Tile &t) const {
        if constexpr (BT == 2) {
            f32x16 v;
            unpack_tile16<T>(t, mul, v);
            return v;
        } else if constexpr (BT == 3 || BT == 5) {
            f32x16 v;
#pragma unroll
            for (int r = 0; r < 16; ++r) v[r] = t[r] * mul;
            return v;
        } else if constexpr (BT == 4) {
            f32x16 v;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                float lo, hi;
                if (COLS) unpack2<T>(t.w[r], lo, hi);
                else unpack2<T>(t.w[r >> 1], lo, hi);
                v[r] = (COLS || r % 2 == 0 ? lo : hi) * mul;
            }
            return v;
        } else {
            return t;
        }
    }
    // For a tile that is a C operand as it lies (BT = 1): the wait for it, here; and, once the chain that begins with it is under way, the next one
    // into its registers (which that chain's first instruction must then not have taken for its result: 16 copies a tile otherwise).
    __device__ __forceinline__ void arrived(Tile &t) const {
#ifdef __HIP_DEVICE_COMPILE__   // (the host's own pass, which has no such registers, drops kernels' entries over it)
        if constexpr (BT == 1) asm volatile("" : "+v"(t));
#endif
    }
    __device__ __forceinline__ void refill(int n, Tile &t) const {
        if constexpr (BT == 1) {
#ifdef __HIP_DEVICE_COMPILE__
            asm volatile("" ::"v"(t));
#endif
            load(n, t);
        }
    }
    __device__ __forceinline__ const f32x16 &lies(const Tile &t, const f32x16 &taken) const {
        if constexpr (BT == 1) return t;
        else return taken;
    }
    // `value`, formed here: the wait for the tile stands before whatever the wave asks for next
    __device__ __forceinline__ f32x16 take(const Tile &t) const {
        f32x16 v = value(t);
        asm volatile("" : "+v"(v));
        return v;
    }
};
template <typename T, bool COLS>
struct BiasStream<T, 0, COLS> {
    struct Tile {};
    __device__ __forceinline__ BiasStream(const EvoAttnParams &, const Extra &, const Prob &, int, int, bool, int) {}
    __device__ __forceinline__ void load(int, Tile &) const {}
    __device__ __forceinline__ f32x16 value(const Tile &) const {
        f32x16 z;
#pragma unroll
        for (int r = 0; r < 16; ++r) z[r] = 0.0f;
        return z;
    }
    __device__ __forceinline__ f32x16 take(const Tile &t) const { return value(t); }
    __device__ __forceinline__ void arrived(Tile &) const {}
    __device__ __forceinline__ void refill(int, Tile &) const {}
};

}  // namespace evo
