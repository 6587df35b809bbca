// Pieces shared by the fp32 kernels, and their bodies on the fp32 matrix instruction (`v_mfma_f32_32x32x2_f32`, 256 flop per clock and CU, a fused
// multiply-add per product like the vector ALU's).
//
// A wave owns 32 rows of the result and walks over the other side's 32-row tiles, which its workgroup stages through LDS; nothing is prepared
// beforehand, and the mask, its shift and delta are formed where they are used, which keeps a small call at one launch forward and three or four
// backward.  Operands (lane l, g = l / 32): A holds row l % 32, B column l % 32, each one value of the two-deep contraction
// index g; C holds column l % 32, register r <-> row crow(r, g).  The order in which the contraction index is walked is
// free: where rows lie in memory (head dim contiguous) four steps take columns 8 j + 4 g .. + 3, i.e. one 16-byte read;
// a C tile goes back in as B operand register by register (step r: rows crow(r, 0) and crow(r, 1)), with no traffic between
// lanes, the other operand then read from row crow(r, g) of the staged tile, 32 consecutive columns at a time.
// LDS rows lie D + 4 floats apart: both kinds of read are free of bank conflicts.
#pragma once

#include "kernels.h"
#include "stream_common.h"

namespace evo {

__device__ __forceinline__ f32x16 mfma2(float a, float b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0); }
__device__ __forceinline__ f32x16 zero16() {
    f32x16 z;
#pragma unroll
    for (int i = 0; i < 16; ++i) z[i] = 0.0f;
    return z;
}

// Memory is addressed as a base that is the same for the workgroup plus a lane's 32-bit offset (one register instead
// of two; a problem's rows and a (b, h) bias matrix lie within 2^32 bytes, csrc/api.hip checks).
__device__ __forceinline__ f32x4 at4(const float *base, unsigned o) {
    return *reinterpret_cast<const f32x4 *>(reinterpret_cast<const char *>(base) + o * 4u);
}
__device__ __forceinline__ float at1(const float *base, unsigned o) {
    return *reinterpret_cast<const float *>(reinterpret_cast<const char *>(base) + o * 4u);
}
__device__ __forceinline__ void put4(float *base, unsigned o, f32x4 v) { *reinterpret_cast<f32x4 *>(reinterpret_cast<char *>(base) + o * 4u) = v; }

// A tile is 32 rows in LDS (`put`: four columns of a row; `clear`: the columns beyond D of `rows` rows); `Frag` is a row in registers, this
// lane's half of it in NP pieces of four columns (`col`); `rows` adds the tile's rows times the lane's, `cols` the tile's columns times a
// tile of results (its 32 rows).
template <int D>
struct Direct {
    static constexpr int DP = D < 32 ? 32 : D;      // columns of a staged row (zeros beyond D: a C tile has 32 rows of the head dim)
    static constexpr int PITCH = DP + 4, TILE = 32 * PITCH * 4, DT = DP / 32, NP = D / 8;
    static constexpr int NB = D <= 64 ? 2 : 1;      // stages in LDS (one barrier per tile with two)
    struct Frag { f32x4 f[NP]; };
    static __device__ __forceinline__ int col(int i, int g) { return 8 * i + 4 * g; }
    static __device__ __forceinline__ void put(unsigned char *tile, int row, int c, f32x4 v) { *reinterpret_cast<f32x4 *>(tile + (row * PITCH + c) * 4) = v; }
    static __device__ __forceinline__ void clear(unsigned char *tile, int rows, int threads) {
        if (D >= 32) return;
        constexpr int PAD = DP - D;
        for (int k = threadIdx.x; k < rows * PAD; k += threads) reinterpret_cast<float *>(tile)[k / PAD * PITCH + D + k % PAD] = 0.0f;
    }
    static __device__ __forceinline__ Frag frag(const f32x4 (&v)[NP]) {
        Frag r;
#pragma unroll
        for (int j = 0; j < NP; ++j) r.f[j] = v[j];
        return r;
    }
    static __device__ __forceinline__ Frag staged(const unsigned char *tile, int lane) {
        Frag r;
#pragma unroll
        for (int j = 0; j < NP; ++j) r.f[j] = *reinterpret_cast<const f32x4 *>(tile + ((lane & 31) * PITCH + col(j, lane >> 5)) * 4);
        return r;
    }
    // Operand reads stay one group of four steps ahead of the matrix instructions and no further (the scheduling barriers): left alone the
    // compiler asks for all of a tile's operands at once, which costs the registers of a fourth wave per SIMD.
    static __device__ __forceinline__ void rows(const unsigned char *tile, int lane, const Frag &b, f32x16 &c) {
        const float *row = reinterpret_cast<const float *>(tile) + (lane & 31) * PITCH + 4 * (lane >> 5);
        f32x4 a = *reinterpret_cast<const f32x4 *>(row);
#pragma unroll
        for (int j = 0; j < NP; ++j) {
            f32x4 next = a;
            if (j + 1 < NP) next = *reinterpret_cast<const f32x4 *>(row + 8 * (j + 1));
#pragma unroll
            for (int i = 0; i < 4; ++i) c = mfma2(a[i], b.f[j][i], c);
            a = next;
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    static __device__ __forceinline__ void cols(const unsigned char *tile, int lane, const f32x16 &w, f32x16 (&acc)[DT]) {
        const float *col0 = reinterpret_cast<const float *>(tile) + 4 * (lane >> 5) * PITCH + (lane & 31);
        constexpr int STEP = DT == 1 ? 4 : DT == 2 ? 2 : 1;   // rows per group of four reads
        auto at = [&](int r, int t) { return col0[(8 * (r >> 2) + (r & 3)) * PITCH + 32 * t]; };
        float a[STEP][DT];
#pragma unroll
        for (int i = 0; i < STEP; ++i)
#pragma unroll
            for (int t = 0; t < DT; ++t) a[i][t] = at(i, t);
#pragma unroll
        for (int r0 = 0; r0 < 16; r0 += STEP) {
            float next[STEP][DT];
#pragma unroll
            for (int i = 0; i < STEP; ++i)
#pragma unroll
                for (int t = 0; t < DT; ++t) next[i][t] = r0 + STEP < 16 ? at(r0 + STEP + i, t) : 0.0f;
#pragma unroll
            for (int i = 0; i < STEP; ++i)
#pragma unroll
                for (int t = 0; t < DT; ++t) acc[t] = mfma2(a[i][t], w[r0 + i], acc[t]);
#pragma unroll
            for (int i = 0; i < STEP; ++i)
#pragma unroll
                for (int t = 0; t < DT; ++t) a[i][t] = next[i][t];
            __builtin_amdgcn_sched_barrier(0);
        }
    }
};

// Mask values are carried no lower than this (the softmax's reference point starts there: nothing overflows), shifted where the
// whole row is dropped.
__device__ __forceinline__ float mask_entry(const EvoAttnParams &p, int b, int s, int key, float shift) {
    return fmaxf(mask_add(p, b, s, key) - shift, kMaskFloor);
}
// The same in two steps, so that nothing waits for the load where it is asked for: the entry as it lies in memory (beyond the row its last one), its value.
__device__ __forceinline__ unsigned mask_ask(const EvoAttnParams &p, int b, int s, int key) {
    if (p.mask_kind == EVO_MASK_NONE) return 0;
    const int64_t off = (int64_t)b * p.mask_stride_b + (int64_t)s * p.mask_stride_s + min(key, p.N - 1);
    if (p.mask_kind == EVO_MASK_F32) return ((const unsigned *)p.mask)[off];
    return p.mask_kind == EVO_MASK_BOOL ? ((const uint8_t *)p.mask)[off] : ((const unsigned short *)p.mask)[off];
}
__device__ __forceinline__ float mask_got(const EvoAttnParams &p, unsigned raw, int key, float shift) {
    float v = 0.0f;
    if (p.mask_kind == EVO_MASK_F32) v = __uint_as_float(raw);
    if (p.mask_kind == EVO_MASK_BOOL) v = raw ? 0.0f : -FLT_MAX;
    if (p.mask_kind == EVO_MASK_BF16) v = __uint_as_float(raw << 16);
    if (p.mask_kind == EVO_MASK_F16) v = (float)__builtin_bit_cast(f16_t, (unsigned short)raw);
    return fmaxf((key >= p.N ? -INFINITY : v) - shift, kMaskFloor);
}

// exp(t - m) as 2^(t log2(e) - m log2(e)), `ml` = m log2(e): one rounding of the exponent, like t - m has.
__device__ __forceinline__ float exp_less(float t, float ml) { return fast_exp2(fmaf(t, kLog2e, -ml)); }

// A row's pieces of this lane's half (see `col`; columns beyond D are zero).
template <class E, int D>
__device__ __forceinline__ void load_row(const float *base, unsigned row, int g, f32x4 (&f)[E::NP]) {
#pragma unroll
    for (int j = 0; j < E::NP; ++j) {
        f32x4 z = {0.0f, 0.0f, 0.0f, 0.0f};
        if (E::NP * 8 <= D || E::col(j, g) < D) z = at4(base, row + (unsigned)E::col(j, g));
        f[j] = z;
    }
}

// ROWS rows of two arrays through registers into LDS: `load` asks for rows r0 .. (zeros at and beyond N), `put` writes them.
template <class E, int D, int THREADS, int ROWS = 32>
struct Stage {
    static constexpr int PIECES = ROWS * D / 4, PER = (PIECES + THREADS - 1) / THREADS;
    f32x4 v[2][PER];
    __device__ __forceinline__ void load(const float *const (&src)[2], unsigned stride_n, int r0, int N) {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int k = threadIdx.x + i * THREADS, row = r0 + k / (D / 4);
            const bool ok = row < N && (PIECES % THREADS == 0 || k < PIECES);
            const unsigned o = (unsigned)row * stride_n + (unsigned)(k % (D / 4) * 4);
#pragma unroll
            for (int a = 0; a < 2; ++a) {
                f32x4 z = {0.0f, 0.0f, 0.0f, 0.0f};
                if (ok) z = at4(src[a], o);
                v[a][i] = z;
            }
        }
    }
    __device__ __forceinline__ void put(unsigned char *dst0, unsigned char *dst1) const {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int k = threadIdx.x + i * THREADS;
            if (PIECES % THREADS == 0 || k < PIECES) {
                E::put(dst0, k / (D / 4), k % (D / 4) * 4, v[0][i]);
                E::put(dst1, k / (D / 4), k % (D / 4) * 4, v[1][i]);
            }
        }
    }
};

// The shift of a problem's mask row (see common.h), from the row itself: every thread of the workgroup gets it.
template <int W>
__device__ __forceinline__ float block_shift(const EvoAttnParams &p, int b, int s, float *red) {
    if (p.mask_kind == EVO_MASK_NONE) return 0.0f;
    float mx = -INFINITY;
    for (int j = threadIdx.x; j < p.N; j += 64 * W) mx = fmaxf(mx, mask_add(p, b, s, j));
    mx = wave_max(mx);
    if (threadIdx.x % 64 == 0) red[threadIdx.x / 64] = mx;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < W; ++w) mx = fmaxf(mx, red[w]);
    return shift_from_max(mx);
}

// Four bias entries of one row at columns c .. c + 3; columns past the row's end repeat entries (their keys are masked).
__device__ __forceinline__ f32x4 bias4(const float *mat, unsigned row, int c, int N, bool vec) {
    f32x4 v;
    if (vec) return at4(mat, row + (unsigned)min(c, N - 4));
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = at1(mat, row + (unsigned)min(c + i, N - 1));
    return v;
}

__device__ __forceinline__ float both_halves(float x) { return x + __shfl_xor(x, 32); }

// What a workgroup keeps in LDS: tiles of two arrays, two values for each of a stage's rows, a value per wave.
template <int D>
struct DirectShared {
    typedef Direct<D> E;
    static constexpr int TILES = E::NB * 2 * E::TILE, BYTES = TILES + E::NB * 2 * 32 * 4 + 64;
    unsigned char *lds;
    __device__ __forceinline__ unsigned char *tile(int buf, int a) const { return lds + (buf * 2 + a) * E::TILE; }
    __device__ __forceinline__ float *row(int buf, int a) const { return reinterpret_cast<float *>(lds + TILES) + (buf * 2 + a) * 32; }
    __device__ __forceinline__ float *red() const { return reinterpret_cast<float *>(lds + TILES) + E::NB * 2 * 32; }
};

// Forward: a wave has 32 queries (lane = query), the keys come by tiles.
template <int D, int W, bool BIAS>
__device__ __forceinline__ void direct_fwd(const EvoAttnParams &p, int vec, unsigned char *lds) {
    typedef Direct<D> E;
    constexpr int NB = E::NB;
    const DirectShared<D> sh{lds};
    const unsigned nqb = (p.N + 32 * W - 1) / (32 * W), bid = xcd_remap(blockIdx.x, gridDim.x);
    const Prob pr = walk_problem(p, bid / nqb);
    const int wave = threadIdx.x / 64, l = threadIdx.x % 64, li = l % 32, g = l / 32;
    const int row = (bid % nqb) * 32 * W + wave * 32 + li, rowc = min(row, p.N - 1);
    const float *const src[2] = {(const float *)p.k + pr.base, (const float *)p.v + pr.base};
    Stage<E, D, 64 * W> st;
    const unsigned stride_n = (unsigned)p.stride_n, off = (unsigned)rowc * stride_n;
    st.load(src, stride_n, 0, p.N);
    f32x4 qv[E::NP];
    load_row<E, D>((const float *)p.q + pr.base, off, g, qv);
    const float *const bmat = BIAS ? (const float *)p.bias + pr.b * p.bias_stride_b + pr.h * p.bias_stride_h : nullptr;
    const unsigned brow = BIAS ? (unsigned)rowc * (unsigned)p.bias_stride_row : 0;
    E::clear(lds, NB * 2 * 32, 64 * W);
    const float shift = block_shift<W>(p, pr.b, pr.s, sh.red());
    const bool dead = shift != 0.0f;   // (of such a row the scores are the mask's)
    const float scale = dead ? 0.0f : p.scale;
    float mk = threadIdx.x < 32 ? mask_entry(p, pr.b, pr.s, threadIdx.x, shift) : 0.0f;
    const typename E::Frag q = E::frag(qv);
    f32x16 acc[E::DT];
#pragma unroll
    for (int t = 0; t < E::DT; ++t) acc[t] = zero16();
    float m = kMaskFloor, ml = kMaskFloor * kLog2e, sum = 0.0f;
    const int nt = (p.N + 31) / 32;
    for (int kt = 0; kt < nt; ++kt) {
        const int buf = NB == 2 ? kt & 1 : 0;
        if (NB == 1) __syncthreads();
        st.put(sh.tile(buf, 0), sh.tile(buf, 1));
        if (threadIdx.x < 32) sh.row(buf, 0)[threadIdx.x] = mk;
        __syncthreads();
        if (kt + 1 < nt) {
            st.load(src, stride_n, (kt + 1) * 32, p.N);
            if (threadIdx.x < 32) mk = mask_entry(p, pr.b, pr.s, (kt + 1) * 32 + threadIdx.x, shift);
        }
        f32x4 b[4] = {};
        if (BIAS && !dead) {
#pragma unroll
            for (int j = 0; j < 4; ++j) b[j] = bias4(bmat, brow, kt * 32 + 8 * j + 4 * g, p.N, vec);
        }
        f32x16 x = zero16();
        E::rows(sh.tile(buf, 0), l, q, x);
        float tmax = kMaskFloor;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const f32x4 mv = *reinterpret_cast<const f32x4 *>(sh.row(buf, 0) + 8 * j + 4 * g);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float t = fmaf(x[4 * j + i], scale, BIAS ? b[j][i] : 0.0f) + mv[i];
                x[4 * j + i] = t;
                tmax = fmaxf(tmax, t);
            }
        }
        tmax = fmaxf(tmax, __shfl_xor(tmax, 32));
        if (__any(tmax > m)) {   // (the sums are brought to a new maximum; most tiles have none)
            const float mn = fmaxf(m, tmax), alpha = exp_less(m, mn * kLog2e);
            m = mn;
            ml = mn * kLog2e;
            sum *= alpha;
#pragma unroll
            for (int t = 0; t < E::DT; ++t) acc[t] *= alpha;
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            x[r] = exp_less(x[r], ml);
            sum += x[r];
        }
        E::cols(sh.tile(buf, 1), l, x, acc);
    }
    sum = both_halves(sum);
    if (row < p.N) {
        const float inv = 1.0f / sum;
#pragma unroll
        for (int t = 0; t < E::DT; ++t)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int c = 32 * t + 8 * j + 4 * g;
                if (c >= D) continue;
                f32x4 o;
#pragma unroll
                for (int i = 0; i < 4; ++i) o[i] = acc[t][4 * j + i] * inv;
                if (p.o) put4((float *)p.o + pr.base, off + c, o);   // (with a gate the gated output may stand alone)
                if (p.gate) {
                    const f32x4 gl = at4((const float *)p.gate + pr.base, off + c);
#pragma unroll
                    for (int i = 0; i < 4; ++i) o[i] = o[i] / (1.0f + expf(-gl[i]));
                    put4((float *)p.o_gated + pr.base, off + c, o);
                }
            }
        if (g == 0) p.lse[pr.row0 + row] = m + logf(sum);
    }
}

// dQ: a wave has 32 queries, like the forward.  Also writes delta = rowsum(dO * O) unless the gate's pass has, and
// the mask shift of its (b, s) for the dBias kernel.
template <int D, int W, bool BIAS>
__device__ __forceinline__ void direct_dq(const EvoAttnParams &p, int vec, float *delta, float *shift_tab, int delta_given, unsigned char *lds) {
    typedef Direct<D> E;
    constexpr int NB = E::NB;
    const DirectShared<D> sh{lds};
    const unsigned nqb = (p.N + 32 * W - 1) / (32 * W), bid = xcd_remap(blockIdx.x, gridDim.x);
    const Prob pr = walk_problem(p, bid / nqb);
    const int wave = threadIdx.x / 64, l = threadIdx.x % 64, li = l % 32, g = l / 32;
    const int row = (bid % nqb) * 32 * W + wave * 32 + li, rowc = min(row, p.N - 1);
    const float *const src[2] = {(const float *)p.k + pr.base, (const float *)p.v + pr.base};
    Stage<E, D, 64 * W> st;
    const unsigned stride_n = (unsigned)p.stride_n, off = (unsigned)rowc * stride_n;
    st.load(src, stride_n, 0, p.N);
    f32x4 qv[E::NP], gv[E::NP];
    load_row<E, D>((const float *)p.q + pr.base, off, g, qv);
    load_row<E, D>((const float *)p.dout + pr.base, off, g, gv);
    const float lse = p.lse[pr.row0 + rowc];
    float dl = 0.0f;
    if (delta_given) {
        dl = delta[pr.row0 + rowc];
    } else {
        f32x4 ov[E::NP];
        load_row<E, D>((const float *)p.o + pr.base, off, g, ov);
#pragma unroll
        for (int j = 0; j < E::NP; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) dl = fmaf(gv[j][i], ov[j][i], dl);
        dl = both_halves(dl);
        if (g == 0 && row < p.N) delta[pr.row0 + row] = dl;
    }
    const float *const bmat = BIAS ? (const float *)p.bias + pr.b * p.bias_stride_b + pr.h * p.bias_stride_h : nullptr;
    const unsigned brow = BIAS ? (unsigned)rowc * (unsigned)p.bias_stride_row : 0;
    E::clear(lds, NB * 2 * 32, 64 * W);
    const float shift = block_shift<W>(p, pr.b, pr.s, sh.red());
    if (threadIdx.x == 0 && pr.h == 0 && bid % nqb == 0) shift_tab[pr.b * p.S + pr.s] = shift;
    const bool dead = shift != 0.0f;
    const float scale = dead ? 0.0f : p.scale;
    const float ll = ds_blocked(p, shift) ? INFINITY : lse * kLog2e;   // (no gradient through replaced scores: dS is zero)
    unsigned mk = threadIdx.x < 32 ? mask_ask(p, pr.b, pr.s, threadIdx.x) : 0;
    f32x4 b[4] = {};   // of the next tile: asked for once this one's are used
    auto ask_bias = [&](int kt) {
        if (!BIAS || dead) return;
#pragma unroll
        for (int j = 0; j < 4; ++j) b[j] = bias4(bmat, brow, kt * 32 + 8 * j + 4 * g, p.N, vec);
    };
    ask_bias(0);
    const typename E::Frag q = E::frag(qv), go = E::frag(gv);
    f32x16 acc[E::DT];
#pragma unroll
    for (int t = 0; t < E::DT; ++t) acc[t] = zero16();
    const int nt = (p.N + 31) / 32;
    for (int kt = 0; kt < nt; ++kt) {
        const int buf = NB == 2 ? kt & 1 : 0;
        if (NB == 1) __syncthreads();
        st.put(sh.tile(buf, 0), sh.tile(buf, 1));
        if (threadIdx.x < 32) sh.row(buf, 0)[threadIdx.x] = mask_got(p, mk, kt * 32 + threadIdx.x, shift);
        __syncthreads();
        if (kt + 1 < nt) {
            st.load(src, stride_n, (kt + 1) * 32, p.N);
            if (threadIdx.x < 32) mk = mask_ask(p, pr.b, pr.s, (kt + 1) * 32 + threadIdx.x);
        }
        f32x16 x = zero16();
        E::rows(sh.tile(buf, 0), l, q, x);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const f32x4 mv = *reinterpret_cast<const f32x4 *>(sh.row(buf, 0) + 8 * j + 4 * g);
#pragma unroll
            for (int i = 0; i < 4; ++i) x[4 * j + i] = exp_less(fmaf(x[4 * j + i], scale, BIAS ? b[j][i] : 0.0f) + mv[i], ll);
        }
        if (kt + 1 < nt) ask_bias(kt + 1);
        f32x16 dp = zero16();
        E::rows(sh.tile(buf, 1), l, go, dp);
#pragma unroll
        for (int r = 0; r < 16; ++r) x[r] *= dp[r] - dl;
        E::cols(sh.tile(buf, 0), l, x, acc);
    }
    if (row < p.N) {
#pragma unroll
        for (int t = 0; t < E::DT; ++t)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int c = 32 * t + 8 * j + 4 * g;
                if (c >= D) continue;
                f32x4 o;
#pragma unroll
                for (int i = 0; i < 4; ++i) o[i] = acc[t][4 * j + i] * p.scale;
                put4((float *)p.dq + pr.base, off + c, o);
            }
    }
}

// dK and dV: a wave has 32 keys (lane = key), the queries come by tiles with their dO, LSE and delta.  Also sums the dBias
// partials of the kernel before it (no launch of its own for that).
template <int D, int W, bool BIAS>
__device__ __forceinline__ void direct_dkdv(const EvoAttnParams &p, const Extra &e, unsigned char *lds) {
    const float *const delta = e.delta;
    typedef Direct<D> E;
    constexpr int NB = E::NB;
    const DirectShared<D> sh{lds};
    const unsigned nkb = (p.N + 32 * W - 1) / (32 * W), bid = xcd_remap(blockIdx.x, gridDim.x);
    const Prob pr = walk_problem(p, bid / nkb);
    const int wave = threadIdx.x / 64, l = threadIdx.x % 64, li = l % 32, g = l / 32;
    const int key = (bid % nkb) * 32 * W + wave * 32 + li, keyc = min(key, p.N - 1);
    const float *const src[2] = {(const float *)p.q + pr.base, (const float *)p.dout + pr.base};
    Stage<E, D, 64 * W> st;
    const unsigned stride_n = (unsigned)p.stride_n, off = (unsigned)keyc * stride_n;
    st.load(src, stride_n, 0, p.N);
    // LSE and delta of a stage's rows as asked for; LSE log2(e) (+inf at and beyond N: probability zero), delta
    auto row_ask = [&](int r0) {
        const int r = min(r0 + (int)(threadIdx.x & 31), p.N - 1);
        return threadIdx.x < 64 ? (threadIdx.x < 32 ? p.lse : delta)[pr.row0 + r] : 0.0f;
    };
    auto row_got = [&](float v, int r0) {
        const bool in = r0 + (int)(threadIdx.x & 31) < p.N;
        return threadIdx.x < 32 ? (in ? v * kLog2e : INFINITY) : (in ? v : 0.0f);
    };
    float rv = row_ask(0);
    f32x4 kv[E::NP], vv[E::NP];
    load_row<E, D>((const float *)p.k + pr.base, off, g, kv);
    load_row<E, D>((const float *)p.v + pr.base, off, g, vv);
    const float *const bmat = BIAS ? (const float *)p.bias + pr.b * p.bias_stride_b + pr.h * p.bias_stride_h : nullptr;
    E::clear(lds, NB * 2 * 32, 64 * W);
    const float shift = block_shift<W>(p, pr.b, pr.s, sh.red());
    const bool dead = shift != 0.0f, blocked = ds_blocked(p, shift);
    const float scale = dead ? 0.0f : p.scale, mk = mask_entry(p, pr.b, pr.s, keyc, shift);
    const typename E::Frag k = E::frag(kv), v = E::frag(vv);
    f32x16 dk[E::DT], dv[E::DT];
#pragma unroll
    for (int t = 0; t < E::DT; ++t) dk[t] = dv[t] = zero16();
    float dm = 0.0f;
    float b[16] = {};
    auto ask_bias = [&](int qt) {
        if (!BIAS || dead) return;
#pragma unroll
        for (int r = 0; r < 16; ++r) b[r] = at1(bmat, (unsigned)min(qt * 32 + crow(r, g), p.N - 1) * (unsigned)p.bias_stride_row + (unsigned)keyc);
    };
    // The bias a tile ahead, but not at head dim 64: its 16 registers are then live beside dP and dV, and 29 spilled (S = 512, N = 64, H = 8, a step: 367 us without,
    // 393 with; N = 32 196 / 208.  D = 128, N = 64 811 with, 882 without, D = 16 131 / 138, D = 8 114 / 118).
    constexpr bool AHEAD = D != 64;
    if (AHEAD) ask_bias(0);
    const int nt = (p.N + 31) / 32;
    for (int qt = 0; qt < nt; ++qt) {
        const int buf = NB == 2 ? qt & 1 : 0;
        if (NB == 1) __syncthreads();
        st.put(sh.tile(buf, 0), sh.tile(buf, 1));
        if (threadIdx.x < 64) sh.row(buf, 0)[threadIdx.x] = row_got(rv, qt * 32);
        __syncthreads();
        if (qt + 1 < nt) {
            st.load(src, stride_n, (qt + 1) * 32, p.N);
            rv = row_ask((qt + 1) * 32);
        }
        if (!AHEAD) {
#pragma unroll
            for (int r = 0; r < 16; ++r) b[r] = 0.0f;
            ask_bias(qt);
        }
        f32x16 x = zero16();
        E::rows(sh.tile(buf, 0), l, k, x);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const f32x4 lse = *reinterpret_cast<const f32x4 *>(sh.row(buf, 0) + 8 * j + 4 * g);
#pragma unroll
            for (int i = 0; i < 4; ++i) x[4 * j + i] = exp_less(fmaf(x[4 * j + i], scale, BIAS ? b[4 * j + i] : 0.0f) + mk, lse[i]);
        }
        if (AHEAD && qt + 1 < nt) ask_bias(qt + 1);
        if (!AHEAD) __builtin_amdgcn_sched_barrier(0);   // (the bias is used up before dP takes its registers)
        E::cols(sh.tile(buf, 1), l, x, dv);
        f32x16 ds = zero16();
        E::rows(sh.tile(buf, 1), l, v, ds);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const f32x4 dl = *reinterpret_cast<const f32x4 *>(sh.row(buf, 1) + 8 * j + 4 * g);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int r = 4 * j + i;
                ds[r] = blocked ? 0.0f : x[r] * (ds[r] - dl[i]);
                dm += ds[r];
            }
        }
        E::cols(sh.tile(buf, 0), l, ds, dk);
    }
    dm = both_halves(dm);
    if (key < p.N) {
        if (p.dmask && g == 0) e.dmask_part[pr.row0 + key] = dm;
#pragma unroll
        for (int t = 0; t < E::DT; ++t)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int c = 32 * t + 8 * j + 4 * g;
                if (c >= D) continue;
                f32x4 a, o;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    a[i] = dk[t][4 * j + i] * p.scale;
                    o[i] = dv[t][4 * j + i];
                }
                put4((float *)p.dk + pr.base, off + c, a);
                put4((float *)p.dv + pr.base, off + c, o);
            }
    }
}

// dBias partials: a workgroup has a block of queries and keys of one (b, h), a wave 32 queries and KT key tiles of it, and walks over a chunk of S rows with
// the sums in registers.  Forms S and dP again (two products): next to the dQ kernel's three that costs less than
// the partial results of workgroups that kept dBias for all the keys of their queries (N = 256: as many matrix
// instructions' time as 64 MB of partials take to write and sum).  Reads delta and the mask shifts that the dQ kernel wrote.
// (waves: two columns of KT key tiles)
template <int D, int KT>
struct DBiasGeo {
    static constexpr int BLK = 64 * KT, W = 2 * BLK / 32;
};
template <int D, int KT, bool BIAS>
__device__ __forceinline__ void direct_dbias(const EvoAttnParams &p, const float *delta, const float *shift_tab, float *part, int chunk, unsigned char *lds) {
    typedef Direct<D> E;
    typedef DBiasGeo<D, KT> R;
    constexpr int ROWS = R::BLK, TH = 64 * R::W, ARRAY = ROWS / 32 * E::TILE;
    float *const small = reinterpret_cast<float *>(lds + 4 * ARRAY);
    const int nb = (p.N + ROWS - 1) / ROWS;
    unsigned t = xcd_remap(blockIdx.x, gridDim.x);
    const int kb = t % nb; t /= nb;
    const int qb = t % nb; t /= nb;
    const int h = t % p.H; t /= p.H;
    const int b = t % p.B, ck = t / p.B;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), l = threadIdx.x % 64, li = l % 32, g = l / 32;
    const int q0 = qb * ROWS, k0 = kb * ROWS, qw = (wave >> 1) * 32, kw = (wave & 1) * 32 * KT;
    f32x16 acc[KT], bz[KT];
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) {
        acc[kt] = bz[kt] = zero16();
        if (BIAS) {
            const float *bmat = (const float *)p.bias + b * p.bias_stride_b + h * p.bias_stride_h;
#pragma unroll
            for (int r = 0; r < 16; ++r)
                bz[kt][r] = at1(bmat, (unsigned)min(q0 + qw + crow(r, g), p.N - 1) * (unsigned)p.bias_stride_row + (unsigned)min(k0 + kw + 32 * kt + li, p.N - 1));
        }
    }
    const int s0 = ck * chunk, s1 = min(s0 + chunk, p.S);
    Stage<E, D, TH, ROWS> sq, sk;
    constexpr int SV = (3 * ROWS + TH - 1) / TH;
    unsigned sv[SV];
    float shift, next_shift;
    auto load = [&](int s) {
        const unsigned pid = ((unsigned)b * p.H + h) * p.S + s;
        const Prob pr = decode_problem(p, pid);
        const float *const a[2] = {(const float *)p.q + pr.base, (const float *)p.dout + pr.base};
        const float *const c[2] = {(const float *)p.k + pr.base, (const float *)p.v + pr.base};
        sq.load(a, (unsigned)p.stride_n, q0, p.N);
        sk.load(c, (unsigned)p.stride_n, k0, p.N);
        next_shift = __int_as_float(uniform_load((const int *)shift_tab + b * p.S + s));
#pragma unroll
        for (int j = 0; j < SV; ++j) {
            const int k = threadIdx.x + j * TH, i = k % ROWS, q = min(q0 + i, p.N - 1);
            if (k < 2 * ROWS) sv[j] = __float_as_uint((k < ROWS ? p.lse : delta)[pr.row0 + q]);
            else if (k < 3 * ROWS) sv[j] = mask_ask(p, b, s, k0 + i);
        }
    };
    auto put_rows = [&] {
        shift = next_shift;
#pragma unroll
        for (int j = 0; j < SV; ++j) {
            const int k = threadIdx.x + j * TH, i = k % ROWS;
            const float f = __uint_as_float(sv[j]);
            if (k < ROWS) small[k] = q0 + i < p.N ? f * kLog2e : INFINITY;
            else if (k < 2 * ROWS) small[k] = q0 + i < p.N ? f : 0.0f;
            else if (k < 3 * ROWS) small[k] = mask_got(p, sv[j], k0 + i, shift);
        }
    };
    load(s0);   // (nothing reads the columns beyond D)
    for (int s = s0; s < s1; ++s) {
        __syncthreads();
        sq.put(lds, lds + ARRAY);
        sk.put(lds + 2 * ARRAY, lds + 3 * ARRAY);
        put_rows();
        __syncthreads();
        if (s + 1 < s1) load(s + 1);
        if (ds_blocked(p, shift)) continue;
        const float scale = shift != 0.0f ? 0.0f : p.scale, bs = shift != 0.0f ? 0.0f : 1.0f;
        if (q0 + qw >= p.N) continue;
        const unsigned char *const qt = lds + qw / 32 * E::TILE, *const kt0 = lds + 2 * ARRAY + kw / 32 * E::TILE;
#pragma unroll
        for (int kt = 0; kt < KT; ++kt) {
            if (k0 + kw + 32 * kt >= p.N) break;
            const float mk = small[2 * ROWS + kw + 32 * kt + li];
            f32x16 x = zero16();
            E::rows(qt, l, E::staged(kt0 + kt * E::TILE, l), x);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const f32x4 lse = *reinterpret_cast<const f32x4 *>(&small[qw + 8 * j + 4 * g]);
#pragma unroll
                for (int i = 0; i < 4; ++i) x[4 * j + i] = exp_less(fmaf(bz[kt][4 * j + i], bs, x[4 * j + i] * scale) + mk, lse[i]);
            }
            f32x16 dp = zero16();
            E::rows(qt + ARRAY, l, E::staged(kt0 + ARRAY + kt * E::TILE, l), dp);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const f32x4 dl = *reinterpret_cast<const f32x4 *>(&small[ROWS + qw + 8 * j + 4 * g]);
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[kt][4 * j + i] = fmaf(x[4 * j + i], dp[4 * j + i] - dl[i], acc[kt][4 * j + i]);
            }
        }
    }
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) {
        const int key = k0 + kw + 32 * kt + li;
        if (key >= p.N) break;
        float *out = part + (((int64_t)ck * p.B + b) * p.H + h) * p.N * p.N + key;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int q = q0 + qw + crow(r, g);
            if (q < p.N) out[(int64_t)q * p.N] = acc[kt][r];
        }
    }
}

}  // namespace evo
