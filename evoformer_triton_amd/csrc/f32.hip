// The fp32 kernels: every product and sum in fp32, on the fp32 matrix instruction (`v_mfma_f32_32x32x2_f32`,
// 256 flop per clock and CU, a fused multiply-add per product like the vector ALU's).
//
// What bounds them is that instruction: a 32 x 32 tile of scores at head dim 32 takes 16 of them (1024 clocks
// of a SIMD) per product, two products in the forward, three for dQ, four for dK/dV and two for dBias, against
// some 600 clocks of vector work (one exponential per score and kernel).  So the work is split by
// tiles alone: a wave owns 32 rows of the result and walks over the other side's 32-row tiles, which its workgroup
// stages through LDS; nothing is prepared beforehand, and the mask, its shift and delta are formed where they are
// used, which keeps a small call at one launch forward and three or four backward.
//
// Operands (lane l, g = l / 32): A holds row l % 32, B column l % 32, each one value of the two-deep contraction
// index g; C holds column l % 32, register r <-> row crow(r, g).  The order in which the contraction index is walked is
// free: where rows lie in memory (head dim contiguous) four steps take columns 8 j + 4 g .. + 3, i.e. one 16-byte read;
// a C tile goes back in as B operand register by register (step r: rows crow(r, 0) and crow(r, 1)), with no traffic between
// lanes, the other operand then read from row crow(r, g) of the staged tile, 32 consecutive columns at a time.
// LDS rows lie D + 4 floats apart: both kinds of read are free of bank conflicts.
//
// B = 1, S = 64, N = 256, H = 8, D = 32, against one row per thread on the vector ALU (csrc/generic.hip): forward 304 -> 54 us, dQ
// (with delta) 325 -> 76 us, dK/dV 375 -> 97 us, dBias 913 -> 64 us; with S = 512 the forward runs at 98 TFLOP/s (a large fp32
// matrix product of the library: 135) and the whole backward's nine products at 102.  What is left is the vector work that does
// not overlap, and about 10 us per launch that do not depend on the rows.
#include "bwd_common.h"
#include "kernels.h"

namespace evo {

template <int D>
struct F32 {
    static constexpr int DP = D < 32 ? 32 : D;      // columns of a staged row (zeros beyond D: a C tile has 32 rows of the head dim)
    static constexpr int PITCH = DP + 4;
    static constexpr int J = D / 8;                 // 16-byte pieces of a row in one half of a wave
    static constexpr int DT = DP / 32;
    static constexpr int TILE = 32 * PITCH;
};

__device__ __forceinline__ f32x16 mfma2(float a, float b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0); }
__device__ __forceinline__ f32x16 zero16() {
    f32x16 z;
#pragma unroll
    for (int i = 0; i < 16; ++i) z[i] = 0.0f;
    return z;
}

// Mask values are carried no lower than this (the softmax's reference point starts there: nothing overflows), shifted where the
// whole row is dropped.
__device__ __forceinline__ float mask_entry(const EvoAttnParams &p, int b, int s, int key, float shift) {
    return fmaxf(mask_add(p, b, s, key) - shift, kMaskFloor);
}

// exp(t - m) as 2^(t log2(e) - m log2(e)), `ml` = m log2(e): one rounding of the exponent, like t - m has.
__device__ __forceinline__ float exp_less(float t, float ml) { return fast_exp2(fmaf(t, kLog2e, -ml)); }

// Memory is addressed as a base that is the same for the workgroup plus a lane's 32-bit offset (one register instead
// of two; a problem's rows and a (b, h) bias matrix lie within 2^32 bytes, csrc/api.hip checks).
__device__ __forceinline__ f32x4 at4(const float *base, unsigned o) {
    return *reinterpret_cast<const f32x4 *>(reinterpret_cast<const char *>(base) + o * 4u);
}
__device__ __forceinline__ float at1(const float *base, unsigned o) {
    return *reinterpret_cast<const float *>(reinterpret_cast<const char *>(base) + o * 4u);
}
__device__ __forceinline__ void put4(float *base, unsigned o, f32x4 v) { *reinterpret_cast<f32x4 *>(reinterpret_cast<char *>(base) + o * 4u) = v; }

// A row's pieces of this lane's half: columns 8 j + 4 g .. + 3.
template <int D>
__device__ __forceinline__ void load_frag(const float *base, unsigned row, int g, f32x4 (&f)[F32<D>::J]) {
#pragma unroll
    for (int j = 0; j < F32<D>::J; ++j) f[j] = at4(base, row + (unsigned)(8 * j + 4 * g));
}

// c += rows of a staged tile (lane's row at `row`, 4 g included) times the lane's column `b`.  Operand reads stay one group of
// four steps ahead of the matrix instructions and no further (the scheduling barriers): left alone the compiler asks for
// all of a tile's operands at once, which costs the registers of a fourth wave per SIMD.
template <int D>
__device__ __forceinline__ void mma_rows(const float *row, const f32x4 (&b)[F32<D>::J], f32x16 &c) {
    f32x4 a = *reinterpret_cast<const f32x4 *>(row);
#pragma unroll
    for (int j = 0; j < F32<D>::J; ++j) {
        f32x4 next = a;
        if (j + 1 < F32<D>::J) next = *reinterpret_cast<const f32x4 *>(row + 8 * (j + 1));
#pragma unroll
        for (int i = 0; i < 4; ++i) c = mfma2(a[i], b[j][i], c);
        a = next;
        __builtin_amdgcn_sched_barrier(0);
    }
}

// acc[t] += (columns 32 t .. of the staged tile)^T times the tile w (rows of both: the tile's 32 rows); `col` points at row 4 g,
// column l % 32.
template <int D>
__device__ __forceinline__ void mma_cols(const float *col, const f32x16 &w, f32x16 (&acc)[F32<D>::DT]) {
    constexpr int DT = F32<D>::DT, PITCH = F32<D>::PITCH, STEP = DT == 1 ? 4 : DT == 2 ? 2 : 1;   // rows per group of four reads
    auto at = [&](int r, int t) { return col[(8 * (r >> 2) + (r & 3)) * PITCH + 32 * t]; };
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

// 32-row tiles of NA arrays through registers into LDS: `load` asks for rows r0 .. r0 + 31 (zeros at and beyond N), `put`
// writes them.
template <int D, int NA, int THREADS, int ROWS = 32>
struct Stage {
    static constexpr int PIECES = ROWS * D / 4, PER = (PIECES + THREADS - 1) / THREADS;
    f32x4 v[NA][PER];
    __device__ __forceinline__ void load(const float *const (&src)[NA], unsigned stride_n, int r0, int N) {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int k = threadIdx.x + i * THREADS, row = r0 + k / (D / 4);
            const bool ok = row < N && (PIECES % THREADS == 0 || k < PIECES);
            const unsigned o = (unsigned)row * stride_n + (unsigned)(k % (D / 4) * 4);
#pragma unroll
            for (int a = 0; a < NA; ++a) {
                f32x4 z = {0.0f, 0.0f, 0.0f, 0.0f};
                if (ok) z = at4(src[a], o);
                v[a][i] = z;
            }
        }
    }
    template <int PITCH>
    __device__ __forceinline__ void put(float *const (&dst)[NA]) const {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int k = threadIdx.x + i * THREADS;
            if (PIECES % THREADS == 0 || k < PIECES) {
#pragma unroll
                for (int a = 0; a < NA; ++a) *reinterpret_cast<f32x4 *>(dst[a] + k / (D / 4) * PITCH + k % (D / 4) * 4) = v[a][i];
            }
        }
    }
};

// The columns D .. 31 of staged rows (head dims below 32): zero, once.
template <int D>
__device__ __forceinline__ void clear_pad(float *tiles, int rows, int threads) {
    if (D >= 32) return;
    constexpr int PAD = F32<D>::DP - D;
    for (int k = threadIdx.x; k < rows * PAD; k += threads) tiles[k / PAD * F32<D>::PITCH + D + k % PAD] = 0.0f;
}

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

// Forward: a wave has 32 queries (lane = query), the keys come by tiles.
template <int D, int W, bool BIAS>
__global__ void __launch_bounds__(64 * W, D <= 32 && W == 4 ? 4 : D <= 64 ? 2 : 1) f32_fwd(EvoAttnParams p, int vec) {
    typedef F32<D> C;
    constexpr int NB = D <= 64 ? 2 : 1;   // stages in LDS (one barrier per tile with two)
    __shared__ __align__(16) float tiles[NB][2][C::TILE];
    __shared__ __align__(16) float mrow[NB][32];
    __shared__ float red[W];
    const unsigned nqb = (p.N + 32 * W - 1) / (32 * W), bid = xcd_remap(blockIdx.x, gridDim.x);
    const Prob pr = walk_problem(p, bid / nqb);
    const int wave = threadIdx.x / 64, l = threadIdx.x % 64, li = l % 32, g = l / 32;
    const int row = (bid % nqb) * 32 * W + wave * 32 + li, rowc = min(row, p.N - 1);
    const float *const src[2] = {(const float *)p.k + pr.base, (const float *)p.v + pr.base};
    Stage<D, 2, 64 * W> st;
    const unsigned stride_n = (unsigned)p.stride_n, off = (unsigned)rowc * stride_n;
    st.load(src, stride_n, 0, p.N);
    f32x4 q[C::J];
    load_frag<D>((const float *)p.q + pr.base, off, g, q);
    const float *const bmat = BIAS ? (const float *)p.bias + pr.b * p.bias_stride_b + pr.h * p.bias_stride_h : nullptr;
    const unsigned brow = BIAS ? (unsigned)rowc * (unsigned)p.bias_stride_row : 0;
    clear_pad<D>(&tiles[0][0][0], NB * 2 * 32, 64 * W);
    const float shift = block_shift<W>(p, pr.b, pr.s, red);
    const bool dead = shift != 0.0f;   // (of such a row the scores are the mask's)
    const float scale = dead ? 0.0f : p.scale;
    float mk = threadIdx.x < 32 ? mask_entry(p, pr.b, pr.s, threadIdx.x, shift) : 0.0f;
    f32x16 acc[C::DT];
#pragma unroll
    for (int t = 0; t < C::DT; ++t) acc[t] = zero16();
    float m = kMaskFloor, ml = kMaskFloor * kLog2e, sum = 0.0f;
    const int nt = (p.N + 31) / 32;
    for (int kt = 0; kt < nt; ++kt) {
        const int buf = NB == 2 ? kt & 1 : 0;
        if (NB == 1) __syncthreads();
        {
            float *const dst[2] = {tiles[buf][0], tiles[buf][1]};
            st.template put<C::PITCH>(dst);
            if (threadIdx.x < 32) mrow[buf][threadIdx.x] = mk;
        }
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
        mma_rows<D>(&tiles[buf][0][li * C::PITCH + 4 * g], q, x);
        float tmax = kMaskFloor;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const f32x4 mv = *reinterpret_cast<const f32x4 *>(&mrow[buf][8 * j + 4 * g]);
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
            for (int t = 0; t < C::DT; ++t) acc[t] *= alpha;
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            x[r] = exp_less(x[r], ml);
            sum += x[r];
        }
        mma_cols<D>(&tiles[buf][1][4 * g * C::PITCH + li], x, acc);
    }
    sum = both_halves(sum);
    if (row >= p.N) return;
    const float inv = 1.0f / sum;
#pragma unroll
    for (int t = 0; t < C::DT; ++t)
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

// dQ: a wave has 32 queries, like the forward.  Also writes delta = rowsum(dO * O) unless the gate's pass has, and
// the mask shift of its (b, s) for the dBias kernel.
template <int D, int W, bool BIAS>
__global__ void __launch_bounds__(64 * W, D <= 64 ? 2 : 1) f32_dq(EvoAttnParams p, int vec, float *delta, float *shift_tab, int delta_given) {
    typedef F32<D> C;
    constexpr int NB = D <= 64 ? 2 : 1;
    __shared__ __align__(16) float tiles[NB][2][C::TILE];
    __shared__ __align__(16) float mrow[NB][32];
    __shared__ float red[W];
    const unsigned nqb = (p.N + 32 * W - 1) / (32 * W), bid = xcd_remap(blockIdx.x, gridDim.x);
    const Prob pr = walk_problem(p, bid / nqb);
    const int wave = threadIdx.x / 64, l = threadIdx.x % 64, li = l % 32, g = l / 32;
    const int row = (bid % nqb) * 32 * W + wave * 32 + li, rowc = min(row, p.N - 1);
    const float *const src[2] = {(const float *)p.k + pr.base, (const float *)p.v + pr.base};
    Stage<D, 2, 64 * W> st;
    const unsigned stride_n = (unsigned)p.stride_n, off = (unsigned)rowc * stride_n;
    st.load(src, stride_n, 0, p.N);
    f32x4 q[C::J], go[C::J];
    load_frag<D>((const float *)p.q + pr.base, off, g, q);
    load_frag<D>((const float *)p.dout + pr.base, off, g, go);
    const float lse = p.lse[pr.row0 + rowc];
    float dl = 0.0f;
    if (delta_given) {
        dl = delta[pr.row0 + rowc];
    } else {
#pragma unroll
        for (int j = 0; j < C::J; ++j) {
            const f32x4 o = at4((const float *)p.o + pr.base, off + (unsigned)(8 * j + 4 * g));
#pragma unroll
            for (int i = 0; i < 4; ++i) dl = fmaf(go[j][i], o[i], dl);
        }
        dl = both_halves(dl);
        if (g == 0 && row < p.N) delta[pr.row0 + row] = dl;
    }
    const float *const bmat = BIAS ? (const float *)p.bias + pr.b * p.bias_stride_b + pr.h * p.bias_stride_h : nullptr;
    const unsigned brow = BIAS ? (unsigned)rowc * (unsigned)p.bias_stride_row : 0;
    clear_pad<D>(&tiles[0][0][0], NB * 2 * 32, 64 * W);
    const float shift = block_shift<W>(p, pr.b, pr.s, red);
    if (threadIdx.x == 0 && pr.h == 0 && bid % nqb == 0) shift_tab[pr.b * p.S + pr.s] = shift;
    const bool dead = shift != 0.0f;
    const float scale = dead ? 0.0f : p.scale;
    const float ll = ds_blocked(p, shift) ? INFINITY : lse * kLog2e;   // (no gradient through replaced scores: dS is zero)
    float mk = threadIdx.x < 32 ? mask_entry(p, pr.b, pr.s, threadIdx.x, shift) : 0.0f;
    f32x16 acc[C::DT];
#pragma unroll
    for (int t = 0; t < C::DT; ++t) acc[t] = zero16();
    const int nt = (p.N + 31) / 32;
    for (int kt = 0; kt < nt; ++kt) {
        const int buf = NB == 2 ? kt & 1 : 0;
        if (NB == 1) __syncthreads();
        {
            float *const dst[2] = {tiles[buf][0], tiles[buf][1]};
            st.template put<C::PITCH>(dst);
            if (threadIdx.x < 32) mrow[buf][threadIdx.x] = mk;
        }
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
        mma_rows<D>(&tiles[buf][0][li * C::PITCH + 4 * g], q, x);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const f32x4 mv = *reinterpret_cast<const f32x4 *>(&mrow[buf][8 * j + 4 * g]);
#pragma unroll
            for (int i = 0; i < 4; ++i) x[4 * j + i] = exp_less(fmaf(x[4 * j + i], scale, BIAS ? b[j][i] : 0.0f) + mv[i], ll);
        }
        __builtin_amdgcn_sched_barrier(0);   // (the bias is used up before dP takes its registers)
        f32x16 dp = zero16();
        mma_rows<D>(&tiles[buf][1][li * C::PITCH + 4 * g], go, dp);
#pragma unroll
        for (int r = 0; r < 16; ++r) x[r] *= dp[r] - dl;
        mma_cols<D>(&tiles[buf][0][4 * g * C::PITCH + li], x, acc);
    }
    if (row >= p.N) return;
#pragma unroll
    for (int t = 0; t < C::DT; ++t)
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

// dK and dV: a wave has 32 keys (lane = key), the queries come by tiles with their dO, LSE and delta.  Also sums the dBias
// partials of the kernel before it (no launch of its own for that).
template <int D, int W, bool BIAS>
__global__ void __launch_bounds__(64 * W, D <= 64 ? 2 : 1) f32_dkdv(EvoAttnParams p, Extra e) {
    const float *const delta = e.delta;
    typedef F32<D> C;
    constexpr int NB = D <= 64 ? 2 : 1;
    __shared__ __align__(16) float tiles[NB][2][C::TILE];
    __shared__ __align__(16) float rows[NB][2][32];   // LSE log2(e) (+inf at and beyond N: probability zero), delta
    __shared__ float red[W];
    const unsigned nkb = (p.N + 32 * W - 1) / (32 * W), bid = xcd_remap(blockIdx.x, gridDim.x);
    const Prob pr = walk_problem(p, bid / nkb);
    const int wave = threadIdx.x / 64, l = threadIdx.x % 64, li = l % 32, g = l / 32;
    const int key = (bid % nkb) * 32 * W + wave * 32 + li, keyc = min(key, p.N - 1);
    const float *const src[2] = {(const float *)p.q + pr.base, (const float *)p.dout + pr.base};
    Stage<D, 2, 64 * W> st;
    const unsigned stride_n = (unsigned)p.stride_n, off = (unsigned)keyc * stride_n;
    st.load(src, stride_n, 0, p.N);
    auto row_value = [&](int r0) {
        const int r = r0 + (threadIdx.x & 31);
        if (threadIdx.x >= 64) return 0.0f;
        return threadIdx.x < 32 ? (r < p.N ? p.lse[pr.row0 + r] * kLog2e : INFINITY) : (r < p.N ? delta[pr.row0 + r] : 0.0f);
    };
    float rv = row_value(0);
    if (e.dbias_chunks) sum_dbias_partials<64 * W>(p, e, threadIdx.x);
    f32x4 k[C::J], v[C::J];
    load_frag<D>((const float *)p.k + pr.base, off, g, k);
    load_frag<D>((const float *)p.v + pr.base, off, g, v);
    const float *const bmat = BIAS ? (const float *)p.bias + pr.b * p.bias_stride_b + pr.h * p.bias_stride_h : nullptr;
    clear_pad<D>(&tiles[0][0][0], NB * 2 * 32, 64 * W);
    const float shift = block_shift<W>(p, pr.b, pr.s, red);
    const bool dead = shift != 0.0f, blocked = ds_blocked(p, shift);
    const float scale = dead ? 0.0f : p.scale, mk = mask_entry(p, pr.b, pr.s, keyc, shift);
    f32x16 dk[C::DT], dv[C::DT];
#pragma unroll
    for (int t = 0; t < C::DT; ++t) dk[t] = dv[t] = zero16();
    float dm = 0.0f;
    const int nt = (p.N + 31) / 32;
    for (int qt = 0; qt < nt; ++qt) {
        const int buf = NB == 2 ? qt & 1 : 0;
        if (NB == 1) __syncthreads();
        {
            float *const dst[2] = {tiles[buf][0], tiles[buf][1]};
            st.template put<C::PITCH>(dst);
            if (threadIdx.x < 64) rows[buf][threadIdx.x / 32][threadIdx.x & 31] = rv;
        }
        __syncthreads();
        if (qt + 1 < nt) {
            st.load(src, stride_n, (qt + 1) * 32, p.N);
            rv = row_value((qt + 1) * 32);
        }
        float b[16] = {};
        if (BIAS && !dead) {
#pragma unroll
            for (int r = 0; r < 16; ++r) b[r] = at1(bmat, (unsigned)min(qt * 32 + crow(r, g), p.N - 1) * (unsigned)p.bias_stride_row + (unsigned)keyc);
        }
        f32x16 x = zero16();
        mma_rows<D>(&tiles[buf][0][li * C::PITCH + 4 * g], k, x);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const f32x4 lse = *reinterpret_cast<const f32x4 *>(&rows[buf][0][8 * j + 4 * g]);
#pragma unroll
            for (int i = 0; i < 4; ++i) x[4 * j + i] = exp_less(fmaf(x[4 * j + i], scale, BIAS ? b[4 * j + i] : 0.0f) + mk, lse[i]);
        }
        __builtin_amdgcn_sched_barrier(0);   // (the bias is used up before dP takes its registers)
        mma_cols<D>(&tiles[buf][1][4 * g * C::PITCH + li], x, dv);
        f32x16 ds = zero16();
        mma_rows<D>(&tiles[buf][1][li * C::PITCH + 4 * g], v, ds);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const f32x4 dl = *reinterpret_cast<const f32x4 *>(&rows[buf][1][8 * j + 4 * g]);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int r = 4 * j + i;
                ds[r] = blocked ? 0.0f : x[r] * (ds[r] - dl[i]);
                dm += ds[r];
            }
        }
        mma_cols<D>(&tiles[buf][0][4 * g * C::PITCH + li], ds, dk);
    }
    dm = both_halves(dm);
    if (key >= p.N) return;
    if (p.dmask && g == 0) e.dmask_part[pr.row0 + key] = dm;
#pragma unroll
    for (int t = 0; t < C::DT; ++t)
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

// dBias partials: a workgroup has 64 queries x 64 keys of one (b, h), a wave 32 x 32 of them, and walks over a chunk of S rows with
// the sums in registers.  Forms S and dP again (two products): next to the dQ kernel's three that costs less than
// the partial results of workgroups that kept dBias for all the keys of their queries (N = 256: as many matrix
// instructions' time as 64 MB of partials take to write and sum).  Reads delta and the mask shifts that the dQ kernel wrote.
template <int D, bool BIAS>
__global__ void __launch_bounds__(256, D <= 64 ? 2 : 1) f32_dbias(EvoAttnParams p, const float *delta, const float *shift_tab, float *part, int chunk) {
    constexpr int PITCH = D + 4, ROWS = 64;
    extern __shared__ __align__(16) float lds[];   // Q, dO, K, V: ROWS x PITCH each; LSE, delta, mask: 64 each
    float *const tile = lds, *const small = lds + 4 * ROWS * PITCH;
    const int nb = (p.N + 63) / 64;
    unsigned t = xcd_remap(blockIdx.x, gridDim.x);
    const int kb = t % nb; t /= nb;
    const int qb = t % nb; t /= nb;
    const int h = t % p.H; t /= p.H;
    const int b = t % p.B, ck = t / p.B;
    const int wave = threadIdx.x / 64, l = threadIdx.x % 64, li = l % 32, g = l / 32;
    const int q0 = qb * 64, k0 = kb * 64, qw = (wave >> 1) * 32, kw = (wave & 1) * 32;
    const int key = min(k0 + kw + li, p.N - 1);
    f32x16 acc = zero16(), bz = zero16();
    if (BIAS) {
        const float *bmat = (const float *)p.bias + b * p.bias_stride_b + h * p.bias_stride_h;
#pragma unroll
        for (int r = 0; r < 16; ++r) bz[r] = at1(bmat, (unsigned)min(q0 + qw + crow(r, g), p.N - 1) * (unsigned)p.bias_stride_row + (unsigned)key);
    }
    const int s0 = ck * chunk, s1 = min(s0 + chunk, p.S);
    Stage<D, 2, 256, ROWS> sq, sk;
    float sv = 0.0f;
    auto load = [&](int s) {
        const unsigned pid = ((unsigned)b * p.H + h) * p.S + s;
        const Prob pr = decode_problem(p, pid);
        const float *const a[2] = {(const float *)p.q + pr.base, (const float *)p.dout + pr.base};
        const float *const c[2] = {(const float *)p.k + pr.base, (const float *)p.v + pr.base};
        sq.load(a, (unsigned)p.stride_n, q0, p.N);
        sk.load(c, (unsigned)p.stride_n, k0, p.N);
        const int i = threadIdx.x & 63;
        if (threadIdx.x < 64) sv = q0 + i < p.N ? p.lse[pr.row0 + q0 + i] * kLog2e : INFINITY;
        else if (threadIdx.x < 128) sv = q0 + i < p.N ? delta[pr.row0 + q0 + i] : 0.0f;
        else if (threadIdx.x < 192) sv = mask_entry(p, b, s, k0 + i, shift_tab[b * p.S + s]);
    };
    auto mma_pair = [](const float *a, const float *b, f32x16 &c) {   // (operand reads one group ahead, as in mma_rows)
        f32x4 x = *reinterpret_cast<const f32x4 *>(a), y = *reinterpret_cast<const f32x4 *>(b);
#pragma unroll
        for (int j = 0; j < D / 8; ++j) {
            f32x4 nx = x, ny = y;
            if (j + 1 < D / 8) {
                nx = *reinterpret_cast<const f32x4 *>(a + 8 * (j + 1));
                ny = *reinterpret_cast<const f32x4 *>(b + 8 * (j + 1));
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) c = mfma2(x[i], y[i], c);
            x = nx;
            y = ny;
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    load(s0);
    for (int s = s0; s < s1; ++s) {
        __syncthreads();
        {
            float *const a[2] = {tile, tile + ROWS * PITCH}, *const c[2] = {tile + 2 * ROWS * PITCH, tile + 3 * ROWS * PITCH};
            sq.template put<PITCH>(a);
            sk.template put<PITCH>(c);
            if (threadIdx.x < 192) small[threadIdx.x] = sv;
        }
        __syncthreads();
        if (s + 1 < s1) load(s + 1);
        const float shift = shift_tab[b * p.S + s];
        if (ds_blocked(p, shift)) continue;
        const float *qr = tile + (qw + li) * PITCH + 4 * g, *kr = tile + (2 * ROWS + kw + li) * PITCH + 4 * g;
        const float mk = small[128 + kw + li], scale = shift != 0.0f ? 0.0f : p.scale, bs = shift != 0.0f ? 0.0f : 1.0f;
        f32x16 x = zero16();
        mma_pair(qr, kr, x);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const f32x4 lse = *reinterpret_cast<const f32x4 *>(&small[qw + 8 * j + 4 * g]);
#pragma unroll
            for (int i = 0; i < 4; ++i) x[4 * j + i] = exp_less(fmaf(bz[4 * j + i], bs, x[4 * j + i] * scale) + mk, lse[i]);
        }
        f32x16 dp = zero16();
        mma_pair(qr + ROWS * PITCH, kr + ROWS * PITCH, dp);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const f32x4 dl = *reinterpret_cast<const f32x4 *>(&small[64 + qw + 8 * j + 4 * g]);
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[4 * j + i] = fmaf(x[4 * j + i], dp[4 * j + i] - dl[i], acc[4 * j + i]);
        }
    }
    if (k0 + kw + li >= p.N) return;
    float *out = part + (((int64_t)ck * p.B + b) * p.H + h) * p.N * p.N + key;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int q = q0 + qw + crow(r, g);
        if (q < p.N) out[(int64_t)q * p.N] = acc[r];
    }
}

// ---------------------------------------------------------------- host side

#define EVO_LAUNCH_CHECK()                                    \
    do {                                                      \
        hipError_t e_ = hipGetLastError();                    \
        if (e_ != hipSuccess) return EVO_EHIP - (int)e_;      \
    } while (0)

static size_t dbias_lds(int D) { return ((size_t)4 * 64 * (D + 4) + 192) * sizeof(float); }

template <int D, int W, bool BIAS>
static int fwd_launch(const EvoAttnParams &p, int vec, hipStream_t st) {
    const unsigned grid = (unsigned)((p.N + 32 * W - 1) / (32 * W)) * (unsigned)(p.B * p.H * p.S);
    f32_fwd<D, W, BIAS><<<grid, 64 * W, 0, st>>>(p, vec);
    EVO_LAUNCH_CHECK();
    return EVO_OK;
}

template <int D, int W, bool BIAS>
static int bwd_launch(const EvoAttnParams &p, const Extra &e, int vec, hipStream_t st) {
    const unsigned grid = (unsigned)((p.N + 32 * W - 1) / (32 * W)) * (unsigned)(p.B * p.H * p.S);
    f32_dq<D, W, BIAS><<<grid, 64 * W, 0, st>>>(p, vec, e.delta, e.shift, e.delta_given);
    EVO_LAUNCH_CHECK();
    Extra kv = e;
    bool reduce = false;
    if (p.dbias) {
        const size_t lds = dbias_lds(D);
        static PerDevice done;
        if (lds > 64 * 1024)   // (more dynamic LDS than a launch may ask for unannounced)
            if (const int rc = ensure_dynamic_lds((const void *)&f32_dbias<D, BIAS>, (int)lds, done, nullptr)) return rc;
        const unsigned nb = (p.N + 63) / 64;
        const bool direct = e.n_chunks == 1 && p.dbias_dtype == EVO_F32;
        f32_dbias<D, BIAS><<<nb * nb * (unsigned)(p.B * p.H * e.n_chunks), 256, lds, st>>>(p, e.delta, e.shift, direct ? (float *)p.dbias : e.dbias_part,
                                                                                        e.chunk);
        EVO_LAUNCH_CHECK();
        reduce = !direct;
        if (reduce && (uintptr_t)p.dbias % 16 == 0 && ((int64_t)p.B * p.H * p.N * p.N) % 4 == 0) {
            kv.dbias_chunks = e.n_chunks;
            reduce = false;
        }
    }
    f32_dkdv<D, W, BIAS><<<grid, 64 * W, 0, st>>>(p, kv);
    EVO_LAUNCH_CHECK();
    if (reduce)
        if (const int rc = launch_dbias_reduce(p, e, st)) return rc;
    return p.dmask ? launch_dmask_reduce(p, e, st) : EVO_OK;
}

#define EVO_F32_DISPATCH(fn, ...)                                                                          \
    const bool bias = p.bias_dtype != EVO_NONE, two = p.N <= 64;                                           \
    switch (p.D) {                                                                                         \
        case 8: return two ? (bias ? fn<8, 2, true>(__VA_ARGS__) : fn<8, 2, false>(__VA_ARGS__))           \
                           : (bias ? fn<8, 4, true>(__VA_ARGS__) : fn<8, 4, false>(__VA_ARGS__));          \
        case 16: return two ? (bias ? fn<16, 2, true>(__VA_ARGS__) : fn<16, 2, false>(__VA_ARGS__))        \
                            : (bias ? fn<16, 4, true>(__VA_ARGS__) : fn<16, 4, false>(__VA_ARGS__));       \
        case 32: return two ? (bias ? fn<32, 2, true>(__VA_ARGS__) : fn<32, 2, false>(__VA_ARGS__))        \
                            : (bias ? fn<32, 4, true>(__VA_ARGS__) : fn<32, 4, false>(__VA_ARGS__));       \
        case 64: return two ? (bias ? fn<64, 2, true>(__VA_ARGS__) : fn<64, 2, false>(__VA_ARGS__))        \
                            : (bias ? fn<64, 4, true>(__VA_ARGS__) : fn<64, 4, false>(__VA_ARGS__));       \
        case 128: return two ? (bias ? fn<128, 2, true>(__VA_ARGS__) : fn<128, 2, false>(__VA_ARGS__))     \
                             : (bias ? fn<128, 4, true>(__VA_ARGS__) : fn<128, 4, false>(__VA_ARGS__));    \
    }                                                                                                      \
    return EVO_EUNSUPPORTED

static int bias_rows_vec(const EvoAttnParams &p) {
    return p.bias && p.N >= 4 && p.N % 4 == 0 && (uintptr_t)p.bias % 16 == 0 && p.bias_stride_b % 4 == 0 && p.bias_stride_h % 4 == 0 &&
           p.bias_stride_row % 4 == 0;
}

int launch_f32_fwd(const EvoAttnParams &p, hipStream_t st) {
    const int vec = bias_rows_vec(p);
    EVO_F32_DISPATCH(fwd_launch, p, vec, st);
}

int launch_f32_bwd(const EvoAttnParams &p, const Extra &e, hipStream_t st) {
    const int vec = bias_rows_vec(p);
    EVO_F32_DISPATCH(bwd_launch, p, e, vec, st);
}

// Chunks of S rows for the dBias kernel: about four workgroups per CU (256 CUs), no more than there are rows.
int f32_dbias_chunks(const EvoAttnParams &p) {
    const int64_t nb = (p.N + 63) / 64, base = nb * nb * p.B * p.H;
    const int64_t want = (1024 + base - 1) / base;
    return (int)(want < p.S ? want : p.S);
}

}  // namespace evo
