// The Linear layers of the block around the attention, 16-bit: y = x W^T + b, dx = dy W, and dW = dy^T x with the column sums
// of dy (the bias gradient).  W may be up to four matrices stacked (the Q, K, V and gate projections), read where they lie.
//
// Each is one launch (dW two: partial sums over slices of the rows, then their sum).  Through the library a product costs 18 to
// 20 us of host time, which is what bounded the block (nine of them, 480 us per training step from the smallest shapes up to 32 768
// rows), a stacked W a copy of the weights and of the bias, dW a sum of 16-bit partials.  The kernels themselves are bound, at these
// widths (K of 256 to 1024), by what a CU has under way from memory: 32 KB per stage and workgroup take 0.75 us, 18 bytes per clock, also where
// a CU has one workgroup and however many stages are asked for (four in a ring: no change), where the same loads from L2 alone reach 55 bytes per clock in
// any order of the chunks (operands or all of a stage through registers, one or two stages ahead: 2 to 8 % slower; a stage's operands all read
// before its first product, tiles of 128 x 256: no change; a stage asked for between the products instead of ahead of them: 13 -> 15 to 19).  Measured beside the library's, us: 32 768 rows, n = 1024, k = 256: y
// 28 (library 29), dx 25 (23), dW with bias gradient 42 (32 and 11); n = k = 256: 10 (11.5), 10 (12), 23 (25 and 11); 4096 rows, n = 1024: 8, 13, 19.
// With the loads as a builtin, of which the compiler waits for the next stage's ahead of every transposing read, and outputs stored
// 16 bytes of 64 rows at a time, those were 34, 32, 45; 11.5, 12, 24; 8, 18, 20 (a training step of the block, 32 768 rows of 256: 346, now 336).
//
// All three work in 128 x 128 tiles, four waves of 64 x 64 (2 x 2 accumulators of v_mfma_f32_32x32x16), 64 of the
// contraction at a time, both operands brought by the load path into LDS (`global_load_lds_dwordx4`), the next stage on its way
// while one is computed on: 64 KB, two workgroups per CU.  A 16-byte chunk of a staged row is stored at chunk ^ x(row)
// (mfma_stream.hip), so that plain reads of 32 rows and transposing reads both touch all banks evenly.  Output tiles are formed
// transposed (outputs along the accumulator's registers), with the 32 outputs of a tile dealt so that a lane ends up with 16
// consecutive ones of a row, and go to memory by way of LDS, 128 bytes of a row from eight lanes.  The contraction runs in ascending order, with one
// rounding of the fp32 sum.
//
// Large products are the library's business: host.cpp has the lines and both sides.
#include "common.h"
#include "bwd_common.h"
#include "kernels.h"

namespace evo {

constexpr int kLinTile = 128, kLinDepth = 64;   // rows and columns of a workgroup's tile, contraction per stage
constexpr int kLinSliceRows = 256;              // least rows of a slice of a weight gradient
typedef short s16x4l __attribute__((ext_vector_type(4)));

// rows of 64 (128 bytes) and of 128 elements (256 bytes)
__device__ __forceinline__ int at64(int r, int c) { return r * 128 + ((c ^ (((r >> 1) & 1) << 2 | ((r >> 2) & 1) << 1 | ((r >> 3) & 1))) << 4); }
__device__ __forceinline__ int swz128(int r) { return (r & 1) << 3 | ((r >> 1) & 1) << 2 | ((r >> 2) & 1) << 1 | ((r >> 3) & 1); }
__device__ __forceinline__ int at128(int r, int c) { return r * 256 + ((c ^ swz128(r)) << 4); }
__device__ __forceinline__ int swz64(int r) { return ((r >> 1) & 1) << 2 | ((r >> 2) & 1) << 1 | ((r >> 3) & 1); }

// 16 bytes per lane, to dst (uniform) + 16 * lane, as an instruction that the compiler does not know: see dma16 in stream_common.h
__device__ __forceinline__ void lin_dma(const void *src, unsigned char *dst) {
    const unsigned base = (unsigned)(uintptr_t)(__attribute__((address_space(3))) void *)dst;
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 4\n\tglobal_load_lds_dwordx4 %1, off" : : "s"(base), "v"(src) : "m0", "memory");
}
// this wave's loads have landed, everybody's have, and everybody is done with the stage before
__device__ __forceinline__ void lin_sync() { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// output that row `r` of a 32-row accumulator tile holds: lane group g ends up with outputs 16g .. 16g+15 in register order
__device__ __forceinline__ int lin_deal(int r) { return 16 * ((r >> 2) & 1) + 4 * (r >> 3) + (r & 3); }

// eight rows (16 ks + 8g ..) of a staged [64][128] tile at column `col` of each lane's group, transposed
template <typename T>
__device__ __forceinline__ typename Mfma<T>::v8 lin_transposed(const unsigned char *tile, int ks, int col, int lane) {
    typename Mfma<T>::v8 r;
#pragma unroll
    for (int h2 = 0; h2 < 2; ++h2) {
        const int row = 16 * ks + 8 * (lane >> 5) + 4 * h2 + ((lane & 15) >> 2);
        const s16x4l w = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (s16x4l __attribute__((address_space(3))) *)(tile + at128(row, col >> 3) + (col & 7) * 2));
        const typename Mfma<T>::v4 v = __builtin_bit_cast(typename Mfma<T>::v4, w);
#pragma unroll
        for (int i = 0; i < 4; ++i) r[4 * h2 + i] = v[i];
    }
    return r;
}

template <typename T>
struct Stacked {   // up to four [rows, K] matrices on top of each other
    const T *w0, *w1, *w2, *w3;
    int rows;
    __device__ __forceinline__ const T *row(int n, int K) const {   // n uniform; 64 rows from a multiple of 64 on lie in one matrix
        const int i = n / rows;
        return (i == 0 ? w0 : i == 1 ? w1 : i == 2 ? w2 : w3) + (int64_t)(n - i * rows) * K;
    }
};

template <typename T>
struct LinArgs {
    const T *a;          // forward: x [M, K]; dx: dy [M, N]
    Stacked<T> w;        // [N, K]
    const T *bias;       // forward: added to outputs bias_from .. N - 1; or null
    T *out;              // forward: y [M, N]; dx: dx [M, K]
    int64_t lda, ldo;
    int M, N, K, bias_from;
};

// chunk c (8 outputs) of row r of a wave's 64 x 64 outputs on their way to memory
__device__ __forceinline__ int lin_out_at(int r, int c) { return r * 128 + ((c ^ (r & 7)) << 4); }

// FWD: y = x W^T + b, contraction over K, W rows dealt into LDS as outputs.  Else dx = dy W, contraction over N, W rows as
// they come, read transposed.
template <typename T, bool FWD>
__global__ void __launch_bounds__(256, 2) linear_rows(LinArgs<T> p) {
    typedef typename Mfma<T>::v8 v8;
    __shared__ __attribute__((aligned(1024))) unsigned char lds[2][2 * kLinTile * kLinDepth * 2];
    constexpr int OFF_W = kLinTile * kLinDepth * 2;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), li = lane & 31, g = lane >> 5;
    const int outs = FWD ? p.N : p.K, depth = FWD ? p.K : p.N, ot = (outs + kLinTile - 1) / kLinTile;
    const unsigned lid = xcd_remap(blockIdx.x, gridDim.x);   // tiles of the same rows meet in one L2
    const int m0 = (int)(lid / ot) * kLinTile, o0 = (int)(lid % ot) * kLinTile;
    const int wm = (wave & 1) * 64, wo = (wave >> 1) * 64;

    const T *asrc[4], *wsrc[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int r = (wave * 4 + i) * 8 + lane / 8, c = (lane % 8) ^ swz64(r);
        asrc[i] = p.a + (int64_t)min(m0 + r, p.M - 1) * p.lda + c * 8;
        if (FWD) wsrc[i] = p.w.row(min(o0 + wave * 32, p.N - 32), p.K) + lin_deal(r & 31) * p.K + c * 8;
    }
    auto fetch = [&](int s) {
        unsigned char *buf = lds[s & 1] + wave * 4096;
        const T *wrows = FWD ? nullptr : p.w.row(s * kLinDepth, p.K);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            lin_dma(asrc[i] + s * kLinDepth, buf + i * 1024);
            if (FWD) {
                lin_dma(wsrc[i] + s * kLinDepth, buf + OFF_W + i * 1024);
            } else {
                const int r = (wave * 4 + i) * 4 + lane / 16, c = (lane % 16) ^ swz128(r);
                lin_dma(wrows + r * p.K + min(o0 + c * 8, p.K - 8), buf + OFF_W + i * 1024);
            }
        }
    };
    f32x16 acc[2][2];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[t][u][r] = 0.0f;

    const int ns = depth / kLinDepth;
    fetch(0);
    for (int s = 0; s < ns; ++s) {
        lin_sync();
        if (s + 1 < ns) fetch(s + 1);
        const unsigned char *buf = lds[s & 1];
#pragma unroll
        for (int ks = 0; ks < kLinDepth / 16; ++ks) {
            v8 w[2], a[2];
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                if (FWD) w[t] = *reinterpret_cast<const v8 *>(buf + OFF_W + at64(wo + 32 * t + li, 2 * ks + g));
                else w[t] = lin_transposed<T>(buf + OFF_W, ks, wo + 32 * t + 16 * (lane & 1) + 8 * ((lane >> 4) & 1) + 4 * ((lane >> 1) & 1), lane);
            }
#pragma unroll
            for (int u = 0; u < 2; ++u) a[u] = *reinterpret_cast<const v8 *>(buf + at64(wm + 32 * u + li, 2 * ks + g));
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int u = 0; u < 2; ++u) acc[t][u] = Mfma<T>::mma(w[t], a[u], acc[t][u]);
        }
    }
    // through LDS (the other stage's, which nobody reads any more), so that eight lanes store 128 bytes of a row
    unsigned char *mine = lds[ns & 1] + wave * 8192;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const int o = o0 + wo + 32 * t + 16 * g;
        float b[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) b[i] = 0.0f;
        if (FWD && p.bias && o >= p.bias_from && o < outs) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const v8 v = ld8(p.bias + o - p.bias_from + 8 * h);
#pragma unroll
                for (int i = 0; i < 8; ++i) b[8 * h + i] = (float)v[i];
            }
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                v8 v;
#pragma unroll
                for (int i = 0; i < 8; ++i) v[i] = (T)(FWD ? acc[t][u][8 * h + i] + b[8 * h + i] : acc[t][u][8 * h + i]);
                *reinterpret_cast<v8 *>(mine + lin_out_at(32 * u + li, 4 * t + 2 * g + h)) = v;
            }
        }
    }
    const int oc = o0 + wo + lane % 8 * 8;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int r = i * 8 + lane / 8, m = m0 + wm + r;
        const v8 v = *reinterpret_cast<const v8 *>(mine + lin_out_at(r, lane % 8));
        if (m < p.M && oc < outs) *reinterpret_cast<v8 *>(p.out + (int64_t)m * p.ldo + oc) = v;
    }
}

// Partial sums of dW [N, K] and of the column sums of dy [N] over one slice of the rows.  Rows of both operands are staged as
// they lie, 64 at a time, and both are read transposed.
template <typename T>
__global__ void __launch_bounds__(256, 2) linear_dw(const T *dy, const T *x, float *part, int64_t lddy, int64_t ldx, int M, int N, int K,
                                                    int slice_rows, bool sums) {
    typedef typename Mfma<T>::v8 v8;
    __shared__ __attribute__((aligned(1024))) unsigned char lds[2][2 * kLinTile * kLinDepth * 2];
    constexpr int OFF_X = kLinTile * kLinDepth * 2;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), li = lane & 31, g = lane >> 5;
    const int kt = (K + kLinTile - 1) / kLinTile, nt = (N + kLinTile - 1) / kLinTile;
    const unsigned lid = xcd_remap(blockIdx.x, gridDim.x);   // tiles of one slice meet in one L2
    const int slice = lid / (nt * kt), tile = lid % (nt * kt), n0 = tile / kt * kLinTile, k0 = tile % kt * kLinTile;
    const int first = slice * slice_rows, last = min(first + slice_rows, M);
    const int wn = (wave >> 1) * 64, wk = (wave & 1) * 64, cols = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);

    auto fetch = [&](int s) {
        unsigned char *buf = lds[s & 1] + wave * 4096;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int r = (wave * 4 + i) * 4 + lane / 16, c = ((lane % 16) ^ swz128(r)) * 8;
            const int64_t row = min(first + s * kLinDepth + r, last - 1);
            lin_dma(dy + row * lddy + min(n0 + c, N - 8), buf + i * 1024);
            lin_dma(x + row * ldx + min(k0 + c, K - 8), buf + OFF_X + i * 1024);
        }
    };
    f32x16 acc[2][2], accb[2];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[t][0][r] = acc[t][1][r] = accb[t][r] = 0.0f;
    v8 ones;
#pragma unroll
    for (int i = 0; i < 8; ++i) ones[i] = (T)1.0f;
    const bool col_sums = sums && k0 == 0 && wk == 0;   // wave-uniform

    const int ns = (last - first + kLinDepth - 1) / kLinDepth;
    fetch(0);
    for (int s = 0; s < ns; ++s) {
        lin_sync();
        if (s + 1 < ns) fetch(s + 1);
        const unsigned char *buf = lds[s & 1];
        const int left = last - first - s * kLinDepth;   // rows of this stage that count
#pragma unroll
        for (int ks = 0; ks < kLinDepth / 16; ++ks) {
            v8 a[2], b[2];
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                a[t] = lin_transposed<T>(buf, ks, wn + 32 * t + cols, lane);
                b[t] = lin_transposed<T>(buf + OFF_X, ks, wk + 32 * t + cols, lane);
                if (left < kLinDepth) {   // uniform: the last stage repeats the last row
#pragma unroll
                    for (int i = 0; i < 8; ++i)
                        if (16 * ks + 8 * g + i >= left) a[t][i] = (T)0.0f;
                }
            }
#pragma unroll
            for (int t = 0; t < 2; ++t) {
#pragma unroll
                for (int u = 0; u < 2; ++u) acc[t][u] = Mfma<T>::mma(a[t], b[u], acc[t][u]);
                if (col_sums) accb[t] = Mfma<T>::mma(a[t], ones, accb[t]);
            }
        }
    }
    float *out = part + (int64_t)slice * ((int64_t)N * K + N);
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int n = n0 + wn + 32 * t + crow(r, g);
            if (n >= N) continue;
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const int k = k0 + wk + 32 * u + li;
                if (k < K) out[(int64_t)n * K + k] = acc[t][u][r];
            }
            if (col_sums && li == 0) out[(int64_t)N * K + n] = accb[t][r];
        }
}

// The slices' sums, four columns per thread.
template <typename T>
__global__ void __launch_bounds__(256) linear_dw_sum(const float *part, T *out, int64_t cols, int64_t pitch, int slices) {
    const int64_t c = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
    if (c >= cols) return;
    float4 s = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 8
    for (int i = 0; i < slices; ++i) {
        const float4 v = *reinterpret_cast<const float4 *>(part + (int64_t)i * pitch + c);
        s.x += v.x;
        s.y += v.y;
        s.z += v.z;
        s.w += v.w;
    }
    typename Mfma<T>::v4 o;
    o[0] = (T)s.x;
    o[1] = (T)s.y;
    o[2] = (T)s.z;
    o[3] = (T)s.w;
    *reinterpret_cast<typename Mfma<T>::v4 *>(out + c) = o;
}

static bool lin_ok(int64_t rows, int n, int k, int nw, int w_rows, int dtype) {
    return (dtype == EVO_BF16 || dtype == EVO_F16) && rows > 0 && rows <= INT32_MAX - kLinTile && n >= 64 && k >= 64 && n % 64 == 0 && k % 64 == 0 &&
           n <= 1 << 16 && k <= 1 << 16 && nw >= 1 && nw <= 4 && (int64_t)nw * w_rows == n && w_rows % 64 == 0 &&
           ((rows + kLinTile - 1) / kLinTile) * ((n > k ? n : k) / 64) <= INT32_MAX;
}

// Slices of the rows that dW is summed over: two workgroups per CU, and enough rows in each for the load path to run ahead.
static int lin_slice_rows(int64_t rows, int n, int k) {
    const int64_t tiles = (int64_t)((n + kLinTile - 1) / kLinTile) * ((k + kLinTile - 1) / kLinTile);
    int64_t slices = (512 + tiles - 1) / tiles;
    if (slices > rows / kLinSliceRows) slices = rows / kLinSliceRows;
    if (slices < 1) slices = 1;
    return (int)((rows + slices * kLinDepth - 1) / (slices * kLinDepth) * kLinDepth);
}

static bool lin_misaligned(const void *p) { return ((uintptr_t)p & 15) != 0; }

static int lin_rc() {
    const hipError_t err = hipGetLastError();
    return err == hipSuccess ? EVO_OK : EVO_EHIP - (int)err;
}

template <bool FWD>
static int lin_rows(const void *a, int64_t lda, const void *const *w, int nw, int w_rows, const void *bias, int bias_from, void *out, int64_t ldo,
                    int64_t rows, int n, int k, int dtype, hipStream_t st) {
    if (!lin_ok(rows, n, k, nw, w_rows, dtype)) return EVO_EUNSUPPORTED;
    if (!a || !w || !out) return EVO_EINVAL;
    if (lda < (FWD ? k : n) || ldo < (FWD ? n : k) || bias_from < 0 || bias_from > n) return EVO_EINVAL;
    if (lin_misaligned(a) || lin_misaligned(out) || lin_misaligned(bias) || lda % 8 || ldo % 8 || bias_from % 16) return EVO_EALIGN;
    for (int i = 0; i < nw; ++i) {
        if (!w[i]) return EVO_EINVAL;
        if (lin_misaligned(w[i])) return EVO_EALIGN;
    }
    const unsigned grid = (unsigned)((rows + kLinTile - 1) / kLinTile * (((FWD ? n : k) + kLinTile - 1) / kLinTile));
    auto go = [&](auto t) {
        typedef decltype(t) T;
        auto at = [&](int i) { return (const T *)w[i < nw ? i : 0]; };
        linear_rows<T, FWD><<<grid, 256, 0, st>>>({(const T *)a, {at(0), at(1), at(2), at(3), w_rows}, (const T *)bias, (T *)out, lda, ldo, (int)rows, n, k, bias_from});
        return lin_rc();
    };
    return dtype == EVO_BF16 ? go(bf16_t()) : go(f16_t());
}

}  // namespace evo

extern "C" {

int evoattn_linear_fwd(const void *x, int64_t ldx, const void *const *w, int32_t nw, int32_t w_rows, const void *bias, int32_t bias_from, void *y,
                       int64_t ldy, int64_t rows, int32_t n, int32_t k, int32_t dtype, void *hip_stream) {
    return evo::lin_rows<true>(x, ldx, w, nw, w_rows, bias, bias_from, y, ldy, rows, n, k, dtype, (hipStream_t)hip_stream);
}

int evoattn_linear_dx(const void *dy, int64_t lddy, const void *const *w, int32_t nw, int32_t w_rows, void *dx, int64_t lddx, int64_t rows, int32_t n,
                      int32_t k, int32_t dtype, void *hip_stream) {
    return evo::lin_rows<false>(dy, lddy, w, nw, w_rows, nullptr, 0, dx, lddx, rows, n, k, dtype, (hipStream_t)hip_stream);
}

size_t evoattn_linear_dw_workspace_bytes(int64_t rows, int32_t n, int32_t k, int32_t dtype) {
    using namespace evo;
    if (!lin_ok(rows, n, k, 1, n, dtype)) return 0;
    const int per = lin_slice_rows(rows, n, k);
    return (size_t)((rows + per - 1) / per) * ((size_t)n * k + n) * sizeof(float);
}

int evoattn_linear_dw(const void *dy, int64_t lddy, const void *x, int64_t ldx, void *out, int32_t sums, void *workspace, size_t workspace_bytes,
                      int64_t rows, int32_t n, int32_t k, int32_t dtype, void *hip_stream) {
    using namespace evo;
    if (!lin_ok(rows, n, k, 1, n, dtype)) return EVO_EUNSUPPORTED;
    if (!dy || !x || !out || lddy < n || ldx < k) return EVO_EINVAL;
    if (lin_misaligned(dy) || lin_misaligned(x) || lin_misaligned(out) || lin_misaligned(workspace) || lddy % 8 || ldx % 8) return EVO_EALIGN;
    if (!workspace || workspace_bytes < evoattn_linear_dw_workspace_bytes(rows, n, k, dtype)) return EVO_EWORKSPACE;
    const int per = lin_slice_rows(rows, n, k), slices = (int)((rows + per - 1) / per);
    const unsigned grid = (unsigned)(((n + kLinTile - 1) / kLinTile) * ((k + kLinTile - 1) / kLinTile) * slices);
    const int64_t all = (int64_t)n * k + n, cols = sums ? all : (int64_t)n * k;
    hipStream_t st = (hipStream_t)hip_stream;
    auto go = [&](auto t) {
        typedef decltype(t) T;
        linear_dw<T><<<grid, 256, 0, st>>>((const T *)dy, (const T *)x, (float *)workspace, lddy, ldx, (int)rows, n, k, per, sums != 0);
        if (const int rc = lin_rc()) return rc;
        linear_dw_sum<T><<<(unsigned)((cols + 1023) / 1024), 256, 0, st>>>((const float *)workspace, (T *)out, cols, all, slices);
        return lin_rc();
    };
    return dtype == EVO_BF16 ? go(bf16_t()) : go(f16_t());
}

}  // extern "C"
