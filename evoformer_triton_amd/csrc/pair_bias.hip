// The pair bias of the block around the attention, z [B,N,N,C] -> LayerNorm -> Linear (C -> H) -> [B,1,H,N,N], as one kernel
// forward and one (with the sum of its partials) backward.  16-bit, C of 64, 128 or 256, up to 16 heads; other shapes
// keep the LayerNorm kernels, the library's products and a permute.
//
// Bound by HBM: z is read once forward; z and the bias gradient are read and dz is written once backward.  Apart they cost
// (z of 65 536 rows of 128, H = 8, bf16) 12 us LayerNorm, 9 product and 5 permute forward, and 5 permute, 10 + 14 products,
// 11 sum of slices, 16 + 6 LayerNorm backward, each a launch or two with an array of z's size in between, the products
// at 18 us of host time each; here 9.5 forward, 17.5 + 6 backward.
//
// The rounding is that of the separate steps: the normalised row to 16 bits before the product, the gradient of the
// normalised row after it, and the LayerNorm sums in layernorm.hip's order; the matrix instruction adds in the order of the
// library's kernels seen at these shapes.  (It matters for comparisons: the gradient of the LayerNorm's bias is zero but for
// those roundings, since a constant added to a query's bias changes no probability.)
//
// A wave owns 32 rows (pairs) at a time.  LayerNorm steps work as in layernorm.hip: C / 8 lanes per row, 16 bytes each.  The
// products are v_mfma_f32_16x16x32 with the heads as one side (lane l, q = l / 16: operands row l % 16, contraction
// 8q .. 8q+7; accumulator column l % 16, rows 4q .. 4q+3); rows cross between the two forms through a wave's own LDS tile
// [32][C], a 16-byte chunk stored at chunk ^ x(row) so that 16 rows of one chunk touch all banks once.
#include <type_traits>

#include "common.h"
#include "bwd_common.h"
#include "kernels.h"

namespace evo {

constexpr int kPbWaves = 4, kPbRows = 32;      // waves per workgroup, rows per wave and turn
constexpr int kPbBwdBlocks = 512;              // most workgroups of the backward = partial sums of the parameter gradients

typedef float f32x4p __attribute__((ext_vector_type(4)));
typedef short s16x4p __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4p mma16(bf16x8 a, bf16x8 b, f32x4p c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }
__device__ __forceinline__ f32x4p mma16(f16x8 a, f16x8 b, f32x4p c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }

template <int C>
struct PbTile {
    static constexpr int ROW = C * 2, BYTES = kPbRows * ROW;
    static __device__ __forceinline__ int x(int r) { return C == 64 ? (r >> 1) & 7 : r & 15; }   // (64: two rows share the banks)
    static __device__ __forceinline__ int at(int r, int c) { return r * ROW + ((c ^ x(r)) << 4); }
};

template <int LANES>
__device__ __forceinline__ float pb_add_xor(float s) {
    return s + __shfl_xor(s, LANES);
}
template <int N>
__device__ __forceinline__ float pb_add_ror(float s) {   // + the value N lanes further within 16
    return s + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(s), 0x120 | N, 0xf, 0xf, false));
}
// Sum over groups of LPR lanes, in the order of a butterfly over halves (rotations pair the same values once the halves are equal).
template <int LPR>
__device__ __forceinline__ float pb_group_sum(float s) {
    if (LPR == 8) return pb_add_xor<1>(pb_add_xor<2>(pb_add_xor<4>(s)));
    if (LPR == 32) s = pb_add_xor<16>(s);
    return pb_add_ror<1>(pb_add_ror<2>(pb_add_ror<4>(pb_add_ror<8>(s))));
}

template <typename T>
struct PairBiasFwd {
    const T *z, *gamma, *beta, *w;
    T *bias;
    float *mean, *rstd;
    unsigned rows, pairs;   // B * N * N, N * N
    int heads;
    float eps;
};

// SPLIT: every 32 channels of a product are summed apart and the sums added, as the library was seen to do for so few rows (of 128 channels).
template <typename T, int C, bool SPLIT>
__global__ void __launch_bounds__(kPbWaves * 64) pair_bias_fwd(PairBiasFwd<T> p) {
    typedef typename Mfma<T>::v8 v8;
    constexpr int LPR = C / 8, RPI = 64 / LPR, ITS = kPbRows / RPI, KS = C / 32;
    __shared__ __attribute__((aligned(16))) unsigned char lds[kPbWaves][PbTile<C>::BYTES];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), q = lane >> 4, li = lane & 15;
    const int sub = lane % LPR, grp = lane / LPR;
    unsigned char *tile = lds[wave];
    const unsigned row0 = (blockIdx.x * kPbWaves + wave) * kPbRows;
    if (row0 >= p.rows) return;

    v8 x[ITS];
#pragma unroll
    for (int it = 0; it < ITS; ++it) x[it] = ld8(p.z + (int64_t)min(row0 + it * RPI + grp, p.rows - 1) * C + sub * 8);
    v8 wf[KS];   // head li
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) wf[ks] = li < p.heads ? ld8(p.w + li * C + ks * 32 + q * 8) : zero8<T>();
    float g[8], b[8];
    {
        v8 gv, bv;
        if (p.gamma) gv = ld8(p.gamma + sub * 8);
        if (p.beta) bv = ld8(p.beta + sub * 8);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            g[e] = p.gamma ? (float)gv[e] : 1.0f;
            b[e] = p.beta ? (float)bv[e] : 0.0f;
        }
    }
    const float inv = 1.0f / (float)C;
#pragma unroll
    for (int it = 0; it < ITS; ++it) {
        float v[8], s = 0.0f, d2 = 0.0f;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            v[e] = (float)x[it][e];
            s += v[e];
        }
        const float mu = pb_group_sum<LPR>(s) * inv;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float d = v[e] - mu;
            d2 += d * d;
        }
        const float r = 1.0f / sqrtf(pb_group_sum<LPR>(d2) * inv + p.eps);
        v8 y;
#pragma unroll
        for (int e = 0; e < 8; ++e) y[e] = (T)((v[e] - mu) * r * g[e] + b[e]);
        *reinterpret_cast<v8 *>(tile + PbTile<C>::at(it * RPI + grp, sub)) = y;
        const unsigned row = row0 + it * RPI + grp;
        if (sub == 0 && row < p.rows) {
            p.mean[row] = mu;
            p.rstd[row] = r;
        }
    }
    // (the wave's own tile: its reads follow its writes)
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        f32x4p acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const v8 y = *reinterpret_cast<const v8 *>(tile + PbTile<C>::at(16 * u + li, 4 * ks + q));
            if (SPLIT) acc += mma16(wf[ks], y, f32x4p{0.0f, 0.0f, 0.0f, 0.0f});
            else acc = mma16(wf[ks], y, acc);
        }
        const unsigned row = row0 + 16 * u + li;
        if (row >= p.rows) continue;
        const unsigned batch = row / p.pairs, pair = row - batch * p.pairs;
        T *out = p.bias + ((int64_t)batch * p.heads + 4 * q) * p.pairs + pair;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (4 * q + i < p.heads) out[(int64_t)i * p.pairs] = (T)acc[i];
    }
}

template <typename T>
struct PairBiasBwd {
    const T *dbias, *z, *gamma, *beta, *w;
    const float *mean, *rstd;
    T *dz;          // may be null
    float *part;    // [gridDim.x][2 + heads][C]: sums of dy * xhat, of dy, of dbias x y; may be null
    unsigned rows, pairs;
    int heads;
};

template <typename T, int C>
__global__ void __launch_bounds__(kPbWaves * 64, C == 256 ? 1 : 3) pair_bias_bwd(PairBiasBwd<T> p) {
    typedef typename Mfma<T>::v8 v8;
    typedef typename Mfma<T>::v4 v4;
    constexpr int LPR = C / 8, RPI = 64 / LPR, ITS = kPbRows / RPI, CT = C / 16, DP = kPbRows + 8, WP = 24, LD = 2;
    __shared__ __attribute__((aligned(16))) unsigned char lds[kPbWaves * PbTile<C>::BYTES];
    __shared__ __attribute__((aligned(16))) T dts[kPbWaves][16 * DP], wt[C * WP];   // [head][pair]; the weight as [channel][head]
    static_assert(PbTile<C>::BYTES >= 16 * C * 4 && kPbWaves * PbTile<C>::BYTES >= kPbWaves * RPI * C * 4, "the sums meet in the tiles");
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), q = lane >> 4, li = lane & 15;
    const int sub = lane % LPR, grp = lane / LPR;
    unsigned char *tile = lds + wave * PbTile<C>::BYTES;
    T *dt = dts[wave];

    for (int i = threadIdx.x; i < 16 * C; i += kPbWaves * 64) wt[(i % C) * WP + i / C] = i / C < p.heads ? p.w[i] : (T)0.0f;
    __syncthreads();
    v8 gv, bv;
    float dg[8], db[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        gv[e] = (T)1.0f;
        bv[e] = (T)0.0f;
        dg[e] = db[e] = 0.0f;
    }
    if (p.gamma) gv = ld8(p.gamma + sub * 8);
    if (p.beta) bv = ld8(p.beta + sub * 8);
    f32x4p dw[CT];
#pragma unroll
    for (int t = 0; t < CT; ++t) dw[t] = {0.0f, 0.0f, 0.0f, 0.0f};
    const float inv = 1.0f / (float)C;

    for (unsigned row0 = (blockIdx.x * kPbWaves + wave) * kPbRows; row0 < p.rows; row0 += gridDim.x * kPbWaves * kPbRows) {
        // z and its moments, LD turns of the LayerNorm ahead of the one that is computed on
        v8 xn[LD];
        float mun[LD], rsn[LD];
        auto fetch = [&](unsigned from) {
#pragma unroll
            for (int k = 0; k < LD; ++k) {
                const unsigned row = min(from + k * RPI + grp, p.rows - 1);
                xn[k] = ld8(p.z + (int64_t)row * C + sub * 8);
                mun[k] = p.mean[row];
                rsn[k] = p.rstd[row];
            }
        };
        fetch(row0);
        // the bias gradient of the rows, zero beyond the last: [pair][head] as an operand, [head][pair] in LDS
        v8 d[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            d[u] = zero8<T>();
            const unsigned row = row0 + 16 * u + li;
            if (row < p.rows && q < 2) {
                const unsigned batch = row / p.pairs, pair = row - batch * p.pairs;
                const T *src = p.dbias + (int64_t)batch * p.heads * p.pairs + pair;
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    if (8 * q + i < p.heads) d[u][i] = src[(int64_t)(8 * q + i) * p.pairs];
            }
            if (q < 2) {
#pragma unroll
                for (int i = 0; i < 8; ++i) dt[(8 * q + i) * DP + 16 * u + li] = d[u][i];
            }
        }
        // gradient of the normalised rows
#pragma unroll 4
        for (int t = 0; t < CT; ++t) {
            v8 wf = zero8<T>();   // channel 16 t + li against heads 8q .. 8q+7
            if (q < 2) wf = ld8(wt + (16 * t + li) * WP + 8 * q);
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const f32x4p a = mma16(wf, d[u], f32x4p{0.0f, 0.0f, 0.0f, 0.0f});
                v4 y;
#pragma unroll
                for (int i = 0; i < 4; ++i) y[i] = (T)a[i];
                *reinterpret_cast<v4 *>(tile + PbTile<C>::at(16 * u + li, 2 * t + (q >> 1)) + (q & 1) * 8) = y;   // channels 16t + 4q ..
            }
        }
        // LayerNorm's backward (layernorm.hip); the normalised row takes the gradient's place in the tile
#pragma unroll 1
        for (int it0 = 0; it0 < ITS; it0 += LD) {
            v8 x[LD];
            float mu[LD], rs[LD];
#pragma unroll
            for (int k = 0; k < LD; ++k) {
                x[k] = xn[k];
                mu[k] = mun[k];
                rs[k] = rsn[k];
            }
            fetch(row0 + min(it0 + LD, ITS - LD) * RPI);
#pragma unroll
            for (int k = 0; k < LD; ++k) {
            const int it = it0 + k;
            const unsigned row = row0 + it * RPI + grp;
            v8 *cell = reinterpret_cast<v8 *>(tile + PbTile<C>::at(it * RPI + grp, sub));
            const v8 dy = *cell;
            float xh[8], gy[8], s1 = 0.0f, s2 = 0.0f;
            v8 y;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float de = (float)dy[e];
                xh[e] = ((float)x[k][e] - mu[k]) * rs[k];
                gy[e] = de * (float)gv[e];
                s1 += gy[e];
                s2 += gy[e] * xh[e];
                dg[e] += de * xh[e];
                db[e] += de;
                y[e] = (T)(((float)x[k][e] - mu[k]) * rs[k] * (float)gv[e] + (float)bv[e]);
            }
            *cell = y;
            if (p.dz) {   // uniform
                const float c1 = pb_group_sum<LPR>(s1) * inv, c2 = pb_group_sum<LPR>(s2) * inv;
                v8 out;
#pragma unroll
                for (int e = 0; e < 8; ++e) out[e] = (T)((gy[e] - c1 - xh[e] * c2) * rs[k]);
                if (row < p.rows) *reinterpret_cast<v8 *>(p.dz + (int64_t)row * C + sub * 8) = out;
            }
        }
        }
        if (!p.part) continue;   // uniform
        const v8 da = *reinterpret_cast<const v8 *>(dt + li * DP + 8 * q);   // head li against pairs 8q .. 8q+7
#pragma unroll
        for (int t = 0; t < CT; ++t) {
            v8 yb;   // channel 16 t + li, pairs 8q .. 8q+7
#pragma unroll
            for (int h2 = 0; h2 < 2; ++h2) {
                const int row = 8 * q + 4 * h2 + (li >> 2), col = 16 * t + 4 * (li & 3);
                const s16x4p r = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                    (s16x4p __attribute__((address_space(3))) *)(tile + PbTile<C>::at(row, col >> 3) + (col & 7) * 2));
                const v4 v = __builtin_bit_cast(v4, r);
#pragma unroll
                for (int i = 0; i < 4; ++i) yb[4 * h2 + i] = v[i];
            }
            dw[t] = mma16(da, yb, dw[t]);
        }
    }
    if (!p.part) return;
    // the workgroup's sums meet in LDS: LayerNorm weight and bias, then the projection's weight
    float *part = p.part + (int64_t)blockIdx.x * (2 + p.heads) * C, *red = reinterpret_cast<float *>(lds);
#pragma unroll
    for (int pass = 0; pass < 2; ++pass) {
        __syncthreads();
#pragma unroll
        for (int e = 0; e < 8; ++e) red[(wave * RPI + grp) * C + sub * 8 + e] = pass == 0 ? dg[e] : db[e];
        __syncthreads();
        for (int c = threadIdx.x; c < C; c += kPbWaves * 64) {
            float s = 0.0f;
            for (int r = 0; r < kPbWaves * RPI; ++r) s += red[r * C + c];
            part[pass * C + c] = s;
        }
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < CT; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) red[(wave * 16 + 4 * q + i) * C + 16 * t + li] = dw[t][i];
    __syncthreads();
    for (int c = threadIdx.x; c < p.heads * C; c += kPbWaves * 64) {
        float s = 0.0f;
#pragma unroll
        for (int w = 0; w < kPbWaves; ++w) s += red[w * 16 * C + c];
        part[2 * C + c] = s;
    }
}

static bool pb_ok(int64_t batches, int64_t pairs, int cols, int heads, int dtype) {
    return (dtype == EVO_BF16 || dtype == EVO_F16) && (cols == 64 || cols == 128 || cols == 256) && heads >= 1 && heads <= 16 && batches > 0 &&
           pairs > 0 && pairs <= INT32_MAX && batches <= INT32_MAX / pairs;
}

static unsigned pb_bwd_blocks(int64_t rows) {
    const int64_t want = (rows + kPbWaves * kPbRows - 1) / (kPbWaves * kPbRows);
    return (unsigned)(want < kPbBwdBlocks ? want : kPbBwdBlocks);
}

template <typename T>
static int pb_fwd(const PairBiasFwd<T> &p, int cols, hipStream_t st) {
    const unsigned grid = (p.rows + kPbWaves * kPbRows - 1) / (kPbWaves * kPbRows);
    auto go = [&](auto split) {
        constexpr bool SPLIT = decltype(split)::value;
        if (cols == 64) pair_bias_fwd<T, 64, SPLIT><<<grid, kPbWaves * 64, 0, st>>>(p);
        else if (cols == 128) pair_bias_fwd<T, 128, SPLIT><<<grid, kPbWaves * 64, 0, st>>>(p);
        else pair_bias_fwd<T, 256, SPLIT><<<grid, kPbWaves * 64, 0, st>>>(p);
    };
    if (p.rows <= 7424) go(std::true_type());   // (29 x 256: seen in the library's results for rows of 128; it changes roundings, not the time)
    else go(std::false_type());
    const hipError_t err = hipGetLastError();
    return err == hipSuccess ? EVO_OK : EVO_EHIP - (int)err;
}

template <typename T>
static int pb_bwd(const PairBiasBwd<T> &p, int cols, void *dparams, hipStream_t st) {
    const unsigned grid = pb_bwd_blocks(p.rows);
    if (cols == 64) pair_bias_bwd<T, 64><<<grid, kPbWaves * 64, 0, st>>>(p);
    else if (cols == 128) pair_bias_bwd<T, 128><<<grid, kPbWaves * 64, 0, st>>>(p);
    else pair_bias_bwd<T, 256><<<grid, kPbWaves * 64, 0, st>>>(p);
    const hipError_t err = hipGetLastError();
    if (err != hipSuccess) return EVO_EHIP - (int)err;
    return p.part ? launch_column_reduce(p.part, (int)grid, (2 + p.heads) * cols, dparams, std::is_same<T, bf16_t>::value ? EVO_BF16 : EVO_F16, st) : EVO_OK;
}

static bool pb_misaligned(const void *p) { return ((uintptr_t)p & 15) != 0; }

}  // namespace evo

extern "C" {

size_t evoattn_pair_bias_workspace_bytes(int64_t batches, int64_t pairs, int32_t cols, int32_t heads, int32_t dtype) {
    using namespace evo;
    if (!pb_ok(batches, pairs, cols, heads, dtype)) return 0;
    return (size_t)pb_bwd_blocks(batches * pairs) * (2 + (size_t)heads) * (size_t)cols * sizeof(float);
}

int evoattn_pair_bias_fwd(const void *z, const void *gamma, const void *beta, const void *w, void *bias, float *mean, float *rstd,
                          int64_t batches, int64_t pairs, int32_t cols, int32_t heads, int32_t dtype, float eps, void *hip_stream) {
    using namespace evo;
    if (!pb_ok(batches, pairs, cols, heads, dtype)) return EVO_EUNSUPPORTED;
    if (!z || !w || !bias || !mean || !rstd || !(eps >= 0.0f)) return EVO_EINVAL;
    if (pb_misaligned(z) || pb_misaligned(gamma) || pb_misaligned(beta) || pb_misaligned(w)) return EVO_EALIGN;
    hipStream_t st = (hipStream_t)hip_stream;
    auto go = [&](auto t) {
        typedef decltype(t) T;
        return pb_fwd<T>({(const T *)z, (const T *)gamma, (const T *)beta, (const T *)w, (T *)bias, mean, rstd, (unsigned)(batches * pairs),
                          (unsigned)pairs, heads, eps}, cols, st);
    };
    return dtype == EVO_BF16 ? go(bf16_t()) : go(f16_t());
}

int evoattn_pair_bias_bwd(const void *dbias, const void *z, const void *gamma, const void *beta, const void *w, const float *mean,
                          const float *rstd, void *dz, void *dparams, void *workspace, size_t workspace_bytes, int64_t batches, int64_t pairs,
                          int32_t cols, int32_t heads, int32_t dtype, void *hip_stream) {
    using namespace evo;
    if (!pb_ok(batches, pairs, cols, heads, dtype)) return EVO_EUNSUPPORTED;
    if (!dbias || !z || !w || !mean || !rstd || (!dz && !dparams)) return EVO_EINVAL;
    if (pb_misaligned(z) || pb_misaligned(gamma) || pb_misaligned(beta) || pb_misaligned(dz) || pb_misaligned(workspace)) return EVO_EALIGN;
    if (dparams && (!workspace || workspace_bytes < evoattn_pair_bias_workspace_bytes(batches, pairs, cols, heads, dtype))) return EVO_EWORKSPACE;
    hipStream_t st = (hipStream_t)hip_stream;
    auto go = [&](auto t) {
        typedef decltype(t) T;
        return pb_bwd<T>({(const T *)dbias, (const T *)z, (const T *)gamma, (const T *)beta, (const T *)w, mean, rstd, (T *)dz,
                          dparams ? (float *)workspace : nullptr, (unsigned)(batches * pairs), (unsigned)pairs, heads}, cols, dparams, st);
    };
    return dtype == EVO_BF16 ? go(bf16_t()) : go(f16_t());
}

}  // extern "C"
