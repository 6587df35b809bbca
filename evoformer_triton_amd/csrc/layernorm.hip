// LayerNorm over the last dimension, forward and backward, for the block around the attention
// (the normalisation of the representation before the Q, K, V and gate projections and of the
// pair representation before the bias projection).  The reference's operator starts at Q, K, V
// (evoformer.py:640-651); the model code around it normalises with the framework's LayerNorm.
//
// The work is bound by HBM: the forward reads x and writes y once, the backward reads x and dy
// and writes dx once.  A row is held in registers by a group of lanes (16 bytes per lane and
// piece, one to four pieces per lane), so mean, variance and the two sums of the backward are
// register sums followed by a few cross-lane steps; a workgroup walks over rows with a grid
// stride.  The gradients of weight and bias are summed per lane over the rows a workgroup
// visits, then over the workgroup in LDS, written as one partial per workgroup and added up
// by a second small kernel in a fixed order: no atomics, bit-reproducible.
#include <type_traits>

#include "common.h"
#include "bwd_common.h"
#include "kernels.h"

namespace evo {

constexpr int kLnThreads = 256;
constexpr int kLnMaxPieces = 4;       // 16-byte pieces of a row per lane
// Most workgroups: of the forward (1024 to 4096 within 3 %), of the backward and of plain column sums = partial sums of the weight and bias gradients
// (the backward with the partials' sum, 32 768 / 8192 / 98 304 rows of 256 bf16, 256 workgroups 18.1 / 11.9 / 52 us, 512 16.8 / 12.0 / 36, 1024 19.2 / 15.0 / 36).
// In fp32 1024, too: of 512 each adds up twice as many rows one after the other, and where there are many the result was 1.1 times as far from 64 bits (98 304 rows
// of 256; 3 000 000 of 4: 1.24; in 16 bits the result's own rounding is a thousand times that).
constexpr int kLnFwdBlocks = 2048, kLnSumBlocks = 1024;
template <typename T> constexpr int kLnBwdBlocks = sizeof(T) == 4 ? 1024 : 512;
constexpr int kLnPartials = 1024;   // that the workspace's size allows for: what callers of earlier builds were told, more than is written
static_assert(kLnBwdBlocks<float> <= kLnPartials && kLnSumBlocks <= kLnPartials, "a partial sum per workgroup");

template <typename T>
struct LnVec {
    static constexpr int N = 16 / sizeof(T);
    typedef T type __attribute__((ext_vector_type(16 / sizeof(T))));
};

// how a row is spread over lanes: `lpr` lanes (a power of two, at most 64), `pieces` 16-byte pieces per lane
struct LnShape {
    int lpr, pieces;
};

static LnShape ln_shape(int cols, int vec) {
    const int n = cols / vec;          // 16-byte pieces per row
    int lpr = 1;
    while (lpr < 64 && lpr < n) lpr *= 2;
    return {lpr, (n + lpr - 1) / lpr};
}

// The value of lane i ^ O, where the lanes of a group of LPR hold the same value with a period of 2 O lanes (sums made so far), or where O is 1 or 2.
template <int O, int LPR>
__device__ __forceinline__ float ln_other(float s) {
    const int u = __float_as_int(s);
    if constexpr (O == 1) return __int_as_float(__builtin_amdgcn_mov_dpp(u, 0xB1, 0xF, 0xF, true));        // quad_perm 1 0 3 2
    else if constexpr (O == 2) return __int_as_float(__builtin_amdgcn_mov_dpp(u, 0x4E, 0xF, 0xF, true));   // quad_perm 2 3 0 1
    else if constexpr (O == 4 && LPR >= 16) return __int_as_float(__builtin_amdgcn_mov_dpp(u, 0x124, 0xF, 0xF, true));   // row_ror 4
    else if constexpr (O == 8) return __int_as_float(__builtin_amdgcn_mov_dpp(u, 0x128, 0xF, 0xF, true));  // row_ror 8
    else return __shfl_xor(s, O);
}

// The sums over the LPR lanes of a group, by xor from half a group down: steps in the vector ALU instead of through LDS.
template <int LPR>
__device__ __forceinline__ float ln_group_sum(float s) {
    if constexpr (LPR >= 64) {
        const auto w = __builtin_amdgcn_permlane32_swap(__float_as_uint(s), __float_as_uint(s), false, false);
        s = __uint_as_float(w[0]) + __uint_as_float(w[1]);
    }
    if constexpr (LPR >= 32) {
        const auto w = __builtin_amdgcn_permlane16_swap(__float_as_uint(s), __float_as_uint(s), false, false);
        s = __uint_as_float(w[0]) + __uint_as_float(w[1]);
    }
    if constexpr (LPR >= 16) s += ln_other<8, LPR>(s);
    if constexpr (LPR >= 8) s += ln_other<4, LPR>(s);
    if constexpr (LPR >= 4) s += ln_other<2, LPR>(s);
    if constexpr (LPR >= 2) s += ln_other<1, LPR>(s);
    return s;
}

// Bound, where a row is long, by memory.  What a row costs beside its elements is kept low: lanes per row known when compiled, sums without LDS, a workgroup
// over several rows with the next one's elements on their way.  32 768 rows of 256, bf16: 10.1 -> 8.5 us, backward with the
// partials' sum 22.9 -> 16.8; 16 384 rows of 640 13.2 -> 10.6 and 27.7 -> 20.4.
template <typename T, int PIECES, int LPR>
__global__ void __launch_bounds__(kLnThreads)
ln_fwd_kernel(const T *__restrict__ x, const T *__restrict__ gamma, const T *__restrict__ beta, T *__restrict__ y,
              float *__restrict__ mean, float *__restrict__ rstd, int64_t rows, int cols, float eps) {
    constexpr int VEC = LnVec<T>::N, RPB = kLnThreads / LPR;
    typedef typename LnVec<T>::type vT;
    const int tid = threadIdx.x, sub = tid % LPR, grp = tid / LPR;
    const int npieces = cols / VEC;
    float g[PIECES][VEC], b[PIECES][VEC];
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
        const int pc = i * LPR + sub;
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
            g[i][e] = 1.0f;
            b[i][e] = 0.0f;
        }
        if (pc < npieces) {
            if (gamma) {
                const vT w = *reinterpret_cast<const vT *>(gamma + pc * VEC);
#pragma unroll
                for (int e = 0; e < VEC; ++e) g[i][e] = (float)w[e];
            }
            if (beta) {
                const vT w = *reinterpret_cast<const vT *>(beta + pc * VEC);
#pragma unroll
                for (int e = 0; e < VEC; ++e) b[i][e] = (float)w[e];
            }
        }
    }
    const float inv = 1.0f / (float)cols;
    const int64_t step = (int64_t)gridDim.x * RPB;
    vT raw[PIECES];
    auto fetch = [&](int64_t row) {   // (lanes and rows past the end repeat the last)
#pragma unroll
        for (int i = 0; i < PIECES; ++i) raw[i] = *reinterpret_cast<const vT *>(x + min(row, rows - 1) * cols + min(i * LPR + sub, npieces - 1) * VEC);
    };
    fetch((int64_t)blockIdx.x * RPB + grp);
    for (int64_t row = (int64_t)blockIdx.x * RPB + grp; row < rows; row += step) {
        float v[PIECES][VEC];
        float s = 0.0f;
#pragma unroll
        for (int i = 0; i < PIECES; ++i) {
            const bool in = i * LPR + sub < npieces;
#pragma unroll
            for (int e = 0; e < VEC; ++e) {
                v[i][e] = in ? (float)raw[i][e] : 0.0f;
                s += v[i][e];
            }
        }
        fetch(row + step);
        const float mu = ln_group_sum<LPR>(s) * inv;
        float q = 0.0f;
#pragma unroll
        for (int i = 0; i < PIECES; ++i) {
            if (i * LPR + sub < npieces) {
#pragma unroll
                for (int e = 0; e < VEC; ++e) {
                    const float d = v[i][e] - mu;
                    q += d * d;
                }
            }
        }
        const float r = 1.0f / sqrtf(ln_group_sum<LPR>(q) * inv + eps);
#pragma unroll
        for (int i = 0; i < PIECES; ++i) {
            const int pc = i * LPR + sub;
            if (pc < npieces) {
                vT out;
#pragma unroll
                for (int e = 0; e < VEC; ++e) out[e] = (T)((v[i][e] - mu) * r * g[i][e] + b[i][e]);
                *reinterpret_cast<vT *>(y + row * cols + pc * VEC) = out;
            }
        }
        if (sub == 0) {
            mean[row] = mu;
            rstd[row] = r;
        }
    }
}

// part: [gridDim.x][2][cols] fp32, the workgroup's sums of dy * xhat (weight) and of dy (bias)
template <typename T, int PIECES, int LPR>
__global__ void __launch_bounds__(kLnThreads)
ln_bwd_kernel(const T *__restrict__ dy, const T *__restrict__ x, const T *__restrict__ gamma, const float *__restrict__ mean,
              const float *__restrict__ rstd, T *__restrict__ dx, float *__restrict__ part, int64_t rows, int cols) {
    constexpr int VEC = LnVec<T>::N, lpr = LPR, rpb = kLnThreads / LPR;
    typedef typename LnVec<T>::type vT;
    __shared__ float red[kLnThreads * PIECES * VEC];      // [rows per workgroup][lpr * PIECES * VEC]
    const int tid = threadIdx.x, sub = tid % lpr, grp = tid / lpr;
    const int npieces = cols / VEC;
    float g[PIECES][VEC], dg[PIECES][VEC], db[PIECES][VEC];
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
        const int pc = i * lpr + sub;
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
            g[i][e] = 1.0f;
            dg[i][e] = 0.0f;
            db[i][e] = 0.0f;
        }
        if (gamma && pc < npieces) {
            const vT w = *reinterpret_cast<const vT *>(gamma + pc * VEC);
#pragma unroll
            for (int e = 0; e < VEC; ++e) g[i][e] = (float)w[e];
        }
    }
    const float inv = 1.0f / (float)cols;
    const int64_t step = (int64_t)gridDim.x * rpb;
    vT xr[PIECES], dr[PIECES];
    float mu_next, r_next;
    auto fetch = [&](int64_t row) {   // (lanes and rows past the end repeat the last)
        row = min(row, rows - 1);
#pragma unroll
        for (int i = 0; i < PIECES; ++i) {
            const int64_t at = row * cols + min(i * lpr + sub, npieces - 1) * VEC;
            xr[i] = *reinterpret_cast<const vT *>(x + at);
            dr[i] = *reinterpret_cast<const vT *>(dy + at);
        }
        mu_next = mean[row];
        r_next = rstd[row];
    };
    fetch((int64_t)blockIdx.x * rpb + grp);
    for (int64_t row = (int64_t)blockIdx.x * rpb + grp; row < rows; row += step) {
        const float mu = mu_next, r = r_next;
        float xh[PIECES][VEC], gy[PIECES][VEC];
        float s1 = 0.0f, s2 = 0.0f;
#pragma unroll
        for (int i = 0; i < PIECES; ++i) {
            if (i * lpr + sub < npieces) {
#pragma unroll
                for (int e = 0; e < VEC; ++e) {
                    const float d = (float)dr[i][e];
                    xh[i][e] = ((float)xr[i][e] - mu) * r;
                    gy[i][e] = d * g[i][e];
                    s1 += gy[i][e];
                    s2 += gy[i][e] * xh[i][e];
                    dg[i][e] += d * xh[i][e];
                    db[i][e] += d;
                }
            } else {
#pragma unroll
                for (int e = 0; e < VEC; ++e) xh[i][e] = gy[i][e] = 0.0f;
            }
        }
        fetch(row + step);
        if (dx) {   // uniform
            const float c1 = ln_group_sum<LPR>(s1) * inv, c2 = ln_group_sum<LPR>(s2) * inv;
#pragma unroll
            for (int i = 0; i < PIECES; ++i) {
                const int pc = i * lpr + sub;
                if (pc < npieces) {
                    vT out;
#pragma unroll
                    for (int e = 0; e < VEC; ++e) out[e] = (T)((gy[i][e] - c1 - xh[i][e] * c2) * r);
                    *reinterpret_cast<vT *>(dx + row * cols + pc * VEC) = out;
                }
            }
        }
    }
    if (!part) return;   // uniform
    // the workgroup's sums: the row groups meet in LDS, first for the weight, then for the bias
    const int pitch = lpr * PIECES * VEC;
#pragma unroll
    for (int pass = 0; pass < 2; ++pass) {
#pragma unroll
        for (int i = 0; i < PIECES; ++i)
#pragma unroll
            for (int e = 0; e < VEC; ++e) red[grp * pitch + (i * lpr + sub) * VEC + e] = pass == 0 ? dg[i][e] : db[i][e];
        __syncthreads();
        for (int c = tid; c < cols; c += kLnThreads) {
            float s = 0.0f;
            for (int r2 = 0; r2 < rpb; ++r2) s += red[r2 * pitch + c];
            part[((int64_t)blockIdx.x * 2 + pass) * cols + c] = s;
        }
        __syncthreads();
    }
}

// Column sums of a dense [rows, cols] array (the bias gradient of a Linear layer): the same walk over
// the rows as the LayerNorm backward, one partial [cols] per workgroup.
template <typename T, int PIECES>
__global__ void __launch_bounds__(kLnThreads)
colsum_kernel(const T *__restrict__ a, float *__restrict__ part, int64_t rows, int cols, int64_t row_stride, int lpr) {
    constexpr int VEC = LnVec<T>::N;
    typedef typename LnVec<T>::type vT;
    __shared__ float red[kLnThreads * PIECES * VEC];
    const int tid = threadIdx.x, sub = tid % lpr, grp = tid / lpr, rpb = kLnThreads / lpr;
    const int npieces = cols / VEC;
    float acc[PIECES][VEC];
#pragma unroll
    for (int i = 0; i < PIECES; ++i)
#pragma unroll
        for (int e = 0; e < VEC; ++e) acc[i][e] = 0.0f;
    for (int64_t row = (int64_t)blockIdx.x * rpb + grp; row < rows; row += (int64_t)gridDim.x * rpb) {
#pragma unroll
        for (int i = 0; i < PIECES; ++i) {
            const int pc = i * lpr + sub;
            if (pc < npieces) {
                const vT v = *reinterpret_cast<const vT *>(a + row * row_stride + pc * VEC);
#pragma unroll
                for (int e = 0; e < VEC; ++e) acc[i][e] += (float)v[e];
            }
        }
    }
    const int pitch = lpr * PIECES * VEC;
#pragma unroll
    for (int i = 0; i < PIECES; ++i)
#pragma unroll
        for (int e = 0; e < VEC; ++e) red[grp * pitch + (i * lpr + sub) * VEC + e] = acc[i][e];
    __syncthreads();
    for (int c = tid; c < cols; c += kLnThreads) {
        float s = 0.0f;
        for (int r2 = 0; r2 < rpb; ++r2) s += red[r2 * pitch + c];
        part[(int64_t)blockIdx.x * cols + c] = s;
    }
}

// dgamma, dbeta = the sums of the partials over the workgroups, in a fixed order (`narr` arrays per partial:
// two for the LayerNorm backward, one for plain column sums, whose result goes to `dgamma`).  A workgroup takes 4
// columns and splits the partials over 64 threads per column, four rows in flight per thread (one
// thread per column walking over a thousand partials waits for a thousand loads in turn: 64 us).
constexpr int kLnRedCols = 4, kLnRedSlices = 64;
template <typename T>
__global__ void __launch_bounds__(kLnRedCols * kLnRedSlices)
ln_reduce_kernel(const float *__restrict__ part, int nblk, int narr, int cols, T *__restrict__ dgamma, T *__restrict__ dbeta) {
    __shared__ float red[2][kLnRedCols][kLnRedSlices];
    const int cq = threadIdx.x % kLnRedCols, rs = threadIdx.x / kLnRedCols, c = blockIdx.x * kLnRedCols + cq;
    float a[4] = {0.0f, 0.0f, 0.0f, 0.0f}, b[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    if (c < cols) {
        int k = rs;
        for (; k + 3 * kLnRedSlices < nblk; k += 4 * kLnRedSlices) {
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const float *row = part + (int64_t)(k + u * kLnRedSlices) * narr * cols;
                a[u] += row[c];
                if (narr == 2) b[u] += row[cols + c];
            }
        }
        for (; k < nblk; k += kLnRedSlices) {
            const float *row = part + (int64_t)k * narr * cols;
            a[0] += row[c];
            if (narr == 2) b[0] += row[cols + c];
        }
    }
    red[0][cq][rs] = (a[0] + a[1]) + (a[2] + a[3]);
    red[1][cq][rs] = (b[0] + b[1]) + (b[2] + b[3]);
    __syncthreads();
    if (threadIdx.x < 2 * kLnRedCols) {
        const int which = threadIdx.x / kLnRedCols, col = blockIdx.x * kLnRedCols + threadIdx.x % kLnRedCols;
        float s = 0.0f;
        for (int i = 0; i < kLnRedSlices; ++i) s += red[which][threadIdx.x % kLnRedCols][i];
        T *out = which == 0 ? dgamma : dbeta;
        if (col < cols && out) out[col] = (T)s;
    }
}

static int ln_elem_bytes(int dtype) { return dtype == EVO_F32 ? 4 : (dtype == EVO_BF16 || dtype == EVO_F16) ? 2 : 0; }

static int ln_check(int64_t rows, int cols, int dtype) {
    const int eb = ln_elem_bytes(dtype);
    if (!eb || rows < 0 || cols <= 0) return EVO_EINVAL;
    const int vec = 16 / eb;
    if (cols % vec) return EVO_EALIGN;
    if (cols / vec > 64 * kLnMaxPieces) return EVO_EUNSUPPORTED;
    if (rows > ((int64_t)1 << 40)) return EVO_EOVERFLOW;
    return EVO_OK;
}

static bool ln_misaligned(const void *p) { return p && ((uintptr_t)p & 15) != 0; }

static unsigned ln_blocks(int64_t rows, int lpr, int most) {
    const int64_t rpb = kLnThreads / lpr, want = (rows + rpb - 1) / rpb;
    return (unsigned)(want < most ? want : most);
}

// `go` with a row's pieces per lane and lanes as constants
template <typename F>
static void ln_forms(const LnShape &s, F go) {
    typedef std::integral_constant<int, 1> One;
    if (s.pieces > 2) go(std::integral_constant<int, 4>(), std::integral_constant<int, 64>());
    else if (s.pieces == 2) go(std::integral_constant<int, 2>(), std::integral_constant<int, 64>());
    else if (s.lpr == 64) go(One(), std::integral_constant<int, 64>());
    else if (s.lpr == 32) go(One(), std::integral_constant<int, 32>());
    else if (s.lpr == 16) go(One(), std::integral_constant<int, 16>());
    else if (s.lpr == 8) go(One(), std::integral_constant<int, 8>());
    else if (s.lpr == 4) go(One(), std::integral_constant<int, 4>());
    else if (s.lpr == 2) go(One(), std::integral_constant<int, 2>());
    else go(One(), One());
}

template <typename T>
static int ln_fwd_launch(const void *x, const void *gamma, const void *beta, void *y, float *mean, float *rstd, int64_t rows,
                         int cols, float eps, hipStream_t st) {
    const LnShape s = ln_shape(cols, LnVec<T>::N);
    const unsigned grid = ln_blocks(rows, s.lpr, kLnFwdBlocks);
    ln_forms(s, [&](auto pieces, auto lpr) {
        ln_fwd_kernel<T, decltype(pieces)::value, decltype(lpr)::value>
            <<<grid, kLnThreads, 0, st>>>((const T *)x, (const T *)gamma, (const T *)beta, (T *)y, mean, rstd, rows, cols, eps);
    });
    return hip_rc();
}

template <typename T>
static int ln_bwd_launch(const void *dy, const void *x, const void *gamma, const float *mean, const float *rstd, void *dx,
                         void *dgamma, void *dbeta, float *part, int64_t rows, int cols, hipStream_t st) {
    const LnShape s = ln_shape(cols, LnVec<T>::N);
    const unsigned grid = ln_blocks(rows, s.lpr, kLnBwdBlocks<T>);
    const bool sums = dgamma || dbeta;
    if (rows > 0) {
        ln_forms(s, [&](auto pieces, auto lpr) {
            ln_bwd_kernel<T, decltype(pieces)::value, decltype(lpr)::value>
                <<<grid, kLnThreads, 0, st>>>((const T *)dy, (const T *)x, (const T *)gamma, mean, rstd, (T *)dx, sums ? part : nullptr, rows, cols);
        });
        if (const int rc = hip_rc()) return rc;
    }
    if (sums) {   // (no rows: no partials, the sums are zero)
        ln_reduce_kernel<T><<<(cols + kLnRedCols - 1) / kLnRedCols, kLnRedCols * kLnRedSlices, 0, st>>>(part, rows > 0 ? (int)grid : 0, 2, cols, (T *)dgamma, (T *)dbeta);
        return hip_rc();
    }
    return EVO_OK;
}

template <typename T>
static int colsum_launch(const void *a, void *out, float *part, int64_t rows, int cols, int64_t row_stride, hipStream_t st) {
    const LnShape s = ln_shape(cols, LnVec<T>::N);
    const unsigned grid = ln_blocks(rows, s.lpr, kLnSumBlocks);
    auto go = [&](auto kern) { kern<<<grid, kLnThreads, 0, st>>>((const T *)a, part, rows, cols, row_stride, s.lpr); };
    if (rows > 0) {
        if (s.pieces == 1) go(colsum_kernel<T, 1>);
        else if (s.pieces == 2) go(colsum_kernel<T, 2>);
        else go(colsum_kernel<T, 4>);
        if (const int rc = hip_rc()) return rc;
    }
    ln_reduce_kernel<T><<<(cols + kLnRedCols - 1) / kLnRedCols, kLnRedCols * kLnRedSlices, 0, st>>>(part, rows > 0 ? (int)grid : 0, 1, cols,
                                                                                                  (T *)out, (T *)nullptr);
    return hip_rc();
}

__global__ void __launch_bounds__(256) keep_mask_kernel(const float *__restrict__ keep, float *__restrict__ out, int64_t n, float inf) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) out[i] = inf * (keep[i] - 1.0f);
}

int launch_column_reduce(const float *part, int blocks, int cols, void *out, int dtype, hipStream_t st) {
    const unsigned grid = (cols + kLnRedCols - 1) / kLnRedCols;
    if (dtype == EVO_BF16) ln_reduce_kernel<bf16_t><<<grid, kLnRedCols * kLnRedSlices, 0, st>>>(part, blocks, 1, cols, (bf16_t *)out, (bf16_t *)nullptr);
    else ln_reduce_kernel<f16_t><<<grid, kLnRedCols * kLnRedSlices, 0, st>>>(part, blocks, 1, cols, (f16_t *)out, (f16_t *)nullptr);
    return hip_rc();
}

}  // namespace evo

extern "C" {

int evoattn_layernorm_fwd(const void *x, const void *gamma, const void *beta, void *y, float *mean, float *rstd, int64_t rows,
                          int32_t cols, int32_t dtype, float eps, void *hip_stream) {
    using namespace evo;
    if (const int rc = ln_check(rows, cols, dtype)) return rc;
    if (!x || !y || !mean || !rstd || !(eps >= 0.0f)) return EVO_EINVAL;
    if (ln_misaligned(x) || ln_misaligned(y) || ln_misaligned(gamma) || ln_misaligned(beta)) return EVO_EALIGN;
    if (rows == 0) return EVO_OK;
    hipStream_t st = (hipStream_t)hip_stream;
    switch (dtype) {
        case EVO_BF16: return ln_fwd_launch<bf16_t>(x, gamma, beta, y, mean, rstd, rows, cols, eps, st);
        case EVO_F16: return ln_fwd_launch<f16_t>(x, gamma, beta, y, mean, rstd, rows, cols, eps, st);
        default: return ln_fwd_launch<float>(x, gamma, beta, y, mean, rstd, rows, cols, eps, st);
    }
}

size_t evoattn_layernorm_bwd_workspace_bytes(int64_t rows, int32_t cols, int32_t dtype) {
    using namespace evo;
    if (ln_check(rows, cols, dtype) != EVO_OK) return 0;
    return (size_t)kLnPartials * 2 * (size_t)cols * sizeof(float);
}

int evoattn_layernorm_bwd(const void *dy, const void *x, const void *gamma, const float *mean, const float *rstd, void *dx,
                          void *dgamma, void *dbeta, void *workspace, size_t workspace_bytes, int64_t rows, int32_t cols,
                          int32_t dtype, void *hip_stream) {
    using namespace evo;
    if (const int rc = ln_check(rows, cols, dtype)) return rc;
    if (!dy || !x || !mean || !rstd || (!dx && !dgamma && !dbeta)) return EVO_EINVAL;
    if (ln_misaligned(dy) || ln_misaligned(x) || ln_misaligned(gamma) || ln_misaligned(dx)) return EVO_EALIGN;
    if ((dgamma || dbeta) && (!workspace || workspace_bytes < evoattn_layernorm_bwd_workspace_bytes(rows, cols, dtype)))
        return EVO_EWORKSPACE;
    if (ln_misaligned(workspace)) return EVO_EALIGN;
    hipStream_t st = (hipStream_t)hip_stream;
    float *part = (float *)workspace;
    switch (dtype) {
        case EVO_BF16: return ln_bwd_launch<bf16_t>(dy, x, gamma, mean, rstd, dx, dgamma, dbeta, part, rows, cols, st);
        case EVO_F16: return ln_bwd_launch<f16_t>(dy, x, gamma, mean, rstd, dx, dgamma, dbeta, part, rows, cols, st);
        default: return ln_bwd_launch<float>(dy, x, gamma, mean, rstd, dx, dgamma, dbeta, part, rows, cols, st);
    }
}

int evoattn_keep_mask(const float *keep, float *out, int64_t n, float inf, void *hip_stream) {
    using namespace evo;
    if (n < 0 || (n && (!keep || !out))) return EVO_EINVAL;
    if (n == 0) return EVO_OK;
    const int64_t want = (n + 255) / 256;
    keep_mask_kernel<<<(unsigned)(want < 2048 ? want : 2048), 256, 0, (hipStream_t)hip_stream>>>(keep, out, n, inf);
    return hip_rc();
}

size_t evoattn_colsum_workspace_bytes(int64_t rows, int32_t cols, int32_t dtype) {
    using namespace evo;
    if (ln_check(rows, cols, dtype) != EVO_OK) return 0;
    return (size_t)kLnPartials * (size_t)cols * sizeof(float);
}

int evoattn_colsum(const void *a, int64_t row_stride, void *out, void *workspace, size_t workspace_bytes, int64_t rows, int32_t cols,
                   int32_t dtype, void *hip_stream) {
    using namespace evo;
    if (const int rc = ln_check(rows, cols, dtype)) return rc;
    if (!a || !out || row_stride < cols) return EVO_EINVAL;
    if (row_stride % (16 / ln_elem_bytes(dtype))) return EVO_EALIGN;
    if (ln_misaligned(a) || ln_misaligned(workspace)) return EVO_EALIGN;
    if (!workspace || workspace_bytes < evoattn_colsum_workspace_bytes(rows, cols, dtype)) return EVO_EWORKSPACE;
    hipStream_t st = (hipStream_t)hip_stream;
    float *part = (float *)workspace;
    switch (dtype) {
        case EVO_BF16: return colsum_launch<bf16_t>(a, out, part, rows, cols, row_stride, st);
        case EVO_F16: return colsum_launch<f16_t>(a, out, part, rows, cols, row_stride, st);
        default: return colsum_launch<float>(a, out, part, rows, cols, row_stride, st);
    }
}

}  // extern "C"
