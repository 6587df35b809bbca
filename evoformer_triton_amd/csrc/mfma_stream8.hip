// Kernels whose rows stream through LDS, head dim 8 (larger ones: mfma_stream.hip).  A row is 16 bytes, one piece of a lane, and a product over 16
// columns holds a row's 8 numbers and, in its upper half, the columns that add mask, LSE and delta; what rounding the scaled Q
// leaves is a second product.
#include "kernels.h"
#include "stream_common.h"

namespace evo {

// ------------------------------------------------------------------ dBias partials

// stream_dbias (mfma_stream.hip) for this head dim: a workgroup has 128 queries x 128 keys of one (b, h) for a chunk of S rows, a wave 32
// queries x 4 key tiles, whose sums and bias (fp32, log2 units: the first C of the score product) stay in registers.
// Bound by vector and matrix issue together at two waves per SIMD.  S = 1024, N = 384, H = 8: mfma_dbias.hip's kernel 300 us (96 vector instructions per
// tile and row), this 285 (34, and 75 per row to prepare the operands); two tiles per wave and three waves per SIMD 302; three tiles 475 (spills).
struct Db8 {
    static constexpr int TPW = 4, KB = TPW * 32, QB = 128, ARR = KB * 16;   // K, V and the mask's columns
    static constexpr int KEYS = 3 * ARR;
};

template <typename T, bool BF32>
__global__ void __launch_bounds__(256, 2) stream_dbias8(EvoAttnParams p, Extra e) {
    typedef Db8 R;
    constexpr int D = 8;
    typedef typename Mfma<T>::v8 v8;
    __shared__ __attribute__((aligned(1024))) unsigned char lds[2 * R::KEYS];

    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), li = lane & 31, g = lane >> 5;
    const int NT = (p.N + 31) / 32, nqb = (p.N + R::QB - 1) / R::QB, nkb = (p.N + R::KB - 1) / R::KB;
    const unsigned lid = xcd_remap(blockIdx.x, gridDim.x);
    const int kbi = lid % nkb, qbi = (lid / nkb) % nqb;
    const unsigned bh = (lid / (nkb * nqb)) % (unsigned)(p.B * p.H);
    const int c = lid / (nkb * nqb) / (unsigned)(p.B * p.H), b = bh / p.H, h = bh % p.H;
    const int q0 = qbi * R::QB + wave * 32, k0 = kbi * R::KB, qrow = min(q0 + li, p.N - 1);
    const bool active = q0 < p.N;                    // wave-uniform
    const int tiles = min(R::TPW, NT - k0 / 32);     // of the block's keys that exist
    const int sn2 = (int)p.stride_n * 2, valid = (p.N - 1) * sn2 + D * 2, np256 = (p.N + 255) / 256 * 256;
    const float cs = p.scale * kLog2e;
    const uint2 one3 = ones3<T>(), zero3 = {0u, 0u};

    const int bb = e.bias_batches > 1 ? b : 0;
    f32x16 bias[R::TPW], sum[R::TPW];
#pragma unroll
    for (int j = 0; j < R::TPW; ++j) {
        const int64_t o = ((((int64_t)bb * p.H + h) * NT + min(q0 >> 5, NT - 1)) * NT + min(k0 / 32 + j, NT - 1)) * 1024;
        if constexpr (BF32) {
            load_tile32(e.bq + o + lane * 4, bias[j]);
        } else {
            Tile16 t;
            load_tile16(e.bq16 + o + lane * 8, t);
            unpack_tile16<T>(t, kLog2e, bias[j]);
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) sum[j][r] = 0.0f;
    }
    const int s_begin = c * e.chunk, s_end = min(p.S, s_begin + e.chunk);
    if (s_begin >= s_end) return;   // uniform over the workgroup

    const int64_t base0 = (int64_t)b * p.stride_b + (int64_t)h * p.stride_h;
    // K, V and the mask's columns of a row: pieces of 64 keys in turn over the waves.  (Rows past the end: zeros.  Their keys are not stored.)
    int off[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int n = wave + 4 * i, r = n / 3 * 64 + lane;
        off[i] = n % 3 == 2 ? r * 16 : r * sn2;
    }
    auto fetch_keys = [&](int s) {
        unsigned char *dst = lds + ((s - s_begin) & 1) * R::KEYS;
        const int64_t row = base0 + (int64_t)s * p.stride_s;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int n = wave + 4 * i, a = n % 3;
            if (n >= 3 * R::ARR / 1024) break;   // uniform
            const void *x = a == 0 ? (const void *)((const T *)p.k + row + (int64_t)k0 * p.stride_n)
                            : a == 1 ? (const void *)((const T *)p.v + row + (int64_t)k0 * p.stride_n)
                                     : (const void *)(e.m2a + ((int64_t)b * p.S + s) * np256 + k0);
            dma16(__builtin_amdgcn_make_buffer_rsrc((void *)x, 0, a == 2 ? (np256 - k0) * 16 : valid - k0 * sn2, 0x00020000), dst + a * R::ARR + n / 3 * 1024, off[i]);
        }
    };
    // this lane's row of Q and of dO, LSE and delta of row s
    v8 q_n, g_n;
    float lse_n, delta_n;
    auto fetch_queries = [&](int s) {
        const int64_t row = base0 + (int64_t)s * p.stride_s, row0 = ((int64_t)bh * p.S + s) * p.N;
        const unsigned at = (unsigned)qrow * (unsigned)p.stride_n;
        q_n = ld8((const T *)p.q + row + at);
        g_n = ld8((const T *)p.dout + row + at);
        lse_n = (p.lse + row0)[(unsigned)qrow];
        delta_n = (e.delta + row0)[(unsigned)qrow];
    };
    const int ka = (g ? 2 * R::ARR : 0) + li * 16, va = (g ? 2 * R::ARR : R::ARR) + li * 16;   // upper half of the columns: the mask's chunk (mask in three parts, 1 1 1)
    fetch_keys(s_begin);
    fetch_queries(s_begin);
    for (int s = s_begin; s < s_end; ++s) {
        const bool dead = uniform_load(e.dead + b * p.S + s) != 0, kill = dead && p.mask_kind == EVO_MASK_BOOL;
        wait_loads();
        wait_lds_barrier();
        if (s + 1 < s_end) fetch_keys(s + 1);   // (everybody has left that buffer: it held row s - 1)
        v8 qf, ql, gf;
        scaled_hilo8<T>(q_n, dead ? 0.0f : cs, qf, ql);
        const v8 qa = aug8<T>(one3, pack_split3<T>(-lse_n * kLog2e)), ga = aug8<T>(zero3, pack_split3<T>(-delta_n));
        qf = g ? qa : qf;
        ql = g ? zero8<T>() : ql;
        gf = g ? ga : g_n;
        asm volatile("" : "+v"(qf), "+v"(ql), "+v"(gf));   // (formed before what they are made of is asked for again)
        if (s + 1 < s_end) fetch_queries(s + 1);
        if (!active || kill) continue;
        const unsigned char *buf = lds + ((s - s_begin) & 1) * R::KEYS;
        auto walk = [&](auto plain) {
#pragma unroll
            for (int j = 0; j < R::TPW; ++j) {
                if (j < tiles) {   // uniform
                    f32x16 z;
#pragma unroll
                    for (int r = 0; r < 16; ++r) z[r] = 0.0f;
                    const v8 k = *reinterpret_cast<const v8 *>(buf + ka + j * 512);
                    f32x16 a = Mfma<T>::mma(k, qf, plain ? bias[j] : z), dp;                                // log2 P^T
                    dp = Mfma<T>::mma(*reinterpret_cast<const v8 *>(buf + va + j * 512), gf, z);          // dP^T - delta
                    a = Mfma<T>::mma(k, ql, a);
#pragma unroll
                    for (int r = 0; r < 16; ++r) sum[j][r] += fast_exp2(a[r]) * dp[r];
                }
                __builtin_amdgcn_sched_barrier(0);   // (the next tile's operands would take the registers)
            }
        };
        if (!dead) walk(std::true_type());
        else walk(std::false_type());   // (a row with every key masked takes no bias)
    }
    // the partial of this chunk: lane = query li, registers 4 rr .. 4 rr + 3 = keys 8 rr + 4 g ..
    if (active && q0 + li < p.N) {
        float *part = e.dbias_part + ((((int64_t)c * p.B + b) * p.H + h) * p.N + (q0 + li)) * p.N;
#pragma unroll
        for (int j = 0; j < R::TPW; ++j)
#pragma unroll
            for (int rr = 0; rr < 4; ++rr) {
                const int kg = k0 + 32 * j + 8 * rr + 4 * g;
                if ((p.N & 3) == 0 && kg + 4 <= p.N) {
                    f32x4 v;
                    v[0] = sum[j][4 * rr]; v[1] = sum[j][4 * rr + 1]; v[2] = sum[j][4 * rr + 2]; v[3] = sum[j][4 * rr + 3];
                    *reinterpret_cast<f32x4 *>(part + kg) = v;
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (kg + i < p.N) part[kg + i] = sum[j][4 * rr + i];
                }
            }
    }
}

int launch_mfma_dbias_d8(const EvoAttnParams &p, const Extra &e, hipStream_t st) {
    typedef Db8 R;
    const int64_t grid = (int64_t)((p.N + R::QB - 1) / R::QB) * ((p.N + R::KB - 1) / R::KB) * p.B * p.H * e.n_chunks;
    if (grid <= 0 || grid > 0x7fffffff) return EVO_EOVERFLOW;
    const bool f = p.bias_dtype == EVO_F32;
    if (p.dtype == EVO_BF16) {
        if (f) stream_dbias8<bf16_t, true><<<(unsigned)grid, 256, 0, st>>>(p, e);
        else stream_dbias8<bf16_t, false><<<(unsigned)grid, 256, 0, st>>>(p, e);
    } else {
        if (f) stream_dbias8<f16_t, true><<<(unsigned)grid, 256, 0, st>>>(p, e);
        else stream_dbias8<f16_t, false><<<(unsigned)grid, 256, 0, st>>>(p, e);
    }
    return hip_rc();
}

}  // namespace evo
