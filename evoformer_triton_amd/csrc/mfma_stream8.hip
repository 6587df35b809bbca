// Kernels whose rows stream through LDS, head dim 8 (larger ones: mfma_stream.hip).  A row is 16 bytes, one piece of a lane, and a product over 16
// columns holds a row's 8 numbers and, in its upper half, the columns that add mask, LSE and delta; what rounding the scaled Q
// leaves is a second product.
#include "fused_common.h"
#include "kernels.h"
#include "stream_common.h"

namespace evo {

// ------------------------------------------------------------------ forward, two S rows at a time

// As in stream_fwd_pair (mfma_stream.hip) a workgroup takes 128 queries of two S rows, whose bias is the same and unpacked once.  The
// matrix instruction is 16x16x32, whose 32 columns hold the scaled Q, the mask and what rounding the scaled Q left: one instruction per 16 x 16
// scores (32x32x16: two per 32 x 32, the same time), and P V, of whose 16 rows the head dim fills half, takes half of the time it
// takes with 32.  A wave's 32 queries are two halves, for which K and V are read once.
// Bound by the vector ALU, busy all the time (92 instructions per tile of 32 x 32 where there were 104, a third of them before and after the loop; each lane prepares one
// row of Q and they are dealt out through LDS: 264 -> 248).  us, mfma_fwd.hip or, up to 256 keys, mfma_fwd_ring.hip / this, H = 8: S = 1024, N = 384 277 / 248;
// S = 1000: N = 96 48 / 38, 192 104 / 95, 256 125 / 116, 768 967 / 818; with an fp32 bias S = 512, N = 384 169 / 152, N = 768 600 / 483.  (Three waves per SIMD
// cost 4 spilled registers, with an fp32 bias up to 28.)
struct Fwd8 {
    static constexpr int KS = 128, ARR = KS * 16, ROW = 3 * ARR, BYTES = 2 * ROW;   // keys per stage; K, V and the mask's columns of a row; two rows
};

template <typename T, int BT>
__global__ void __launch_bounds__(256, 3) stream_fwd8(EvoAttnParams p, Extra e) {
    typedef Fwd8 R;
    constexpr int D = 8, BES = BT == 2 ? 2 : 4;
    typedef typename Mfma<T>::v8 v8;
    typedef typename Mfma<T>::v4 v4;
    typedef Mfma16<T> M;
    __shared__ __attribute__((aligned(1024))) unsigned char lds[2][R::BYTES], qlds[4 * 4096];

    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), c = lane & 15, j = lane >> 4;
    const int N = p.N, NT = (N + 31) / 32, nqb = (N + 127) / 128, nst = (N + R::KS - 1) / R::KS;
    const unsigned lid = xcd_remap(blockIdx.x, gridDim.x);
    unsigned pid;   // of the pair's first row
    {
        // (pairs in the order in which walk_problem takes problems)
        const unsigned t = lid / nqb, S2 = (unsigned)(p.S + 1) / 2, H = (unsigned)p.H;
        const bool heads_first = p.stride_h < p.stride_n;
        const unsigned bh = heads_first ? t / H / S2 * H + t % H : t / S2, i = heads_first ? t / H % S2 : t % S2;
        pid = bh * (unsigned)p.S + 2 * i;
    }
    const Prob pr = decode_problem(p, pid);
    const int n = pr.s + 1 < p.S ? 2 : 1;   // rows of this pair (uniform; a last single row is computed twice and stored once)
    const int q0 = (lid % nqb) * 128 + wave * 32;
    const bool active = q0 < N;   // wave-uniform
    const int sn2 = (int)p.stride_n * 2, valid = (N - 1) * sn2 + D * 2, np256 = (N + 255) / 256 * 256;
    const bool dead[2] = {uniform_load(e.dead + pr.b * p.S + pr.s) != 0, uniform_load(e.dead + pr.b * p.S + pr.s + n - 1) != 0};

    // A stage's rows: wave w fetches 64 keys of row w / 2 of the pair (of the first one once more where there is no second).
    // Rows 8 .. 15 and 0 .. 7 of every second 16 lie swapped: a product's operand is rows 0 .. 7 and 16 .. 23, which then meet other banks.
    const int fr = (wave >> 1) < n ? wave >> 1 : 0, fpos = (wave & 1) * 64 + lane, frow = fpos ^ ((fpos >> 1) & 8);
    const int64_t fbase = pr.base + (int64_t)fr * p.stride_s;
    const __amdgpu_buffer_rsrc_t krs = __builtin_amdgcn_make_buffer_rsrc((void *)((const T *)p.k + fbase), 0, valid, 0x00020000);
    const __amdgpu_buffer_rsrc_t vrs = __builtin_amdgcn_make_buffer_rsrc((void *)((const T *)p.v + fbase), 0, valid, 0x00020000);
    const __amdgpu_buffer_rsrc_t mrs = __builtin_amdgcn_make_buffer_rsrc((void *)(e.m2a + ((int64_t)pr.b * p.S + pr.s + fr) * np256), 0, np256 * 16, 0x00020000);
    auto fetch = [&](int stage) {   // (rows past the end repeat the last one; the mask has its floor there)
        unsigned char *dst = lds[stage & 1] + (wave >> 1) * R::ROW + (wave & 1) * 1024;
        const int off = min(stage * R::KS + frow, N - 1) * sn2;
        dma16(krs, dst, off);
        dma16(vrs, dst + R::ARR, off);
        dma16(mrs, dst + 2 * R::ARR, min(stage * R::KS + frow, np256 - 1) * 16);
    };
    fetch(0);

    // The query operand, 32 columns: Q scaled, (1 1 1 -maximum) against the mask's, what rounding the scaled Q left, nothing.  Index: 2 row + half of the queries.
    const float cs = p.scale * kLog2e;
    const uint2 one3 = ones3<T>(), zero3 = {0u, 0u};
    // (Each lane prepares the row of index j and leaves the four quarters in LDS of its wave.)
    v8 qb[4];
    {
        const int s = (j >> 1) < n ? j >> 1 : 0;
        const v8 raw = ld8((const T *)p.q + pr.base + (int64_t)s * p.stride_s + (int64_t)min(q0 + 16 * (j & 1) + c, N - 1) * p.stride_n);
        v8 hi, lo;
        scaled_hilo8<T>(raw, (s ? dead[1] : dead[0]) ? 0.0f : cs, hi, lo);
        unsigned char *const own = qlds + wave * 4096;
        v8 *const at = reinterpret_cast<v8 *>(own + j * 1024 + c * 16);
        at[0] = hi;
        at[16] = aug8<T>(one3, zero3);
        at[32] = lo;
        at[48] = zero8<T>();
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
        for (int i = 0; i < 4; ++i) qb[i] = *reinterpret_cast<const v8 *>(own + i * 1024 + lane * 16);
    }
    // bias tiles of these 32 queries in accumulator order: this lane's eight entries of 16 queries x 32 keys are one piece of 16 bytes (fp32: two)
    const int64_t tile0 = ((((int64_t)(e.bias_batches > 1 ? pr.b : 0) * p.H + pr.h) * NT + min(q0 >> 5, NT - 1)) * NT) * 1024;
    const __amdgpu_buffer_rsrc_t brs = __builtin_amdgcn_make_buffer_rsrc(BT == 2 ? (void *)(e.bq16 + tile0) : (void *)(e.bq + tile0), 0, NT * 1024 * BES, 0x00020000);
    const int boff = (j >> 1) * (512 * BES) + (c + 32 * (j & 1)) * 16;
    struct Raw { uint4 w[2]; f32x4 f[2][2]; };
    struct Init { f32x4 v[2][2]; };   // [half of the queries][product]
    auto load_bias = [&](int kt, Raw &r) __attribute__((always_inline)) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int at = min(kt, NT - 1) * 1024 * BES + h * 256;
            if (BT == 2) r.w[h] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(brs, boff, at, 0));
            else {
                r.f[h][0] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(brs, boff, at, 0));
                r.f[h][1] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(brs, boff, at + 1024, 0));
            }
        }
    };
    auto value = [&](const Raw &r) __attribute__((always_inline)) {
        Init v;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            if (BT == 2) {
                const unsigned w[4] = {r.w[h].x, r.w[h].y, r.w[h].z, r.w[h].w};
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    float lo, hi;
                    unpack2<T>(w[i], lo, hi);
                    v.v[h][i >> 1][2 * (i & 1)] = lo * kLog2e;
                    v.v[h][i >> 1][2 * (i & 1) + 1] = hi * kLog2e;
                }
            } else {
                v.v[h][0] = r.f[h][0];
                v.v[h][1] = r.f[h][1];
            }
        }
        return v;
    };
    auto take = [&](const Raw &r) __attribute__((always_inline)) {   // (formed here: the wait for the tile stands before whatever the wave asks for next)
        Init v = value(r);
        asm volatile("" : "+v"(v.v[0][0]), "+v"(v.v[0][1]), "+v"(v.v[1][0]), "+v"(v.v[1][1]));
        return v;
    };
    Raw ct, c1;
    load_bias(0, ct);
    load_bias(1, c1);

    // m, mf, l as in stream_fwd (mfma_stream.hip), of the lane's query; `level`: m == mf everywhere
    float m[4] = {0.f, 0.f, 0.f, 0.f}, mf[4] = {0.f, 0.f, 0.f, 0.f}, l[4] = {0.f, 0.f, 0.f, 0.f};
    f32x4 o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = f32x4{0.f, 0.f, 0.f, 0.f};

    // rows of an operand: keys 16 (c / 8) + 8 t + c % 8 of the tile; transposed ones: the keys of this lane's eight entries, columns 0 .. 7 of V and, from 8 on,
    // twice the second half of the mask's chunk, 1 1 0 0: row 8 of O^T is the sum of the probabilities as they are rounded, by which O is divided.  (Divided
    // by the sum of the unrounded ones O is 4 % further from 64 bits: S = 64, N = 256 2.24e-3 against 2.17e-3.  LSE keeps that sum, and O with an fp32 bias, where
    // the forwards that served these calls before divide by it too and the other reads cost 2 %: columns 0 .. 7 again.)
    const int ka = (j == 1 ? 2 * R::ARR : 0) + (24 * (c >> 3) + (c & 7)) * 16, kstep = c < 8 ? 128 : -128;
    const int va = (BT == 2 && (c & 2) ? 2 * R::ARR + 8 : R::ARR + (c & 1) * 8) + (24 * (j >> 1) + 4 * (j & 1) + (c >> 2)) * 16, vstep = j < 2 ? 128 : -128;
    auto score = [&](const unsigned char *buf, int kb, int row, bool plain, const Init &init, f32x4 (&a)[2][2]) __attribute__((always_inline)) {   // both halves of the queries
        const unsigned char *x = buf + row * R::ROW + ka + kb * 16;
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const v8 k = *reinterpret_cast<const v8 *>(x + t * kstep);
#pragma unroll
            for (int h = 0; h < 2; ++h) a[h][t] = M::mma(k, qb[2 * row + h], plain || !dead[row] ? init.v[h][t] : f32x4{0.f, 0.f, 0.f, 0.f});
        }
    };
    auto settle = [&](int i, bool first, f32x4 *a, int count, float used) __attribute__((always_inline)) {
        float mloc = a[0][0];
#pragma unroll
        for (int t = 0; t < count; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) mloc = fmaxf(mloc, a[t][r]);
        {
            auto x = __builtin_amdgcn_permlane16_swap(__float_as_uint(mloc), __float_as_uint(mloc), false, false);
            mloc = fmaxf(__uint_as_float(x[0]), __uint_as_float(x[1]));
            x = __builtin_amdgcn_permlane32_swap(__float_as_uint(mloc), __float_as_uint(mloc), false, false);
            mloc = fmaxf(__uint_as_float(x[0]), __uint_as_float(x[1]));
        }
        // (not below the floor of masked keys: the scores of a step are -inf where the bias is, and -inf less -inf is no number)
        const float cand = fmaxf(mloc + used, kMaskFloor);
        const bool grow = first || cand > m[i] + 8.0f;   // (moved only when it grows by more than 2^8)
        if (__any(grow || m[i] != used)) {
            const float mn = grow ? cand : m[i];
            if (!first) {
                const float alpha = fast_exp2(m[i] - mn);
                l[i] *= alpha;
#pragma unroll
                for (int r = 0; r < 4; ++r) o[i][r] *= alpha;
            }
            m[i] = mn;
            const float dsub = mn - used;
#pragma unroll
            for (int t = 0; t < count; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) a[t][r] -= dsub;
            mf[i] = fabsf(mn) <= 1024.0f ? mn : 0.0f;
            const v8 qa = aug8<T>(one3, pack_split3<T>(-mf[i]));
            if (j == 1) qb[i] = qa;
        }
    };
    auto probs = [&](f32x4 *a, v8 &pf) __attribute__((always_inline)) {
        float s = 0.0f;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float x = fast_exp2(a[t][r]);
                s += x;
                pf[4 * t + r] = (T)x;
            }
        return s;
    };
    auto values = [&](const unsigned char *buf, int kb, int row) __attribute__((always_inline)) {   // V transposed
        v8 v;
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const v4 w = fused_tr<T>(buf + row * R::ROW + va + kb * 16 + t * vstep);
#pragma unroll
            for (int r = 0; r < 4; ++r) v[4 * t + r] = w[r];
        }
        return v;
    };
    bool level = true;
    auto settled = [&] { level = !__any(m[0] != mf[0] || m[1] != mf[1] || m[2] != mf[2] || m[3] != mf[3]); };
    // the first two tiles, row after row, each row relative to its maximum over both; `between`: what is asked for once the bias has arrived
    auto first = [&](const unsigned char *buf, auto plain, auto between) __attribute__((always_inline)) {
        const Init i0 = take(ct), i1 = take(c1);
        between();
        load_bias(2, ct);
#pragma unroll
        for (int row = 0; row < 2; ++row) {
            f32x4 a[2][2], b[2][2];
            score(buf, 0, row, plain, i0, a);
            score(buf, 32, row, plain, i1, b);
            const v8 v0 = values(buf, 0, row), v1 = values(buf, 32, row);
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int i = 2 * row + h;
                f32x4 ab[4] = {a[h][0], a[h][1], b[h][0], b[h][1]};
                settle(i, true, ab, 4, 0.0f);
                v8 pf;
                l[i] += probs(ab, pf);
                o[i] = M::mma(v0, pf, o[i]);
                l[i] += probs(ab + 2, pf);
                o[i] = M::mma(v1, pf, o[i]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        settled();
    };
    // a key tile of all rows: kt, from row kb of the stage on
    auto step = [&](const unsigned char *buf, int kt, int kb, auto plain, auto between) __attribute__((always_inline)) {
        constexpr int ROWS = 2;
        const Init init = take(ct);
        between();
        load_bias(kt + 1, ct);
        f32x4 a[ROWS][2][2];
        float s[2 * ROWS], top = 0.0f;
        v8 pf[2 * ROWS];
#pragma unroll
        for (int row = 0; row < ROWS; ++row) score(buf, kb, row, plain, init, a[row]);
        const bool lazy = level;
        if (!lazy) {
#pragma unroll
            for (int i = 0; i < 2 * ROWS; ++i) settle(i, false, a[i >> 1][i & 1], 2, mf[i]);
            settled();
        }
#pragma unroll
        for (int i = 0; i < 2 * ROWS; ++i) {
            s[i] = probs(a[i >> 1][i & 1], pf[i]);
            top = i ? fmaxf(top, s[i]) : s[i];
        }
        if (__builtin_expect(lazy && __any(!(top <= 8192.0f)), 0)) {   // some score stands far above m: once more, the long way
            Raw again;
            load_bias(kt, again);
            const Init v = value(again);
#pragma unroll
            for (int row = 0; row < ROWS; ++row) score(buf, kb, row, plain, v, a[row]);
#pragma unroll
            for (int i = 0; i < 2 * ROWS; ++i) {
                settle(i, false, a[i >> 1][i & 1], 2, mf[i]);
                s[i] = probs(a[i >> 1][i & 1], pf[i]);
            }
            settled();
        }
#pragma unroll
        for (int row = 0; row < ROWS; ++row) {
            const v8 v = values(buf, kb, row);
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                l[2 * row + h] += s[2 * row + h];
                o[2 * row + h] = M::mma(v, pf[2 * row + h], o[2 * row + h]);
            }
        }
    };

    wait_loads();
    wait_lds_barrier();
    auto walk = [&](auto plain) __attribute__((always_inline)) {
        auto rest = [&](int s, const unsigned char *buf) __attribute__((always_inline)) {
            if (4 * s + 2 < NT) step(buf, 4 * s + 2, 64, plain, [] {});
            if (4 * s + 3 < NT) step(buf, 4 * s + 3, 96, plain, [] {});
        };
        auto next = [&](int s) { if (s + 1 < nst) fetch(s + 1); };
        if (active) {
            first(lds[0], plain, [&] { next(0); });
            rest(0, lds[0]);
        } else {
            next(0);
        }
        for (int s = 1; s < nst; ++s) {
            wait_loads();
            wait_lds_barrier();
            if (active) {
                const unsigned char *buf = lds[s & 1];
                step(buf, 4 * s, 0, plain, [&] { next(s); });
                if (4 * s + 1 < NT) step(buf, 4 * s + 1, 32, plain, [] {});
                rest(s, buf);
            } else {
                next(s);
            }
        }
    };
    if (!dead[0] && !dead[1]) walk(std::true_type());
    else walk(std::false_type());

    if (!active) return;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if (i / 2 >= n) break;   // uniform
        auto x = __builtin_amdgcn_permlane16_swap(__float_as_uint(l[i]), __float_as_uint(l[i]), false, false);
        float sum = __uint_as_float(x[0]) + __uint_as_float(x[1]);
        x = __builtin_amdgcn_permlane32_swap(__float_as_uint(sum), __float_as_uint(sum), false, false);
        sum = __uint_as_float(x[0]) + __uint_as_float(x[1]);
        const float inv = 1.0f / (BT == 2 ? __shfl(o[i][0], 32 + c) : sum);
        const int q = q0 + 16 * (i & 1) + c;
        if (q < N) {
            if (j == 0) p.lse[pr.row0 + (int64_t)(i / 2) * N + q] = (m[i] + __log2f(sum)) * kLn2;
            if (j < 2) store4<T>((T *)p.o + pr.base + (int64_t)(i / 2) * p.stride_s + (int64_t)q * p.stride_n + 4 * j, o[i][0] * inv, o[i][1] * inv, o[i][2] * inv, o[i][3] * inv);
        }
    }
}

int launch_stream_fwd8(const EvoAttnParams &p, const Extra &e, hipStream_t st) {
    const unsigned pairs = (unsigned)((p.N + 127) / 128) * (unsigned)(p.B * p.H) * (unsigned)((p.S + 1) / 2);
    const bool h = p.dtype == EVO_BF16;
    if (e.bq16) h ? stream_fwd8<bf16_t, 2><<<pairs, 256, 0, st>>>(p, e) : stream_fwd8<f16_t, 2><<<pairs, 256, 0, st>>>(p, e);
    else h ? stream_fwd8<bf16_t, 1><<<pairs, 256, 0, st>>>(p, e) : stream_fwd8<f16_t, 1><<<pairs, 256, 0, st>>>(p, e);
    return hip_rc();
}

// ------------------------------------------------------------------ dBias partials

// stream_dbias (mfma_stream.hip) for this head dim: a workgroup has 128 queries x 128 keys of one (b, h) for a chunk of S rows, a wave 32
// queries x 4 key tiles, whose sums and bias (fp32, log2 units: the first C of the score product) stay in registers.
// The vector ALU is busy for .66 of the time, the matrix core .18, at two waves per SIMD.  S = 1024, N = 384, H = 8: mfma_dbias.hip's kernel 300 us (96 vector instructions per
// tile and row), this 285 (34, and 75 per row to prepare the operands) and 247 since no sum is copied around a tile's branch; two tiles per wave and three waves per SIMD 302; three tiles 475 (spills).
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
    int dead_n;
    auto fetch_queries = [&](int s) {
        const int64_t row = base0 + (int64_t)s * p.stride_s, row0 = ((int64_t)bh * p.S + s) * p.N;
        const unsigned at = (unsigned)qrow * (unsigned)p.stride_n;
        q_n = ld8((const T *)p.q + row + at);
        g_n = ld8((const T *)p.dout + row + at);
        lse_n = (p.lse + row0)[(unsigned)qrow];
        delta_n = (e.delta + row0)[(unsigned)qrow];
        dead_n = e.dead[b * p.S + s];   // (with the rest: as a scalar load it would be waited for at the top of each row)
    };
    const int ka = (g ? 2 * R::ARR : 0) + li * 16, va = (g ? 2 * R::ARR : R::ARR) + li * 16;   // upper half of the columns: the mask's chunk (mask in three parts, 1 1 1)
    fetch_keys(s_begin);
    fetch_queries(s_begin);
    for (int s = s_begin; s < s_end; ++s) {
        wait_loads();
        asm volatile("" : "+v"(q_n), "+v"(g_n), "+v"(lse_n), "+v"(delta_n), "+v"(dead_n));   // (the compiler's own wait for them: here, not behind the next keys' loads)
        const bool dead = __builtin_amdgcn_readfirstlane(dead_n) != 0, kill = dead && p.mask_kind == EVO_MASK_BOOL;
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
#pragma unroll
        for (int j = 0; j < R::TPW; ++j) {
            if (j < tiles) {   // uniform
                f32x16 z;
#pragma unroll
                for (int r = 0; r < 16; ++r) z[r] = 0.0f;
                const v8 k = *reinterpret_cast<const v8 *>(buf + ka + j * 512);
                f32x16 a;
                if (__builtin_expect(!dead, 1)) a = Mfma<T>::mma(k, qf, bias[j]);                             // log2 P^T
                else a = Mfma<T>::mma(k, qf, z);   // (a row with every key masked takes no bias)
                const f32x16 dp = Mfma<T>::mma(*reinterpret_cast<const v8 *>(buf + va + j * 512), gf, z);     // dP^T - delta
                a = Mfma<T>::mma(k, ql, a);
#pragma unroll
                for (int r = 0; r < 16; ++r) sum[j][r] += fast_exp2(a[r]) * dp[r];
            } else {
                asm volatile("");   // (a block of its own for the sums that stay: without one they are copied ahead of the branch, 16 moves a tile)
            }
            __builtin_amdgcn_sched_barrier(0);   // (the next tile's operands would take the registers)
        }
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
