// Forward, dQ, dK/dV and dBias for head dims 32, 64 and 128: one workgroup per block of rows of a problem
// (b, h, s), the other side's rows streamed through LDS.  Compiled once per head dim (-DEVO_D=32|64|128).
//
// The arithmetic is that of the one-workgroup-per-problem kernels for smaller head dims (mfma_fwd.hip, mfma_bwd.hip,
// mfma_dq_wide.hip: every additive term of the score rides in the matrix instruction, the scaled Q rounded once in the
// same way everywhere), and so is a wave's part: 32 rows, and 32 x 32 tiles against the other side.  What differs is how the
// other side arrives.  At these head dims a wave keeps 110 to 250 registers, a SIMD two to four waves, and kernels that staged
// 128 rows at a time between two barriers waited 60 to 85 % of their time for memory with every unit less than 35 %
// busy.  Here
//   * rows go from memory into LDS by the load path itself (`buffer_load_dwordx4 ... lds`), no register in between, a stage of
//     64 (head dim 128 in the dK/dV kernel: 32) rows ahead of the one that is computed on: one barrier per stage, and the
//     wait before it finds the rows there;
//   * V, K, dO and Q lie row-major; the operands that need them transposed read them by `ds_read_b64_tr_b16`;
//   * a lane's 16-byte piece of a row is stored at chunk c ^ x(row), x the row's low bits reversed: reads of one chunk of
//     consecutive rows and transposing reads of four chunks of eight rows both touch all banks evenly (with the bits in
//     order the eight rows met in half of the banks).
#include "kernels.h"
#include "stream_common.h"

#ifndef EVO_D
#error "compile with -DEVO_D=<head dim>"
#endif

namespace evo {

// ------------------------------------------------------------------ forward

template <int D>
struct FwdStream {
    static constexpr int ROWS = 64, OFF_V = ROWS * D * 2, OFF_A = 2 * ROWS * D * 2, BYTES = OFF_A + ROWS * 16;
};

template <typename T, int D, int BT>
__global__ void __launch_bounds__(256, D == 32 ? (BT == 0 ? 4 : 3) : D == 64 && BT < 3 ? 3 : 2) stream_fwd(EvoAttnParams p, Extra e) {
    typedef StreamGeo<D> G;
    typedef FwdStream<D> R;
    constexpr int NW = 4, KSD = D / 16, KS = KSD + 1, DT = D / 32;
    constexpr int ST = D == 32 ? 2 : 1;
    // ST: key tiles per step.  Wider heads leave no registers for a second tile of scores.  Two tiles
    // add up exactly as in mfma_fwd.hip.
    // (Three waves per SIMD: S = N = 384, H = 4 97 us; at four the second tile spills, 124 us; mfma_fwd.hip's form 124 us.)
    typedef typename Mfma<T>::v8 v8;
    __shared__ __attribute__((aligned(1024))) unsigned char lds[2][R::BYTES];

    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), li = lane & 31, g = lane >> 5;
    const int NT = (p.N + 31) / 32, nqb = (p.N + 127) / 128;
    const unsigned lid = xcd_remap(blockIdx.x, gridDim.x);
    const Prob pr = walk_problem(p, lid / nqb);
    const int q0 = (lid % nqb) * 128 + wave * 32, qrow = min(q0 + li, p.N - 1);
    const bool active = q0 < p.N;   // wave-uniform
    const bool dead = e.dead[pr.b * p.S + pr.s] != 0;
    const int sn2 = (int)p.stride_n * 2, valid = (p.N - 1) * sn2 + D * 2;
    const __amdgpu_buffer_rsrc_t krs = __builtin_amdgcn_make_buffer_rsrc((void *)((const T *)p.k + pr.base), 0, valid, 0x00020000);
    const __amdgpu_buffer_rsrc_t vrs = __builtin_amdgcn_make_buffer_rsrc((void *)((const T *)p.v + pr.base), 0, valid, 0x00020000);
    const int np256 = (p.N + 255) / 256 * 256;
    const __amdgpu_buffer_rsrc_t mrs =
        __builtin_amdgcn_make_buffer_rsrc((void *)(e.m2a + ((int64_t)pr.b * p.S + pr.s) * np256), 0, np256 * 16, 0x00020000);
    auto fetch = [&](int stage) {
        unsigned char *dst = lds[stage & 1];
        dma_rows<D, R::ROWS, NW>(krs, vrs, dst, stage * R::ROWS, p.N, sn2, wave, lane);
        if (wave == 0) dma16(mrs, dst + R::OFF_A, (stage * R::ROWS + lane) * 16);
    };
    fetch(0);

    // Q operand: data times scale * log2(e), rounded once; ones against the mask columns
    const float c = p.scale * kLog2e;
    v8 qf[KS];
    {
        const T *Q = (const T *)p.q + pr.base + (int64_t)qrow * p.stride_n;
#pragma unroll
        for (int ks = 0; ks < KSD; ++ks) qf[ks] = ld8(Q + ks * 16 + g * 8);
    }
    const BiasStream<T, BT, false> bias(p, e, pr, min(q0 >> 5, NT - 1), qrow, dead, lane);
    // AHEAD: tiles whose bias is asked for together.  Where few S rows leave the caller's bias rows as the traffic (head dim 64) it is
    // both tiles of a stage, 256 bytes of a row at a time, which memory serves better than 128: B = 4, S = 1, N = 1024, H = 32, fp32 164 -> 148 us.  They are asked
    // for when the stage before is half done: at its beginning they took 16 registers more than three waves per SIMD have (at two waves N = 1024 147 us, 768 89,
    // 725 114; at three, so, 143, 84, 87; at three with what does not fit spilled 211, 106).  (Prepared tiles lie whole: S = 200, N = 640, H = 5, fp32 190 / 204.)
    constexpr int AHEAD = D == 64 && BT >= 3 ? 2 : ST;
    typename BiasStream<T, BT, false>::Tile ct[AHEAD];
#pragma unroll
    for (int t = 0; t < AHEAD; ++t) bias.load(t, ct[t]);
    asked_together<KSD>(qf);
#pragma unroll
    for (int ks = 0; ks < KSD; ++ks) qf[ks] = dead ? zero8<T>() : scaled8<T>(qf[ks], c);
    qf[KSD] = zero8<T>();
    if (g == 0) qf[KSD][0] = qf[KSD][1] = qf[KSD][2] = (T)1.0f;

    // m: the maximum the probabilities are relative to; mf: what the mask step subtracts inside the product (m, or 0 while
    // m is unknown or too large for three 16-bit columns): after the first step the scores arrive relative to m, and
    // a later one searches its maximum only when its sums show that it stands far above (see mfma_fwd.hip).
    float m = 0.0f, mf = 0.0f, l = 0.0f;
    f32x16 o[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[dt][r] = 0.0f;

    auto score = [&](const unsigned char *buf, int kb, const f32x16 &init, f32x16 &a) {
        a = init;
#pragma unroll
        for (int ks = 0; ks < KSD; ++ks) a = Mfma<T>::mma(*reinterpret_cast<const v8 *>(buf + G::at(kb + li, 2 * ks + g)), qf[ks], a);
        a = Mfma<T>::mma(*reinterpret_cast<const v8 *>(buf + R::OFF_A + (kb + li) * 16), qf[KSD], a);   // (zero in the step's upper half)
    };
    auto settle = [&](bool first, f32x16 (&a)[ST], float used) {
        float mloc = a[0][0];
#pragma unroll
        for (int t = 0; t < ST; ++t)
#pragma unroll
            for (int r = 0; r < 16; ++r) mloc = fmaxf(mloc, a[t][r]);
        const unsigned u = __float_as_uint(mloc);
        auto sw = __builtin_amdgcn_permlane32_swap(u, u, false, false);
        // (not below the floor of masked keys: the scores of a step are -inf where the bias is, and -inf less -inf is no number)
        const float cand = fmaxf(fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1])) + used, kMaskFloor);
        const bool grow = first || cand > m + 8.0f;   // (moved only when it grows by more than 2^8)
        if (__any(grow || m != used)) {
            const float mn = grow ? cand : m;
            if (!first) {
                const float alpha = fast_exp2(m - mn);
                l *= alpha;
#pragma unroll
                for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                    for (int r = 0; r < 16; ++r) o[dt][r] *= alpha;
            }
            m = mn;
            const float dsub = m - used;
#pragma unroll
            for (int t = 0; t < ST; ++t)
#pragma unroll
                for (int r = 0; r < 16; ++r) a[t][r] -= dsub;
            mf = fabsf(m) <= 1024.0f ? m : 0.0f;
            const v8 qa = aug8<T>(ones3<T>(), pack_split3<T>(-mf));
            if (g == 0) qf[KSD] = qa;
        }
    };
    auto probs = [&](f32x16 (&a)[ST], v8 (&pf)[2 * ST]) {
        float s = 0.0f;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            float x = 0.0f;
#pragma unroll
            for (int t = 0; t < ST; ++t) {
                a[t][r] = fast_exp2(a[t][r]);
                x = t ? x + a[t][r] : a[t][r];
            }
            s += x;
        }
#pragma unroll
        for (int ts = 0; ts < 2 * ST; ++ts)
#pragma unroll
            for (int i = 0; i < 8; ++i) pf[ts][i] = (T)a[ts / 2][8 * (ts & 1) + i];
        return s;
    };
    // AHEAD tiles' bias, from tile kt on, and the next ones asked for; `between`: what is asked for once these have arrived
    // (a tile that is a C operand as it lies: `step` asks for the next one where this one's chain has begun)
    constexpr bool IN_PLACE = BT == 1;
    auto biases = [&](int kt, f32x16 (&init)[AHEAD], auto between) {
        if constexpr (IN_PLACE) {
#pragma unroll
            for (int t = 0; t < AHEAD; ++t) bias.arrived(ct[t]);
            between();
        } else {
#pragma unroll
            for (int t = 0; t < AHEAD; ++t) init[t] = bias.take(ct[t]);
            between();
#pragma unroll
            for (int t = 0; t < AHEAD; ++t) bias.load(kt + AHEAD + t, ct[t]);
        }
    };
    // ST tiles, from tile kt and row kb of the stage on
    auto step = [&](const unsigned char *buf, int kt, int kb, const f32x16 *init, auto first) __attribute__((always_inline)) {
        const float used = mf;
        f32x16 a[ST];
        if constexpr (IN_PLACE) {
#pragma unroll
            for (int t = 0; t < ST; ++t) score(buf, kb + 32 * t, ct[t], a[t]);
#pragma unroll
            for (int t = 0; t < ST; ++t) bias.refill(kt + ST + t, ct[t]);
        } else {
#pragma unroll
            for (int t = 0; t < ST; ++t) score(buf, kb + 32 * t, init[t], a[t]);
        }
        const bool lazy = !first && !__any(m != used);
        if (!lazy) settle(first, a, used);
        v8 pf[2 * ST];
        float s = probs(a, pf);
        if (__builtin_expect(lazy && __any(!(s <= 8192.0f)), 0)) {   // some score stands far above m: once more, the long way
#pragma unroll
            for (int t = 0; t < ST; ++t) {
                typename BiasStream<T, BT, false>::Tile again;
                bias.load(kt + t, again);
                score(buf, kb + 32 * t, bias.value(again), a[t]);
            }
            settle(false, a, used);
            s = probs(a, pf);
        }
        l += s;
#pragma unroll
        for (int ts = 0; ts < 2 * ST; ++ts)
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
                o[dt] = Mfma<T>::mma(transposed<T, D>(buf + R::OFF_V, kb + (ts / 2) * 32, ts & 1, dt, lane), pf[ts], o[dt]);
    };

    const int nst = (p.N + R::ROWS - 1) / R::ROWS;
    wait_loads();
    wait_lds_barrier();
    auto stage = [&](int s, auto first) __attribute__((always_inline)) {
        auto next = [&] { if (s + 1 < nst) fetch(s + 1); };
        if (AHEAD > ST && active) {   // (the next stage's bias is asked for in the middle of this one, when both of this one's tiles have left their registers)
            const unsigned char *buf = lds[s & 1];
            f32x16 init = bias.take(ct[0]);
            next();
            step(buf, 2 * s, 0, &init, first);
            if (2 * s + 1 < NT) {
                init = bias.take(ct[AHEAD - 1]);
                bias.load(2 * s + 2, ct[0]);
                bias.load(2 * s + 3, ct[AHEAD - 1]);
                step(buf, 2 * s + 1, 32, &init, std::false_type());
            }
        } else if (active) {
            const unsigned char *buf = lds[s & 1];
            f32x16 init[AHEAD];
            biases(2 * s, init, next);
            step(buf, 2 * s, 0, init, first);
            if (ST == 1 && 2 * s + 1 < NT) {
                biases(2 * s + 1, init, [] {});
                step(buf, 2 * s + 1, 32, init, std::false_type());
            }
        } else {
            next();
        }
        if (s + 1 < nst) {
            // (a stage before the last has two tiles, and the bias asked for there, four pieces or more for each, is younger than the rows)
            if (AHEAD > ST && active) wait_loads_but<8>();
            else wait_loads();
            wait_lds_barrier();
        }
    };
    // (Head dim 128, 16-bit tiles: the first stage by itself; with bf16 the compiler left its test in the loop otherwise.  us, S = 120, N = 58, H = 32 62.6 -> 59.7, S = 187,
    // N = 56, H = 16 49.2 -> 47.2; some 600 calls of 33 to 64 keys .96 of the time at the median, longer ones 1.00.)
    if constexpr (D == 128 && BT == 2) {
        stage(0, std::true_type());
        for (int s = 1; s < nst; ++s) stage(s, std::false_type());
    } else {
        for (int s = 0; s < nst; ++s) stage(s, s == 0);
    }

    if (!active) return;
    l += __shfl_xor(l, 32);
    const float inv = 1.0f / l;
    if (q0 + li >= p.N) return;
    if (g == 0) p.lse[pr.row0 + q0 + li] = (m + __log2f(l)) * kLn2;
    const int64_t off = pr.base + (int64_t)(q0 + li) * p.stride_n;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
        if (p.o) store_row_tile<T>((T *)p.o + off, dt * 32, D, o[dt], inv, g);
        if (p.gate) {
#pragma unroll
            for (int r = 0; r < 16; ++r) o[dt][r] *= inv;
            gate_row_tile<T>((const T *)p.gate + off, dt * 32, D, o[dt], g);
            store_row_tile<T>((T *)p.o_gated + off, dt * 32, D, o[dt], 1.0f, g);
        }
    }
}

#if EVO_D == 32
// ------------------------------------------------------------------ forward, two S rows at a time

// stream_fwd for head dim 32 where the vector unit's issue is the bound (0.86 of the time, 101 instructions per tile, 32 of them to unpack and
// scale 16 bit bias entries): a workgroup takes the same 128 queries of two S rows, which have the same bias, so a tile of it is
// unpacked once and is the first C of both rows' chains.  After the first two tiles a step takes one key tile of
// both rows instead of two of one: the scores of two tiles are what the registers of three waves per SIMD hold, and two rows keep the units
// as busy.  (The probabilities are stream_fwd's, their sums are added in another order.  Gated calls keep stream_fwd: the bias of a block's pair norm
// has a gradient that is zero but for the rounding of O.)
// us, stream_fwd / this: H = 4, S = N = 768 501 / 455, 512 168 / 153, 384 81 / 75; H = 8, S = 128, N = 384 53.7 / 50.6; S = 300, N = 224 54.5 / 51.1; with
// an fp32 bias S = N = 768, H = 4 536 / 486.  (Three waves per SIMD cost 6 spilled registers, with an fp32 bias in bf16 23.)
template <typename T, int BT>
__global__ void __launch_bounds__(256, 3) stream_fwd_pair(EvoAttnParams p, Extra e) {
    constexpr int D = 32, NW = 4, KSD = D / 16, KS = KSD + 1;
    typedef StreamGeo<D> G;
    typedef FwdStream<D> R;
    typedef typename Mfma<T>::v8 v8;
    __shared__ __attribute__((aligned(1024))) unsigned char lds[2][2][R::BYTES];   // stage parity, S row

    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), li = lane & 31, g = lane >> 5;
    const int NT = (p.N + 31) / 32, nqb = (p.N + 127) / 128;
    const unsigned lid = xcd_remap(blockIdx.x, gridDim.x);
    unsigned pid;   // of the pair's first row
    {
        // (pairs in the order in which walk_problem takes problems)
        const unsigned t = lid / nqb, S2 = (unsigned)(p.S + 1) / 2, H = (unsigned)p.H;
        const bool heads_first = p.stride_h < p.stride_n && p.N <= 512;
        const unsigned bh = heads_first ? t / H / S2 * H + t % H : t / S2, i = heads_first ? t / H % S2 : t % S2;
        pid = bh * (unsigned)p.S + 2 * i;
    }
    const Prob pr = decode_problem(p, pid);
    const int n = pr.s + 1 < p.S ? 2 : 1;   // rows of this pair (uniform)
    const int q0 = (lid % nqb) * 128 + wave * 32, qrow = min(q0 + li, p.N - 1);
    const bool active = q0 < p.N;   // wave-uniform
    const int sn2 = (int)p.stride_n * 2, valid = (p.N - 1) * sn2 + D * 2, np256 = (p.N + 255) / 256 * 256;
    bool dead[2];
    int64_t base[2];
    __amdgpu_buffer_rsrc_t krs[2], vrs[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int s = j < n ? pr.s + j : pr.s;
        dead[j] = uniform_load(e.dead + pr.b * p.S + s) != 0;
        base[j] = pr.base + (int64_t)(s - pr.s) * p.stride_s;
        krs[j] = __builtin_amdgcn_make_buffer_rsrc((void *)((const T *)p.k + base[j]), 0, valid, 0x00020000);
        vrs[j] = __builtin_amdgcn_make_buffer_rsrc((void *)((const T *)p.v + base[j]), 0, valid, 0x00020000);
    }
    const int sm = pr.s + (wave < n ? wave : 0);   // the first two waves fetch a row's mask each
    const __amdgpu_buffer_rsrc_t mrs = __builtin_amdgcn_make_buffer_rsrc((void *)(e.m2a + ((int64_t)pr.b * p.S + sm) * np256), 0, np256 * 16, 0x00020000);
    auto fetch = [&](int stage) {
#pragma unroll
        for (int j = 0; j < 2; ++j)
            if (j < n) dma_rows<D, R::ROWS, NW>(krs[j], vrs[j], lds[stage & 1][j], stage * R::ROWS, p.N, sn2, wave, lane);
        if (wave < n) dma16(mrs, lds[stage & 1][wave] + R::OFF_A, (stage * R::ROWS + lane) * 16);
    };
    fetch(0);

    const float c = p.scale * kLog2e;
    v8 qf[2][KS];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const T *Q = (const T *)p.q + base[j] + (int64_t)qrow * p.stride_n;
#pragma unroll
        for (int ks = 0; ks < KSD; ++ks) qf[j][ks] = ld8(Q + ks * 16 + g * 8);
    }
    const BiasStream<T, BT, false> bias(p, e, pr, min(q0 >> 5, NT - 1), qrow, false, lane);
    typename BiasStream<T, BT, false>::Tile ct, c1;
    bias.load(0, ct);
    bias.load(1, c1);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        asked_together<KSD>(qf[j]);
#pragma unroll
        for (int ks = 0; ks < KSD; ++ks) qf[j][ks] = dead[j] ? zero8<T>() : scaled8<T>(qf[j][ks], c);
        qf[j][KSD] = zero8<T>();
        if (g == 0) qf[j][KSD][0] = qf[j][KSD][1] = qf[j][KSD][2] = (T)1.0f;
    }

    float m[2] = {0.0f, 0.0f}, mf[2] = {0.0f, 0.0f}, l[2] = {0.0f, 0.0f};   // as in stream_fwd
    f32x16 o[2];
#pragma unroll
    for (int r = 0; r < 16; ++r) o[0][r] = o[1][r] = 0.0f;

    auto score = [&](int j, bool plain, const unsigned char *buf, int kb, const f32x16 &init, f32x16 &a) {
        const v8 k0 = *reinterpret_cast<const v8 *>(buf + G::at(kb + li, g));
        if (plain || !dead[j]) {
            a = Mfma<T>::mma(k0, qf[j][0], init);
        } else {   // (a row with every key masked takes no bias)
            f32x16 z;
#pragma unroll
            for (int r = 0; r < 16; ++r) z[r] = 0.0f;
            a = Mfma<T>::mma(k0, qf[j][0], z);
        }
#pragma unroll
        for (int ks = 1; ks < KSD; ++ks) a = Mfma<T>::mma(*reinterpret_cast<const v8 *>(buf + G::at(kb + li, 2 * ks + g)), qf[j][ks], a);
        a = Mfma<T>::mma(*reinterpret_cast<const v8 *>(buf + R::OFF_A + (kb + li) * 16), qf[j][KSD], a);   // (zero in the step's upper half)
    };
    // (`a`: the one or two tiles of a step)
    auto settle = [&](int j, bool first, auto &a, float used) {
        constexpr int ST = sizeof(a) / sizeof(f32x16);
        float mloc = a[0][0];
#pragma unroll
        for (int t = 0; t < ST; ++t)
#pragma unroll
            for (int r = 0; r < 16; ++r) mloc = fmaxf(mloc, a[t][r]);
        const unsigned u = __float_as_uint(mloc);
        auto sw = __builtin_amdgcn_permlane32_swap(u, u, false, false);
        const float cand = fmaxf(fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1])) + used, kMaskFloor);
        const bool grow = first || cand > m[j] + 8.0f;
        if (__any(grow || m[j] != used)) {
            const float mn = grow ? cand : m[j];
            if (!first) {
                const float alpha = fast_exp2(m[j] - mn);
                l[j] *= alpha;
#pragma unroll
                for (int r = 0; r < 16; ++r) o[j][r] *= alpha;
            }
            m[j] = mn;
            const float dsub = mn - used;
#pragma unroll
            for (int t = 0; t < ST; ++t)
#pragma unroll
                for (int r = 0; r < 16; ++r) a[t][r] -= dsub;
            mf[j] = fabsf(mn) <= 1024.0f ? mn : 0.0f;
            const v8 qa = aug8<T>(ones3<T>(), pack_split3<T>(-mf[j]));
            if (g == 0) qf[j][KSD] = qa;
        }
    };
    auto probs = [&](f32x16 &a, v8 (&pf)[2]) {
        float s = 0.0f;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            a[r] = fast_exp2(a[r]);
            s += a[r];
        }
#pragma unroll
        for (int ts = 0; ts < 2; ++ts)
#pragma unroll
            for (int i = 0; i < 8; ++i) pf[ts][i] = (T)a[8 * ts + i];
        return s;
    };
    auto add = [&](int j, const unsigned char *buf, int kb, const v8 (&pf)[2]) {
#pragma unroll
        for (int ts = 0; ts < 2; ++ts) o[j] = Mfma<T>::mma(transposed<T, D>(buf + R::OFF_V, kb, ts, 0, lane), pf[ts], o[j]);
    };
    // The first two tiles, row after row, each row relative to its maximum over both, as in stream_fwd (its probabilities
    // are then that kernel's to the bit); `between`: what is asked for once the bias has arrived
    auto first = [&](const unsigned char *buf, auto rows, auto plain, auto between) {
        constexpr int ROWS = decltype(rows)::value;
#pragma unroll
        for (int j = 0; j < ROWS; ++j) {
            f32x16 a[2];
            v8 pf[2];
            {
                const f32x16 i0 = bias.take(ct), i1 = bias.take(c1);
                if (j == 0) between();
                score(j, plain, buf + j * R::BYTES, 0, i0, a[0]);
                score(j, plain, buf + j * R::BYTES, 32, i1, a[1]);
            }
            settle(j, true, a, 0.0f);
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                l[j] += probs(a[t], pf);
                add(j, buf + j * R::BYTES, 32 * t, pf);
            }
            __builtin_amdgcn_sched_barrier(0);   // (both rows' tiles at once would not fit the registers)
        }
        bias.load(2, ct);
    };
    // a key tile of all (one or both) rows: kt, from row kb of the stage on
    auto step = [&](const unsigned char *buf, int kt, int kb, auto rows, auto plain, auto between) {
        constexpr int ROWS = decltype(rows)::value;
        f32x16 init;
        if (BT == 1) bias.arrived(ct);   // (the C operand as it lies)
        else init = bias.take(ct);
        between();
        if (BT != 1) bias.load(kt + 1, ct);
        f32x16 a[ROWS][1];
        float used[ROWS], s[ROWS];
        v8 pf[ROWS][2];
#pragma unroll
        for (int j = 0; j < ROWS; ++j) {
            used[j] = mf[j];
            score(j, plain, buf + j * R::BYTES, kb, bias.lies(ct, init), a[j][0]);
        }
        if (BT == 1) bias.refill(kt + 1, ct);
        const bool lazy = !__any(m[0] != mf[0] || m[ROWS - 1] != mf[ROWS - 1]);
        if (!lazy)
#pragma unroll
            for (int j = 0; j < ROWS; ++j) settle(j, false, a[j], used[j]);
#pragma unroll
        for (int j = 0; j < ROWS; ++j) s[j] = probs(a[j][0], pf[j]);
        if (__builtin_expect(lazy && __any(!(s[0] <= 8192.0f) || !(s[ROWS - 1] <= 8192.0f)), 0)) {   // some score stands far above m: once more, the long way
            typename BiasStream<T, BT, false>::Tile again;
            bias.load(kt, again);
#pragma unroll
            for (int j = 0; j < ROWS; ++j) {
                score(j, plain, buf + j * R::BYTES, kb, bias.value(again), a[j][0]);
                settle(j, false, a[j], used[j]);
                s[j] = probs(a[j][0], pf[j]);
            }
        }
#pragma unroll
        for (int j = 0; j < ROWS; ++j) {
            l[j] += s[j];
            add(j, buf + j * R::BYTES, kb, pf[j]);
        }
    };

    const int nst = (p.N + R::ROWS - 1) / R::ROWS;
    wait_loads();
    wait_lds_barrier();
    auto walk = [&](auto rows, auto plain) {
        if (active) first(lds[0][0], rows, plain, [&] { fetch(1); });
        else fetch(1);
        for (int s = 1; s < nst; ++s) {   // (at least two stages)
            wait_loads();
            wait_lds_barrier();
            auto next = [&] { if (s + 1 < nst) fetch(s + 1); };
            if (active) {
                const unsigned char *buf = lds[s & 1][0];
                step(buf, 2 * s, 0, rows, plain, next);
                if (2 * s + 1 < NT) step(buf, 2 * s + 1, 32, rows, plain, [] {});
            } else {
                next();
            }
        }
    };
    // (fp32 tiles: another copy of the loop spills 350 registers)
    if (BT == 2 && n == 2 && !dead[0] && !dead[1]) walk(std::integral_constant<int, 2>(), std::integral_constant<bool, BT == 2>());
    else if (n == 2) walk(std::integral_constant<int, 2>(), std::false_type());
    else walk(std::integral_constant<int, 1>(), std::false_type());

    if (!active) return;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        if (j >= n) break;   // uniform
        const float sum = l[j] + __shfl_xor(l[j], 32);
        if (q0 + li < p.N) {
            if (g == 0) p.lse[pr.row0 + (int64_t)j * p.N + q0 + li] = (m[j] + __log2f(sum)) * kLn2;
            store_row_tile<T>((T *)p.o + base[j] + (int64_t)(q0 + li) * p.stride_n, 0, D, o[j], 1.0f / sum, g);
        }
    }
}

#endif

// ------------------------------------------------------------------ forward of few problems

// A call whose problems leave most of the chip idle is bound by the chain of one wave: in stream_fwd a wave takes 2.3 us per 64
// keys of its row, one after the other (16 problems of 128 keys at D = 64: 8.3 us, of 512 keys: 22 us).  Here a workgroup's four
// waves share 32 queries and split the keys, every fourth tile each, and their partial sums meet in LDS.  A wave needs nobody
// until then: K comes from memory into the operand's registers, V by the load path into LDS of the wave's own, the next
// tile's on their way while one is computed on, and no barrier.  The mask is read as given (its largest entry by
// every wave), so the prep kernel has nothing to do for this one, and a call without a backward skips it.  16 problems,
// D = 64, fp32 bias, prep and forward before / this: 128 keys 10.7 / 6.7 us, 256 15.4 / 8.1, 512 26.6 / 11.6.  It ends where one
// workgroup per 128 queries has the chip full: 252 of those 30.5 / 29.6 us.
// BF: 0 no bias, 1 fp32, 2 in the dtype of q; read as given, four at a time where the rows allow it.
template <int D>
struct SplitFwd {
    static constexpr int TILE = 32 * D * 2, V_BYTES = 4 * 2 * TILE, O_BYTES = 4 * D * 32 * 4, BYTES = (V_BYTES > O_BYTES ? V_BYTES : O_BYTES) + 4 * 2 * 32 * 4;
};

// mask entries (additive form) of keys j0 + 64 i, i < 8, of one row; keys past the end repeat the last.  (Asked for per
// kind, so that the eight loads are under way together.)
__device__ __forceinline__ void mask8(const EvoAttnParams &p, int64_t off, int j0, float (&v)[8]) {
    int64_t at[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) at[i] = off + min(j0 + 64 * i, p.N - 1);
    if (p.mask_kind == EVO_MASK_BOOL) {
        uint8_t x[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) x[i] = ((const uint8_t *)p.mask)[at[i]];
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = x[i] ? 0.0f : -FLT_MAX;
    } else if (p.mask_kind == EVO_MASK_F32) {
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = ((const float *)p.mask)[at[i]];
    } else {
        unsigned short x[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) x[i] = ((const unsigned short *)p.mask)[at[i]];
#pragma unroll
        for (int i = 0; i < 8; ++i)
            v[i] = p.mask_kind == EVO_MASK_BF16 ? (float)__builtin_bit_cast(bf16_t, x[i]) : (float)__builtin_bit_cast(f16_t, x[i]);
    }
}

template <typename T, int D, int BF>
__global__ void __launch_bounds__(256, D == 32 ? 3 : D == 64 ? 2 : 1) split_fwd(EvoAttnParams p, bool vec) {
    typedef StreamGeo<D> G;
    typedef SplitFwd<D> R;
    typedef typename Mfma<T>::v8 v8;
    constexpr int KSD = D / 16, DT = D / 32, PIECES = R::TILE / 1024, RPP = 1024 / G::ROW;
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
    float *stats = reinterpret_cast<float *>(lds + R::BYTES - 4 * 2 * 32 * 4);   // [wave][m, l][query]
    float *masks = reinterpret_cast<float *>(lds + R::BYTES);                    // [key], not below the floor

    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), li = lane & 31, g = lane >> 5;
    const int NT = (p.N + 31) / 32;
    const unsigned lid = xcd_remap(blockIdx.x, gridDim.x);
    const Prob pr = walk_problem(p, lid / NT);
    const int q0 = (lid % NT) * 32, qrow = min(q0 + li, p.N - 1), sn = (int)p.stride_n;
    const T *K = (const T *)p.k + pr.base, *V = (const T *)p.v + pr.base;
    const int valid = ((p.N - 1) * sn + D) * 2;
    const __amdgpu_buffer_rsrc_t vrs = __builtin_amdgcn_make_buffer_rsrc((void *)V, 0, valid, 0x00020000);
    const int64_t bias_row = (int64_t)(p.bias_stride_b ? pr.b : 0) * p.bias_stride_b + (int64_t)pr.h * p.bias_stride_h + (int64_t)qrow * p.bias_stride_row;
    unsigned char *vbuf = lds + wave * 2 * R::TILE;

    struct Tile {
        v8 k[KSD];
        f32x16 bias;
    };
    auto fetch = [&](int t, Tile &d) {   // keys 32 t ..; V to the buffer of the parity of t / 4
        const int k0 = t * 32;
        unsigned char *dst = vbuf + ((t >> 2) & 1) * R::TILE;
#pragma unroll
        for (int i = 0; i < PIECES; ++i) {
            const int r = i * RPP + lane / G::C, c = (lane % G::C) ^ G::x(r);
            dma16(vrs, dst + i * 1024, min(k0 + r, p.N - 1) * sn * 2 + c * 16);
        }
        const T *krow = K + (int64_t)min(k0 + li, p.N - 1) * sn + g * 8;
#pragma unroll
        for (int ks = 0; ks < KSD; ++ks) d.k[ks] = ld8(krow + ks * 16);
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) {
            const int key = k0 + 8 * rr + 4 * g;
            if (BF == 1 && vec) {
                const f32x4 v = *reinterpret_cast<const f32x4 *>((const float *)p.bias + bias_row + min(key, p.N - 4));
#pragma unroll
                for (int i = 0; i < 4; ++i) d.bias[4 * rr + i] = v[i];
            } else if (BF == 2 && vec) {
                const typename Mfma<T>::v4 v = *reinterpret_cast<const typename Mfma<T>::v4 *>((const T *)p.bias + bias_row + min(key, p.N - 4));
#pragma unroll
                for (int i = 0; i < 4; ++i) d.bias[4 * rr + i] = (float)v[i];
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int kk = min(key + i, p.N - 1);
                if (BF == 1 && !vec) d.bias[4 * rr + i] = ((const float *)p.bias)[bias_row + kk];
                if (BF == 2 && !vec) d.bias[4 * rr + i] = (float)((const T *)p.bias)[bias_row + kk];
            }
        }
    };
    Tile next;
    if (wave < NT) fetch(wave, next);
    v8 qf[KSD];
#pragma unroll
    for (int ks = 0; ks < KSD; ++ks) qf[ks] = ld8((const T *)p.q + pr.base + (int64_t)qrow * sn + ks * 16 + g * 8);
    // The mask into LDS (every wave all of it, the same values: no wave waits for another), and its largest entry: in a row
    // masked throughout the scores are the mask alone, relative to that (prep.hip).
    float mx = -INFINITY;
    if (p.mask_kind != EVO_MASK_NONE) {   // uniform
        const int64_t off = (int64_t)pr.b * p.mask_stride_b + (int64_t)pr.s * p.mask_stride_s;
        for (int j0 = 0; j0 < NT * 32; j0 += 512) {
            float v[8];
            mask8(p, off, j0 + lane, v);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int j = j0 + lane + 64 * i;
                v[i] = j < p.N ? fmaxf(v[i], kMaskFloor) : kMaskFloor;
                mx = fmaxf(mx, v[i]);
                if (j < NT * 32) masks[j] = v[i];
            }
        }
        mx = wave_max(mx);
    } else {
        for (int j = lane; j < NT * 32; j += 64) masks[j] = j < p.N ? 0.0f : kMaskFloor;
    }
    const bool dead = p.mask_kind != EVO_MASK_NONE && mx < kShiftThreshold;
    const float c = dead ? 0.0f : p.scale * kLog2e, shift = dead ? mx : 0.0f;
#pragma unroll
    for (int ks = 0; ks < KSD; ++ks) qf[ks] = dead ? zero8<T>() : scaled8<T>(qf[ks], c);

    // (not from -inf: against a tile whose every bias entry is -inf the maximum stays where it starts, and -inf less -inf is no number)
    float m = kMaskFloor, l = 0.0f;
    f32x16 o[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[dt][r] = 0.0f;
    for (int t = wave; t < NT; t += 4) {
        const Tile now = next;
        // V of this tile has landed; and the reads of the tile before have left the buffer that the next fetch writes (nothing else
        // orders a read of LDS before the load path's write to it: the products that use the reads may come after the fetch)
        wait_loads_and_lds();
        if (t + 4 < NT) fetch(t + 4, next);
        f32x16 a;
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) {
            const f32x4 mk = *reinterpret_cast<const f32x4 *>(masks + 32 * t + 8 * rr + 4 * g);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float mask = 32 * t + 8 * rr + 4 * g + i < p.N ? fmaxf((mk[i] - shift) * kLog2e, kMaskFloor) : kMaskFloor;
                a[4 * rr + i] = BF && !dead ? now.bias[4 * rr + i] * kLog2e + mask : mask;   // (dropped, not times zero: it may be infinite)
            }
        }
#pragma unroll
        for (int ks = 0; ks < KSD; ++ks) a = Mfma<T>::mma(now.k[ks], qf[ks], a);
        float x = a[0];
#pragma unroll
        for (int r = 1; r < 16; ++r) x = fmaxf(x, a[r]);
        const unsigned u = __float_as_uint(x);
        auto sw = __builtin_amdgcn_permlane32_swap(u, u, false, false);
        const float mn = fmaxf(m, fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1]))), alpha = fast_exp2(m - mn);
        m = mn;
        float s = 0.0f;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            a[r] = fast_exp2(a[r] - m);
            s += a[r];
        }
        l = l * alpha + s;
        v8 pf[2];
#pragma unroll
        for (int ts = 0; ts < 2; ++ts)
#pragma unroll
            for (int i = 0; i < 8; ++i) pf[ts][i] = (T)a[8 * ts + i];
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int r = 0; r < 16; ++r) o[dt][r] *= alpha;
        const unsigned char *vt = vbuf + ((t >> 2) & 1) * R::TILE;
#pragma unroll
        for (int ts = 0; ts < 2; ++ts)
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) o[dt] = Mfma<T>::mma(transposed<T, D>(vt, 0, ts, dt, lane), pf[ts], o[dt]);
    }
    l += __shfl_xor(l, 32);

    // the waves' parts: [wave][d][query]
    __syncthreads();
    float *part = reinterpret_cast<float *>(lds);
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) part[(wave * D + dt * 32 + crow(r, g)) * 32 + li] = o[dt][r];
    if (g == 0) {
        stats[(wave * 2) * 32 + li] = m;
        stats[(wave * 2 + 1) * 32 + li] = l;
    }
    __syncthreads();
    const int q = threadIdx.x & 31, d0 = (threadIdx.x >> 5) * (D / 8);
    float w[4], top = kMaskFloor, sum = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i) top = fmaxf(top, stats[(i * 2) * 32 + q]);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        w[i] = fast_exp2(stats[(i * 2) * 32 + q] - top);
        sum += w[i] * stats[(i * 2 + 1) * 32 + q];
    }
    if (q0 + q >= p.N) return;
    if (threadIdx.x < 32) p.lse[pr.row0 + q0 + q] = (top + __log2f(sum)) * kLn2;
    const float inv = 1.0f / sum;
    const int64_t off = pr.base + (int64_t)(q0 + q) * sn + d0;
#pragma unroll
    for (int d = 0; d < D / 8; d += 4) {
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            v[i] = 0.0f;
#pragma unroll
            for (int k = 0; k < 4; ++k) v[i] += w[k] * part[(k * D + d0 + d + i) * 32 + q];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] *= inv;
        if (p.o) store4<T>((T *)p.o + off + d, v[0], v[1], v[2], v[3]);
        if (p.gate) {
            const typename Mfma<T>::v4 gv = *reinterpret_cast<const typename Mfma<T>::v4 *>((const T *)p.gate + off + d);
            store4<T>((T *)p.o_gated + off + d, v[0] * sigmoidf((float)gv[0]), v[1] * sigmoidf((float)gv[1]), v[2] * sigmoidf((float)gv[2]),
                      v[3] * sigmoidf((float)gv[3]));
        }
    }
}

// ------------------------------------------------------------------ dQ

// As mfma_dq_wide.hip, whose place it takes at these head dims: where dBias is no sum over S rows, or its sum comes from a
// kernel of its own.  A wave has 32 queries for all keys; with WRITE_DS (S = 1) dBias is dS and goes out as it is formed.
// Block `block` of 128 queries of problem `problem`, in `lds` of 2 R::BYTES.
constexpr int kDsBytes = 32 * 32 * 4;   // a wave's tile of dS in fp32
template <typename T, int D, int BT, bool WRITE_DS>
__device__ __forceinline__ void dq_rows(const EvoAttnParams &p, const Extra &e, unsigned char *lds, unsigned problem, int block) {
    typedef StreamGeo<D> G;
    typedef FwdStream<D> R;
    constexpr int NW = 4, KSD = D / 16, KS = KSD + 1, DT = D / 32;
    typedef typename Mfma<T>::v8 v8;

    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), li = lane & 31, g = lane >> 5;
    const int NT = (p.N + 31) / 32;
    const Prob pr = walk_problem(p, problem);
    const int q0 = block * 128 + wave * 32, qrow = min(q0 + li, p.N - 1);
    const bool active = q0 < p.N;
    const bool dead = e.dead[pr.b * p.S + pr.s] != 0, kill = dead && p.mask_kind == EVO_MASK_BOOL;
    const int sn2 = (int)p.stride_n * 2, valid = (p.N - 1) * sn2 + D * 2;
    const __amdgpu_buffer_rsrc_t krs = __builtin_amdgcn_make_buffer_rsrc((void *)((const T *)p.k + pr.base), 0, valid, 0x00020000);
    const __amdgpu_buffer_rsrc_t vrs = __builtin_amdgcn_make_buffer_rsrc((void *)((const T *)p.v + pr.base), 0, valid, 0x00020000);
    const int np256 = (p.N + 255) / 256 * 256;
    const __amdgpu_buffer_rsrc_t mrs =
        __builtin_amdgcn_make_buffer_rsrc((void *)(e.m2a + ((int64_t)pr.b * p.S + pr.s) * np256), 0, np256 * 16, 0x00020000);
    auto fetch = [&](int stage) {
        unsigned char *dst = lds + (stage & 1) * R::BYTES;
        dma_rows<D, R::ROWS, NW>(krs, vrs, dst, stage * R::ROWS, p.N, sn2, wave, lane);
        if (wave == 0) dma16(mrs, dst + R::OFF_A, (stage * R::ROWS + lane) * 16);
    };
    fetch(0);

    // this lane's half of the query row: Q (scaled), dO, and delta = <dO, O>
    const float cs = p.scale * kLog2e;
    v8 qf[KS], gf[KS], of[KSD];
    const int64_t row = pr.base + (int64_t)qrow * p.stride_n + g * 8;
    // (where delta is given, by the gate's pass, there may be no ungated O: dO is read in its place and the sum dropped)
    const T *O = e.delta_given ? (const T *)p.dout : (const T *)p.o;
#pragma unroll
    for (int ks = 0; ks < KSD; ++ks) {
        qf[ks] = ld8((const T *)p.q + row + ks * 16);
        gf[ks] = ld8((const T *)p.dout + row + ks * 16);
        of[ks] = ld8(O + row + ks * 16);
    }
    float lse2 = p.lse[pr.row0 + qrow], dgiven = 0.0f;
    if (e.delta_given) dgiven = e.delta[pr.row0 + qrow];
    const v8 vaug = aug8<T>(ones3<T>(), {0u, 0u});
    const BiasStream<T, BT, false> bias(p, e, pr, min(q0 >> 5, NT - 1), qrow, dead, lane);
    // PAIR: the caller's rows of a stage's two tiles are asked for together, and its dBias is stored together: 256 bytes of a row at a time (see
    // stream_fwd; B = 4, S = 1, N = 1024, H = 32, fp32 312 -> 285 us).  (Loads and stores that bypass the caches: 348, 731: pieces of a line meet there.)
    constexpr bool PAIR = D == 64 && BT >= 3;
    typename BiasStream<T, BT, false>::Tile ct, c1;
    bias.load(0, ct);
    if (PAIR) bias.load(1, c1);
    {
        asked_together<KSD>(qf);
        asked_together<KSD>(gf);
        asked_together<KSD>(of);
        float dl = 0.0f;
#pragma unroll
        for (int ks = 0; ks < KSD; ++ks) {
            qf[ks] = dead ? zero8<T>() : scaled8<T>(qf[ks], cs);
            dl = dot8<T>(gf[ks], of[ks], dl);
        }
        dl += __shfl_xor(dl, 32);
        if (e.delta_given) dl = dgiven;
        else if (g == 0 && q0 + li < p.N) e.delta[pr.row0 + q0 + li] = dl;
        lse2 *= kLog2e;
        const uint2 one3 = ones3<T>(), zero3 = {0u, 0u};
        qf[KSD] = g == 0 ? aug8<T>(one3, pack_split3<T>(-lse2)) : zero8<T>();   // ones x mask, -lse x ones
        gf[KSD] = g == 0 ? aug8<T>(pack_split3<T>(-dl), zero3) : zero8<T>();    // -delta x ones
        if (kill) {   // no gradient through replaced scores: dP - delta is then zero, and dS with it
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) gf[ks] = zero8<T>();
        }
    }

    // S = 1: this lane's row of dBias[b][h]
    const int64_t dsrow = (((int64_t)pr.b * p.H + pr.h) * p.N + qrow) * p.N;
    const bool ds_vec = (p.N & 3) == 0 && ((uintptr_t)p.dbias & 15) == 0, ds_f32 = p.dbias_dtype == EVO_F32;

    float *const dstile = (float *)p.dbias + (((int64_t)pr.b * p.H + pr.h) * p.N + q0 + (lane >> 3)) * p.N + 4 * (lane & 7);   // (fp32; where this lane stores of a tile: its row of eight, its four columns)

    f32x16 dq[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) dq[dt][r] = 0.0f;

    auto tile = [&](const unsigned char *buf, int kb, f32x16 a, auto begun, auto leave) {   // `begun`: the chains are; `leave` takes dS
        f32x16 dp;
#pragma unroll
        for (int r = 0; r < 16; ++r) dp[r] = 0.0f;
#pragma unroll
        for (int ks = 0; ks < KSD; ++ks) {
            const int o = G::at(kb + li, 2 * ks + g);
            a = Mfma<T>::mma(*reinterpret_cast<const v8 *>(buf + o), qf[ks], a);                  // log2 P^T
            dp = Mfma<T>::mma(*reinterpret_cast<const v8 *>(buf + R::OFF_V + o), gf[ks], dp);     // dP^T - delta
        }
        a = Mfma<T>::mma(*reinterpret_cast<const v8 *>(buf + R::OFF_A + (kb + li) * 16), qf[KSD], a);
        dp = Mfma<T>::mma(vaug, gf[KSD], dp);
        begun();
#pragma unroll
        for (int r = 0; r < 16; ++r) a[r] = fast_exp2(a[r]) * dp[r];
        leave(a);
        v8 ds[2];
#pragma unroll
        for (int ts = 0; ts < 2; ++ts)
#pragma unroll
            for (int i = 0; i < 8; ++i) ds[ts][i] = (T)a[8 * ts + i];
#pragma unroll
        for (int ts = 0; ts < 2; ++ts)
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) dq[dt] = Mfma<T>::mma(transposed<T, D>(buf, kb, ts, dt, lane), ds[ts], dq[dt]);
    };
    auto write = [&](int kt, const f32x16 &a) {
        if (!WRITE_DS) return;
        if (PAIR && ds_f32) {   // through LDS of the wave's own, so that a store covers 128 bytes of eight rows each
            unsigned char *const own = lds + 2 * R::BYTES + wave * kDsBytes;
            auto at = [](int r, int c) { return r * 128 + ((c ^ (r >> 1 & 7)) << 4); };   // (two rows share the 64 banks)
#pragma unroll
            for (int rr = 0; rr < 4; ++rr) {
                f32x4 v;
                v[0] = a[4 * rr]; v[1] = a[4 * rr + 1]; v[2] = a[4 * rr + 2]; v[3] = a[4 * rr + 3];
                *reinterpret_cast<f32x4 *>(own + at(li, 2 * rr + g)) = v;
            }
            const int c = lane & 7, col = kt * 32 + 4 * c;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int r = 8 * j + (lane >> 3);
                const f32x4 v = *reinterpret_cast<const f32x4 *>(own + at(r, c));
                if (q0 + r >= p.N) continue;
                float *const d = dstile + (int64_t)(8 * j) * p.N + kt * 32;
                if (col + 4 <= p.N) {
                    *reinterpret_cast<f32x4_at4 *>(d) = v;   // (16 bytes wherever they start)
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (col + i < p.N) d[i] = v[i];
                }
            }
            return;
        }
        if (q0 + li >= p.N) return;
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) {
            const int kg = kt * 32 + 8 * rr + 4 * g;   // registers 4 rr .. 4 rr + 3 hold keys kg .. kg + 3
            if ((ds_vec || ds_f32) && kg + 4 <= p.N) {   // (16 bytes in fp32 wherever they start)
                if (ds_f32) {
                    f32x4 v;
                    v[0] = a[4 * rr]; v[1] = a[4 * rr + 1]; v[2] = a[4 * rr + 2]; v[3] = a[4 * rr + 3];
                    *reinterpret_cast<f32x4_at4 *>((float *)p.dbias + dsrow + kg) = v;
                } else {
                    store4<T>((T *)p.dbias + dsrow + kg, a[4 * rr], a[4 * rr + 1], a[4 * rr + 2], a[4 * rr + 3]);
                }
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (kg + i < p.N) {
                        if (ds_f32) ((float *)p.dbias)[dsrow + kg + i] = a[4 * rr + i];
                        else ((T *)p.dbias)[dsrow + kg + i] = (T)a[4 * rr + i];
                    }
            }
        }
    };

    const int nst = (p.N + R::ROWS - 1) / R::ROWS;
    wait_loads();
    wait_lds_barrier();
    for (int s = 0; s < nst; ++s) {
        auto next = [&] {
            if (s + 1 < nst) fetch(s + 1);
            if (WRITE_DS) asm volatile("" ::: "memory");   // (this stage's stores are younger than what is asked for here)
        };
        if (active) {
            const unsigned char *buf = lds + (s & 1) * R::BYTES;
            if constexpr (PAIR) {
                const f32x16 b0 = bias.take(ct), b1 = bias.take(c1);
                next();
                bias.load(2 * s + 2, ct);
                bias.load(2 * s + 3, c1);
                tile(buf, 0, b0, [] {}, [&](const f32x16 &d) { write(2 * s, d); });
                if (2 * s + 1 < NT) tile(buf, 32, b1, [] {}, [&](const f32x16 &d) { write(2 * s + 1, d); });
            } else if constexpr (BT == 1) {
                bias.arrived(ct);
                next();
                tile(buf, 0, ct, [&] { bias.refill(2 * s + 1, ct); }, [&](const f32x16 &d) { write(2 * s, d); });
                if (2 * s + 1 < NT) tile(buf, 32, ct, [&] { bias.refill(2 * s + 2, ct); }, [&](const f32x16 &d) { write(2 * s + 1, d); });
            } else {
                const f32x16 b0 = bias.take(ct);
                next();
                bias.load(2 * s + 1, ct);
                tile(buf, 0, b0, [] {}, [&](const f32x16 &d) { write(2 * s, d); });
                if (2 * s + 1 < NT) {
                    const f32x16 b1 = bias.take(ct);
                    bias.load(2 * s + 2, ct);
                    tile(buf, 32, b1, [] {}, [&](const f32x16 &d) { write(2 * s + 1, d); });
                }
            }
        } else {
            next();
        }
        if (s + 1 < nst) {
            // A stage before the last has two whole tiles: a wave with 32 queries (with fewer, a store of eight rows may have none) stored at least
            // eight pieces of dBias after it had asked for the next stage, and need not wait for them.
            if (WRITE_DS && q0 + 32 <= p.N) wait_loads_but<8>();
            else wait_loads();
            wait_lds_barrier();
        }
    }
    if (active && q0 + li < p.N) {
        T *dQ = (T *)p.dq + pr.base + (int64_t)(q0 + li) * p.stride_n;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) store_row_tile<T>(dQ, dt * 32, D, dq[dt], p.scale, g);
    }
}

template <typename T, int D, int BT, bool WRITE_DS>
__global__ void __launch_bounds__(256, D == 32 ? 4 : D == 64 && BT < 3 ? 3 : 2) stream_dq(EvoAttnParams p, Extra e) {
    __shared__ __attribute__((aligned(1024))) unsigned char lds[2 * FwdStream<D>::BYTES + (D == 64 && BT >= 3 && WRITE_DS ? 4 * kDsBytes : 0)];
    const unsigned nqb = (p.N + 127) / 128, lid = xcd_remap(blockIdx.x, gridDim.x);
    dq_rows<T, D, BT, WRITE_DS>(p, e, lds, lid / nqb, lid % nqb);
}

// ------------------------------------------------------------------ dK and dV

// A wave has 32 keys, the queries stream by.  The score product wants Q scaled and rounded, dK wants it as given: a wave
// scales the pieces it has fetched itself, from LDS to LDS, between the wait and the barrier.  At head dim 128 the keys'
// K operand lies in LDS (next to V, dK and dV it would not fit the registers of two waves per SIMD).
template <int D, int NW>
struct KvStream {
    static constexpr int ROWS = D <= 64 ? 64 : 32, BLK = ROWS * D * 2;
    static constexpr bool K_LDS = D == 128;
    static constexpr int OFF_G = BLK, OFF_QS = 2 * BLK, OFF_AQ = 3 * BLK, OFF_AG = OFF_AQ + ROWS * 16, STAGE = (OFF_AG + ROWS * 16 + 1023) / 1024 * 1024;
    static constexpr int OFF_K = 2 * STAGE, BYTES = OFF_K + (K_LDS ? NW * 32 * D * 2 : 0);
};

// Block `block` of NW * 32 keys of problem `problem`.  OWN_DELTA: delta = <dO, O> is formed here, by four threads per row of a stage; else read.
// DM: the row sums of dS that a mask's gradient is summed from are wanted (head dim 64; the other head dims ask at run time).
template <typename T, int D, int BT, int NW, bool OWN_DELTA, bool DM>
__device__ __forceinline__ void dkdv_rows(const EvoAttnParams &p, const Extra &e, unsigned char *lds, unsigned problem, int block) {
    typedef StreamGeo<D> G;
    typedef KvStream<D, NW> R;
    constexpr int KSD = D / 16, DT = D / 32, ROWS = R::ROWS;
    constexpr int TPR = OWN_DELTA ? 4 : 1, OC = G::C / TPR;   // threads per row of a stage, chunks of O of each
    static_assert(!OWN_DELTA || (NW == 4 && D == 64), "every thread has a quarter of a row of its wave's two pieces of eight");
    typedef typename Mfma<T>::v8 v8;

    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), li = lane & 31, g = lane >> 5;
    const int NT = (p.N + 31) / 32;
    const Prob pr = walk_problem(p, problem);
    const int key0 = block * NW * 32 + wave * 32, key = key0 + li, keyc = min(key, p.N - 1);
    const bool active = key0 < p.N;
    const bool dead = e.dead[pr.b * p.S + pr.s] != 0, kill = dead && p.mask_kind == EVO_MASK_BOOL;
    const bool want_dm = DM || (D != 64 && e.dmask_part != nullptr && p.dmask != nullptr);
    const float cs = p.scale * kLog2e;
    const uint2 one3 = ones3<T>(), zero3 = {0u, 0u};
    const int sn2 = (int)p.stride_n * 2, valid = (p.N - 1) * sn2 + D * 2;
    const __amdgpu_buffer_rsrc_t qrs = __builtin_amdgcn_make_buffer_rsrc((void *)((const T *)p.q + pr.base), 0, valid, 0x00020000);
    const __amdgpu_buffer_rsrc_t grs = __builtin_amdgcn_make_buffer_rsrc((void *)((const T *)p.dout + pr.base), 0, valid, 0x00020000);

    // this thread's row of a stage (OWN_DELTA: of those that its wave fetches)
    const int myrow = OWN_DELTA ? wave * 8 + (lane >> 2 & 7) + (lane >> 5) * 32 : (int)threadIdx.x;
    float nl = 0.0f, nd = 0.0f;   // -LSE log2(e) and -delta of that row of the stage on its way (myrow < ROWS)
    v8 orow[OWN_DELTA ? OC : 1];  // (or this thread's part of O)
    auto fetch = [&](int stage) {
        dma_rows<D, ROWS, NW>(qrs, grs, lds + (stage & 1) * R::STAGE, stage * ROWS, p.N, sn2, wave, lane);
        const int q = stage * ROWS + myrow;
        if constexpr (OWN_DELTA) {
#pragma unroll
            for (int i = 0; i < OC; ++i) orow[i] = ld8((const T *)p.o + pr.base + (int64_t)min(q, p.N - 1) * p.stride_n + (threadIdx.x % TPR * OC + i) * 8);
            nl = q < p.N ? -p.lse[pr.row0 + q] * kLog2e : kMaskFloor;
        } else if (myrow < ROWS) {   // rows at and beyond N: probability zero
            nl = q < p.N ? -p.lse[pr.row0 + q] * kLog2e : kMaskFloor;
            nd = q < p.N ? -e.delta[pr.row0 + q] : 0.0f;
        }
    };
    auto finish = [&](int stage, bool bias_behind) {   // what this wave fetched is there: its pieces of Q scaled, the extra columns
        unsigned char *buf = lds + (stage & 1) * R::STAGE;
        if (bias_behind) wait_loads_but<8>();   // (two tiles of the bias, in four pieces each, are younger than the stage)
        else wait_loads();
        constexpr int PIECES = R::BLK / 1024;
#pragma unroll
        for (int i = 0; i < (PIECES + NW - 1) / NW; ++i) {
            const int m = wave + i * NW;
            if (PIECES % NW != 0 && m >= PIECES) break;
            const v8 a = *reinterpret_cast<const v8 *>(buf + m * 1024 + lane * 16);
            *reinterpret_cast<v8 *>(buf + R::OFF_QS + m * 1024 + lane * 16) = scaled8<T>(a, cs);
        }
        bool mine = myrow < ROWS;
        if constexpr (OWN_DELTA) {
            float d = 0.0f;
#pragma unroll
            for (int i = 0; i < OC; ++i) d = dot8<T>(*reinterpret_cast<const v8 *>(buf + R::OFF_G + G::at(myrow, threadIdx.x % TPR * OC + i)), orow[i], d);
            d += __shfl_xor(d, 1);
            d += __shfl_xor(d, 2);
            nd = -d;
            mine = threadIdx.x % TPR == 0;
        }
        if (mine) {
            *reinterpret_cast<v8 *>(buf + R::OFF_AQ + myrow * 16) = aug8<T>(one3, pack_split3<T>(nl));
            *reinterpret_cast<v8 *>(buf + R::OFF_AG + myrow * 16) = aug8<T>(pack_split3<T>(nd), zero3);
        }
        wait_lds_barrier();
    };
    fetch(0);

    // this wave's keys: K with the mask columns, V with ones against -delta
    // (all asked for before any is used, but not where the caller's bias rows come to head dim 128 as well: the loop then spills others, dK/dV of one row, N = 1 008, H = 4,
    // fp32 90 -> 100 us; a step of it so 170 and with all together 184, of 16 bits at N = 2 048, H = 2 362 and 377.  With prepared tiles S = 64, N = 512 294 / 285.)
    constexpr bool TOGETHER = !(D == 128 && BT >= 3);
    v8 kf[KSD], vf[KSD], kaug, vaug;
    uint2 mraw;
    {
        const int64_t row = pr.base + (int64_t)keyc * p.stride_n + g * 8;
#pragma unroll
        for (int ks = 0; ks < KSD; ++ks) {
            if constexpr (TOGETHER) {
                kf[ks] = ld8((const T *)p.k + row + ks * 16);
                vf[ks] = ld8((const T *)p.v + row + ks * 16);
            } else {
                kf[ks] = dead ? zero8<T>() : ld8((const T *)p.k + row + ks * 16);
                *reinterpret_cast<v8 *>(lds + R::OFF_K + wave * 32 * G::ROW + G::at(li, 2 * ks + g)) = kf[ks];
                vf[ks] = kill ? zero8<T>() : ld8((const T *)p.v + row + ks * 16);
            }
        }
        mraw = e.m2[((int64_t)pr.b * p.S + pr.s) * (NT * 32) + min(key, NT * 32 - 1)];
    }
    const BiasStream<T, BT, true> bias(p, e, pr, min(key0 >> 5, NT - 1), keyc, dead, lane);
    // TWO: the bias of a stage's two tiles is asked for when the stage before begins, which its end waits for anyway, and nothing in a tile is waited
    // for or branched on.  S = 200, N = 640, H = 5, fp32 bias 331 -> 321 us; B = 4, S = 1, N = 1024, H = 32 with dQ 387 -> 378.  (Head dim 32 spills with
    // a second tile under way.  Every read of LDS four or six matrix instructions ahead of its use, by groups of the scheduler: 320; two waves
    // per SIMD hide these already.)
    constexpr bool TWO = D == 64;
    typename BiasStream<T, BT, true>::Tile ct, c1;
    bias.load(0, ct);
    if (TWO) bias.load(1, c1);
    if constexpr (TOGETHER) {
        asked_together<KSD>(kf);
        asked_together<KSD>(vf);
    }
#pragma unroll
    for (int ks = 0; ks < KSD; ++ks) {
        if (TOGETHER && dead) kf[ks] = zero8<T>();
        if (TOGETHER && kill) vf[ks] = zero8<T>();   // (no gradient through replaced scores: dS is then zero)
        if constexpr (TOGETHER && R::K_LDS) *reinterpret_cast<v8 *>(lds + R::OFF_K + wave * 32 * G::ROW + G::at(li, 2 * ks + g)) = kf[ks];
    }
    kaug = g == 0 ? aug8<T>(mraw, one3) : zero8<T>();     // mask x ones, ones x -lse
    vaug = g == 0 && !kill ? aug8<T>(one3, zero3) : zero8<T>();    // ones x -delta
    // (the dBias partials of the kernels before this one, summed on the way in where the caller asks for it)
    if (e.dbias_chunks > 0) sum_dbias_partials<NW * 64>(p, e, threadIdx.x);

    f32x16 dk[DT], dv[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) dk[dt][r] = dv[dt][r] = 0.0f;
    float dm = 0.0f;

    auto tile = [&](const unsigned char *buf, int qb, auto begin, auto behind) {   // `begin`: the bias, and what is asked for once it is there
        f32x16 a = begin(), dp;
#pragma unroll
        for (int r = 0; r < 16; ++r) dp[r] = 0.0f;
#pragma unroll
        for (int ks = 0; ks < KSD; ++ks) {
            const int o = G::at(qb + li, 2 * ks + g);
            v8 k;
            if constexpr (R::K_LDS) k = *reinterpret_cast<const v8 *>(lds + R::OFF_K + wave * 32 * G::ROW + G::at(li, 2 * ks + g));
            else k = kf[ks];
            a = Mfma<T>::mma(*reinterpret_cast<const v8 *>(buf + R::OFF_QS + o), k, a);          // log2 P
            dp = Mfma<T>::mma(*reinterpret_cast<const v8 *>(buf + R::OFF_G + o), vf[ks], dp);    // dP - delta
        }
        a = Mfma<T>::mma(*reinterpret_cast<const v8 *>(buf + R::OFF_AQ + (qb + li) * 16), kaug, a);
        dp = Mfma<T>::mma(*reinterpret_cast<const v8 *>(buf + R::OFF_AG + (qb + li) * 16), vaug, dp);
        behind();
        v8 pf[2], ds[2];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            a[r] = fast_exp2(a[r]);
            dp[r] *= a[r];
        }
        if (want_dm) {
#pragma unroll
            for (int r = 0; r < 16; ++r) dm += dp[r];
        }
#pragma unroll
        for (int ts = 0; ts < 2; ++ts)
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                pf[ts][i] = (T)a[8 * ts + i];
                ds[ts][i] = (T)dp[8 * ts + i];
            }
#pragma unroll
        for (int ts = 0; ts < 2; ++ts)
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) {
                dv[dt] = Mfma<T>::mma(transposed<T, D>(buf + R::OFF_G, qb, ts, dt, lane), pf[ts], dv[dt]);
                dk[dt] = Mfma<T>::mma(transposed<T, D>(buf, qb, ts, dt, lane), ds[ts], dk[dt]);
            }
    };

    const int nst = (p.N + ROWS - 1) / ROWS;
    finish(0, false);
    for (int s = 0; s < nst; ++s) {
        auto next = [&] { if (s + 1 < nst) fetch(s + 1); };
        if (active) {
            const unsigned char *buf = lds + (s & 1) * R::STAGE;
            const int qt = s * (ROWS / 32);
            if constexpr (TWO && BT == 1) {
                bias.arrived(ct);
                bias.arrived(c1);
                next();
                tile(buf, 0, [&] { return ct; }, [&] { bias.refill(qt + 2, ct); });
                if (qt + 1 < NT) tile(buf, 32, [&] { return c1; }, [&] { bias.refill(qt + 3, c1); });
            } else if constexpr (TWO) {
                const f32x16 b0 = bias.take(ct), b1 = bias.take(c1);
                next();
                bias.load(qt + 2, ct);
                bias.load(qt + 3, c1);
                tile(buf, 0, [&] { return b0; }, [] {});
                if (qt + 1 < NT) tile(buf, 32, [&] { return b1; }, [] {});
            } else {
                auto one = [&](int t, int qb, auto then) {
                    tile(buf, qb, [&] {
                        const f32x16 b = bias.take(ct);
                        then();
                        if (D < 128) bias.load(t + 1, ct);
                        return b;
                    }, [&] { if (D == 128) bias.load(t + 1, ct); });   // (no registers for it any sooner)
                };
                one(qt, 0, next);
                if (ROWS == 64 && qt + 1 < NT) one(qt + 1, 32, [] {});
            }
        } else {
            next();
        }
        if (s + 1 < nst) finish(s + 1, TWO && BT == 1 && active);   // (a stage before the last has two tiles)
    }

    if (!active) return;
    if (want_dm) {
        dm += __shfl_xor(dm, 32);
        if (g == 0 && key < p.N) e.dmask_part[pr.row0 + key] = dm;
    }
    if (key < p.N) {
        T *dK = (T *)p.dk + pr.base + (int64_t)key * p.stride_n, *dV = (T *)p.dv + pr.base + (int64_t)key * p.stride_n;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
            store_row_tile<T>(dK, dt * 32, D, dk[dt], p.scale, g);
            store_row_tile<T>(dV, dt * 32, D, dv[dt], 1.0f, g);
        }
    }
}

template <typename T, int D, int BT, int NW, bool DM>
__global__ void __launch_bounds__(NW * 64, D == 32 ? 3 : 2) stream_dkdv(EvoAttnParams p, Extra e) {
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
    const unsigned nkb = (p.N + NW * 32 - 1) / (NW * 32), lid = xcd_remap(blockIdx.x, gridDim.x);
    dkdv_rows<T, D, BT, NW, false, DM>(p, e, lds, lid / nkb, lid % nkb);
}

// ------------------------------------------------------------------ dQ, dK, dV and dBias of one S row

// With one S row the traffic is the bias, which both kernels read, and dBias, and few problems do not fill the chip with either kernel.
// Here the workgroups of both are one launch, those of a problem next to each other on one XCD: what one has read of the bias the other finds in
// the memory-side cache, the one that waits for memory shares the chip with the one that computes, and a last round is
// one instead of two.  dK/dV forms delta for itself.  The last problems come first: what the forward has left in the caches.
// H = 32, fp32 bias, dQ and dK/dV one after the other / this, us: B = 1, N = 128 19.6 / 11.2, 256 28.7 / 16.8, 512 51 / 29, 1024 101 / 90; B = 3, N = 724
// 220 / 171; B = 4, N = 1024 424 / 378 (337 since dBias is stored 128 bytes of a row at a time, 5.3 TB/s past L2; problems in order the next call's forward takes 161 instead of 144;
// sweeps turned so that both kinds meet in the same tile at the same time: no change); H = 8, B = 1, N = 2048 176 / 93.
// Also without dBias (WRITE_DS) and with delta from the gate's pass (GIVEN), for rows that start or end within a group of four: as two launches, whose bias is read
// entry by entry, these lost to the prepared tiles where there are few workgroups.
template <typename T, int BT, bool WRITE_DS, bool GIVEN>
__global__ void __launch_bounds__(256, 2) stream_bwd_one(EvoAttnParams p, Extra e) {
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
    const unsigned nb = (p.N + 127) / 128, lid = gridDim.x - 1 - xcd_remap(blockIdx.x, gridDim.x), problem = lid / (2 * nb), r = lid % (2 * nb);
    if (r >= nb) dkdv_rows<T, 64, BT == 5 ? 3 : BT, 4, !GIVEN, false>(p, e, lds, problem, r - nb);
    else dq_rows<T, 64, BT, WRITE_DS>(p, e, lds, problem, r);
}

// ------------------------------------------------------------------ dBias partials

// What mfma_dbias.hip is for head dim 16: dS a second time, summed over a chunk of S rows in registers.  A
// workgroup has 128 queries x 64 keys (head dim 32: 128) of one (b, h), a wave 32 queries x all of the block's key tiles.  Keys (K, V, mask
// columns) are shared and double-buffered in LDS; a wave's own rows of Q and dO come into LDS of its own, which it reads into registers at the
// top of a row and refills at once, so they need no second buffer and no barrier.
// The vector ALU is busy for .55 of the time and the matrix core for .29 at two waves per SIMD (S = N = 768, H = 4, D = 32), so what can be said once is: the bias of a wave's tiles
// stays in registers in fp32, log2 units, the first operand C of a tile's chain where it lies (as 16-bit pairs it was unpacked and multiplied
// per tile and row, 32 instructions of 131); -delta, one value per lane, is the C of the other chain, in place of a matrix step of
// its own; array bases advance by the scalar unit and a lane's offsets are formed once.  dBias of S = N = 768, H = 4, D = 32 (mfma_dbias.hip
// before) 595 -> 455 us, of S = 200, N = 640, H = 5, D = 64 with an fp32 bias 238 -> 193; S = 64, N = 512, H = 4, D = 128 78 -> 65.
// Two tiles per wave and three waves per SIMD at head dim 32: 596; -delta in a matrix step: 516.
template <int D>
struct DbStream {
    static constexpr int TPW = D == 32 ? 4 : 2, KB = TPW * 32, QB = 128, BLK = KB * D * 2;   // key tiles per wave; keys, queries per workgroup
    static constexpr int OFF_V = BLK, OFF_A = 2 * BLK, KEYS = OFF_A + KB * 16;
    static constexpr int OFF_Q = 2 * KEYS, WAVE = 2 * 32 * D * 2, BYTES = OFF_Q + 4 * WAVE;
    static constexpr int KP = BLK / 4096, QP = 32 * D * 2 / 1024, RPP = 1024 / (D * 2);   // pieces of 1 KB per wave: of an array of keys, of one of queries; rows of one
};

template <typename T, int D, bool BF32>
__global__ void __launch_bounds__(256, D <= 64 ? 2 : 1) stream_dbias(EvoAttnParams p, Extra e) {
    typedef StreamGeo<D> G;
    typedef DbStream<D> R;
    constexpr int KSD = D / 16, KS = KSD + 1;
    typedef typename Mfma<T>::v8 v8;
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];

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
    const uint2 one3 = ones3<T>();

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

    // offsets of this lane's 16 bytes of a piece of keys and of queries (rows past the end repeat the last one), from row 0 of the problem on
    int koff[R::KP], qoff[R::QP];
#pragma unroll
    for (int i = 0; i < R::KP; ++i) {
        const int r = (wave + 4 * i) * R::RPP + lane / G::C;
        koff[i] = min(k0 + r, p.N - 1) * sn2 + (((lane % G::C) ^ G::x(r)) << 4);
    }
#pragma unroll
    for (int i = 0; i < R::QP; ++i) {
        const int r = i * R::RPP + lane / G::C;
        qoff[i] = min(q0 + r, p.N - 1) * sn2 + (((lane % G::C) ^ G::x(r)) << 4);
    }
    const int64_t base0 = (int64_t)b * p.stride_b + (int64_t)h * p.stride_h;
    auto rows = [&](const void *x, int s) { return __builtin_amdgcn_make_buffer_rsrc((void *)((const T *)x + base0 + (int64_t)s * p.stride_s), 0, valid, 0x00020000); };
    unsigned char *const own = lds + R::OFF_Q + wave * R::WAVE;
    float lse_n = 0.0f, delta_n = 0.0f;
    int dead_n = 0;
    auto fetch_keys = [&](int s) {
        const __amdgpu_buffer_rsrc_t krs = rows(p.k, s), vrs = rows(p.v, s);
        unsigned char *dst = lds + ((s - s_begin) & 1) * R::KEYS;
#pragma unroll
        for (int i = 0; i < R::KP; ++i) {
            dma16(krs, dst + (wave + 4 * i) * 1024, koff[i]);
            dma16(vrs, dst + R::OFF_V + (wave + 4 * i) * 1024, koff[i]);
        }
        if (wave < R::KB / 64) {
            const __amdgpu_buffer_rsrc_t mrs = __builtin_amdgcn_make_buffer_rsrc((void *)(e.m2a + ((int64_t)b * p.S + s) * np256 + k0), 0, R::KB * 16, 0x00020000);
            dma16(mrs, dst + R::OFF_A + wave * 1024, (wave * 64 + lane) * 16);
        }
    };
    auto fetch_query_pieces = [&](int s, int i0, int i1) __attribute__((always_inline)) {   // [i0, i1) of Q's and as many of dO's
        const __amdgpu_buffer_rsrc_t qrs = rows(p.q, s), grs = rows(p.dout, s);
#pragma unroll
        for (int i = 0; i < R::QP; ++i) {
            if (i < i0 || i >= i1) continue;
            dma16(qrs, own + i * 1024, qoff[i]);
            dma16(grs, own + 32 * G::ROW + i * 1024, qoff[i]);
        }
    };
    auto fetch_query_values = [&](int s) {
        const int64_t row0 = ((int64_t)bh * p.S + s) * p.N;
        lse_n = (p.lse + row0)[(unsigned)qrow];
        delta_n = (e.delta + row0)[(unsigned)qrow];
        // (With the rest: as a scalar load it is waited for at the top of each row.  S = N = 768, H = 4, D = 32 495 -> 455 us, S = 64, N = 512, H = 4, D = 128
        // 71 -> 65; at head dim 64 203 / 209.)
        if (D != 64) dead_n = e.dead[b * p.S + s];
    };
    fetch_keys(s_begin);
    fetch_query_pieces(s_begin, 0, R::QP);
    fetch_query_values(s_begin);
    for (int s = s_begin; s < s_end; ++s) {
        wait_loads();
        asm volatile("" : "+v"(lse_n), "+v"(delta_n), "+v"(dead_n));   // (the compiler's own wait for them: here, not behind the next keys' loads)
        const bool dead = (D != 64 ? __builtin_amdgcn_readfirstlane(dead_n) : uniform_load(e.dead + b * p.S + s)) != 0, kill = dead && p.mask_kind == EVO_MASK_BOOL;
        wait_lds_barrier();
        if (s + 1 < s_end) fetch_keys(s + 1);   // (everybody has left that buffer: it held row s - 1)
        v8 qf[KS], gf[KSD];
#pragma unroll
        for (int ks = 0; ks < KSD; ++ks) {
            const int o = G::at(li, 2 * ks + g);
            qf[ks] = *reinterpret_cast<const v8 *>(own + o);
            gf[ks] = *reinterpret_cast<const v8 *>(own + 32 * G::ROW + o);
        }
        qf[KSD] = g == 0 ? aug8<T>(one3, pack_split3<T>(-lse_n * kLog2e)) : zero8<T>();
        f32x16 nd;
#pragma unroll
        for (int r = 0; r < 16; ++r) nd[r] = -delta_n;
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (s + 1 < s_end) {
            if (!active || kill) fetch_query_pieces(s + 1, 0, R::QP);
            fetch_query_values(s + 1);
        }
#pragma unroll
        for (int ks = 0; ks < KSD; ++ks) qf[ks] = scaled8<T>(qf[ks], dead ? 0.0f : cs);
        if (!active || kill) continue;
        const unsigned char *buf = lds + ((s - s_begin) & 1) * R::KEYS;
#pragma unroll
        for (int j = 0; j < R::TPW; ++j) {
            // uniform.  Head dim 128, a wave per SIMD: both tiles together, also where the second's keys do not exist (masked, and
            // not stored): 78 -> 74 us; at head dim 64 that is slower, 193 -> 205.
            if (D == 128 || j < tiles) {
                f32x16 a, dp;
                v8 k = *reinterpret_cast<const v8 *>(buf + G::at(32 * j + li, g)), v = *reinterpret_cast<const v8 *>(buf + R::OFF_V + G::at(32 * j + li, g));
#pragma unroll
                for (int ks = 0; ks < KSD; ++ks) {
                    v8 k1, v1;
                    if (ks + 1 < KSD) {
                        const int o = G::at(32 * j + li, 2 * ks + 2 + g);
                        k1 = *reinterpret_cast<const v8 *>(buf + o);
                        v1 = *reinterpret_cast<const v8 *>(buf + R::OFF_V + o);
                    }
                    // The next row's queries a few pieces per step of the first tile: all at once they hold up the wave that asks, behind the CU's load
                    // path.  S = 64, N = 512, H = 4, D = 128 (a wave per SIMD) 78 -> 74 us, S = N = 768, D = 32 468 -> 458, S = 200, N = 640, H = 5, D = 64 211 -> 209.
                    if (j == 0 && s + 1 < s_end) fetch_query_pieces(s + 1, ks * R::QP / KSD, (ks + 1) * R::QP / KSD);
                    if (ks) {
                        a = Mfma<T>::mma(k, qf[ks], a);                                                        // log2 P^T
                    } else if (__builtin_expect(!dead, 1)) {
                        a = Mfma<T>::mma(k, qf[0], bias[j]);
                    } else {   // (a row with every key masked takes no bias)
                        f32x16 z;
#pragma unroll
                        for (int r = 0; r < 16; ++r) z[r] = 0.0f;
                        a = Mfma<T>::mma(k, qf[0], z);
                    }
                    dp = Mfma<T>::mma(v, gf[ks], ks ? dp : nd);         // dP^T - delta
                    if (ks + 1 < KSD) {
                        k = k1;
                        v = v1;
                    }
                }
                a = Mfma<T>::mma(*reinterpret_cast<const v8 *>(buf + R::OFF_A + (32 * j + li) * 16), qf[KSD], a);
#pragma unroll
                for (int r = 0; r < 16; ++r) sum[j][r] += fast_exp2(a[r]) * dp[r];
            } else {
                asm volatile("");   // (a block of its own for the sums that stay: without one they are copied ahead of the branch, 16 moves a tile)
            }
            if (D < 128) __builtin_amdgcn_sched_barrier(0);   // (the next tile's operands would take the registers)
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

// ------------------------------------------------------------------ launchers

// the caller's bias rows start or end within a group of four (fp32, head dim 64: bias_ragged in api.hip)
static bool ragged_rows(const EvoAttnParams &p, const Extra &e) { return p.N % 4 != 0 || !e.vec_ok; }

template <typename T, int D>
static int fwd_launch(const EvoAttnParams &p, const Extra &e, hipStream_t st) {
    const unsigned grid = (unsigned)((p.N + 127) / 128) * (unsigned)(p.B * p.H * p.S);
#if EVO_D == 32
    if (mfma_fwd_pair_ok(p, e.bias_direct)) {
        const unsigned pairs = (unsigned)mfma_fwd_pairs(p);
        if (e.bq16) stream_fwd_pair<T, 2><<<pairs, 256, 0, st>>>(p, e);
        else stream_fwd_pair<T, 1><<<pairs, 256, 0, st>>>(p, e);
        return hip_rc();
    }
#endif
    if (p.bias_dtype == EVO_NONE) stream_fwd<T, D, 0><<<grid, 256, 0, st>>>(p, e);
    else if (e.bias_direct && p.bias_dtype == EVO_F32 && ragged_rows(p, e)) stream_fwd<T, D, D == 64 ? 5 : 3><<<grid, 256, 0, st>>>(p, e);
    else if (e.bias_direct && p.bias_dtype == EVO_F32) stream_fwd<T, D, 3><<<grid, 256, 0, st>>>(p, e);
    else if (e.bias_direct) stream_fwd<T, D, 4><<<grid, 256, 0, st>>>(p, e);
    else if (e.bq16) stream_fwd<T, D, 2><<<grid, 256, 0, st>>>(p, e);
    else stream_fwd<T, D, 1><<<grid, 256, 0, st>>>(p, e);
    return hip_rc();
}

int EVO_CAT(launch_mfma_fwd_d, EVO_D)(const EvoAttnParams &p, const Extra &e, hipStream_t st) {
    return p.dtype == EVO_BF16 ? fwd_launch<bf16_t, EVO_D>(p, e, st) : fwd_launch<f16_t, EVO_D>(p, e, st);
}

template <typename T, int D>
static int split_launch(const EvoAttnParams &p, hipStream_t st) {
    const unsigned grid = (unsigned)((p.N + 31) / 32) * (unsigned)(p.B * p.H * p.S);
    const int es = p.bias_dtype == EVO_F32 ? 4 : 2;
    const bool vec = p.N % 4 == 0 && ((uintptr_t)p.bias % (4 * es)) == 0 && p.bias_stride_b % 4 == 0 && p.bias_stride_h % 4 == 0 && p.bias_stride_row % 4 == 0;
    auto go = [&](auto kern, PerDevice &done) {
        constexpr int most = SplitFwd<D>::BYTES + kSplitFwdMaxN * 4;
        if (most > 64 * 1024)
            if (const int rc = ensure_dynamic_lds((const void *)kern, most, done, nullptr)) return rc;
        kern<<<grid, 256, SplitFwd<D>::BYTES + (p.N + 31) / 32 * 128, st>>>(p, vec);
        return hip_rc();
    };
    static PerDevice done[3]{};
    if (p.bias_dtype == EVO_NONE) return go(split_fwd<T, D, 0>, done[0]);
    return p.bias_dtype == EVO_F32 ? go(split_fwd<T, D, 1>, done[1]) : go(split_fwd<T, D, 2>, done[2]);
}

int EVO_CAT(launch_split_fwd_d, EVO_D)(const EvoAttnParams &p, hipStream_t st) {
    return p.dtype == EVO_BF16 ? split_launch<bf16_t, EVO_D>(p, st) : split_launch<f16_t, EVO_D>(p, st);
}

template <typename T, int D>
static int dq_launch(const EvoAttnParams &p, const Extra &e, hipStream_t st) {
    const unsigned grid = (unsigned)((p.N + 127) / 128) * (unsigned)(p.B * p.H * p.S);
    const bool f32_rows = e.bias_direct && p.bias_dtype == EVO_F32, t16_rows = e.bias_direct && !f32_rows, t16 = e.bq16 != nullptr;
    if (p.dbias && p.S != 1) return EVO_EUNSUPPORTED;   // (a sum over S rows is the other kernels' business)
    if (p.bias_dtype == EVO_NONE) stream_dq<T, D, 0, false><<<grid, 256, 0, st>>>(p, e);
    else if (!p.dbias && f32_rows && ragged_rows(p, e)) stream_dq<T, D, D == 64 ? 5 : 3, false><<<grid, 256, 0, st>>>(p, e);
    else if (!p.dbias && f32_rows) stream_dq<T, D, 3, false><<<grid, 256, 0, st>>>(p, e);
    else if (!p.dbias && t16_rows) stream_dq<T, D, 4, false><<<grid, 256, 0, st>>>(p, e);
    else if (!p.dbias && t16) stream_dq<T, D, 2, false><<<grid, 256, 0, st>>>(p, e);
    else if (!p.dbias) stream_dq<T, D, 1, false><<<grid, 256, 0, st>>>(p, e);
    else if (f32_rows && ragged_rows(p, e)) stream_dq<T, D, D == 64 ? 5 : 3, true><<<grid, 256, 0, st>>>(p, e);
    else if (f32_rows) stream_dq<T, D, 3, true><<<grid, 256, 0, st>>>(p, e);
    else if (t16_rows) stream_dq<T, D, 4, true><<<grid, 256, 0, st>>>(p, e);
    else if (t16) stream_dq<T, D, 2, true><<<grid, 256, 0, st>>>(p, e);
    else stream_dq<T, D, 1, true><<<grid, 256, 0, st>>>(p, e);
    return hip_rc();
}

int EVO_CAT(launch_mfma_dqw_d, EVO_D)(const EvoAttnParams &p, const Extra &e, hipStream_t st) {
    return p.dtype == EVO_BF16 ? dq_launch<bf16_t, EVO_D>(p, e, st) : dq_launch<f16_t, EVO_D>(p, e, st);
}

template <typename T, int D, int BT, int NW>
static int dkdv_launch(const EvoAttnParams &p, const Extra &e, hipStream_t st) {
    const unsigned grid = (unsigned)((p.N + NW * 32 - 1) / (NW * 32)) * (unsigned)(p.B * p.H * p.S);
    constexpr int lds = KvStream<D, NW>::BYTES;
    auto kern = stream_dkdv<T, D, BT, NW, false>;
    if constexpr (D == 64) {
        if (p.dmask) kern = stream_dkdv<T, D, BT, NW, true>;
    }
    if constexpr (lds > 64 * 1024) {
        static PerDevice done{};
        if (const int rc = ensure_dynamic_lds((const void *)kern, lds, done, nullptr)) return rc;
    }
    kern<<<grid, NW * 64, lds, st>>>(p, e);
    return hip_rc();
}

template <typename T, int D, int NW>
static int dkdv_bias(const EvoAttnParams &p, const Extra &e, hipStream_t st) {
    if (p.bias_dtype == EVO_NONE) return dkdv_launch<T, D, 0, NW>(p, e, st);
    if (e.bias_direct) return p.bias_dtype == EVO_F32 ? dkdv_launch<T, D, 3, NW>(p, e, st) : dkdv_launch<T, D, 4, NW>(p, e, st);
    return e.bk16 ? dkdv_launch<T, D, 2, NW>(p, e, st) : dkdv_launch<T, D, 1, NW>(p, e, st);
}

// Eight waves share a stage of queries at head dim 128 (the keys' K operand takes their LDS then).
template <typename T, int D>
static int dkdv_waves(const EvoAttnParams &p, const Extra &e, hipStream_t st) {
    if constexpr (D == 128) {
        if (p.N > 128) return dkdv_bias<T, D, 8>(p, e, st);
    }
    return dkdv_bias<T, D, 4>(p, e, st);
}

#if EVO_D == 64
template <typename T>
static int bwd_one_launch(const EvoAttnParams &p, const Extra &e, hipStream_t st) {
    const unsigned grid = 2 * (unsigned)((p.N + 127) / 128) * (unsigned)(p.B * p.H);
    auto go = [&](auto kern) {
        constexpr int lds = KvStream<64, 4>::BYTES;
        static_assert(lds >= 2 * FwdStream<64>::BYTES + 4 * kDsBytes && lds <= 64 * 1024, "the larger of the two");
        kern<<<grid, 256, lds, st>>>(p, e);
        return hip_rc();
    };
    if (p.bias_dtype != EVO_F32) return go(stream_bwd_one<T, 4, true, false>);
    if (!ragged_rows(p, e)) return go(stream_bwd_one<T, 3, true, false>);
    if (e.delta_given) return p.dbias ? go(stream_bwd_one<T, 5, true, true>) : go(stream_bwd_one<T, 5, false, true>);
    return p.dbias ? go(stream_bwd_one<T, 5, true, false>) : go(stream_bwd_one<T, 5, false, false>);
}
int launch_stream_bwd_one_d64(const EvoAttnParams &p, const Extra &e, hipStream_t st) {
    return p.dtype == EVO_BF16 ? bwd_one_launch<bf16_t>(p, e, st) : bwd_one_launch<f16_t>(p, e, st);
}
#endif

#if EVO_D == 32   // (mfma_bwd.hip chooses between its kernel of eight waves and this one)
int launch_stream_dkdv_d32(const EvoAttnParams &p, const Extra &e, hipStream_t st) {
#else
int EVO_CAT(launch_mfma_dkdv_d, EVO_D)(const EvoAttnParams &p, const Extra &e, hipStream_t st) {
#endif
    return p.dtype == EVO_BF16 ? dkdv_waves<bf16_t, EVO_D>(p, e, st) : dkdv_waves<f16_t, EVO_D>(p, e, st);
}

template <typename T, int D, bool BF32>
static int dbias_launch(const EvoAttnParams &p, const Extra &e, hipStream_t st) {
    typedef DbStream<D> R;
    const int64_t grid = (int64_t)((p.N + R::QB - 1) / R::QB) * ((p.N + R::KB - 1) / R::KB) * p.B * p.H * e.n_chunks;
    if (grid <= 0 || grid > 0x7fffffff) return EVO_EOVERFLOW;
    static PerDevice done{};
    if (const int rc = ensure_dynamic_lds((const void *)&stream_dbias<T, D, BF32>, R::BYTES, done, nullptr)) return rc;
    stream_dbias<T, D, BF32><<<(unsigned)grid, 256, R::BYTES, st>>>(p, e);
    return hip_rc();
}

int EVO_CAT(launch_mfma_dbias_d, EVO_D)(const EvoAttnParams &p, const Extra &e, hipStream_t st) {
    const bool f = p.bias_dtype == EVO_F32;
    if (p.dtype == EVO_BF16) return f ? dbias_launch<bf16_t, EVO_D, true>(p, e, st) : dbias_launch<bf16_t, EVO_D, false>(p, e, st);
    return f ? dbias_launch<f16_t, EVO_D, true>(p, e, st) : dbias_launch<f16_t, EVO_D, false>(p, e, st);
}

}  // namespace evo
