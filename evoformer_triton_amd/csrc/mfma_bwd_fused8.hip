// dQ, dK and dV in one kernel, head dim 8.
//
// mfma_bwd_fused.hip for rows of 16 bytes, where one instruction has room for more than a row: of its 32 columns the score product uses 8 for the
// scaled Q, 8 for mask and LSE and 8 for what rounding the scaled Q left, and the last 8 of the key operand hold V, so that one register set
// of the keys serves both products.  dK and dV of a tile are 8 registers, and a workgroup keeps up to 384 keys (KT = 6 tiles of 16 per wave):
// rows up to that length are one block, their queries pass once.  A group's dQ is two tiles of 16 queries: two waves share one, each with half of the
// keys, and meet in LDS.
// Bound by the vector ALU, busy .79 of the time at S = 1024, N = 384, H = 8 (counters, at 2.1 GHz; 42 instructions per wave, tile and group, 16 of them for the bias); LDS
// .50, a fifth of it bank conflicts, matrix core .32, at two waves per SIMD.
// S = 1024, N = 384, H = 8, without dBias: dQ and dK/dV kernels 663 us, this 400.  Blocks of 192 keys (KT = 3) 495, at three waves per SIMD
// with 29 registers spilled 575; KT = 2, three waves, 495; more workgroups than are resident at a time (768) 517.
#include "fused_common.h"
#include "kernels.h"

namespace evo {

// KT: key tiles of 16 per wave
template <int KT>
struct Fused8 {
    static constexpr int D = 8, NW = 4, KB = NW * KT * 16;   // waves; keys per block
    static constexpr int QR = 128, BLK = QR * 16;            // query rows per stage, bytes of an array of them
    // of a stage: Q and dO as given, Q scaled and what its rounding left, (1 1 1 -LSE in three parts), zeros, -delta
    static constexpr int OFF_G = BLK, OFF_H = 2 * BLK, OFF_R = 3 * BLK, OFF_L = 4 * BLK, OFF_Z = 5 * BLK, OFF_D = 6 * BLK, STAGE = OFF_D + QR * 4;
    static constexpr int EX = KB * 64, OFF_EX = 2 * STAGE;   // dS of 32 queries x the block's keys, two of them; before there is any, the block's keys
    static constexpr int OFF_X = OFF_EX + 2 * EX, BYTES = OFF_X + 2 * 1024;   // half of a group's dQ, two of them
    static constexpr int AHEAD = KT == 6 ? 3 : KT;           // tiles that the bias is asked for ahead
    static __device__ __forceinline__ int ate(int r, int c) { return r * 64 + ((c ^ (((r >> 3) & 1) | ((r >> 2) & 1) << 1)) << 4); }
};

template <typename T, int KT, int BT>
__global__ void __launch_bounds__(256, KT == 2 ? 3 : 2) bwd_fused8(EvoAttnParams p, Extra e, unsigned problems, int nb) {
    typedef Fused8<KT> R;
    typedef typename Mfma<T>::v8 v8;
    typedef typename Mfma<T>::v4 v4;
    typedef Mfma16<T> M;
    constexpr int D = R::D, BES = BT == 2 ? 2 : 4, GPS = R::QR / 32;   // GPS: groups of 32 queries per stage
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];

    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), c = lane & 15, j = lane >> 4;
    const int N = p.N, NT = (N + 31) / 32, nst = (N + R::QR - 1) / R::QR, sn2 = (int)p.stride_n * 2, valid = (N - 1) * sn2 + D * 2;
    unsigned char *const ex = lds + R::OFF_EX, *const xch = lds + R::OFF_X;
    const int np256 = (N + 255) / 256 * 256;
    const uint2 one3 = ones3<T>();
    // (floor, floor, floor, 1) of the mask's chunk
    const uint2 floor3 = pack_split3<T>(kMaskFloor), floor2 = make_uint2(floor3.x, (floor3.y & 0xffffu) | one3.x << 16);
    // A stage is fetched and prepared by all waves: two have 64 rows of Q each, two of dO and O.
    const bool has_q = wave < 2;
    // Rows 8 .. 15 and 0 .. 7 of every second 16 lie swapped: the product's operands are rows 0 .. 7 and 16 .. 23 at once, which then meet
    // other banks.  dpos: where this lane's row lies.
    const int dpos = (wave & 1) * 64 + lane, drow = dpos ^ ((dpos >> 1) & 8), doff = drow * sn2;
    const unsigned ooff = has_q ? kFusedPast : (unsigned)doff, loff = has_q ? (unsigned)drow * 4u : kFusedPast;
    // A group's dQ: 16 of its 32 queries and half of the block's keys per wave
    const int sl0 = (wave & 1) * 16, kk0 = (wave >> 1) * KT;
    // the query of slot sl0 + c: slot 8 j + i holds query 16 (j / 2) + 8 (i / 4) + 4 (j % 2) + i % 4
    const int slq = sl0 + 8 * ((c >> 2) & 1) + 4 * ((c >> 3) & 1) + (c & 3);
    // (lane's place in a bias tile: key c of 16 (the tile's second 16 lie 16 lanes on), half a tile of queries, every other four of it)
    const int boff = BT == 2 ? (j >> 1) * 1024 + (c + 32 * (j & 1)) * 16 : (j >> 1) * 2048 + (c + 32 * (j & 1)) * 16;
    // The 32 columns of the key operand are K, (mask 1 1 1), K, V: of the score product Q scaled, (1 1 1 -LSE), the rest of Q, zeros
    // meet them, of dP zeros three times and dO.
    const int arow = (24 * (c >> 3) + (c & 7)) * 16, aoff = (j == 0 ? R::OFF_H : j == 1 ? R::OFF_L : j == 2 ? R::OFF_R : R::OFF_Z) + arow, goff = (j == 3 ? R::OFF_G : R::OFF_Z) + arow;
    const int toff = (24 * (j >> 1) + 4 * (j & 1) + (c >> 2)) * 16 + (c & 1) * 8;   // rows read transposed (columns 8 .. 15: 0 .. 7 again)
    const int astep = c < 8 ? 128 : -128, tstep = j < 2 ? 128 : -128;               // from the operand's first eight rows of each 16 to its others
    const bool has_d = j < 2;                                                       // lanes whose four rows of a result are columns of D

    // problems in order per XCD, one after the other where the grid is smaller
    const unsigned xcd = blockIdx.x % 8, per = gridDim.x / 8;
    const bool spread = gridDim.x < problems;
    unsigned t = spread ? (unsigned)((uint64_t)problems * xcd / 8) + blockIdx.x / 8 : xcd_remap(blockIdx.x, gridDim.x);
    const unsigned t_end = spread ? (unsigned)((uint64_t)problems * (xcd + 1) / 8) : t + 1;
    const __amdgpu_buffer_rsrc_t prs = __builtin_amdgcn_make_buffer_rsrc((void *)(e.dq_part + (nb > 1 ? (int64_t)blockIdx.x * N * D : 0)), 0, nb > 1 ? N * D * 4 : 0, 0x00020000);
    const unsigned poff = has_d && wave < 2 ? (unsigned)(slq * D + 4 * j) * 4u : kFusedPast, qoff = has_d && wave < 2 ? (unsigned)(slq * sn2 + 4 * j * 2) : kFusedPast;

    *reinterpret_cast<uint4 *>(lds + (wave >> 1) * R::STAGE + R::OFF_Z + ((wave & 1) * 64 + lane) * 16) = make_uint4(0u, 0u, 0u, 0u);
    for (; t < t_end; t += per) {
        const Prob pr = walk_problem(p, t);
        const bool dead = uniform_load(e.dead + pr.b * p.S + pr.s) != 0, kill = dead && p.mask_kind == EVO_MASK_BOOL;
        const __amdgpu_buffer_rsrc_t frs = __builtin_amdgcn_make_buffer_rsrc((void *)((const T *)(has_q ? p.q : p.dout) + pr.base), 0, valid, 0x00020000);
        const __amdgpu_buffer_rsrc_t krs = __builtin_amdgcn_make_buffer_rsrc((void *)((const T *)p.k + pr.base), 0, valid, 0x00020000);
        const __amdgpu_buffer_rsrc_t vrs = __builtin_amdgcn_make_buffer_rsrc((void *)((const T *)p.v + pr.base), 0, valid, 0x00020000);
        const __amdgpu_buffer_rsrc_t mrs = __builtin_amdgcn_make_buffer_rsrc((void *)(e.m2a + ((int64_t)pr.b * p.S + pr.s) * np256), 0, np256 * 16, 0x00020000);
        const __amdgpu_buffer_rsrc_t ors = __builtin_amdgcn_make_buffer_rsrc((void *)((const T *)p.o + pr.base), 0, valid, 0x00020000);
        const __amdgpu_buffer_rsrc_t lrs = __builtin_amdgcn_make_buffer_rsrc((void *)(p.lse + pr.row0), 0, N * 4, 0x00020000);
        const __amdgpu_buffer_rsrc_t drs = __builtin_amdgcn_make_buffer_rsrc((void *)(e.delta + pr.row0), 0, N * 4, 0x00020000);
        const __amdgpu_buffer_rsrc_t dqrs = __builtin_amdgcn_make_buffer_rsrc((void *)((T *)p.dq + pr.base), 0, valid, 0x00020000);
        const __amdgpu_buffer_rsrc_t dkrs = __builtin_amdgcn_make_buffer_rsrc((void *)((T *)p.dk + pr.base), 0, valid, 0x00020000);
        const __amdgpu_buffer_rsrc_t dvrs = __builtin_amdgcn_make_buffer_rsrc((void *)((T *)p.dv + pr.base), 0, valid, 0x00020000);
        const float mul = dead ? 0.0f : kLog2e, qscale = dead ? 0.0f : p.scale * kLog2e;   // (a row with every key masked has neither bias nor scores)
        const int64_t btile = dead ? e.zero_tile : ((int64_t)(e.bias_batches > 1 ? pr.b : 0) * p.H + pr.h) * NT * NT * 1024;
        const __amdgpu_buffer_rsrc_t brs = __builtin_amdgcn_make_buffer_rsrc(
            BT == 2 ? (void *)(e.bk16 + btile) : (void *)(e.bk + btile), 0, BT == 0 ? 0 : dead ? 1024 * BES : NT * NT * 1024 * BES, 0x00020000);

        for (int kb = 0; kb < nb; ++kb) {
            const int key0 = kb * R::KB + wave * KT * 16;
            v8 orow;
            float lse;
            auto fetch = [&](int stage, int parity, bool ask) {   // (rows past the end: zeros)
                const int from = stage * R::QR * sn2;
                if (ask) fused_dma(frs, lds + parity * R::STAGE + (has_q ? 0 : R::OFF_G) + (wave & 1) * 1024, doff, from);
                orow = __builtin_bit_cast(v8, __builtin_amdgcn_raw_buffer_load_b128(ors, ooff, from, 0));
                lse = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(lrs, loff, stage * R::QR * 4, 0));
            };
            auto finish = [&](int stage, int parity, auto younger) {   // what this wave asked for is there
                unsigned char *const buf = lds + parity * R::STAGE;
                fused_wait_but<decltype(younger)::value>();
                const int q = stage * R::QR + drow;
                if (has_q) {
                    v8 hi, lo;
                    scaled_hilo8<T>(*reinterpret_cast<const v8 *>(buf + dpos * 16), qscale, hi, lo);
                    *reinterpret_cast<v8 *>(buf + R::OFF_H + dpos * 16) = hi;
                    *reinterpret_cast<v8 *>(buf + R::OFF_R + dpos * 16) = lo;
                    *reinterpret_cast<v8 *>(buf + R::OFF_L + dpos * 16) = aug8<T>(one3, pack_split3<T>(q < N ? -lse * kLog2e : kMaskFloor));   // (rows past the end: probability zero)
                } else {
                    const float d = dot8<T>(*reinterpret_cast<const v8 *>(buf + R::OFF_G + dpos * 16), orow, 0.0f);
                    reinterpret_cast<float *>(buf + R::OFF_D)[drow] = kill ? 0.0f : -d;   // (no gradient through replaced scores)
                    if (kb == 0) __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(d), drs, drow * 4, stage * R::QR * 4, 0);
                }
            };
            // the block's keys in LDS
            for (int i = wave; i < KT; i += R::NW) fused_dma(krs, ex + i * 1024, (i * 64 + lane) * sn2, kb * R::KB * sn2);
            fetch(0, 0, true);
            v8 kv[KT];
#pragma unroll
            for (int kt = 0; kt < KT; ++kt) {
                // (keys past the end: V zero, the mask's floor; the uniform offsets stay inside)
                const int k16 = key0 + kt * 16;
                const u32x4f v = __builtin_amdgcn_raw_buffer_load_b128(vrs, c * sn2, min(k16, N - 1) * sn2, 0);
                u32x4f m = __builtin_amdgcn_raw_buffer_load_b128(mrs, c * 16, min(k16, np256 - 16) * 16, 0);
                if (k16 + c >= N) {
                    m[0] = floor2.x;
                    m[1] = floor2.y;
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) m[i] = j == 1 ? m[i] : kill ? 0u : v[i];
                kv[kt] = __builtin_bit_cast(v8, m);
            }
            // bias tiles in 32 x 32 accumulator order: this lane's eight entries of 32 queries x 16 keys are one piece of 16 bytes (fp32: two)
            uint4 bt[R::AHEAD];
            f32x4 bf[R::AHEAD][2];
            const int brow = dead ? 0 : NT * 1024 * BES;   // from one group of queries to the next
            auto load_bias = [&](int n, int kt) {
                const int k16 = (key0 >> 4) + kt, tile = min(k16 >> 1, NT - 1);
                const int at = min(n, NT - 1) * brow + (dead ? 0 : tile * 1024 * BES) + (k16 & 1) * 256;
                if (BT == 2) bt[kt % R::AHEAD] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(brs, boff, at, 0));
                if (BT == 1) {
                    bf[kt % R::AHEAD][0] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(brs, boff, at, 0));
                    bf[kt % R::AHEAD][1] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(brs, boff, at + 1024, 0));
                }
            };
#pragma unroll
            for (int kt = 0; kt < R::AHEAD; ++kt) load_bias(0, kt);
            finish(0, 0, std::integral_constant<int, 0>());
            fused_barrier();
#pragma unroll
            for (int kt = 0; kt < KT; ++kt) {
                const v8 k = *reinterpret_cast<const v8 *>(ex + (wave * KT * 16 + kt * 16 + c) * 16);
                if ((j & 1) == 0) kv[kt] = k;
            }
            v8 ktr[KT];   // K transposed, of this wave's half of the keys
#pragma unroll
            for (int i = 0; i < KT; ++i)
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const v4 w = fused_tr<T>(ex + ((kk0 + i) * 32 + 16 * h + 4 * j + (c >> 2)) * 16 + (c & 1) * 8);
#pragma unroll
                    for (int r = 0; r < 4; ++r) ktr[i][4 * h + r] = w[r];
                }
            fused_barrier();

            f32x4 dk[KT], dv[KT];
#pragma unroll
            for (int kt = 0; kt < KT; ++kt) dk[kt] = dv[kt] = f32x4{0.f, 0.f, 0.f, 0.f};

            // dQ of a group follows one group behind, a step of 32 keys behind every tile, and is stored one group later yet: the two halves of
            // the keys meet in LDS then.
            f32x4 dq = {0.f, 0.f, 0.f, 0.f}, before = dq;
            auto dq_step = [&](const unsigned char *exb, int i) {
                v8 b;
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int row = (kk0 + i) * 32 + 16 * h + 4 * j + (c >> 2), col = sl0 + 4 * (c & 3);
                    const v4 w = fused_tr<T>(exb + R::ate(row, col >> 3) + (col & 7) * 2);
#pragma unroll
                    for (int r = 0; r < 4; ++r) b[4 * h + r] = w[r];
                }
                dq = M::mma(ktr[i], b, dq);
            };
            auto dq_leave = [&](int par) {
                if (wave >= 2 && has_d) *reinterpret_cast<f32x4 *>(xch + par * 1024 + (wave & 1) * 512 + c * 32 + j * 16) = dq;
            };
            // (Every load and store of a group is issued whatever the group: the compiler counts what is under way, and takes the least of what
            // may be.  What there is nothing to do for lies past the end of its array: nothing is stored, zeros are read.)
            auto dq_store = [&](int n, int par) {
                const f32x4 v = dq + before + *reinterpret_cast<const f32x4 *>(xch + par * 1024 + (wave & 1) * 512 + c * 32 + (j & 1) * 16);
                if (kb + 1 < nb) {
                    // (no uniform offset: see kFusedPast)
                    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4f, v), prs, n < 0 ? kFusedPast : poff + (unsigned)(n * 32 * D * 4), 0, 0);
                } else {
                    v4 w;
#pragma unroll
                    for (int i = 0; i < 4; ++i) w[i] = (T)(v[i] * p.scale);
                    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2f, w), dqrs, n < 0 ? kFusedPast : qoff + (unsigned)(n * 32 * sn2), 0, 0);
                }
            };
            auto dq_begin = [&](int n) {   // what the blocks before have left of it
                dq = f32x4{0.f, 0.f, 0.f, 0.f};
                before = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(prs, kb > 0 && n >= 0 ? poff + (unsigned)(n * 32 * D * 4) : kFusedPast, 0, 0));
            };

            for (int n0 = 0; n0 < NT; n0 += 2 * GPS) {   // two stages
#pragma unroll
                for (int u = 0; u < 2 * GPS; ++u) {
                    const int n = n0 + u, s1 = min(n / GPS + 1, nst - 1), gb = u % GPS * 32, parity = u / GPS;
                    const bool first = u % GPS == 0, last = u % GPS == GPS - 1, more = n / GPS + 1 < nst;   // group of its stage; a stage follows (this one is whole)
                    if (n < NT) {   // uniform
                        const unsigned char *buf = lds + parity * R::STAGE;
                        unsigned char *const exb = ex + (u & 1) * R::EX, *const exq = ex + ((u & 1) ^ 1) * R::EX;
                        dq_store(n - 2, (u & 1) ^ 1);
                        if (first) fetch(s1, parity ^ 1, more);
                        dq_begin(n - 1);
                        asm volatile("" ::: "memory");   // (the bias asked for below is younger: `finish` counts on it)

                        v8 aq[2], ag[2], qt, gt;
                        f32x4 ndl[2];
#pragma unroll
                        for (int t2 = 0; t2 < 2; ++t2) {
                            aq[t2] = *reinterpret_cast<const v8 *>(buf + aoff + gb * 16 + t2 * astep);
                            ag[t2] = *reinterpret_cast<const v8 *>(buf + goff + gb * 16 + t2 * astep);
                            ndl[t2] = *reinterpret_cast<const f32x4 *>(buf + R::OFF_D + (gb + 16 * (j >> 1) + 8 * t2 + 4 * (j & 1)) * 4);
                        }
#pragma unroll
                        for (int h = 0; h < 2; ++h) {
                            const v4 w = fused_tr<T>(buf + toff + gb * 16 + h * tstep), v = fused_tr<T>(buf + R::OFF_G + toff + gb * 16 + h * tstep);
#pragma unroll
                            for (int i = 0; i < 4; ++i) {
                                qt[4 * h + i] = w[i];
                                gt[4 * h + i] = v[i];
                            }
                        }
#pragma unroll
                        for (int kt = 0; kt < KT; ++kt) {
                            // since `fetch`, GPS - 1 groups before, this wave has asked for the bias of the tiles between, a load or, in fp32, two for each
                            if (kt == KT - 1 && last && more)
                                finish(s1, parity ^ 1, std::integral_constant<int, (BT == 0 ? 0 : BT == 1 ? 2 : 1) * (KT * GPS - 1)>());
                            f32x4 a[2], dp[2];
                            if (BT == 2) {
                                const uint4 raw = bt[kt % R::AHEAD];
                                const unsigned w[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
                                for (int i = 0; i < 4; ++i) {
                                    float lo, hi;
                                    unpack2<T>(w[i], lo, hi);
                                    a[i >> 1][2 * (i & 1)] = lo * mul;
                                    a[i >> 1][2 * (i & 1) + 1] = hi * mul;
                                }
                            } else if (BT == 1) {
                                a[0] = bf[kt % R::AHEAD][0];
                                a[1] = bf[kt % R::AHEAD][1];
                            } else {
                                a[0] = a[1] = f32x4{0.f, 0.f, 0.f, 0.f};
                            }
                            if (kt + R::AHEAD < KT) load_bias(n, kt + R::AHEAD);
                            else load_bias(n + 1, kt + R::AHEAD - KT);
#pragma unroll
                            for (int t2 = 0; t2 < 2; ++t2) {
                                a[t2] = M::mma(aq[t2], kv[kt], a[t2]);        // log2 P
                                dp[t2] = M::mma(ag[t2], kv[kt], ndl[t2]);     // dP - delta
                            }
                            dq_step(exq, kt);
                            v8 pf, ds;
#pragma unroll
                            for (int t2 = 0; t2 < 2; ++t2)
#pragma unroll
                                for (int r = 0; r < 4; ++r) {
                                    const float pv = fast_exp2(a[t2][r]);
                                    pf[4 * t2 + r] = (T)pv;
                                    ds[4 * t2 + r] = (T)(pv * dp[t2][r]);
                                }
                            *reinterpret_cast<v8 *>(exb + R::ate(wave * KT * 16 + kt * 16 + c, j)) = ds;
                            dv[kt] = M::mma(gt, pf, dv[kt]);
                            dk[kt] = M::mma(qt, ds, dk[kt]);
                            __builtin_amdgcn_sched_barrier(0);
                        }
                        dq_leave(u & 1);
                        fused_barrier();
                    }
                }
            }
            dq_store(NT - 2, (NT & 1) ^ 1);
            dq_begin(NT - 1);
#pragma unroll
            for (int i = 0; i < KT; ++i) dq_step(ex + ((NT - 1) & 1) * R::EX, i);
            dq_leave(NT & 1);
            fused_barrier();   // (everybody has left dS before the next keys come)
            dq_store(NT - 1, NT & 1);
#pragma unroll
            for (int kt = 0; kt < KT; ++kt) {
                const int k16 = key0 + kt * 16;
                const unsigned at = k16 < N && has_d ? (unsigned)(c * sn2 + 8 * j) : kFusedPast;   // (rows from N on lie past the end)
                const int from = min(k16, N - 1) * sn2;
                v4 wk, wv;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    wk[r] = (T)(dk[kt][r] * p.scale);
                    wv[r] = (T)dv[kt][r];
                }
                __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2f, wk), dkrs, at, from, 0);
                __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2f, wv), dvrs, at, from, 0);
            }
        }
    }
}

template <typename T, int KT>
static int fused8_launch(const EvoAttnParams &p, const Extra &e, hipStream_t st) {
    typedef Fused8<KT> R;
    const unsigned grid = (unsigned)mfma_fused_wgs(p), problems = (unsigned)((int64_t)p.B * p.H * p.S);
    const int nb = mfma_fused_blocks(p);
    auto go = [&](auto kern, PerDevice &done) {
        if (const int rc = ensure_dynamic_lds((const void *)kern, R::BYTES, done, nullptr)) return rc;
        kern<<<grid, 256, R::BYTES, st>>>(p, e, problems, nb);
        return hip_rc();
    };
    static PerDevice done[3]{};
    if (p.bias_dtype == EVO_NONE) return go(bwd_fused8<T, KT, 0>, done[0]);
    return e.bk16 ? go(bwd_fused8<T, KT, 2>, done[2]) : go(bwd_fused8<T, KT, 1>, done[1]);
}

template <typename T>
static int fused8_width(const EvoAttnParams &p, const Extra &e, hipStream_t st) {
    switch (mfma_fused8_tiles(p.N)) {
        case 2: return fused8_launch<T, 2>(p, e, st);
        case 3: return fused8_launch<T, 3>(p, e, st);
        case 4: return fused8_launch<T, 4>(p, e, st);
        case 5: return fused8_launch<T, 5>(p, e, st);
        default: return fused8_launch<T, 6>(p, e, st);
    }
}

int launch_mfma_fused8(const EvoAttnParams &p, const Extra &e, hipStream_t st) {
    return p.dtype == EVO_BF16 ? fused8_width<bf16_t>(p, e, st) : fused8_width<f16_t>(p, e, st);
}

}  // namespace evo
