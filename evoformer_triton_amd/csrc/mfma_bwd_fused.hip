// dQ, dK and dV in one kernel, head dim 32.
//
// Two kernels, one whose waves keep queries (dQ) and one whose waves keep keys (dK, dV), form every score, P and dP twice: 32 of 96 vector
// instructions per 32 x 32 tile for the bias, 32 issue slots for exp2.  Here they are formed once: a workgroup of 4 waves has a (b, h, s) problem, a wave
// KT key tiles of 16, whose dK and dV stay in registers while the queries stream by in groups of 32, two groups to a stage in LDS,
// double-buffered.  The matrix instruction is 16x16x32: a lane's eight probabilities of a group are eight consecutive operand columns of the
// dK and dV products as they lie.  dQ needs the sum over all keys of the block, which are four waves': they leave dS in LDS, and one
// group later each wave multiplies a quarter of the group's dQ out of it, two steps of 32 keys behind every tile of its own, so that the exchange
// costs the barrier that the stages need anyway.  Rows of more than 256 keys take blocks of keys, one after the other; dQ of the blocks before
// lies in fp32 in a scratch of the workgroup's own (512 workgroups then share the problems), read back and added in the same order every time.
// LSE rides in a matrix step with the mask (three 16-bit parts each, exact), -delta is the first C of dP.  delta = <dO, O> is formed where a wave
// prepares a stage, and written for the dBias kernel.
// No single bound: at S = N = 768, H = 4 the vector ALU is busy for .50 of the time, the matrix core .32, LDS .56, a fifth of that bank conflicts (counters, at
// 2.1 GHz), at two waves per SIMD (the registers of a wave's 64 keys), which wait for .30 of their life; 3.6 GB of traffic where once through the tensors is 1.2.  Per wave,
// group and tile 42 vector and 12 matrix instructions.  S = N = 768, H = 4 without dBias 1292 -> 992 us (dQ and dK/dV kernels before), S = N = 384 180 -> 143,
// N = 256, S = 512, H = 8 281 -> 209.  Four tiles per wave spill 12 registers (with an fp32 bias 28, and three 9), read back once per
// block of keys, outside the loop over queries.  Two tiles per wave and three waves per SIMD spill (1650); the next block's keys and first stage fetched
// during this one's last: more scalar registers than there are, 1035; head dim 64, of 32-query stages, 960 against the two kernels' 560.
#include "fused_common.h"
#include "kernels.h"

namespace evo {

// KT: key tiles of 16 per wave
template <int KT>
struct Fused {
    static constexpr int D = 32, NW = 4, C = D / 8, ROW = D * 2;    // waves; 16-byte chunks and bytes of a row
    static constexpr int KB = NW * KT * 16;                         // keys per block
    static constexpr int QR = 64, BLK = QR * ROW;    // query rows per stage
    static constexpr bool K_LDS = KT == 4;                          // the transposed keys are read from LDS again for every group
    static constexpr int OFF_G = BLK, OFF_QS = 2 * BLK, OFF_L = 3 * BLK, OFF_D = OFF_L + QR * 16, STAGE = (OFF_D + QR * 4 + 255) / 256 * 256;
    static constexpr int EX = KB * 64, OFF_EX = 2 * STAGE;          // dS of 32 queries x the block's keys, two of them
    static constexpr int KBYTES = KB * ROW, OFF_K = K_LDS ? OFF_EX + 2 * EX : OFF_EX;   // (else in the place of dS, before there is any)
    static constexpr int BYTES = K_LDS ? OFF_K + KBYTES : OFF_EX + (2 * EX > KBYTES ? 2 * EX : KBYTES);
    static constexpr int RPP = 1024 / ROW;                          // rows of a piece of 1 KB: a wave fetches one of each array and stage
    static_assert(BLK == NW * 1024, "one piece per wave");
    // where chunk c of row r lies: query rows (groups of four rows 16 and 4 apart meet other banks), and rows of keys and of dS
    static __device__ __forceinline__ int xq(int r) { return ((r >> 4) & 1) | ((r >> 2) & 1) << 1; }
    static __device__ __forceinline__ int xk(int r) { return ((r >> 3) & 1) | ((r >> 2) & 1) << 1; }
    static __device__ __forceinline__ int atq(int r, int c) { return r * ROW + ((c ^ xq(r)) << 4); }
    static __device__ __forceinline__ int atk(int r, int c) { return r * ROW + ((c ^ xk(r)) << 4); }
    static __device__ __forceinline__ int ate(int r, int c) { return r * 64 + ((c ^ xk(r)) << 4); }
};

template <typename T, int KT, int BT>
__global__ void __launch_bounds__(256, 2) bwd_fused(EvoAttnParams p, Extra e, unsigned problems, int nb) {
    typedef Fused<KT> R;
    typedef typename Mfma<T>::v8 v8;
    typedef typename Mfma<T>::v4 v4;
    typedef Mfma16<T> M;
    constexpr int D = R::D, BES = BT == 2 ? 2 : 4, DT = D / 16, KK = R::KB / 32, GPS = R::QR / 32;   // GPS: groups of 32 queries per stage
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];

    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), c = lane & 15, j = lane >> 4;
    const int N = p.N, NT = (N + 31) / 32, nst = (N + R::QR - 1) / R::QR, sn2 = (int)p.stride_n * 2, valid = (N - 1) * sn2 + D * 2;
    unsigned char *const ex = lds + R::OFF_EX, *const keys = lds + R::OFF_K;
    const uint2 one3 = ones3<T>();
    // this lane's row of a stage (its wave's first piece of 1 KB) and the offset of its 16 bytes of it
    const int drow = wave * R::RPP + lane / R::C, doff = drow * sn2 + (((lane % R::C) ^ R::xq(drow)) << 4);
    // this wave's tile of a group's dQ: 16 of its 32 queries, 16 columns
    const int sl0 = (wave & 1) * 16, d0 = (wave >> 1) * 16;
    // the query of slot sl0 + c: slot 8 j + i holds query 16 (j / 2) + 8 (i / 4) + 4 (j % 2) + i % 4
    // (lane's place in a bias tile: key c of 16 (the tile's second 16 lie 16 lanes on), half a tile of queries, every other four of it)
    const int boff = BT == 2 ? (j >> 1) * 1024 + (c + 32 * (j & 1)) * 16 : (j >> 1) * 2048 + (c + 32 * (j & 1)) * 16;
    const int slq = sl0 + 8 * ((c >> 2) & 1) + 4 * ((c >> 3) & 1) + (c & 3);

    // problems in order per XCD, one after the other where the grid is smaller
    const unsigned xcd = blockIdx.x % 8, per = gridDim.x / 8;
    const bool spread = gridDim.x < problems;
    unsigned t = spread ? (unsigned)((uint64_t)problems * xcd / 8) + blockIdx.x / 8 : xcd_remap(blockIdx.x, gridDim.x);
    const unsigned t_end = spread ? (unsigned)((uint64_t)problems * (xcd + 1) / 8) : t + 1;
    const __amdgpu_buffer_rsrc_t prs = __builtin_amdgcn_make_buffer_rsrc((void *)(e.dq_part + (nb > 1 ? (int64_t)blockIdx.x * N * D : 0)), 0, nb > 1 ? N * D * 4 : 0, 0x00020000);
    const int poff = (slq * D + d0 + 4 * j) * 4, qoff = slq * sn2 + (d0 + 4 * j) * 2;

    for (; t < t_end; t += per) {
        const Prob pr = walk_problem(p, t);
        const bool dead = uniform_load(e.dead + pr.b * p.S + pr.s) != 0, kill = dead && p.mask_kind == EVO_MASK_BOOL;
        const __amdgpu_buffer_rsrc_t qrs = __builtin_amdgcn_make_buffer_rsrc((void *)((const T *)p.q + pr.base), 0, valid, 0x00020000);
        const __amdgpu_buffer_rsrc_t grs = __builtin_amdgcn_make_buffer_rsrc((void *)((const T *)p.dout + pr.base), 0, valid, 0x00020000);
        const __amdgpu_buffer_rsrc_t krs = __builtin_amdgcn_make_buffer_rsrc((void *)((const T *)p.k + pr.base), 0, valid, 0x00020000);
        const __amdgpu_buffer_rsrc_t ors = __builtin_amdgcn_make_buffer_rsrc((void *)((const T *)p.o + pr.base), 0, valid, 0x00020000);
        const __amdgpu_buffer_rsrc_t lrs = __builtin_amdgcn_make_buffer_rsrc((void *)(p.lse + pr.row0), 0, N * 4, 0x00020000);
        const __amdgpu_buffer_rsrc_t drs = __builtin_amdgcn_make_buffer_rsrc((void *)(e.delta + pr.row0), 0, N * 4, 0x00020000);
        const __amdgpu_buffer_rsrc_t dqrs = __builtin_amdgcn_make_buffer_rsrc((void *)((T *)p.dq + pr.base), 0, valid, 0x00020000);
        const float mul = dead ? 0.0f : kLog2e, qscale = dead ? 0.0f : p.scale * kLog2e;   // (a row with every key masked has neither bias nor scores)
        const int64_t btile = dead ? e.zero_tile : ((int64_t)(e.bias_batches > 1 ? pr.b : 0) * p.H + pr.h) * NT * NT * 1024;
        const __amdgpu_buffer_rsrc_t brs = __builtin_amdgcn_make_buffer_rsrc(
            BT == 2 ? (void *)(e.bk16 + btile) : (void *)(e.bk + btile), 0, BT == 0 ? 0 : dead ? 1024 * BES : NT * NT * 1024 * BES, 0x00020000);

        for (int kb = 0; kb < nb; ++kb) {
            const int key0 = kb * R::KB + wave * KT * 16;
            v8 orow;
            float lse;
            auto fetch = [&](int stage, int parity, bool ask) {   // (rows past the end: zeros)
                unsigned char *dst = lds + parity * R::STAGE + wave * 1024;
                const int from = stage * R::QR * sn2;
                if (ask) {
                    fused_dma(qrs, dst, doff, from);
                    fused_dma(grs, dst + R::OFF_G, doff, from);
                }
                orow = __builtin_bit_cast(v8, __builtin_amdgcn_raw_buffer_load_b128(ors, doff, from, 0));
                lse = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(lrs, drow * 4, stage * R::QR * 4, 0));
            };
            auto finish = [&](int stage, int parity, auto younger) {   // what this wave asked for is there: Q scaled, the rows' -LSE (log2 units) and -delta
                unsigned char *const buf = lds + parity * R::STAGE, *const piece = buf + wave * 1024 + lane * 16;
                fused_wait_but<decltype(younger)::value>();
                const v8 q8 = *reinterpret_cast<const v8 *>(piece), g8 = *reinterpret_cast<const v8 *>(piece + R::OFF_G);
                *reinterpret_cast<v8 *>(piece + R::OFF_QS) = scaled8<T>(q8, qscale);
                float d = dot8<T>(g8, orow, 0.0f);
#pragma unroll
                for (int o = 1; o < R::C; o *= 2) d += fused_xor(d, o);
                if (lane % R::C == 0) {
                    const int q = stage * R::QR + drow;
                    *reinterpret_cast<v8 *>(buf + R::OFF_L + drow * 16) = aug8<T>(one3, pack_split3<T>(q < N ? -lse * kLog2e : kMaskFloor));   // (rows past the end: probability zero)
                    reinterpret_cast<float *>(buf + R::OFF_D)[drow] = kill ? 0.0f : -d;   // (no gradient through replaced scores)
                    if (kb == 0) __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(d), drs, drow * 4, stage * R::QR * 4, 0);
                }
            };
            // the block's keys in LDS
#pragma unroll
            for (int i = 0; i < R::KBYTES / 4096; ++i) {
                const int m = wave * (R::KBYTES / 4096) + i, r = m * R::RPP + lane / R::C, ch = (lane % R::C) ^ R::xk(r);
                fused_dma(krs, keys + m * 1024, r * sn2 + ch * 16, kb * R::KB * sn2);
            }
            fetch(0, 0, true);
            v8 kf[KT], vf[KT];
            v8 mk[KT];   // the keys' columns of the step that adds mask and -LSE: in its first eight, of lanes 0 to 15, alone
#pragma unroll
            for (int kt = 0; kt < KT; ++kt) {
                const int key = key0 + kt * 16 + c;
                vf[kt] = ld8((const T *)p.v + pr.base + (int64_t)min(key, N - 1) * p.stride_n + j * 8);
                uint2 m = e.m2[((int64_t)pr.b * p.S + pr.s) * (NT * 32) + min(key, NT * 32 - 1)];
                if (key >= NT * 32) m = pack_split3<T>(kMaskFloor);
                mk[kt] = j == 0 ? aug8<T>(m, one3) : zero8<T>();
            }
            // bias tiles in 32 x 32 accumulator order: this lane's eight entries of 32 queries x 16 keys are one piece of 16 bytes (fp32: two)
            uint4 bt[KT];
            f32x4 bf[KT][2];
            const int brow = dead ? 0 : NT * 1024 * BES;   // from one group of queries to the next
            auto load_bias = [&](int n, int kt) {
                const int k16 = (key0 >> 4) + kt, tile = min(k16 >> 1, NT - 1);
                const int at = min(n, NT - 1) * brow + (dead ? 0 : tile * 1024 * BES) + (k16 & 1) * 256;
                if (BT == 2) bt[kt] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(brs, boff, at, 0));
                if (BT == 1) {
                    bf[kt][0] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(brs, boff, at, 0));
                    bf[kt][1] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(brs, boff, at + 1024, 0));
                }
            };
#pragma unroll
            for (int kt = 0; kt < KT; ++kt) load_bias(0, kt);
            finish(0, 0, std::integral_constant<int, 0>());
            fused_barrier();
#pragma unroll
            for (int kt = 0; kt < KT; ++kt) {
                if (!R::K_LDS) kf[kt] = *reinterpret_cast<const v8 *>(keys + R::atk(wave * KT * 16 + kt * 16 + c, j));
                if (kill) vf[kt] = zero8<T>();
            }
            auto key_operand = [&](int kk) {   // K transposed: columns d0 .., keys 32 kk ..
                v8 r;
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int row = kk * 32 + 16 * h + 4 * j + (c >> 2), col = d0 + 4 * (c & 3);
                    const v4 w = fused_tr<T>(keys + R::atk(row, col >> 3) + (col & 7) * 2);
#pragma unroll
                    for (int i = 0; i < 4; ++i) r[4 * h + i] = w[i];
                }
                return r;
            };
            v8 ktr[R::K_LDS ? 1 : KK];
            if constexpr (!R::K_LDS) {
#pragma unroll
                for (int kk = 0; kk < KK; ++kk) ktr[kk] = key_operand(kk);
                fused_barrier();
            }

            f32x4 dk[KT][DT], dv[KT][DT];
#pragma unroll
            for (int kt = 0; kt < KT; ++kt)
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) dk[kt][dt] = dv[kt][dt] = f32x4{0.f, 0.f, 0.f, 0.f};

            // dQ of a group follows one group behind, two steps of 32 keys behind every tile, and is stored one group later yet: behind the
            // wait for that group's bias, which would wait for the stores as well.
            f32x4 dq = {0.f, 0.f, 0.f, 0.f}, before = dq;
            auto dq_step = [&](const unsigned char *exb, int kk) {
                v8 b;
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int row = kk * 32 + 16 * h + 4 * j + (c >> 2), col = sl0 + 4 * (c & 3);
                    const v4 w = fused_tr<T>(exb + R::ate(row, col >> 3) + (col & 7) * 2);
#pragma unroll
                    for (int i = 0; i < 4; ++i) b[4 * h + i] = w[i];
                }
                if constexpr (R::K_LDS) dq = M::mma(key_operand(kk), b, dq);
                else dq = M::mma(ktr[kk], b, dq);
            };
            // (Every load and store of a group is issued whatever the group: the compiler counts what is under way, and takes the least of what
            // may be.  What there is nothing to do for lies past the end of its array: nothing is stored, zeros are read.)
            auto dq_store = [&](int n) {
                const f32x4 v = dq + before;
                if (kb + 1 < nb) {
                    // (no uniform offset: see kFusedPast)
                    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4f, v), prs, (unsigned)poff + (n < 0 ? kFusedPast : (unsigned)(n * 32 * D * 4)), 0, 0);
                } else {
                    v4 w;
#pragma unroll
                    for (int i = 0; i < 4; ++i) w[i] = (T)(v[i] * p.scale);
                    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2f, w), dqrs, (unsigned)qoff + (n < 0 ? kFusedPast : (unsigned)(n * 32 * sn2)), 0, 0);
                }
            };
            auto dq_begin = [&](int n) {   // what the blocks before have left of it
                dq = f32x4{0.f, 0.f, 0.f, 0.f};
                before = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(prs, (unsigned)poff + (kb > 0 && n >= 0 ? (unsigned)(n * 32 * D * 4) : kFusedPast), 0, 0));
            };

            for (int n0 = 0; n0 < NT; n0 += 2 * GPS) {   // two stages
#pragma unroll
                for (int u = 0; u < 2 * GPS; ++u) {
                    const int n = n0 + u, s1 = min(n / GPS + 1, nst - 1), gb = u % GPS * 32, parity = u / GPS;
                    const bool first = u % GPS == 0, last = u % GPS == GPS - 1, more = n / GPS + 1 < nst;   // group of its stage; a stage follows (this one is whole)
                    if (n < NT) {
                    const unsigned char *buf = lds + parity * R::STAGE;
                    unsigned char *const exb = ex + (u & 1) * R::EX, *const exq = ex + ((u & 1) ^ 1) * R::EX;
                    dq_store(n - 2);
                    if (first) fetch(s1, parity ^ 1, more);
                    dq_begin(n - 1);
                    asm volatile("" ::: "memory");   // (the bias asked for below is younger: `finish` counts on it)

                    v8 aq[2], ag[2], al[2], qt[DT], gt[DT];
                    f32x4 ndl[2];
#pragma unroll
                    for (int t2 = 0; t2 < 2; ++t2) {
                        const int row = gb + 16 * (c >> 3) + 8 * t2 + (c & 7);
                        aq[t2] = *reinterpret_cast<const v8 *>(buf + R::OFF_QS + R::atq(row, j));
                        ag[t2] = *reinterpret_cast<const v8 *>(buf + R::OFF_G + R::atq(row, j));
                        al[t2] = *reinterpret_cast<const v8 *>(buf + R::OFF_L + row * 16);
                        ndl[t2] = *reinterpret_cast<const f32x4 *>(buf + R::OFF_D + (gb + 16 * (j >> 1) + 8 * t2 + 4 * (j & 1)) * 4);
                    }
#pragma unroll
                    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                        for (int h = 0; h < 2; ++h) {
                            const int row = gb + 16 * (j >> 1) + 8 * h + 4 * (j & 1) + (c >> 2), col = dt * 16 + 4 * (c & 3);
                            const int o = R::atq(row, col >> 3) + (col & 7) * 2;
                            const v4 w = fused_tr<T>(buf + o), v = fused_tr<T>(buf + R::OFF_G + o);
#pragma unroll
                            for (int i = 0; i < 4; ++i) {
                                qt[dt][4 * h + i] = w[i];
                                gt[dt][4 * h + i] = v[i];
                            }
                        }
#pragma unroll
                    for (int kt = 0; kt < KT; ++kt) {
                        // since `fetch`, GPS - 1 groups before, this wave has asked for the bias of the tiles between, a load or, in fp32, two for each
                        if (kt == KT - 1 && last && more)
                            finish(s1, parity ^ 1, std::integral_constant<int, (BT == 0 ? 0 : BT == 1 ? 2 : 1) * (KT * GPS - 1)>());
                        f32x4 a[2], dp[2];
                        if (BT == 2) {
                            const unsigned w[4] = {bt[kt].x, bt[kt].y, bt[kt].z, bt[kt].w};
#pragma unroll
                            for (int i = 0; i < 4; ++i) {
                                float lo, hi;
                                unpack2<T>(w[i], lo, hi);
                                a[i >> 1][2 * (i & 1)] = lo * mul;
                                a[i >> 1][2 * (i & 1) + 1] = hi * mul;
                            }
                        } else if (BT == 1) {
                            a[0] = bf[kt][0];
                            a[1] = bf[kt][1];
                        } else {
                            a[0] = a[1] = f32x4{0.f, 0.f, 0.f, 0.f};
                        }
                        load_bias(n + 1, kt);
                        if constexpr (R::K_LDS) kf[kt] = *reinterpret_cast<const v8 *>(keys + R::atk(wave * KT * 16 + kt * 16 + c, j));
#pragma unroll
                        for (int t2 = 0; t2 < 2; ++t2) {
                            a[t2] = M::mma(aq[t2], kf[kt], a[t2]);
                            dp[t2] = M::mma(ag[t2], vf[kt], ndl[t2]);
                            a[t2] = M::mma(al[t2], mk[kt], a[t2]);   // log2 P; dP - delta
                        }
                        dq_step(exq, 2 * kt);
                        dq_step(exq, 2 * kt + 1);
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
#pragma unroll
                        for (int dt = 0; dt < DT; ++dt) {
                            dv[kt][dt] = M::mma(gt[dt], pf, dv[kt][dt]);
                            dk[kt][dt] = M::mma(qt[dt], ds, dk[kt][dt]);
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    fused_barrier();
                    }
                }
            }
            dq_store(NT - 2);
            dq_begin(NT - 1);
#pragma unroll
            for (int kk = 0; kk < KK; ++kk) dq_step(ex + ((NT - 1) & 1) * R::EX, kk);
            dq_store(NT - 1);
#pragma unroll
            for (int kt = 0; kt < KT; ++kt) {
                const int key = key0 + kt * 16 + c;
                if (key < N) {
                    const int64_t o = pr.base + (int64_t)key * p.stride_n + 4 * j;
#pragma unroll
                    for (int dt = 0; dt < DT; ++dt) {
                        store4<T>((T *)p.dk + o + dt * 16, dk[kt][dt][0] * p.scale, dk[kt][dt][1] * p.scale, dk[kt][dt][2] * p.scale, dk[kt][dt][3] * p.scale);
                        store4<T>((T *)p.dv + o + dt * 16, dv[kt][dt][0], dv[kt][dt][1], dv[kt][dt][2], dv[kt][dt][3]);
                    }
                }
            }
            fused_barrier();   // (everybody has left dS before the next keys come)
        }
    }
}

template <typename T, int KT>
static int fused_launch(const EvoAttnParams &p, const Extra &e, hipStream_t st) {
    typedef Fused<KT> R;
    const unsigned grid = (unsigned)mfma_fused_wgs(p), problems = (unsigned)((int64_t)p.B * p.H * p.S);
    const int nb = mfma_fused_blocks(p);
    auto go = [&](auto kern, PerDevice &done) {
        if (const int rc = ensure_dynamic_lds((const void *)kern, R::BYTES, done, nullptr)) return rc;
        kern<<<grid, 256, R::BYTES, st>>>(p, e, problems, nb);
        return hip_rc();
    };
    static PerDevice done[3]{};
    if (p.bias_dtype == EVO_NONE) return go(bwd_fused<T, KT, 0>, done[0]);
    return e.bk16 ? go(bwd_fused<T, KT, 2>, done[2]) : go(bwd_fused<T, KT, 1>, done[1]);
}

template <typename T>
static int fused_width(const EvoAttnParams &p, const Extra &e, hipStream_t st) {
    switch (mfma_fused_tiles(p.N)) {
        case 2: return fused_launch<T, 2>(p, e, st);
        case 3: return fused_launch<T, 3>(p, e, st);
        default: return fused_launch<T, 4>(p, e, st);
    }
}

int launch_mfma_fused(const EvoAttnParams &p, const Extra &e, hipStream_t st) {
    return p.dtype == EVO_BF16 ? fused_width<bf16_t>(p, e, st) : fused_width<f16_t>(p, e, st);
}

}  // namespace evo
