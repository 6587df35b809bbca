// The fp32 kernels: operands and results in fp32, products on the bf16 matrix instruction out of three bf16 parts of every operand.
//
// The fp32 matrix instruction does 256 flop per clock and CU, the bf16 one sixteen times as many.  A value is the sum of three bf16 numbers (each the
// rest rounded), and of the nine products of parts the three smallest, below 2^-26 of the whole, are left out: six instructions in the place of sixteen,
// with fewer roundings on the way (a product of 32 x 32 x K by this / by the fp32 instruction, error against 64 bits over the result's norm:
// K = 32 6.8e-8 / 1.02e-7, 256 2.4e-7 / 2.9e-7, 1 024 4.9e-7 / 5.8e-7).  At head dim 32 a 32 x 32 tile takes 384 clocks of a SIMD per product
// instead of 1 024.
//
// What bounds the kernels then is the matrix instructions and the vector ones one after the other (the two barely overlap: 8 matrix and 64 fused
// multiply-adds take 171 ns a wave at four waves per SIMD, 109 and 106 by themselves), so what surrounds the products is kept off the vector ALU:
// Q is scaled by log2 e / sqrt(D) before it is split; mask, -maximum, -LSE and -delta (three parts each, exact) come in by one more step of a chain. Scores and
// bias are summed alike in every kernel, the large terms last: their roundings are the same in P and in the LSE that it is relative to.
//
// The work is split by tiles alone: a wave owns 32 rows of the result and walks over the other side's 32-row tiles, which its workgroup brings
// from memory through registers, splits (3.5 instructions per value) and leaves in LDS, a plane for each part; nothing is prepared beforehand, which
// keeps a small call at one launch forward and three or four backward.  Bias, mask and rows of the next tile are asked for before this one is computed on
// and nothing is done to them until then: with a conversion behind a load, every tile waited for memory (forward 56 -> 39 us of the case below).
//
// us, fp32 instruction / this, B = 1: S = 64, N = 256, H = 8, D = 32 forward 48 / 36, backward 228 / 151 (counters: a forward's SIMD is busy 67 k clocks, 33 k of
// them with vector and 26 k with matrix instructions; with one tile of keys instead of eight 22 k; in dQ, dBias and dK/dV, at 1.6 waves per SIMD, vector instructions
// take 0.31 to 0.33 of the time and matrix instructions 0.28 to 0.34); S = 4, N = 1 024, H = 4 76 / 47, 231 / 139; S = 100, N = 160, H = 4 31 / 19, 135 / 103;
// D = 64, S = 64, N = 256, H = 8 90 / 62, 384 / 330.  Not taken up: 64 rows per stage, all of a tile's operands read ahead, a priority of half
// the waves (each within 3 %), eight waves in the backward (161 / 154).
// Error against 64 bits over that of the fp32 instruction, N = 32 to 256, 160 calls: .65 to .78 at the median for every result, none above 1.
//
// Infinite operands, and those beyond bf16's range: `either_way`.
#include "f32_direct.h"

namespace evo {

// Two values as three bf16 pairs each whose sums are the values: every part is the rest rounded, so the third is exact down to 2^-102; below, the
// smaller parts run out of exponents.  A rest comes from one v_dot2c: x + (-1) part of this half + 0 part of the other.
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
struct Parts2 { bf16x2 p[3]; };
// So operands are split 2^24 times as large, every normal fp32 number whole, and results divided by it: of a dO or a V around 1e-36 nothing is lost, and dS,
// formed of the two, is 2^48 times itself (split as they are, dQ of a dO around 1e-34 was 6 times, around 1e-36 600 times as far from 64 bits as by the fp32
// instruction).  A score's two factors can't both be: the staged one is, the other one is split 2^24 times as small.  Where that takes a value of it
// below 2^-102 (`begin`; the dBias kernel, which stages both, asks whether the larger one is so large that it could tell), `either_way` has the fp32 instruction.
// Of the probabilities the forward's are relative to a sum in which one is 2^-8 at least; dV's, where a key may have only small ones, are split 2^24 times as
// large as well.
constexpr float kUp = 0x1p24f, kDown = 0x1p-24f, kUp2 = 0x1p48f, kDown2 = 0x1p-48f, kDown3 = 0x1p-72f, kWhole = 0x1p-102f, kMostStaged = 0x1p84f;
__device__ __forceinline__ Parts2 parts2(float x, float y) {
    // (-1, 0) and (0, -1), kept from the compiler: it writes the first as the inline constant -1.0, which the instruction reads as (0, -1)
    unsigned lo = 0x0000bf80u, hi = 0xbf800000u;
    asm("" : "+s"(lo), "+s"(hi));
    Parts2 r;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        r.p[i][0] = (bf16_t)x;
        r.p[i][1] = (bf16_t)y;
        if (i == 2) break;
        x = __builtin_amdgcn_fdot2_f32_bf16(r.p[i], __builtin_bit_cast(bf16x2, lo), x, false);
        y = __builtin_amdgcn_fdot2_f32_bf16(r.p[i], __builtin_bit_cast(bf16x2, hi), y, false);
    }
    return r;
}

// A tile is 32 rows in LDS, a plane for each part (`put`: four columns of a row; `clear`: the columns beyond D); `Frag` is a row in registers, this lane's half
// of it in NP pieces of four columns (`col`); `rows` is the tile's rows times the lane's, `cols` adds the tile's columns times a tile of results.
template <int D>
struct Split {
    typedef Mfma<bf16_t> M;
    typedef M::v8 v8;
    static constexpr int DP = D < 32 ? 32 : D, PLANE = 32 * DP * 2, TILE = 3 * PLANE, DT = DP / 32, KS = D < 16 ? 1 : D / 16, NP = 2 * KS;
    typedef StreamGeo<DP> G;
    struct Frag { v8 p[3][KS]; };
    static __device__ __forceinline__ int col(int i, int g) { return 16 * (i >> 1) + 8 * g + 4 * (i & 1); }   // (head dim 8: the upper half has none)
    static __device__ __forceinline__ void put(unsigned char *tile, int row, int c, f32x4 v) {
        const Parts2 a = parts2(v[0], v[1]), b = parts2(v[2], v[3]);
        tile += (row >> 5) * TILE + G::at(row & 31, c >> 3) + (c & 4) * 2;
#pragma unroll
        for (int i = 0; i < 3; ++i)
            *reinterpret_cast<uint2 *>(tile + i * PLANE) = make_uint2(__builtin_bit_cast(unsigned, a.p[i]), __builtin_bit_cast(unsigned, b.p[i]));
    }
    static __device__ __forceinline__ void clear(unsigned char *tile, int rows, int threads) {
        if (D >= 32) return;
        constexpr int PAD = (DP - D) / 8;
        for (int k = threadIdx.x; k < rows * PAD * 3; k += threads) {
            const int pl = k % 3, c = D / 8 + k / 3 % PAD, r = k / 3 / PAD;
            *reinterpret_cast<uint4 *>(tile + (r >> 5) * TILE + pl * PLANE + G::at(r & 31, c)) = make_uint4(0, 0, 0, 0);
        }
    }
    static __device__ __forceinline__ Frag frag(const f32x4 (&v)[NP], float scale) {
        Frag r;
#pragma unroll
        for (int j = 0; j < NP; ++j)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const Parts2 a = parts2(v[j][2 * h] * scale, v[j][2 * h + 1] * scale);
#pragma unroll
                for (int i = 0; i < 3; ++i) {
                    r.p[i][j >> 1][4 * (j & 1) + 2 * h] = a.p[i][0];
                    r.p[i][j >> 1][4 * (j & 1) + 2 * h + 1] = a.p[i][1];
                }
            }
        return r;
    }
    // Zero, or not a number where a value's parts are not all of it once it has been multiplied by `scale`: what the lane's sums begin with, so that they are
    // not finite then (kept beside them, the answer cost the kernels with a bias 16 registers).
    static __device__ __forceinline__ float begin(const f32x4 (&v)[NP], float scale) {
        bool lacks = false;
#pragma unroll
        for (int j = 0; j < NP; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) lacks |= fabsf(v[j][i] * scale) < kWhole && v[j][i] != 0.0f;
        return lacks && scale != 0.0f ? __int_as_float(0x7fc00000) : 0.0f;
    }
    static __device__ __forceinline__ v8 operand(const unsigned char *tile, int part, int ks, int lane) {
        return *reinterpret_cast<const v8 *>(tile + part * PLANE + G::at(lane & 31, 2 * ks + (lane >> 5)));
    }
    static __device__ __forceinline__ Frag staged(const unsigned char *tile, int lane) {
        Frag r;
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) r.p[i][ks] = operand(tile, i, ks, lane);
        return r;
    }
    // (the smallest products first)
    static __device__ __forceinline__ f32x16 rows(const unsigned char *tile, int lane, const Frag &b) {
        f32x16 c = zero16();
#pragma unroll
        for (int i = 2; i >= 0; --i) {
            v8 a[KS];
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) a[ks] = operand(tile, i, ks, lane);
#pragma unroll
            for (int j = 2 - i; j >= 0; --j)
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) c = M::mma(a[ks], b.p[j][ks], c);
        }
        return c;
    }
    static __device__ __forceinline__ void cols(const unsigned char *tile, int lane, const f32x16 &w, f32x16 (&acc)[DT], float scale = 1.0f) {
        v8 b[3][2];
#pragma unroll
        for (int r = 0; r < 16; r += 2) {
            const Parts2 a = parts2(w[r] * scale, w[r + 1] * scale);
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                b[i][r >> 3][r & 7] = a.p[i][0];
                b[i][r >> 3][(r & 7) + 1] = a.p[i][1];
            }
        }
#pragma unroll
        for (int i = 2; i >= 0; --i)
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                for (int ts = 0; ts < 2; ++ts) {
                    const v8 a = transposed<bf16_t, DP>(tile + i * PLANE, 0, ts, dt, lane);
#pragma unroll
                    for (int j = 2 - i; j >= 0; --j) acc[dt] = M::mma(a, b[j][ts], acc[dt]);
                }
    }
};

// What a workgroup keeps in LDS: tiles of two arrays in two stages (one barrier per tile), an operand chunk for each of a stage's rows and one
// of ones, a value per wave.
template <int D>
struct SplitShared {
    typedef Split<D> E;
    static constexpr int TILES = 4 * E::TILE, BYTES = TILES + (2 * 32 + 1) * 16 + 64;
    unsigned char *lds;
    __device__ __forceinline__ unsigned char *tile(int buf, int a) const { return lds + (buf * 2 + a) * E::TILE; }
    __device__ __forceinline__ uint4 *chunk(int buf) const { return reinterpret_cast<uint4 *>(lds + TILES) + buf * 32; }
    __device__ __forceinline__ uint4 *one() const { return reinterpret_cast<uint4 *>(lds + TILES) + 2 * 32; }
    __device__ __forceinline__ float *red() const { return reinterpret_cast<float *>(one() + 1); }
};

// A value that is the same for the wave.
__device__ __forceinline__ float uniform(float x) { return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(x))); }

// The extra step of a chain: eight columns out of two values' parts, (a a a b b b 0 0).
__device__ __forceinline__ uint4 chunk_of(uint2 a, uint2 b) { return __builtin_bit_cast(uint4, aug8<bf16_t>(a, b)); }
__device__ __forceinline__ bf16x8 as_operand(uint4 v) { return __builtin_bit_cast(bf16x8, v); }
__device__ __forceinline__ uint2 parts_of(float x) { return pack_split3<bf16_t>(x); }

// An array's rows; those at and beyond N read as zero.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rows_of(const void *base, const EvoAttnParams &p) {
    return __builtin_amdgcn_make_buffer_rsrc((void *)base, 0, (int)(((unsigned)(p.N - 1) * (unsigned)p.stride_n + (unsigned)p.D) * 4u), 0x00020000);
}
// ROWS rows of two arrays through registers into LDS: `load` asks for rows r0 .. (r0 < N), `put` splits and writes them, times a factor for each array;
// HUGE_TOO: `huge`, the lanes that have written a value of the first array of kMostStaged or more so far (lacking 2^-102 of the other factor they might show it).
template <int D, int THREADS, int ROWS = 32, bool HUGE_TOO = false>
struct SplitStage {
    typedef Split<D> E;
    static constexpr int PIECES = ROWS * D / 4, PER = (2 * PIECES + THREADS - 1) / THREADS;   // (of one array: a multiple of 64)
    f32x4 v[PER];
    unsigned long long huge = 0;
    __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t a, __amdgpu_buffer_rsrc_t b, unsigned stride_n, int r0) {
        const int first = __builtin_amdgcn_readfirstlane(threadIdx.x & ~63);
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            // (k0: the same for the wave; where there are more waves than pieces, some ask for the others' again: behind a branch the load is waited for at once)
            const int k0 = (first + i * THREADS) & (2 * PIECES - 1), k = (k0 & (PIECES - 1)) + (threadIdx.x & 63);
            v[i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(k0 < PIECES ? a : b, ((unsigned)(k / (D / 4)) * stride_n + (unsigned)(k % (D / 4) * 4)) * 4u,
                                                                                 (unsigned)r0 * stride_n * 4u, 0));
        }
    }
    __device__ __forceinline__ void put(unsigned char *dst0, unsigned char *dst1, float scale0, float scale1) {
        const int first = __builtin_amdgcn_readfirstlane(threadIdx.x & ~63);
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int k0 = first + i * THREADS, k = (k0 & (PIECES - 1)) + (threadIdx.x & 63);
            if (2 * PIECES % THREADS != 0 && k0 >= 2 * PIECES) break;
            const f32x4 x = v[i] * (k0 < PIECES ? scale0 : scale1);
            if (HUGE_TOO && k0 < PIECES)
                huge |= __builtin_amdgcn_ballot_w64(fmaxf(fmaxf(fabsf(x[0]), fabsf(x[1])), fmaxf(fabsf(x[2]), fabsf(x[3]))) >= kMostStaged);
            E::put(k0 < PIECES ? dst0 : dst1, k / (D / 4), k % (D / 4) * 4, x);
        }
    }
};

// The bias of one tile as a lane has it: entries as they come, asked for a tile ahead; ROW: of the lane's row, four columns at a time, else of its column.
// A row with every key masked has none: its matrix is empty, and what is read outside is zero.  (Every load is issued whatever the tile, into the
// registers that the tile before has left: behind a branch around it the compiler copies what may or may not have been loaded, and waits for it.)
template <bool BIAS, bool ROW>
struct BiasAhead {
    __amdgpu_buffer_rsrc_t rs;
    unsigned at, stride;   // bytes: the lane's own row or column (inside the matrix) and, of columns, its half's first row; from row to row
    int N, g;
    f32x16 v;
    __device__ __forceinline__ BiasAhead(const EvoAttnParams &p, int b, int h, int own, bool dead, int lane) {
        if (!BIAS) return;
        stride = (unsigned)p.bias_stride_row * 4u;
        N = p.N;
        g = lane >> 5;
        at = ROW ? (unsigned)own * stride + 16u * g : (unsigned)own * 4u + 4u * g * stride;
        rs = __builtin_amdgcn_make_buffer_rsrc((void *)((const float *)p.bias + b * p.bias_stride_b + h * p.bias_stride_h), 0,
                                               dead ? 0 : (int)((unsigned)(N - 1) * stride + (unsigned)N * 4u), 0x00020000);
        ask(0);
    }
    __device__ __forceinline__ float entry(unsigned lane_at, unsigned uniform_at) const {
        return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, lane_at, uniform_at, 0));
    }
    // tile t, past the last one that one again (not used); entries past the row's end, or of rows past the last, repeat the last: their keys are
    // masked, their queries' probabilities zero
    __device__ __forceinline__ void ask(int t) {
        if (!BIAS) return;
        const int c = min(32 * t, (N - 1) & ~31);
        // (uniform; a last tile's pieces that lie beyond the row are the row's last.  An entry at a time there: S = 64, N = 120 / 248, H = 8, D = 32 forward
        // 18 / 42 us, so 14 / 35, where the fp32 instruction took 17 / 48.  As a branch of its own it is waited for: N = 250, S = 4, D = 8 15 -> 16 us.)
        if (c + 32 <= N || (ROW && N % 4 == 0)) {
            const unsigned last = at - 16u * g + 4u * (unsigned)(N - 4);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if (ROW) {
                    const f32x4 x = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, min(at + 4u * c + 32u * j, last), 0, 0));
#pragma unroll
                    for (int i = 0; i < 4; ++i) v[4 * j + i] = x[i];
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i) v[4 * j + i] = entry(at, (unsigned)(c + 8 * j + i) * stride);
                }
            }
        } else {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const unsigned d = (unsigned)(min(c + crow(r, g), N - 1) - 4 * g);   // (modulo 2^32)
                v[r] = entry(at + d * (ROW ? 4u : stride), 0);
            }
        }
    }
    __device__ __forceinline__ void add(f32x16 &x) const {   // times log2 e
        if (!BIAS) return;
#pragma unroll
        for (int r = 0; r < 16; ++r) x[r] = fmaf(v[r], kLog2e, x[r]);
    }
};

__device__ __forceinline__ float other_half(float x) {   // max with it, or add it: which lane's comes first does not matter there
    const unsigned u = __float_as_uint(x);
    const auto s = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    return (threadIdx.x & 32) ? __uint_as_float(s[0]) : __uint_as_float(s[1]);
}

// (zero, or not a number where some result is infinite or none)
template <int DT>
__device__ __forceinline__ float finite_check(const f32x16 (&acc)[DT]) {
    float x = 0.0f;
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) x = fmaf(acc[t][r], 0.0f, x);
    return x;
}
// Whether a thread of the workgroup's says so (__syncthreads_or takes three times as long: 0.3 us of a call of 5).
template <int W>
__device__ __forceinline__ bool any_wave(bool x, float *red) {
    const bool mine = __any(x);
    if (threadIdx.x % 64 == 0) red[threadIdx.x / 64] = mine ? 1.0f : 0.0f;
    __syncthreads();
    float r = 0.0f;
#pragma unroll
    for (int w = 0; w < W; ++w) r += red[w];
    return uniform(r) != 0.0f;
}
// Which calls form products out of parts, all of a call's kernels or none (P and the LSE then have the same roundings; with two kinds dV of large scores
// was twice as far from 64 bits); the others stay on the fp32 instruction alone.  Head dim 128 has no registers for three parts of every operand.  Rows of up to
// 64, which two waves share: head dims 8 and 16 have little to multiply (S = 256, N = 64, H = 8 forward 13.9 and 15.1 us, in parts 15.5 and 16.4),
// at 64 the backward spills (171, 190).  Above 64 keys parts win at every head dim up to 64, whatever the registers: 131 forwards and steps of 65 to 1 000 keys take
// 0.55 to 0.87 of the instruction's time (S = 64, N = 256, H = 8 a step at D = 8 164 / 124 us with dK/dV at two waves per SIMD instead of four, D = 16 194 / 133, D = 64 472 / 391
// with 36 registers of dK/dV spilled).
constexpr bool splits(int D, int W) { return D == 32 || (D <= 64 && W > 2); }
template <int D, bool SPLITS> constexpr int shared_bytes() {
    // (the second forming writes none of the vote's words, which a wave may still be reading when another has begun with it)
    if constexpr (SPLITS) static_assert(DirectShared<D>::BYTES <= SplitShared<D>::BYTES - 64, "");
    return SPLITS ? SplitShared<D <= 64 ? D : 64>::BYTES : DirectShared<D>::BYTES;
}
// A kernel forms its results in parts and, where some result of the workgroup is then not finite, once more on the fp32 instruction: parts of an infinite
// operand, or of one that is beyond bf16's range when 2^24 times as large, are not numbers, where the value itself may give a number, or an infinite result.
// The same where a score's factors might not be whole (above).  `split` returns, for the whole workgroup, whether one or the other is so, and then has written nothing
// over an operand: these are read again, and O may lie where Q does, dQ where O does, dK and dV where K and V do (a workgroup writes only the rows it alone reads).
template <bool SPLITS, class A, class B>
__device__ __forceinline__ void either_way(A split, B direct) {
    if constexpr (SPLITS) {
        if (__builtin_expect(!split(), 1)) return;
    }
    direct();
}

// Forward: a wave has 32 queries (lane = query), the keys come by tiles.
template <int D, int W, bool BIAS>
__device__ __forceinline__ bool split_body_fwd(const EvoAttnParams &p, unsigned char *lds) {
    typedef Split<D> E;
    const SplitShared<D> sh{lds};
    const unsigned nqb = (p.N + 32 * W - 1) / (32 * W), bid = xcd_remap(blockIdx.x, gridDim.x);
    const Prob pr = walk_problem(p, bid / nqb);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), l = threadIdx.x % 64, li = l % 32, g = l / 32;
    const int row0 = (bid % nqb) * 32 * W + wave * 32, row = row0 + li, rowc = min(row, p.N - 1);
    const bool active = row0 < p.N;   // (uniform over the wave)
    const unsigned stride_n = (unsigned)p.stride_n, off = (unsigned)rowc * stride_n;
    const __amdgpu_buffer_rsrc_t krs = rows_of((const float *)p.k + pr.base, p), vrs = rows_of((const float *)p.v + pr.base, p);
    SplitStage<D, 64 * W> st;
    st.load(krs, vrs, stride_n, 0);
    f32x4 qv[E::NP];
    load_row<E, D>((const float *)p.q + pr.base, off, g, qv);
    unsigned mk = threadIdx.x < 32 ? mask_ask(p, pr.b, pr.s, threadIdx.x) : 0;
    E::clear(lds, 4 * 32, 64 * W);
    const float shift = uniform(block_shift<W>(p, pr.b, pr.s, sh.red()));
    const bool dead = shift != 0.0f;   // (of such a row the scores are the mask's)
    BiasAhead<BIAS, true> bias(p, pr.b, pr.h, rowc, dead, l);
    const float qscale = dead ? 0.0f : p.scale * kLog2e * kDown;
    const typename E::Frag q = E::frag(qv, qscale);
    const uint2 ones = ones3<bf16_t>(), none = make_uint2(0, 0);
    uint4 extra = g == 0 ? chunk_of(ones, none) : make_uint4(0, 0, 0, 0);   // against (mask, 1): adds mask - mf
    f32x16 acc[E::DT];
#pragma unroll
    for (int t = 0; t < E::DT; ++t) acc[t] = zero16();
    // Maximum (log2 units), what of it the extra step subtracts (not where it is so low that a score would be lost beside it), sum.
    float m = 0.0f, mf = 0.0f, sum = E::begin(qv, qscale);
    const int nt = (p.N + 31) / 32;
    for (int kt = 0; kt < nt; ++kt) {
        const int buf = kt & 1;
        st.put(sh.tile(buf, 0), sh.tile(buf, 1), kUp, kUp);
        if (threadIdx.x < 32) sh.chunk(buf)[threadIdx.x] = chunk_of(parts_of(mask_got(p, mk, kt * 32 + threadIdx.x, shift) * kLog2e), ones);
        __syncthreads();
        if (kt + 1 < nt) {
            st.load(krs, vrs, stride_n, (kt + 1) * 32);
            if (threadIdx.x < 32) mk = mask_ask(p, pr.b, pr.s, (kt + 1) * 32 + threadIdx.x);
        }
        if (!active) continue;
        f32x16 x = E::rows(sh.tile(buf, 0), l, q);
        bias.add(x);
        bias.ask(kt + 1);
        x = E::M::mma(as_operand(sh.chunk(buf)[li]), as_operand(extra), x);
        float top = x[0];
#pragma unroll
        for (int r = 1; r < 16; ++r) top = fmaxf(top, x[r]);
        top = fmaxf(top, other_half(top));
        // The sums are brought to a new maximum where it stands 2^8 above the old one (at the first tile, and in few others).
        if (kt == 0 || __any(top > 8.0f || m != mf)) {
            const float cand = fmaxf(top + mf, kMaskFloor * kLog2e);
            const float mn = kt == 0 || cand > m + 8.0f ? cand : m, sub = mn - mf;
            if (kt > 0) {
                const float alpha = fast_exp2(m - mn);
                sum *= alpha;
#pragma unroll
                for (int t = 0; t < E::DT; ++t) acc[t] *= alpha;
            }
#pragma unroll
            for (int r = 0; r < 16; ++r) x[r] -= sub;
            m = mn;
            mf = fabsf(mn) <= 65536.0f ? mn : 0.0f;
            if (g == 0) extra = chunk_of(ones, parts_of(-mf));
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            x[r] = fast_exp2(x[r]);
            sum += x[r];
        }
        E::cols(sh.tile(buf, 1), l, x, acc);
    }
    sum = both_halves(sum);
    if (__builtin_expect(any_wave<W>(active && !(fmaf(sum, 0.0f, finite_check(acc)) == 0.0f), sh.red()), 0)) return true;
    if (row < p.N) {
        const float inv = kDown / sum;
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
        if (g == 0) p.lse[pr.row0 + row] = fmaf(m, kLn2, logf(sum));
    }
    return false;
}
template <int D, int W, bool BIAS>
__global__ void __launch_bounds__(64 * W, D <= 32 && W >= 4 ? (W == 8 ? 4 : 3) : D <= 64 ? 2 : 1) f32_fwd(EvoAttnParams p, int vec) {
    __shared__ __align__(1024) unsigned char lds[shared_bytes<D, splits(D, W)>()];
    either_way<splits(D, W)>([&]() __attribute__((always_inline)) { return split_body_fwd<D, W, BIAS>(p, lds); },
                  [&]() __attribute__((always_inline)) { direct_fwd<D, W, BIAS>(p, vec, lds); });
}

// dQ: a wave has 32 queries, like the forward.  Also writes delta = rowsum(dO * O) unless the gate's pass has, and
// the mask shift of its (b, s) for the dBias kernel.
template <int D, int W, bool BIAS>
__device__ __forceinline__ bool split_body_dq(const EvoAttnParams &p, float *delta, float *shift_tab, int delta_given, unsigned char *lds) {
    typedef Split<D> E;
    const SplitShared<D> sh{lds};
    const unsigned nqb = (p.N + 32 * W - 1) / (32 * W), bid = xcd_remap(blockIdx.x, gridDim.x);
    const Prob pr = walk_problem(p, bid / nqb);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), l = threadIdx.x % 64, li = l % 32, g = l / 32;
    const int row0 = (bid % nqb) * 32 * W + wave * 32, row = row0 + li, rowc = min(row, p.N - 1);
    const bool active = row0 < p.N;
    const unsigned stride_n = (unsigned)p.stride_n, off = (unsigned)rowc * stride_n;
    const __amdgpu_buffer_rsrc_t krs = rows_of((const float *)p.k + pr.base, p), vrs = rows_of((const float *)p.v + pr.base, p);
    SplitStage<D, 64 * W> st;
    st.load(krs, vrs, stride_n, 0);
    f32x4 qv[E::NP], gv[E::NP];
    load_row<E, D>((const float *)p.q + pr.base, off, g, qv);
    load_row<E, D>((const float *)p.dout + pr.base, off, g, gv);
    const float lse = p.lse[pr.row0 + rowc];
    unsigned mk = threadIdx.x < 32 ? mask_ask(p, pr.b, pr.s, threadIdx.x) : 0;
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
    E::clear(lds, 4 * 32, 64 * W);
    const float shift = uniform(block_shift<W>(p, pr.b, pr.s, sh.red()));
    if (threadIdx.x == 0 && pr.h == 0 && bid % nqb == 0) shift_tab[pr.b * p.S + pr.s] = shift;
    const bool dead = shift != 0.0f;
    BiasAhead<BIAS, true> bias(p, pr.b, pr.h, rowc, dead, l);
    const float ll = ds_blocked(p, shift) ? kMaskFloor : -lse * kLog2e;   // (no gradient through replaced scores: dS is zero)
    const float qscale = dead ? 0.0f : p.scale * kLog2e * kDown;
    const typename E::Frag q = E::frag(qv, qscale), go = E::frag(gv, kUp);
    const uint2 ones = ones3<bf16_t>(), none = make_uint2(0, 0);
    const uint4 zero = make_uint4(0, 0, 0, 0), xs = g == 0 ? chunk_of(ones, parts_of(ll)) : zero, xd = g == 0 ? chunk_of(none, parts_of(-dl * kUp2)) : zero;   // against (mask, 1)
    f32x16 acc[E::DT];
#pragma unroll
    for (int t = 0; t < E::DT; ++t) acc[t] = zero16();
    acc[0][0] = E::begin(qv, qscale);
    const int nt = (p.N + 31) / 32;
    for (int kt = 0; kt < nt; ++kt) {
        const int buf = kt & 1;
        st.put(sh.tile(buf, 0), sh.tile(buf, 1), kUp, kUp);
        if (threadIdx.x < 32) sh.chunk(buf)[threadIdx.x] = chunk_of(parts_of(mask_got(p, mk, kt * 32 + threadIdx.x, shift) * kLog2e), ones);
        __syncthreads();
        if (kt + 1 < nt) {
            st.load(krs, vrs, stride_n, (kt + 1) * 32);
            if (threadIdx.x < 32) mk = mask_ask(p, pr.b, pr.s, (kt + 1) * 32 + threadIdx.x);
        }
        if (!active) continue;
        const bf16x8 row = as_operand(sh.chunk(buf)[li]);
        f32x16 x = E::rows(sh.tile(buf, 0), l, q);
        bias.add(x);
        bias.ask(kt + 1);
        x = E::M::mma(row, as_operand(xs), x);
        const f32x16 dp = E::M::mma(row, as_operand(xd), E::rows(sh.tile(buf, 1), l, go));
#pragma unroll
        for (int r = 0; r < 16; ++r) x[r] = fast_exp2(x[r]) * dp[r];
        E::cols(sh.tile(buf, 0), l, x, acc);
    }
    if (__builtin_expect(any_wave<W>(active && !(finite_check(acc) == 0.0f), sh.red()), 0)) return true;
    if (row < p.N) {
#pragma unroll
        for (int t = 0; t < E::DT; ++t)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int c = 32 * t + 8 * j + 4 * g;
                if (c >= D) continue;
                f32x4 o;
#pragma unroll
                for (int i = 0; i < 4; ++i) o[i] = acc[t][4 * j + i] * (p.scale * kDown3);
                put4((float *)p.dq + pr.base, off + c, o);
            }
    }
    return false;
}
template <int D, int W, bool BIAS>
__global__ void __launch_bounds__(64 * W, D <= 64 ? 2 : 1) f32_dq(EvoAttnParams p, int vec, float *delta, float *shift_tab, int delta_given) {
    __shared__ __align__(1024) unsigned char lds[shared_bytes<D, splits(D, W)>()];
    either_way<splits(D, W)>([&]() __attribute__((always_inline)) { return split_body_dq<D, W, BIAS>(p, delta, shift_tab, delta_given, lds); },
                  [&]() __attribute__((always_inline)) { direct_dq<D, W, BIAS>(p, vec, delta, shift_tab, delta_given, lds); });
}

// dK and dV: a wave has 32 keys (lane = key), the queries come by tiles with their dO, LSE and delta.  Also sums the dBias
// partials of the kernel before it (no launch of its own for that).
template <int D, int W, bool BIAS>
__device__ __forceinline__ bool split_body_dkdv(const EvoAttnParams &p, const Extra &e, unsigned char *lds) {
    typedef Split<D> E;
    const SplitShared<D> sh{lds};
    const unsigned nkb = (p.N + 32 * W - 1) / (32 * W), bid = xcd_remap(blockIdx.x, gridDim.x);
    const Prob pr = walk_problem(p, bid / nkb);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), l = threadIdx.x % 64, li = l % 32, g = l / 32;
    const int key0 = (bid % nkb) * 32 * W + wave * 32, key = key0 + li, keyc = min(key, p.N - 1);
    const bool active = key0 < p.N;
    const unsigned stride_n = (unsigned)p.stride_n, off = (unsigned)keyc * stride_n;
    const __amdgpu_buffer_rsrc_t qrs = rows_of((const float *)p.q + pr.base, p), grs = rows_of((const float *)p.dout + pr.base, p);
    SplitStage<D, 64 * W> st;
    st.load(qrs, grs, stride_n, 0);
    float lse = 0.0f, dl = 0.0f;   // of a stage's rows (the first 32 threads)
    auto ask_row = [&](int r0) {
        if (threadIdx.x >= 32) return;
        const int r = min(r0 + (int)threadIdx.x, p.N - 1);
        lse = p.lse[pr.row0 + r];
        dl = e.delta[pr.row0 + r];
    };
    ask_row(0);
    f32x4 kv[E::NP], vv[E::NP];
    load_row<E, D>((const float *)p.k + pr.base, off, g, kv);
    load_row<E, D>((const float *)p.v + pr.base, off, g, vv);
    E::clear(lds, 4 * 32, 64 * W);
    if (threadIdx.x == 0) *sh.one() = chunk_of(ones3<bf16_t>(), make_uint2(0, 0));
    const float shift = uniform(block_shift<W>(p, pr.b, pr.s, sh.red()));
    const bool dead = shift != 0.0f, blocked = ds_blocked(p, shift);   // (blocked: dP - delta is zero)
    BiasAhead<BIAS, false> bias(p, pr.b, pr.h, keyc, dead, l);
    const float mk = mask_entry(p, pr.b, pr.s, keyc, shift) * kLog2e;
    const float kscale = dead ? 0.0f : kDown;
    const typename E::Frag k = E::frag(kv, kscale), v = E::frag(vv, blocked ? 0.0f : kUp);
    const uint2 ones = ones3<bf16_t>(), none = make_uint2(0, 0);
    // against a row's chunk, (-LSE, -delta), and in the upper half's columns ones: LSE and mask; delta
    const uint4 zero = make_uint4(0, 0, 0, 0), xs = chunk_of(g == 0 ? ones : parts_of(mk), none), xd = g == 0 && !blocked ? chunk_of(none, ones) : zero;
    f32x16 dk[E::DT], dv[E::DT];
#pragma unroll
    for (int t = 0; t < E::DT; ++t) dk[t] = dv[t] = zero16();
    float dm = E::begin(kv, kscale);
    const int nt = (p.N + 31) / 32;
    for (int qt = 0; qt < nt; ++qt) {
        const int buf = qt & 1;
        st.put(sh.tile(buf, 0), sh.tile(buf, 1), p.scale * kLog2e * kUp, kUp);
        if (threadIdx.x < 32) {   // (rows at and beyond N: probability zero)
            const bool in = qt * 32 + (int)threadIdx.x < p.N;
            sh.chunk(buf)[threadIdx.x] = chunk_of(parts_of(in ? -lse * kLog2e : kMaskFloor), parts_of(in ? -dl * kUp2 : 0.0f));
        }
        __syncthreads();
        if (qt + 1 < nt) {
            st.load(qrs, grs, stride_n, (qt + 1) * 32);
            ask_row((qt + 1) * 32);
        }
        if (!active) continue;
        const bf16x8 row = as_operand(g == 0 ? sh.chunk(buf)[li] : *sh.one());
        f32x16 x = E::rows(sh.tile(buf, 0), l, k);
        bias.add(x);
        bias.ask(qt + 1);
        x = E::M::mma(row, as_operand(xs), x);
#pragma unroll
        for (int r = 0; r < 16; ++r) x[r] = fast_exp2(x[r]);
        E::cols(sh.tile(buf, 1), l, x, dv, kUp);
        f32x16 ds = E::M::mma(row, as_operand(xd), E::rows(sh.tile(buf, 1), l, v));
#pragma unroll
        for (int r = 0; r < 16; ++r) ds[r] *= x[r];
        if (p.dmask) {
#pragma unroll
            for (int r = 0; r < 16; ++r) dm += ds[r];
        }
        E::cols(sh.tile(buf, 0), l, ds, dk);
    }
    dm = both_halves(dm);
    if (__builtin_expect(any_wave<W>(active && !(fmaf(dm, 0.0f, finite_check(dk) + finite_check(dv)) == 0.0f), sh.red()), 0)) return true;
    if (key < p.N) {
        if (p.dmask && g == 0) e.dmask_part[pr.row0 + key] = dm * kDown2;
#pragma unroll
        for (int t = 0; t < E::DT; ++t)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int c = 32 * t + 8 * j + 4 * g;
                if (c >= D) continue;
                f32x4 a, o;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    a[i] = dk[t][4 * j + i] * (kLn2 * kDown3);   // (of Q as scaled)
                    o[i] = dv[t][4 * j + i] * kDown2;
                }
                put4((float *)p.dk + pr.base, off + c, a);
                put4((float *)p.dv + pr.base, off + c, o);
            }
    }
    return false;
}
template <int D, int W, bool BIAS>
__global__ void __launch_bounds__(64 * W, D <= 64 ? 2 : 1) f32_dkdv(EvoAttnParams p, Extra e) {
    __shared__ __align__(1024) unsigned char lds[shared_bytes<D, splits(D, W)>()];
    if (e.dbias_chunks) sum_dbias_partials<64 * W>(p, e, threadIdx.x);
    either_way<splits(D, W)>([&]() __attribute__((always_inline)) { return split_body_dkdv<D, W, BIAS>(p, e, lds); },
                  [&]() __attribute__((always_inline)) { direct_dkdv<D, W, BIAS>(p, e, lds); });
}

// dBias partials: a workgroup has a block of queries and keys of one (b, h), a wave 32 queries and KT key tiles of it, and walks over a chunk of S rows with
// the sums in registers.  Forms S and dP again (two products): next to the dQ kernel's three that costs less than
// the partial results of workgroups that kept dBias for all the keys of their queries (N = 256: as much time
// as 64 MB of partials take to write and sum).  Reads delta and the mask shifts that the dQ kernel wrote.
template <int D, int KT, bool SPLITS>
struct DBias : DBiasGeo<D, KT> {
    static constexpr int BLK = DBiasGeo<D, KT>::BLK, DIRECT = 4 * (BLK / 32) * Direct<D>::TILE + 3 * BLK * 4;
    static constexpr int CHUNKS = SPLITS ? 4 * (BLK / 32) * Split<D <= 64 ? D : 64>::TILE : 0, SPLIT = CHUNKS + (2 * BLK + 1) * 16 + 64;   // Q, dO, K, V; rows' and keys' chunks, ones, a value per wave
    static_assert(!SPLITS || D > 64 || DIRECT <= SPLIT - 64, "the second forming writes none of the vote's words");
    static constexpr int BYTES = SPLITS ? SPLIT : DIRECT;
};
template <int D, int KT, bool BIAS>
__device__ __forceinline__ bool split_body_dbias(const EvoAttnParams &p, const float *delta, const float *shift_tab, float *part, int chunk, unsigned char *lds) {
    typedef Split<D> E;
    typedef DBias<D, KT, true> R;
    constexpr int ROWS = R::BLK, TH = 64 * R::W, ARRAY = ROWS / 32 * E::TILE;
    uint4 *const qchunk = reinterpret_cast<uint4 *>(lds + R::CHUNKS), *const kchunk = qchunk + ROWS, *const one = kchunk + ROWS;
    const int nb = (p.N + ROWS - 1) / ROWS;
    unsigned t = xcd_remap(blockIdx.x, gridDim.x);
    const int kb = t % nb; t /= nb;
    const int qb = t % nb; t /= nb;
    const int h = t % p.H; t /= p.H;
    const int b = t % p.B, ck = t / p.B;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), l = threadIdx.x % 64, li = l % 32, g = l / 32;
    const int q0 = qb * ROWS, k0 = kb * ROWS, qw = (wave >> 1) * 32, kw = (wave & 1) * 32 * KT;
    const bool active = q0 + qw < p.N;
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
    const uint2 ones = ones3<bf16_t>(), none = make_uint2(0, 0);
    if (threadIdx.x == 0) *one = chunk_of(ones, none);
    SplitStage<D, TH, ROWS> sq;
    SplitStage<D, TH, ROWS, true> sk;
    float lse = 0.0f, dl = 0.0f, shift = 0.0f, next_shift = 0.0f;
    unsigned mk = 0;
    auto load = [&](int s) {
        const unsigned pid = ((unsigned)b * p.H + h) * p.S + s;
        const Prob pr = decode_problem(p, pid);
        sq.load(rows_of((const float *)p.q + pr.base, p), rows_of((const float *)p.dout + pr.base, p), (unsigned)p.stride_n, q0);
        sk.load(rows_of((const float *)p.k + pr.base, p), rows_of((const float *)p.v + pr.base, p), (unsigned)p.stride_n, k0);
        next_shift = __int_as_float(uniform_load((const int *)shift_tab + b * p.S + s));
        const int i = threadIdx.x;
        if (i < ROWS) {
            const int q = min(q0 + i, p.N - 1);
            lse = p.lse[pr.row0 + q];
            dl = delta[pr.row0 + q];
        } else if (i < 2 * ROWS) {
            mk = mask_ask(p, b, s, k0 + i - ROWS);
        }
    };
    static_assert(TH >= 2 * ROWS, "a thread for each row's and each key's chunk");
    if (D < 16) E::clear(lds, 4 * ROWS, TH);   // (no columns beyond 16 are read)
    load(s0);
    const bf16x8 xd = g == 0 ? as_operand(chunk_of(none, ones)) : zero8<bf16_t>();
    for (int s = s0; s < s1; ++s) {
        __syncthreads();
        shift = next_shift;
        const bool dead = shift != 0.0f;
        sq.put(lds, lds + ARRAY, dead ? 0.0f : p.scale * kLog2e * kDown, kUp);
        sk.put(lds + 2 * ARRAY, lds + 3 * ARRAY, kUp, kUp);
        {
            const int i = threadIdx.x;
            if (i < ROWS) qchunk[i] = chunk_of(parts_of(q0 + i < p.N ? -lse * kLog2e : kMaskFloor), parts_of(q0 + i < p.N ? -dl * kUp2 : 0.0f));
            else if (i < 2 * ROWS) qchunk[i] = chunk_of(parts_of(mask_got(p, mk, k0 + i - ROWS, shift) * kLog2e), none);   // (the keys': behind the rows')
        }
        __syncthreads();
        if (s + 1 < s1) load(s + 1);
        if (!active || ds_blocked(p, shift)) continue;
        const unsigned char *const qt = lds + qw / 32 * E::TILE, *const kt0 = lds + 2 * ARRAY + kw / 32 * E::TILE;
        // one more step for LSE and mask: (-LSE, -delta) against (1, 0) in its first eight columns, 1 against mask in the others
        const bf16x8 row = as_operand(g == 0 ? qchunk[qw + li] : *one);
#pragma unroll
        for (int kt = 0; kt < KT; ++kt) {
            if (k0 + kw + 32 * kt >= p.N) break;
            f32x16 x = E::rows(qt, l, E::staged(kt0 + kt * E::TILE, l));
            if (BIAS && !dead) {
#pragma unroll
                for (int r = 0; r < 16; ++r) x[r] = fmaf(bz[kt][r], kLog2e, x[r]);
            }
            x = E::M::mma(row, as_operand(g == 0 ? *one : kchunk[kw + 32 * kt + li]), x);
            const f32x16 dp = E::M::mma(row, xd, E::rows(qt + ARRAY, l, E::staged(kt0 + ARRAY + kt * E::TILE, l)));
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[kt][r] = fmaf(fast_exp2(x[r]), dp[r], acc[kt][r]);
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
            if (q < p.N) out[(int64_t)q * p.N] = acc[kt][r] * kDown2;
        }
    }
    return any_wave<R::W>(sk.huge != 0 || (active && !(finite_check(acc) == 0.0f)), reinterpret_cast<float *>(one + 1));   // (dBias lies where nothing is read any more; asked before the stores, 16 to 38 registers more)
}
template <int D, int KT, bool SPLITS, bool BIAS>
__global__ void __launch_bounds__((64 * DBiasGeo<D, KT>::W), D <= 64 ? 2 : 1) f32_dbias(EvoAttnParams p, const float *delta, const float *shift_tab, float *part, int chunk) {
    extern __shared__ __align__(1024) unsigned char dbias_lds[];
    either_way<SPLITS>([&]() __attribute__((always_inline)) { return split_body_dbias<D, KT, BIAS>(p, delta, shift_tab, part, chunk, dbias_lds); },
                  [&]() __attribute__((always_inline)) { direct_dbias<D, KT, BIAS>(p, delta, shift_tab, part, chunk, dbias_lds); });
}

// ---------------------------------------------------------------- host side

#define EVO_LAUNCH_CHECK()                                    \
    do {                                                      \
        hipError_t e_ = hipGetLastError();                    \
        if (e_ != hipSuccess) return EVO_EHIP - (int)e_;      \
    } while (0)

template <int D, int W, bool BIAS>
static int fwd_launch(const EvoAttnParams &p, int vec, hipStream_t st) {
    const unsigned grid = (unsigned)((p.N + 32 * W - 1) / (32 * W)) * (unsigned)(p.B * p.H * p.S);
    f32_fwd<D, W, BIAS><<<grid, 64 * W, 0, st>>>(p, vec);
    EVO_LAUNCH_CHECK();
    return EVO_OK;
}

// The dBias kernel's blocks: 64 queries and keys, or 128, whose rows are split half as often, where they fit the LDS and a row is longer than 64.
static int dbias_block(const EvoAttnParams &p) { return p.D <= 32 && p.N > 64 ? 128 : 64; }

template <int D, int KT, bool SPLITS, bool BIAS>
static int dbias_launch(const EvoAttnParams &p, const Extra &e, float *out, hipStream_t st) {
    typedef DBias<D, KT, SPLITS> R;
    static PerDevice done;
    if (R::BYTES > 64 * 1024)   // (more dynamic LDS than a launch may ask for unannounced)
        if (const int rc = ensure_dynamic_lds((const void *)&f32_dbias<D, KT, SPLITS, BIAS>, R::BYTES, done, nullptr)) return rc;
    const unsigned nb = (p.N + R::BLK - 1) / R::BLK;
    f32_dbias<D, KT, SPLITS, BIAS><<<nb * nb * (unsigned)(p.B * p.H * e.n_chunks), 64 * R::W, R::BYTES, st>>>(p, e.delta, e.shift, out, e.chunk);
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
        const bool direct = e.n_chunks == 1 && p.dbias_dtype == EVO_F32;
        float *const out = direct ? (float *)p.dbias : e.dbias_part;
        if (const int rc = dbias_launch<D, (D <= 32 && W > 2) ? 2 : 1, splits(D, W), BIAS>(p, e, out, st)) return rc;   // (W follows N as `dbias_block` does)
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

// Waves, of 32 rows each, that share what a workgroup stages: two for short rows, else four; eight in a forward of more than 128 queries and more than 384 workgroups so:
// twice as many of four waves are more than three on each of 256 CUs, what fits at once, while two of eight fit there.  us, H = 4, workgroups of eight waves 320 / 384 / 448 / 512,
// D = 32, N = 256: eight 31 / 33 / 34 / 36, four 28 / 30 / 37 / 39; N = 1 000 97 / 101 / 109 / 112 and 87 / 93 / 119 / 124; D = 8, N = 250 30 / 30 / 30 / 30 and 25 / 25 / 34 / 34; D = 64, N = 400
// 73 / 74 / 75 / 79 and 65 / 66 / 79 / 83.  (193 to 256, one each: eight 4 to 13 % faster at D = 8 and 64, 0 to 9 at 32.  The backward: S = 64, N = 256, H = 8 161 / 154.)
template <int D, bool FWD, class F>
static int by_rows(const EvoAttnParams &p, F go) {
    auto with = [&](auto w) { return p.bias_dtype != EVO_NONE ? go(w, std::true_type()) : go(w, std::false_type()); };
    if (p.N <= 64) return with(std::integral_constant<int, 2>());
    if constexpr (FWD && D <= 64)
        if (p.N > 128 && (int64_t)((p.N + 255) / 256) * p.B * p.H * p.S > 384) return with(std::integral_constant<int, 8>());
    return with(std::integral_constant<int, 4>());
}
#define EVO_F32_DISPATCH(FWD, fn, ...) \
    switch (p.D) { \
        case 8: return by_rows<8, FWD>(p, [&](auto w, auto b) { return fn<8, decltype(w)::value, decltype(b)::value>(__VA_ARGS__); }); \
        case 16: return by_rows<16, FWD>(p, [&](auto w, auto b) { return fn<16, decltype(w)::value, decltype(b)::value>(__VA_ARGS__); }); \
        case 32: return by_rows<32, FWD>(p, [&](auto w, auto b) { return fn<32, decltype(w)::value, decltype(b)::value>(__VA_ARGS__); }); \
        case 64: return by_rows<64, FWD>(p, [&](auto w, auto b) { return fn<64, decltype(w)::value, decltype(b)::value>(__VA_ARGS__); }); \
        case 128: return by_rows<128, FWD>(p, [&](auto w, auto b) { return fn<128, decltype(w)::value, decltype(b)::value>(__VA_ARGS__); }); \
    } \
    return EVO_EUNSUPPORTED

static int bias_rows_vec(const EvoAttnParams &p) {
    return p.bias && p.N >= 4 && p.N % 4 == 0 && (uintptr_t)p.bias % 16 == 0 && p.bias_stride_b % 4 == 0 && p.bias_stride_h % 4 == 0 &&
           p.bias_stride_row % 4 == 0;
}

int launch_f32_fwd(const EvoAttnParams &p, hipStream_t st) {
    const int vec = bias_rows_vec(p);
    EVO_F32_DISPATCH(true, fwd_launch, p, vec, st);
}

int launch_f32_bwd(const EvoAttnParams &p, const Extra &e, hipStream_t st) {
    const int vec = bias_rows_vec(p);
    EVO_F32_DISPATCH(false, bwd_launch, p, e, vec, st);
}

// Chunks of S rows for the dBias kernel: about 1024 blocks of 64 rows, 256 of 128, at a time, no more than there are rows.
int f32_dbias_chunks(const EvoAttnParams &p) {
    const int64_t blk = dbias_block(p), nb = (p.N + blk - 1) / blk, base = nb * nb * p.B * p.H, all = blk == 128 ? 256 : 1024;
    const int64_t want = (all + base - 1) / base;
    return (int)(want < p.S ? want : p.S);
}

}  // namespace evo
