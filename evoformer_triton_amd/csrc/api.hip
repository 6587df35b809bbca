// C ABI of the library: parameter validation, workspace layout and kernel dispatch.
// Everything in this file runs on the host; nothing here needs a GPU except the two
// enqueue entry points.
#include <atomic>

#include "common.h"
#include "kernels.h"

// Prepared operands of evoattn_fwd_static: one array per GPU the library runs on, held until the
// process ends.  In host code the name stands for the symbol only; the array's device address is
// asked for once per device (static_prep below) and only that address is handed to kernels.
static __device__ __align__(256) unsigned char scratch[EVOATTN_STATIC_PREP_BYTES];

namespace evo {

static inline size_t align_up(size_t x, size_t a = 256) { return (x + a - 1) / a * a; }
static inline bool aligned(const void *p, size_t a) { return ((uintptr_t)p % a) == 0; }
static inline int elem_size(int dtype) { return dtype == EVO_F32 ? 4 : 2; }


// Elements from the first to one past the last element of a q-family tensor (= B*H*S*N*D when it is dense).
static int64_t q_span(const EvoAttnParams &p) {
    const int64_t st4[4] = {p.stride_b, p.stride_h, p.stride_s, p.stride_n};
    const int64_t ext[4] = {p.B, p.H, p.S, p.N};
    int64_t span = p.D;
    for (int i = 0; i < 4; ++i) span += (ext[i] - 1) * st4[i];
    return span;
}

static int check_common(const EvoAttnParams *p) {
    if (!p) return EVO_EINVAL;
    if (p->B <= 0 || p->S <= 0 || p->N <= 0 || p->H <= 0 || p->D <= 0) return EVO_EINVAL;
    if (p->dtype != EVO_BF16 && p->dtype != EVO_F16 && p->dtype != EVO_F32) return EVO_EINVAL;
    if (p->bias_dtype != EVO_NONE && p->bias_dtype != EVO_F32 && p->bias_dtype != p->dtype) return EVO_EINVAL;
    if (p->mask_kind < EVO_MASK_NONE || p->mask_kind > EVO_MASK_F16) return EVO_EINVAL;
    if ((p->bias_dtype == EVO_NONE) != (p->bias == nullptr)) return EVO_EINVAL;
    if ((p->mask_kind == EVO_MASK_NONE) != (p->mask == nullptr)) return EVO_EINVAL;
    if (!p->q || !p->k || !p->v || !p->lse) return EVO_EINVAL;
    // (with a gate the gated output may stand alone: the forward then writes no ungated O and the backward,
    // whose gate pass forms delta from the gated output, reads none)
    if (!p->o && !(p->gate && p->o_gated)) return EVO_EINVAL;
    if (!(p->scale == p->scale) || p->scale <= 0.0f) return EVO_EINVAL;
    if (p->flags & ~EVO_FLAG_ALL) return EVO_EINVAL;
    // (a second call on the same dout would apply the gate to it a second time)
    if ((p->flags & EVO_FLAG_GATE_DOUT_INPLACE) && (p->flags & (EVO_FLAG_ONLY_DQ | EVO_FLAG_ONLY_DKDV))) return EVO_EINVAL;
    if (p->gate) {
        // The gate is read and its products written element for element like q; the backward keeps the gradient
        // of the ungated output in the workspace, laid out like q, gaps included: the q-family may be dense or a
        // slot of a buffer of up to 8 such tensors (Q, K, V and the gate as one projection's result), not sparser.
        if (p->D % 8 || p->H > 256) return EVO_EUNSUPPORTED;   // (the gate's backward pass keeps 128 bytes of LDS per head)
        if (q_span(*p) > 8 * (int64_t)p->B * p->H * p->S * p->N * p->D) return EVO_EUNSUPPORTED;
    } else if (p->o_gated || p->dgate) {
        return EVO_EINVAL;
    }
    if (p->D != 8 && p->D != 16 && p->D != 32 && p->D != 64 && p->D != 128) return EVO_EUNSUPPORTED;
    if (p->stride_b < 0 || p->stride_h < 0 || p->stride_s < 0 || p->stride_n < p->D) return EVO_EINVAL;
    if (p->bias && (p->bias_stride_b < 0 || p->bias_stride_h < 0 || p->bias_stride_row < p->N)) return EVO_EINVAL;
    if (p->mask && (p->mask_stride_b < 0 || p->mask_stride_s < 0)) return EVO_EINVAL;
    // index ranges: problems and rows are 32-bit in the kernels, element offsets 64-bit
    const int64_t probs = (int64_t)p->B * p->H * p->S;
    if (probs > (int64_t)1 << 26 || (int64_t)p->N > (int64_t)1 << 20) return EVO_EOVERFLOW;
    if (probs * ((p->N + 31) / 32) > (int64_t)0x7fffffff) return EVO_EOVERFLOW;
    if ((int64_t)p->B * p->H * p->N * ((p->N + 63) / 64) > (int64_t)0x7fffffff) return EVO_EOVERFLOW;
    const int es = elem_size(p->dtype);
    if (!aligned(p->q, es) || !aligned(p->k, es) || !aligned(p->v, es) || !aligned(p->o, es) || !aligned(p->lse, 4))
        return EVO_EALIGN;
    if (p->bias && !aligned(p->bias, elem_size(p->bias_dtype))) return EVO_EALIGN;
    if (p->gate) {
        // The gate's kernels move rows in 8- and 16-byte pieces whichever attention kernels run: every tensor laid out
        // like q starts on a 16-byte boundary and every stride is a whole number of such pieces (o_gated may be NULL
        // in a backward call, o in any call).
        const int64_t per16 = 16 / es;
        if (p->stride_b % per16 || p->stride_h % per16 || p->stride_s % per16 || p->stride_n % per16) return EVO_EALIGN;
        if (!aligned(p->gate, 16) || !aligned(p->o_gated, 16) || !aligned(p->o, 16)) return EVO_EALIGN;
    }
    if (p->mask_kind == EVO_MASK_F32 && !aligned(p->mask, 4)) return EVO_EALIGN;
    if ((p->mask_kind == EVO_MASK_BF16 || p->mask_kind == EVO_MASK_F16) && !aligned(p->mask, 2)) return EVO_EALIGN;
    return EVO_OK;
}

// The matrix-core kernels read rows with 16-byte loads and keep one 32-wide key tile per
// 16 accumulator registers in the dBias kernel (at most 16 tiles per wave, 4 waves).
static bool long_rows_bwd_ok(const EvoAttnParams &p);
static bool mfma_ok(const EvoAttnParams &p, int pass) {
    if (p.flags & EVO_FLAG_FORCE_GENERIC) return false;
    if (p.dtype != EVO_BF16 && p.dtype != EVO_F16) return false;
    if (p.D != 8 && p.D != 16 && p.D != 32 && p.D != 64 && p.D != 128) return false;
    if (p.stride_b % 8 || p.stride_h % 8 || p.stride_s % 8 || p.stride_n % 8) return false;
    // (the kernels address the rows of one (b, h, s) problem by 32-bit byte offsets from its first row, also the rows
    // up to the next multiple of 256 beyond N, which their buffer loads must find out of range rather than wrapped)
    if (((int64_t)(p.N + 511) * p.stride_n + p.D) * 2 >= ((int64_t)1 << 31)) return false;
    if (!aligned(p.q, 16) || !aligned(p.k, 16) || !aligned(p.v, 16) || !aligned(p.o, 16)) return false;
    if (pass == EVO_PASS_BWD) {
        if (p.N > 2048 && !long_rows_bwd_ok(p)) return false;
        if (!aligned(p.dout, 16) || !aligned(p.dq, 16) || !aligned(p.dk, 16) || !aligned(p.dv, 16)) return false;
    }
    return true;
}

// fp32 on the matrix core (f32.hip): rows and their strides in whole 16-byte pieces.  Anything else in fp32 (and 16-bit tensors at odd addresses) takes the plain
// kernels, one row per thread on the vector ALU.
static bool f32_ok(const EvoAttnParams &p, int pass) {
    if (p.dtype != EVO_F32 || (p.flags & EVO_FLAG_FORCE_GENERIC)) return false;
    if (p.stride_b % 4 || p.stride_h % 4 || p.stride_s % 4 || p.stride_n % 4) return false;
    if (!aligned(p.q, 16) || !aligned(p.k, 16) || !aligned(p.v, 16) || !aligned(p.o, 16)) return false;
    // (a problem's rows, whole tiles of them, and a bias matrix lie within 32-bit byte offsets)
    if ((int64_t)(p.N + 64) * p.stride_n + p.D >= ((int64_t)1 << 30)) return false;
    if (p.bias && (int64_t)p.N * p.bias_stride_row >= ((int64_t)1 << 30)) return false;
    const int64_t nb = (p.N + 63) / 64;
    if (pass == EVO_PASS_BWD) {
        if (!aligned(p.dout, 16) || !aligned(p.dq, 16) || !aligned(p.dk, 16) || !aligned(p.dv, 16)) return false;
        if (p.dbias && nb * nb * p.B * p.H * f32_dbias_chunks(p) > (int64_t)0x7fffffff) return false;
    }
    return true;
}

static int bias_vec_ok(const EvoAttnParams &p) {
    if (!p.bias) return 0;
    const size_t a = p.bias_dtype == EVO_F32 ? 16 : 8;
    return aligned(p.bias, a) && p.bias_stride_b % 4 == 0 && p.bias_stride_h % 4 == 0 && p.bias_stride_row % 4 == 0;
}

// The prepared bias tiles (two copies in accumulator order, fp32 or, for a bias in the dtype of q,
// 16 bits per entry) cost 6 to 12 bytes of memory traffic per bias entry before any kernel has
// used one; each kernel then reads 2 or 4 bytes per entry and S row.  With very few S rows per (batch, head) - the reference's own speed benchmark has one -
// the one-workgroup-per-problem kernels read the caller's tensor instead, which needs rows that
// allow 16-byte (fp32) or 8-byte loads.  EVO_FLAG_DEBUG_BIAS_TILES keeps the tiles, for comparison.
//
// One S row of an fp32 bias whose rows start or end within a group of four (any length that is no multiple of 4): the kernels for head
// dim 64 read these in place too, and the tiles, which nobody then needs, are most of such a call.  Forward and backward, us, H = 32, tiles / in place: B = 1, N = 251
// 55 / 36, 517 101 / 78, 1023 284 / 158; B = 2, N = 771 357 / 216; B = 4, N = 517 362 / 211, 1023 1116 / 633 (N = 1024: 525).
// Fewer than 32 workgroups keep the tiles: their backward is another kernel's.  (The forward, which decides, does not know whether dBias will be wanted: without it, and with a
// gate, such a backward is one launch as well, see bwd_one_ok.)
static bool bias_ragged(const EvoAttnParams &p) {
    if (!p.bias || p.S != 1 || p.D != 64 || p.bias_dtype != EVO_F32 || p.dtype == EVO_F32 || (p.flags & EVO_FLAG_DEBUG_BIAS_TILES)) return false;
    if ((p.N % 4 == 0 && bias_vec_ok(p)) || p.N < 4 || (int64_t)p.N * p.bias_stride_row >= ((int64_t)1 << 31)) return false;
    return (int64_t)((p.N + 127) / 128) * p.B * p.H >= 32;
}
static bool bias_direct(const EvoAttnParams &p) {
    if (bias_ragged(p)) return true;
    if (!p.bias || p.S > 4 || (p.flags & EVO_FLAG_DEBUG_BIAS_TILES) || p.N % 4) return false;
    // The 16-bit tiles of a bias in the dtype of q are cheap to prepare (2 + 4 bytes of traffic per entry at
    // streaming rate) and pay from the first S row on where the score work per entry is small: they are taken
    // for rows beyond 256 keys unless S = 1 at head dim 64 or more (whole step, us, tiles against the caller's
    // tensor: H = 8, D = 32, N = 1024, S = 1 / 2 / 4 103 / 111 / 151 against 121 / 142 / 189; N = 2048 210 / 357 / 444
    // against 244 / 418 / 545; B = 4, H = 32, D = 64, N = 1024, S = 1 / 2 / 4 596 / 1383 / 2320 against 536 / 1528 /
    // 2718; up to 256 keys the tiles would bring the chunk-of-rows kernels, which need more S rows: 49 against
    // 40 us at S = 4).  An fp32 bias keeps the direct reads up to 4 rows (S = 1: 257 against 140 us).
    if (p.bias_dtype == p.dtype && p.dtype != EVO_F32 && p.N > 256 && !(p.S == 1 && p.D >= 64)) return false;
    // beyond 2048 keys a dBias summed over several S rows needs the kernel that reads prepared tiles
    // (decided without looking at dbias: the forward, which prepares, has none)
    if (p.N > 2048 && p.S > 1) return false;
    if (p.bias_dtype != EVO_F32 && p.bias_dtype != p.dtype) return false;
    if ((int64_t)p.N * p.bias_stride_row >= ((int64_t)1 << 31)) return false;   // 32-bit offsets inside one (b, h) matrix
    return bias_vec_ok(p) != 0;
}

// The dQ kernel that double-buffers its operands in LDS takes rows of limited length.
static bool dq_ring_ok(const EvoAttnParams &p) {
    return !(p.flags & EVO_FLAG_PER_PROBLEM) && !bias_direct(p) && mfma_dqr_qrows(p.D, p.N) > 0;
}

// Where dBias is not a sum over S rows (no bias, one that takes no gradient, or S = 1, where
// dBias is dS itself) nothing ties a wave of the dQ kernel to a key tile for a chunk of S rows:
// the kernel whose waves own their query rows for all keys takes those problems, and with
// S = 1 writes dBias as it goes (no partials, no reduction).  Its workgroups take 128 query
// rows each and walk over the keys one tile after the other: with very few of them the
// kernels that split a row's keys over the waves finish sooner (N = 300, 6 workgroups: 10.4 us
// against 8.2 us).  EVO_FLAG_DEBUG_NO_DQ_WIDE selects the other kernels, for comparison.
static bool dq_wide_grid_ok(const EvoAttnParams &p) {
    if (bias_ragged(p)) return true;   // (the other dQ kernels read such rows as tiles, which are not made)
    return !(p.flags & (EVO_FLAG_PER_PROBLEM | EVO_FLAG_DEBUG_NO_DQ_WIDE)) && (int64_t)((p.N + 127) / 128) * p.B * p.H * p.S >= 32;
}

// Long rows with a dBias to sum: either the dQ kernel over a chunk of rows, which keeps the sums of its key
// tiles next to dQ (up to 512 keys with two query tiles per workgroup or in one or two stages, beyond in
// blocks of 256 keys with one query tile), or dQ from the kernel whose waves own their query rows for all keys
// and the dBias partials from a kernel of their own that forms dS a second time.  The pair is taken where
// the one kernel has no form (beyond 768 keys; head dim 64 beyond 128 keys; head dim 8 beyond 512) and, between
// 513 and 768 keys, where the row leaves the one kernel's last 256-key block mostly empty.  dQ with dBias, bf16, one kernel / the
// pair (at head dim 32 stream_dq and mfma_dbias), us: H = 4, head dim 32: N = 320 (S = 128) 40 / 58; N = 352, 448, 480, 512
// (S = 256) 79 / 104, 146 / 161, 155 / 169, 158 / 178; N = 576, 704, 736, 768 267 / 250, 363 / 358, 367 / 374, 378 / 390; N = 640
// (B = 2) 650 / 565; S = N = 768 1119 / 1156; head dim 16, H = 8, S = 512: N = 576, 640, 704 881 / 838, 1003 / 915, 1145 / 1196.
// At head dim 128 the one kernel is the one-workgroup-per-problem form, one workgroup per CU without a prefetch: H = 4, N = 512,
// S = 64 241 / 152, N = 201, S = 32 54 / 35.
// EVO_FLAG_DEBUG_NO_DQ_SPLIT selects the one kernel, for comparison.
static bool dq_split_ok(const EvoAttnParams &p) {
    if (p.D == 128 && p.N > 2048) return false;   // (rows that long keep the plain kernels at that head dim)
    const int min_n = p.D == 128 ? 32 : p.D == 64 ? 128 : 512;
    const int rem = p.N % 256;
    const bool full_blocks = rem == 0 || rem >= (p.D == 32 ? 224 : 192);
    const bool ring = dq_ring_ok(p);
    if (full_blocks && ring) return false;
    // Fewest S rows: the second kernel's start-up has to pay.  Where the one kernel over a chunk of rows has no form, against the
    // one-workgroup-per-problem dQ kernel (dQ with dBias, us, that kernel / the pair): D = 8, H = 8, N = 768, S = 8 / 16 / 32 46 / 50,
    // 92 / 70, 158 / 102; D = 64, H = 4, N = 1024, S = 8 / 16 / 32 89 / 56, 152 / 78, 274 / 152; N = 300, S = 16 / 32 29 / 26, 47 / 33;
    // N = 130, S = 64 32 / 27; and from 1024 keys on from 2 rows: D = 32, H = 8, N = 1024, S = 2 / 4 / 7 35 / 38, 65 / 42, 100 / 53;
    // N = 2048, S = 4 / 7 215 / 114, 362 / 175 (at N = 640..768 with S = 5, 6 the one kernel stays ahead, whole step 76 / 103
    // against 88 / 111).  Beyond 2048 keys that kernel has no form either.
    const int min_s = p.D == 128 ? 2 : p.N >= 1024 ? 2 : !ring ? (p.D == 64 ? 16 : 8) : p.D == 32 && p.N > 512 ? 8 : 64;
    if (!p.dbias || p.S < min_s || p.N <= min_n || (p.flags & EVO_FLAG_DEBUG_NO_DQ_SPLIT) || bias_direct(p) || !dq_wide_grid_ok(p)) return false;
    return p.bias_dtype == p.dtype || p.bias_dtype == EVO_F32;   // (the dBias kernel keeps 16-bit pairs or fp32 tiles)
}

// dQ, dK and dV from one kernel (head dims 32 and 8), dBias, where it is wanted, from the kernel that forms dS for it alone.  The scores and dS, which
// two kernels would form, are formed once, or with dBias twice instead of three times.  Backward, bf16, us, the kernels otherwise / this way:
//   no dBias     H = 8: N = 96, S = 256 40 / 34; N = 128, S = 48, 256 14 / 11, 54 / 43; N = 256, S = 48, 128, 256 36 / 25, 68 / 50, 116 / 94; N = 384,
//                S = 256 263 / 196; N = 768, S = 192 668 / 495; N = 2048, S = 192 4305 / 3528
//   with dBias   N = 256 stays with the kernels over a chunk of rows, whose dBias comes with dQ: S = 128 78 / 83; S = 512, N = 300 489 / 482, N = 320,
//                H = 4 149 / 152; N = 340, S = 160 168 / 159; N = 384, S = 256 313 / 292; N = 400, S = 128 232 / 186; N = 512, S = 192 431 / 353;
//                N = S = 768, H = 4 1793 / 1497; N = 1024, S = 192 1649 / 1280
// A problem is one workgroup's, two at a time on each of 256 CUs, so what counts beside is how full its last half round is.  H = 8, S = 48
// (three quarters), 56, 64 (full), 65 (two thirds), 75: N = 512 81 / 70, 92 / 73, 101 / 78, 114 / 109, 121 / 109; N = 2048 1091 / 963, 1265 /
// 1066, 1448 / 1156, 1494 / 1568, 1701 / 1582; with dBias N = 512 109 / 111, 126 / 119, 139 / 127, 152 / 162, 165 / 165; N = 1024 410 / 364,
// 471 / 392, 531 / 438, 561 / 549, 633 / 580.  From 321 to 384 keys, where the gain is least, only whole rounds of at least 1024 problems.
// Head dim 8, H = 8 (up to 384 keys are one block there):
//   no dBias     S = 32, 128, 1024: N = 64 9 / 7, 11 / 11, 58 / 62 (left out); N = 96 10 / 7, 14 / 13, 74 / 71; N = 192 14 / 10, 32 / 23, 215 / 152; N = 384
//                27 / 20, 84 / 54, 663 / 400; N = 1024 135 / 120, 503 / 352, 4190 / 2896; S = 65 N = 256 28 / 25, N = 1024 275 / 249
//   with dBias   N = 192, S = 128, 1024 48 / 53, 289 / 283 (left out); N = 300, S = 64, 65, 96, 256 56 / 56, 58 / 65, 74 / 73, 166 / 156; N = 384
//                66 / 66, 69 / 79, 91 / 87, 206 / 185, S = 1024 774 / 706; N = 512, S = 64, 256 99 / 98, 329 / 321; from 513 keys on the pair of kernels for dQ
//                stands against it: N = 768, S = 32, 65, 256 160 / 150, 279 / 251, 886 / 683; N = 1024, S = 32, 1024 212 / 199, 6352 / 4888
//
// Over sizes drawn at random (some 5000 backwards, heads times batches from 1 to 128) some calls were slower than with the other kernels, and are
// left to them:
//   Rows of several blocks (from 513 keys on, head dim 8 385 without dBias) are also padded to whole blocks, up to 1.3 times, and share 512 workgroups. `fused_share`
//   is the part of the rounds' slots, a last half round at .62, that works on keys that exist.  Median and most of this way / otherwise where it is just
//   below the lines here, and just above: head dim 32 without dBias 1.03, 1.22 and .93, 1.06 up to 768 keys, 1.01, 1.16 and .94, 1.07 up to 1024, 1.01, 1.07 and .90, 1.03
//   beyond; with it .97, 1.06 and .96, .99; head dim 8 .96, 1.06 and .91, 1.04 up to 768 keys, 1.05, 1.17 and .91, 1.03 beyond.  (H = 8, S = 73, N = 784, head dim 32 246 / 298 us.)
//   With dBias and up to 384 keys, where the other way is one kernel whose dBias comes with dQ, few S rows per head leave this one's second kernel with partial sums of a row or
//   two each: up to 64 rows 1.06, 1.58 (B = 2, S = 24, N = 377, H = 16, D = 8 109 / 172), from 65 on .93, 1.06.  One head alone at head dim 8 1.05, 1.09;
//   an fp32 bias of one or two heads at head dim 32 1.03, 1.05.
static double fused_share(const EvoAttnParams &p) {
    const int64_t problems = (int64_t)p.B * p.H * p.S, rest = problems % 512;
    const double rounds = (double)(problems / 512) + (rest == 0 ? 0.0 : rest <= 256 ? 0.62 : 1.0);
    return (double)problems / 512.0 / rounds * p.N / (mfma_fused_blocks(p) * mfma_fused_keys(p));
}
static bool fused_ok(const EvoAttnParams &p) {
    constexpr int apart = EVO_FLAG_PER_PROBLEM | EVO_FLAG_ONLY_DQ | EVO_FLAG_ONLY_DKDV | EVO_FLAG_DEBUG_NO_KV_RING | EVO_FLAG_DEBUG_NO_DQ_WIDE |
                          EVO_FLAG_DEBUG_NO_DQ_SPLIT | EVO_FLAG_DEBUG_OTHER_WIDTH;
    if ((p.flags & apart) || (p.dtype != EVO_BF16 && p.dtype != EVO_F16) || (p.D != 32 && p.D != 8) || p.gate || p.dmask || bias_direct(p)) return false;
    if (p.N < 96 || p.N > 2048) return false;
    if (p.dbias && !p.bias) return false;   // (the dBias kernel keeps bias tiles; dBias without a bias, the sum of dS alone, comes with dQ)
    const int64_t problems = (int64_t)p.B * p.H * p.S;
    const double full = (double)problems / (double)((problems + 255) / 256 * 256);
    const double share = fused_share(p);
    const int heads = p.B * p.H;
    if (p.D == 8) {
        if (problems < 256) return false;
        if (p.N > (p.dbias ? 512 : 384)) return (!p.dbias || p.S >= 8) && share >= (p.N > 768 ? 0.54 : 0.48);
        if (!p.dbias) return true;
        return p.N >= 288 && problems >= 768 && full >= 0.9 && (p.N > 384 ? p.S >= 8 : p.S > 64 && heads > 1);
    }
    if (problems < 384) return false;
    if (!p.dbias) return p.N <= 512 ? full >= 0.7 : share >= (p.N <= 768 ? 0.66 : p.N <= 1024 ? 0.7 : 0.75);
    if (p.S < 8 || p.N <= 320) return false;
    if (p.N <= 384) return problems >= 1024 && full >= 0.95 && p.S > 64 && (p.bias_dtype == p.dtype || heads > 2);
    return full >= (p.N > 768 ? 0.75 : 0.85) && share >= 0.58;
}

static bool dq_wide_ok(const EvoAttnParams &p) {
    // (without a bias that kernel has no form that writes dS)
    return dq_wide_grid_ok(p) && (!p.dbias || (p.S == 1 && p.bias) || dq_split_ok(p));
}
// Rows of more than 2048 keys: the dQ kernels that keep the dBias sums of a wave's key tiles in
// registers have no form that long (16 tiles per wave would be the whole register file).  The
// backward still runs on the matrix core where dQ comes from the kernel without those sums:
// no dBias asked for, S = 1, or the dBias kernel of its own (bias in the dtype of q).
static bool long_rows_bwd_ok(const EvoAttnParams &p) { return dq_wide_ok(p); }
static bool dq_writes_dbias(const EvoAttnParams &p) { return p.dbias && p.S == 1 && dq_wide_ok(p); }

// One S row, its bias read from the caller's tensor, head dim 64: dQ (which writes dBias) and dK/dV from one launch.  512 workgroups are on the chip
// at a time: where each kernel has just one full round of them nothing is left to fill, and two kinds of different length end less
// evenly.  H = 32, fp32 bias, forward and backward, us, two launches / one: B = 4, N = 384 (384 workgroups of each) 95 / 90, B = 2, N = 768 (384) 175 / 169,
// 896 (448) 224 / 221, 1024 (512) 292 / 297, B = 4, N = 512 (512) 133 / 138, 640 (640) 270 / 242, 768 347 / 324, 896 473 / 424, 1024 (1024) 582 / 525.
// Rows that start or end within a group of four are one launch also without dBias and with a gate.  Forward and backward over some 2700 random sizes against the
// prepared tiles that such rows had before, median and most: two launches 32 workgroups 1.19, 1.29, 64 1.06, 1.22 (with a gate 1.11, 1.25 and 1.06,
// 1.18), one launch .84, .96 and .82, .92 (.89, .98 and .89, .96); B = 1, N = 129, H = 16 without dBias 28.0 (tiles) / 36.0 (two) / 26.3 us.
static bool bwd_one_ok(const EvoAttnParams &p) {
    constexpr int apart = EVO_FLAG_PER_PROBLEM | EVO_FLAG_ONLY_DQ | EVO_FLAG_ONLY_DKDV | EVO_FLAG_DEBUG_NO_DQ_WIDE;
    const int64_t wgs = (int64_t)((p.N + 127) / 128) * p.B * p.H;
    if (wgs > 448 && wgs <= 512) return false;
    if (p.D != 64 || p.S != 1 || (p.flags & apart) || p.dmask || !bias_direct(p)) return false;
    return bias_ragged(p) ? dq_wide_ok(p) : !p.gate && dq_writes_dbias(p);
}

// S is split into chunks; one workgroup of the dQ kernel sums dS over one chunk and
// writes one partial dBias tile.  Enough chunks to fill the chip, no more.  The kernel that
// walks over its chunk with one workgroup per CU (256 CUs) runs in rounds of 256 workgroups:
// among the chunk counts that give up to four rounds it takes the cheapest by a count of rows
// per workgroup, rounds and partials (below).
static void chunking(const EvoAttnParams &p, int *n_chunks, int *chunk) {
    const int64_t NT = (p.N + 31) / 32;
    if (p.dtype == EVO_F32) {
        const int want = f32_dbias_chunks(p);
        *chunk = (p.S + want - 1) / want;
        *n_chunks = (p.S + *chunk - 1) / *chunk;
        return;
    }
    if (fused_ok(p) || dq_split_ok(p)) {
        // the dBias kernel: one workgroup per block of 128 queries x 128 keys (64 from head dim 64 on), (b, h) and chunk, two
        // (head dim 128: one) workgroups per CU (256 CUs) at a time; among the chunk counts that give one to four rounds
        // the one that leaves the fewest slots idle in the last round (near ties: the fewest chunks)
        const int64_t kb = p.D >= 64 ? 64 : 128;   // keys per block
        const int64_t base = (int64_t)((p.N + 127) / 128) * ((p.N + kb - 1) / kb) * p.B * p.H, slots = p.D == 128 ? 256 : 512;
        const int64_t lo = slots / base > 0 ? slots / base : 1, hi = (4 * slots + base - 1) / base;
        int64_t want = lo;
        double best = -1.0;
        for (int64_t n = lo; n <= hi; ++n) {
            const int64_t wgs = base * n, rounds = (wgs + slots - 1) / slots;
            const double eff = (double)wgs / (double)(rounds * slots);
            if (eff > best + 0.02) { best = eff; want = n; }
        }
        if (want > p.S) want = p.S;
        *chunk = (int)((p.S + want - 1) / want);
        *n_chunks = (p.S + *chunk - 1) / *chunk;
        return;
    }
    const bool ring = dq_ring_ok(p);
    // workgroups per chunk: one per slab of query rows and head
    const int64_t base = (ring ? (p.N + mfma_dqr_qrows(p.D, p.N) - 1) / mfma_dqr_qrows(p.D, p.N) : NT) * p.B * p.H;
    int64_t want = (1024 + base - 1) / base;
    // The kernel over a chunk of rows: every chunk is a partial dBias to write and to sum again, about a
    // quarter of a row's worth (S = N = 384, H = 4 takes 10 chunks in one round of 240 workgroups over 32 in
    // three full rounds: backward 269 against 298 us; S = N = 768 8 chunks in three rounds over 5 in two:
    // 2.00 against 2.01 ms).
    if (ring) want = chunks_for_rounds(base, p.S, 256, 0.25);
    if (want < 1) want = 1;
    if (want > p.S) want = p.S;
    *chunk = (int)((p.S + want - 1) / want);
    *n_chunks = (p.S + *chunk - 1) / *chunk;
}

struct PrepLayout {
    size_t bq, bk, bq16, bk16, bt, m2, m2a, dead, total;
    int bias_batches;
};

static PrepLayout prep_layout(const EvoAttnParams &p) {
    PrepLayout w{};
    const size_t NT = (size_t)(p.N + 31) / 32;
    w.bias_batches = (p.bias && p.bias_stride_b == 0) ? 1 : p.B;
    // Bias tiles, with one extra all-zero tile at the end of each copy: for a bias in the dtype of q
    // the entries as given, 16 bits each (every kernel that reads tiles multiplies by log2 e
    // itself, in fp32: the product the fp32 tiles hold); else fp32 tiles in log2 units.
    const bool have_tiles = p.bias && !bias_direct(p);
    const bool t16_ok = have_tiles && p.bias_dtype == p.dtype && p.dtype != EVO_F32;
    const size_t tile_elems = have_tiles ? ((size_t)w.bias_batches * p.H * NT * NT + 1) * 1024 : 0;
    size_t off = 0;
    w.bq = off; off += align_up(t16_ok ? 0 : tile_elems * 4);
    w.bk = off; off += align_up(t16_ok ? 0 : tile_elems * 4);
    w.bq16 = w.bk16 = (size_t)-1;
    if (t16_ok) {
        w.bq16 = off; off += align_up(tile_elems * 2);
        w.bk16 = off; off += align_up(tile_elems * 2);
    }
    // transposed 16-bit copy for the kernel that keeps bias columns resident (the chunk-of-rows dK/dV: rows of
    // 129 keys up to its longest)
    const bool bt_ok = p.bias && !bias_direct(p) && p.bias_dtype == p.dtype && p.N % 8 == 0 && p.N > 128 &&
                       p.N <= mfma_kvr_max_n(p.D);
    w.bt = bt_ok ? off : (size_t)-1;
    if (bt_ok) off += align_up((size_t)w.bias_batches * p.H * p.N * p.N * 2);
    w.m2 = off; off += align_up((size_t)p.B * p.S * NT * 32 * 8);
    w.m2a = off; off += align_up((size_t)p.B * p.S * ((p.N + 255) / 256 * 256) * 16);
    w.dead = off; off += align_up((size_t)p.B * p.S * 4);
    w.total = off;
    return w;
}

static void fill_prep(const EvoAttnParams &p, Extra &e) {
    const PrepLayout w = prep_layout(p);
    char *base = (char *)p.prep;
    e.bias_batches = w.bias_batches;
    e.bias_direct = bias_direct(p) ? 1 : 0;
    e.bq = (float *)(base + w.bq);
    e.bk = (float *)(base + w.bk);
    e.bq16 = w.bq16 == (size_t)-1 ? nullptr : (unsigned short *)(base + w.bq16);
    e.bk16 = w.bk16 == (size_t)-1 ? nullptr : (unsigned short *)(base + w.bk16);
    e.bt = w.bt == (size_t)-1 ? nullptr : (void *)(base + w.bt);
    e.m2 = (uint2 *)(base + w.m2);
    e.m2a = (uint4 *)(base + w.m2a);
    e.dead = (int *)(base + w.dead);
    e.zero_tile = (int64_t)w.bias_batches * p.H * ((p.N + 31) / 32) * ((p.N + 31) / 32) * 1024;
}

static int check_prep(const EvoAttnParams &p) {
    if (!p.prep || p.prep_bytes < prep_layout(p).total) return EVO_EWORKSPACE;
    if (!aligned(p.prep, 256)) return EVO_EALIGN;
    return EVO_OK;
}

struct WsLayout {
    size_t delta, shift, dmask_part, dbias_part, dout_ungated, dq_part, total;
    int n_chunks, chunk;
};

static WsLayout ws_layout(const EvoAttnParams &p) {
    WsLayout w{};
    const size_t rows = (size_t)p.B * p.H * p.S * p.N;
    size_t off = 0;
    w.delta = off; off += align_up(rows * 4);
    w.shift = off; off += align_up((size_t)p.B * p.S * 4);
    w.dmask_part = off; if (p.dmask) off += align_up(rows * 4);
    chunking(p, &w.n_chunks, &w.chunk);
    w.dbias_part = off;
    if (p.dbias && !dq_writes_dbias(p)) off += align_up((size_t)w.n_chunks * p.B * p.H * p.N * p.N * 4);
    w.dout_ungated = off;
    if (p.gate && !(p.flags & EVO_FLAG_GATE_DOUT_INPLACE)) off += align_up((size_t)q_span(p) * (size_t)elem_size(p.dtype));
    // dQ of the blocks of keys before, in the place of the dBias partials: those are written when dQ is done (and there is no gate)
    w.dq_part = w.dbias_part;
    if (fused_ok(p) && mfma_fused_blocks(p) > 1) {
        const size_t end = w.dq_part + align_up((size_t)mfma_fused_wgs(p) * p.N * p.D * 4);
        if (end > off) off = end;
    }
    w.total = off;
    return w;
}

static int check_bwd(const EvoAttnParams *p) {
    if (!p->dout || !p->dq || !p->dk || !p->dv) return EVO_EINVAL;
    const int es = elem_size(p->dtype);
    if (!aligned(p->dout, es) || !aligned(p->dq, es) || !aligned(p->dk, es) || !aligned(p->dv, es)) return EVO_EALIGN;
    if (p->dbias) {
        if (p->dbias_dtype != EVO_F32 && p->dbias_dtype != p->dtype) return EVO_EINVAL;
        if (!aligned(p->dbias, elem_size(p->dbias_dtype))) return EVO_EALIGN;
    }
    if (p->dmask && !aligned(p->dmask, 4)) return EVO_EALIGN;
    if (p->gate && (!p->dgate || !aligned(p->dgate, 16) || !aligned(p->dout, 16) || !aligned(p->o, 16) || !aligned(p->o_gated, 16))) return p->dgate ? EVO_EALIGN : EVO_EINVAL;
    const WsLayout w = ws_layout(*p);
    if (!p->workspace || p->workspace_bytes < w.total) return EVO_EWORKSPACE;
    if (!aligned(p->workspace, 256)) return EVO_EALIGN;
    return EVO_OK;
}

}  // namespace evo

using namespace evo;

#ifdef EVO_TRACE
static long long *g_trace = nullptr;
extern "C" void evoattn_set_trace(void *buf) { g_trace = (long long *)buf; }
#define EVO_SET_TRACE(e) (e).trace = g_trace
#else
#define EVO_SET_TRACE(e) do {} while (0)
#endif

extern "C" {

int evoattn_version(void) { return EVOATTN_VERSION; }

const char *evoattn_strerror(int code) {
    switch (code) {
        case EVO_OK: return "ok";
        case EVO_EINVAL: return "invalid argument (null pointer, non-positive size or bad enum)";
        case EVO_EUNSUPPORTED: return "unsupported head dimension or size";
        case EVO_EALIGN: return "pointer or stride not aligned for the dtype";
        case EVO_EWORKSPACE: return "workspace missing or too small";
        case EVO_EOVERFLOW: return "extents overflow the kernels' index range";
    }
    if (code <= EVO_EHIP) return hipGetErrorString((hipError_t)(EVO_EHIP - code));
    return "unknown error";
}

int evoattn_check(const EvoAttnParams *p, int pass) {
    int rc = check_common(p);
    if (rc) return rc;
    if (pass == EVO_PASS_BWD) return check_bwd(p);
    if (pass != EVO_PASS_FWD) return EVO_EINVAL;
    if (p->gate && !p->o_gated) return EVO_EINVAL;   // the forward writes the gated output
    return EVO_OK;
}

// Whether the forward is the one whose waves split a row's keys (mfma_stream.hip): single sequences without a backward, where
// one workgroup per 128 queries leaves some of the CUs without any.
static bool split_fwd_ok(const EvoAttnParams &p) {
    return p.D >= 32 && p.S == 1 && p.N <= kSplitFwdMaxN && (p.flags & EVO_FLAG_FORWARD_ONLY) && !(p.flags & EVO_FLAG_PER_PROBLEM) && (int64_t)p.B * p.H * ((p.N + 127) / 128) < 256;
}

size_t evoattn_prep_bytes(const EvoAttnParams *p) {
    if (!p || p->B <= 0 || p->S <= 0 || p->N <= 0 || p->H <= 0) return 0;
    if (split_fwd_ok(*p) && mfma_ok(*p, EVO_PASS_FWD)) return 0;
    return prep_layout(*p).total;
}

size_t evoattn_bwd_workspace_bytes(const EvoAttnParams *p) {
    if (!p || p->B <= 0 || p->S <= 0 || p->N <= 0 || p->H <= 0) return 0;
    size_t bytes = ws_layout(*p).total;
    if (fused_ok(*p)) {   // (a caller that times the phases of this call alone, by its flags, gets other kernels)
        EvoAttnParams q = *p;
        q.flags |= EVO_FLAG_ONLY_DQ;
        const size_t apart = ws_layout(q).total;
        if (apart > bytes) bytes = apart;
    }
    return bytes;
}

const char *evoattn_path(const EvoAttnParams *p, int pass) {
    if (!p) return "invalid";
    return mfma_ok(*p, pass) ? "mfma" : "generic";
}

// Whether a kernel that walks over a chunk of S rows, one workgroup per CU with the head's bias resident, is ahead of one
// whose workgroups take single problems and stream (head dim 32): it gains a quarter to a fifth per row of 225 to 256 keys (both
// take the same time for all of these) and pays `start` rows' worth per round and the rows that do not fill its last round; shorter
// rows leave waves of its eight idle.  This kernel / the streaming one, us:
//   forward  N = 256, H = 8, S = 16 13.9 / 10.7; 64 19.8 / 18.6; 128 29.3 / 29.3; 192 38.9 / 39.0; 256 46.9 / 49.6; 512 88 / 101; H = 4, S = 256
//            29.5 / 29.1, 512 46.7 / 49.4; N = 248, S = 300, H = 8 67 / 75; N = 216 65 / 66
//   dK/dV    N = 256, H = 8, S = 16 18.2 / 11.4; 64 26.9 / 23.3; 96 33.2 / 30.3; 128 39.0 / 40.8; 192 50.4 / 55.7; 512 130 / 155; N = 232,
//            S = 128 34.4 / 39.1 (left to the other one by this count)
// Rows of exactly 256 keys keep it throughout, a length at which callers of the C ABI (and the tests of capture and of the library's own
// allocations) count on these kernels; below some 100 S rows at 8 heads that costs 1 to 7 us.
static bool ring_pays(const EvoAttnParams &p, double start, double per_row) {
    if (p.N == 256) return true;
    if (p.N <= 224) return false;
    const int64_t bh = (int64_t)p.B * p.H;
    const int n = chunks_for_rounds(bh, p.S, 256, 0.0);
    const double rounds = (double)((bh * n + 255) / 256), rows = (double)((p.S + n - 1) / n);
    return per_row * rounds * (rows + start) * 256.0 < (double)bh * p.S;
}

// Head dim 8 with a bias, no gate: two S rows per workgroup.  With the bias in the dtype of q it is ahead of the kernel over a chunk of rows
// (129..256 keys) from few rows on (H = 8, S = 8 / 64 / 1000, that one / this, us: N = 160 10.5 / 9.9, 14.0 / 12.3, 102 / 86; N = 256 11.9 / 11.5,
// 16.1 / 15.0, 125 / 116; with an fp32 bias N = 192, S = 128 20.4 / 24.6: left to it); of the one-workgroup-per-problem forward where the
// pairs fill two rounds of the three workgroups that a CU holds, for long rows one (H = 8: N = 96, S = 200, 400 15.3 / 14.8, 23.9 / 21.1; N = 384, S = 32, 96,
// 128 17.0 / 19.2, 34.0 / 34.5, 41.9 / 39.3; N = 768, S = 16, 32 30.1 / 33.5, 44.7 / 42.3).
// Left out again after some 2900 forwards of sizes drawn at random (this / that, median and most): an fp32 bias up to 64 keys .96, 1.16 (S = 197, N = 64, 16 heads times batches
// 18.7 / 21.6), and from 97 to 128 of more than 8 heads times batches .96, 1.14; rows of 512 keys and more that overflow one round by little with the bias in the dtype of q
// 1.01, 1.10 (800 pairs: S = 9, B = 2, N = 576, H = 16 45.1 / 49.6), and of three S rows, whose second pair is half empty, 1.05, 1.07.
static bool fwd_pairs8_ok(const EvoAttnParams &p) {
    if (p.D != 8 || !p.bias || p.gate || p.S < 2 || p.N <= 32 || bias_direct(p) || (p.flags & (EVO_FLAG_PER_PROBLEM | EVO_FLAG_DEBUG_FWD_BIAS_TILES))) return false;
    const int64_t pairs = mfma_fwd_pairs(p);
    const bool own = p.bias_dtype == p.dtype;
    if (p.N > 128 && p.N <= 256) return own && pairs >= 64;
    if (p.N >= 512) return p.S != 3 && pairs >= (own ? 900 : 768);
    if (!own && (p.N <= 64 || (p.N > 96 && p.N <= 128 && (int64_t)p.B * p.H > 8))) return false;
    return pairs >= 1536;
}

// rows of 129..256 keys: a workgroup per chunk of S rows with the head's bias resident
static bool fwd_ring_ok(const EvoAttnParams &p) {
    if (fwd_pairs8_ok(p)) return false;
    if ((p.flags & EVO_FLAG_PER_PROBLEM) || bias_direct(p) || p.N <= 128 || p.N > mfma_fwdr_max_n(p.D)) return false;
    // (a gated call keeps it at every length: the bias of a block's pair norm has a gradient that is zero but for
    // the rounding of O, and the two kernels round P against different maxima)
    if (p.D == 32 && !p.gate && !ring_pays(p, 2.4, 0.72)) return false;
    // Resident, a bias in the dtype of q takes 64 registers, an fp32 bias 128, which fit the register file only at
    // head dim 8 without a gate; elsewhere most of them are spilled and the one-workgroup-per-problem forward, which
    // streams the tiles, serves an fp32 bias (B = 1, S = 512, N = 256, H = 8, D = 32: 130 against 214 us).
    // EVO_FLAG_DEBUG_FWD_BIAS_TILES keeps the resident fp32 form, for comparison.
    return !p.bias || p.bias_dtype == p.dtype || (p.D == 8 && !p.gate) || (p.flags & EVO_FLAG_DEBUG_FWD_BIAS_TILES);
}

// The dK/dV kernel that walks over a chunk of S rows keeps 16-bit bias columns resident: it
// takes a bias in the dtype of q (or none) and rows whose length is a multiple of 8.  
// EVO_FLAG_DEBUG_NO_KV_RING selects the other kernel, for comparison.
static bool kv_ring_ok(const EvoAttnParams &p) {
    if ((p.flags & (EVO_FLAG_PER_PROBLEM | EVO_FLAG_DEBUG_NO_KV_RING)) || p.N <= 128 || p.N > mfma_kvr_max_n(p.D) || p.N % 8) return false;
    if (!aligned(p.lse, 16) || bias_direct(p)) return false;   // LSE rows are read four values at a time
    if (p.D == 32 && !ring_pays(p, 1.3, 0.82)) return false;
    return !p.bias || p.bias_dtype == p.dtype;
}

// whether dQ of this call comes from the kernel over a chunk of rows in the form that also does the gate's pass
static bool gate_in_dq(const EvoAttnParams &p) {
    return mfma_ok(p, EVO_PASS_BWD) && !dq_split_ok(p) && !dq_wide_ok(p) && dq_ring_ok(p) && mfma_dqr_gate_ok(p.D, p.N);
}

static int launch_dq(const EvoAttnParams &p, const Extra &e, hipStream_t st) {
    if (dq_split_ok(p)) {
        EvoAttnParams q = p;
        q.dbias = nullptr;                       // dQ and delta first, then the dBias partials, which read delta
        if (const int rc = launch_mfma_dqw(q, e, st)) return rc;
        return launch_mfma_dbias(p, e, st);
    }
    if (dq_wide_ok(p)) return launch_mfma_dqw(p, e, st);
    return dq_ring_ok(p) ? launch_mfma_dqr(p, e, st) : launch_mfma_dq(p, e, st);
}

const char *evoattn_kernels(const EvoAttnParams *p, int pass) {
    if (!p) return "invalid";
    if (f32_ok(*p, pass)) return pass == EVO_PASS_FWD ? "f32_fwd" : p->dbias ? "f32_dq+f32_dbias,f32_dkdv" : "f32_dq,f32_dkdv";
    if (!mfma_ok(*p, pass)) return "generic";
    if (pass == EVO_PASS_FWD) {
        if (split_fwd_ok(*p)) return "split_fwd";
        if (fwd_ring_ok(*p)) return "mfma_fwd_ring";
        return fwd_pairs8_ok(*p) || mfma_fwd_pair_ok(*p, bias_direct(*p)) ? "mfma_fwd_pair" : "mfma_fwd";
    }
    if (fused_ok(*p)) return p->dbias ? "mfma_bwd_fused+mfma_dbias" : "mfma_bwd_fused";
    const bool kvr = kv_ring_ok(*p);
    if (dq_split_ok(*p)) return kvr ? "mfma_dq_wide+mfma_dbias,mfma_dkdv_ring" : "mfma_dq_wide+mfma_dbias,mfma_dkdv";
    if (bwd_one_ok(*p)) return "mfma_dq_wide,mfma_dkdv(one launch)";
    if (dq_wide_ok(*p)) return kvr ? "mfma_dq_wide,mfma_dkdv_ring" : "mfma_dq_wide,mfma_dkdv";
    if (kvr) return dq_ring_ok(*p) ? "mfma_dq_ring,mfma_dkdv_ring" : "mfma_dq,mfma_dkdv_ring";
    return dq_ring_ok(*p) ? "mfma_dq_ring,mfma_dkdv" : "mfma_dq,mfma_dkdv";
}

// the forward's launches for a checked parameter block whose `prep` is in place
static int fwd_launches(const EvoAttnParams &p, hipStream_t st) {
    Extra e{};
    e.vec_ok = bias_vec_ok(p);
    fill_prep(p, e);
    EVO_SET_TRACE(e);
    // Without a backward the copies of the bias that only its kernels read need not be made, nor any where the forward keeps
    // the caller's rows (S = 128, N = 251, H = 8, gated, fp16: 36.1 -> 34.7 us).
    const bool ring = fwd_ring_ok(p), alone = (p.flags & EVO_FLAG_FORWARD_ONLY) != 0;
    if (alone) {
        e.bk = nullptr;
        e.bk16 = nullptr;
        e.bt = nullptr;
    }
    // (that forward then has nothing to wait for: it reads the mask as given, too)
    if (alone && ring && !fwd_pairs8_ok(p) && (!p.bias || mfma_fwdr_reads_rows(p))) e.m2a = nullptr;
    else if (const int rc = launch_prep(p, e, st)) return rc;
    return fwd_pairs8_ok(p) ? launch_stream_fwd8(p, e, st) : ring ? launch_mfma_fwdr(p, e, st) : launch_mfma_fwd(p, e, st);
}

int evoattn_fwd(const EvoAttnParams *p, void *hip_stream) {
    int rc = evoattn_check(p, EVO_PASS_FWD);
    if (rc) return rc;
    hipStream_t st = (hipStream_t)hip_stream;
    if (f32_ok(*p, EVO_PASS_FWD)) return launch_f32_fwd(*p, st);
    if (!mfma_ok(*p, EVO_PASS_FWD)) return launch_generic_fwd(*p, st);
    if (split_fwd_ok(*p)) return launch_split_fwd(*p, st);   // (needs no `prep`)
    if ((rc = check_prep(*p))) return rc;
    return fwd_launches(*p, st);
}

// Device address of this GPU's copy of `scratch`, asked for on the first call on that device.
static int static_prep(void **out) {
    static std::atomic<void *> addr[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return EVO_EHIP - (int)hipGetLastError();
    if (dev < 0 || dev >= 64) return EVO_EUNSUPPORTED;
    void *ptr = addr[dev].load(std::memory_order_acquire);
    if (!ptr) {
        const hipError_t err = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (err != hipSuccess || !ptr) return EVO_EHIP - (int)(err != hipSuccess ? err : hipErrorInvalidSymbol);
        addr[dev].store(ptr, std::memory_order_release);
    }
    *out = ptr;
    return EVO_OK;
}

int evoattn_fwd_static(const EvoAttnParams *p, void *hip_stream) {
    int rc = evoattn_check(p, EVO_PASS_FWD);
    if (rc) return rc;
    hipStream_t st = (hipStream_t)hip_stream;
    if (f32_ok(*p, EVO_PASS_FWD)) return launch_f32_fwd(*p, st);         // (these kernels take no prepared operands,
    if (!mfma_ok(*p, EVO_PASS_FWD)) return launch_generic_fwd(*p, st);   // nor do those)
    if (prep_layout(*p).total > (size_t)EVOATTN_STATIC_PREP_BYTES) return EVO_EWORKSPACE;
    EvoAttnParams q = *p;
    if ((rc = static_prep(&q.prep))) return rc;
    q.prep_bytes = (size_t)EVOATTN_STATIC_PREP_BYTES;
    // The prep kernel writes every byte of the array that this call's kernels read (bias tiles
    // with their zero tile, mask rows, flags), so nothing of an earlier call has to be cleared.
    return fwd_launches(q, st);
}

int evoattn_bwd(const EvoAttnParams *p0, void *hip_stream) {
    int rc = evoattn_check(p0, EVO_PASS_BWD);
    if (rc) return rc;
    hipStream_t st = (hipStream_t)hip_stream;
    const WsLayout w = ws_layout(*p0);
    char *ws = (char *)p0->workspace;
    // With a gate, p0->dout is the gradient of the gated output: one pass over the rows forms the
    // gradient of the ungated output (into the workspace) and of the gate, and the attention
    // backward below runs on the former.
    EvoAttnParams ungated = *p0;
    Extra e{};
    if (p0->gate) {
        // (in place: a thread reads its 8 elements of dout before it writes them)
        void *d_o = (p0->flags & EVO_FLAG_GATE_DOUT_INPLACE) ? const_cast<void *>(p0->dout) : (void *)(ws + w.dout_ungated);
        ungated.dout = d_o;
        ungated.gate = nullptr;
        ungated.o_gated = nullptr;
        ungated.dgate = nullptr;
        // Where dQ comes from the kernel over a chunk of rows in its form for up to 256 keys at head dim 32, that
        // kernel does the gate's pass on the rows it stages anyway (it runs before the dK/dV kernel, which reads
        // the gradient of the ungated output it writes).
        if (gate_in_dq(ungated) && p0->o_gated && !(p0->flags & EVO_FLAG_ONLY_DKDV)) {
            e.gate_dout = p0->dout;
            e.gate_logits = p0->gate;
            e.gate_og = p0->o_gated;
            e.gate_dgate = p0->dgate;
        } else if ((rc = launch_gate_bwd(*p0, d_o, (float *)(ws + w.delta), st))) {
            return rc;
        }
    }
    const EvoAttnParams *p = &ungated;
    e.n_chunks = w.n_chunks;
    e.chunk = w.chunk;
    e.vec_ok = bias_vec_ok(*p);
    e.delta = (float *)(ws + w.delta);
    e.delta_given = p0->gate && !e.gate_dout ? 1 : 0;   // (the gate's pass wrote it; the dQ kernels then read no ungated O)
    e.shift = (float *)(ws + w.shift);
    e.dmask_part = (float *)(ws + w.dmask_part);
    e.dbias_part = (float *)(ws + w.dbias_part);
    e.dq_part = (float *)(ws + w.dq_part);
    if (f32_ok(*p, EVO_PASS_BWD)) return launch_f32_bwd(*p, e, st);
    if (!mfma_ok(*p, EVO_PASS_BWD)) return launch_generic_bwd(*p, e, st);
    if ((rc = check_prep(*p))) return rc;
    fill_prep(*p, e);
    EVO_SET_TRACE(e);
    if (!(p->flags & EVO_FLAG_PREP_VALID) && (rc = launch_prep(*p, e, st))) return rc;
    if (!p0->gate && fused_ok(*p)) {
        if ((rc = p->D == 8 ? launch_mfma_fused8(*p, e, st) : launch_mfma_fused(*p, e, st))) return rc;   // (writes delta as well)
        if (!p->dbias) return EVO_OK;
        if ((rc = launch_mfma_dbias(*p, e, st))) return rc;
        return launch_dbias_reduce(*p, e, st);
    }
    if (bwd_one_ok(*p0)) return launch_stream_bwd_one_d64(*p, e, st);
    if (p->flags & EVO_FLAG_ONLY_DQ) return launch_dq(*p, e, st);
    const bool kvring = kv_ring_ok(*p);
    // that kernel sums the dBias partials on its way in (they lie 16-byte aligned for it)
    const bool partials = p->dbias && !dq_writes_dbias(*p);
    // (both dK/dV kernels do; the one-workgroup-per-problem kernel where the sums come in whole 16-byte pieces)
    const bool fused_reduce = partials && !(p->flags & EVO_FLAG_ONLY_DQ) && aligned(p->dbias, 16) &&
                              (kvring || ((int64_t)p->B * p->H * p->N * p->N) % 4 == 0);
    e.dbias_chunks = fused_reduce ? e.n_chunks : 0;
    if (p->flags & EVO_FLAG_ONLY_DKDV) return kvring ? launch_mfma_kvr(*p, e, st) : launch_mfma_dkdv(*p, e, st);
    // dQ first: it also writes delta, which the dK/dV kernel reads
    if ((rc = launch_dq(*p, e, st))) return rc;
    if ((rc = kvring ? launch_mfma_kvr(*p, e, st) : launch_mfma_dkdv(*p, e, st))) return rc;
    if (partials && !fused_reduce && (rc = launch_dbias_reduce(*p, e, st))) return rc;
    if (p->dmask && (rc = launch_dmask_reduce(*p, e, st))) return rc;
    return EVO_OK;
}

}  // extern "C"
