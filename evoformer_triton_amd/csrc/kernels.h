// Host-side launchers of the kernel families; each enqueues on `st` and returns EVO_OK or
// EVO_EHIP - hipError_t.
#pragma once

#include "common.h"

namespace evo {

int launch_generic_fwd(const EvoAttnParams &p, hipStream_t st);
int launch_generic_bwd(const EvoAttnParams &p, const Extra &e, hipStream_t st);
int launch_f32_fwd(const EvoAttnParams &p, hipStream_t st);
int launch_f32_bwd(const EvoAttnParams &p, const Extra &e, hipStream_t st);
int f32_dbias_chunks(const EvoAttnParams &p);  // chunks of S rows that those kernels split a dBias sum into
int launch_delta_generic(const EvoAttnParams &p, const Extra &e, hipStream_t st);
int launch_dmask_reduce(const EvoAttnParams &p, const Extra &e, hipStream_t st);
int launch_dbias_reduce(const EvoAttnParams &p, const Extra &e, hipStream_t st);
int launch_gate_bwd(const EvoAttnParams &p, void *dout_ungated, float *delta, hipStream_t st);  // dO, dgate and delta from the gradient of the gated output
int launch_mask_shift(const EvoAttnParams &p, const Extra &e, hipStream_t st);

int launch_prep(const EvoAttnParams &p, const Extra &e, hipStream_t st);
int launch_mfma_fwd(const EvoAttnParams &p, const Extra &e, hipStream_t st);
constexpr int kSplitFwdMaxN = 4096;   // (its mask row lies in LDS)
int launch_split_fwd(const EvoAttnParams &p, hipStream_t st);  // the keys of a row split over waves; reads mask and bias as given
// whether that kernel (where it serves the call) keeps the caller's 16-bit bias rows, else prepared tiles
inline bool mfma_fwdr_reads_rows(const EvoAttnParams &p) {
    return p.bias_dtype == p.dtype && !(p.D == 8 && !p.gate) && !(p.flags & EVO_FLAG_DEBUG_FWD_BIAS_TILES);
}
// Workgroups of the forwards that take two S rows (stream_fwd_pair, stream_fwd8), and whether launch_mfma_fwd takes that of head dim 32: two
// rounds of the three workgroups that a CU holds, or the last one is too empty for a workgroup that takes twice as long (stream_fwd / pairs, us, H = 8: N = 384,
// S = 48, 64, 96, 128 26.7 / 27.8, 30.3 / 29.6, 40.4 / 41.2, 50.4 / 47.2; N = 300, S = 96, 128 34.5 / 35.5, 42.3 / 39.9); up to 192 keys what a
// workgroup costs beside its tiles decides (N = 128, S = 200 20.4 / 22.8; N = 192 32.9 / 33.9; N = 224 39.8 / 37.2).
inline int64_t mfma_fwd_pairs(const EvoAttnParams &p) { return (int64_t)((p.N + 127) / 128) * p.B * p.H * ((p.S + 1) / 2); }
inline bool mfma_fwd_pair_ok(const EvoAttnParams &p, bool bias_direct) {
    return p.D == 32 && p.N > 192 && mfma_fwd_pairs(p) >= 2 * 768 && p.bias_dtype != EVO_NONE && !bias_direct && !p.gate && !(p.flags & EVO_FLAG_PER_PROBLEM);
}
int launch_mfma_fwdr(const EvoAttnParams &p, const Extra &e, hipStream_t st);
int mfma_fwdr_max_n(int D);  // largest N the chunk-of-rows forward takes, 0 for a head dim it is not built for
int launch_mfma_dq(const EvoAttnParams &p, const Extra &e, hipStream_t st);
int launch_mfma_dqr(const EvoAttnParams &p, const Extra &e, hipStream_t st);
int launch_mfma_kvr(const EvoAttnParams &p, const Extra &e, hipStream_t st);
int mfma_kvr_max_n(int D);  // largest N the chunk-of-rows dK/dV kernel takes (it takes N > 128 only), 0 where it is not built
// whether the dQ kernel over a chunk of rows, where it serves such rows, also does the gate's backward pass on the
// rows it stages (its form of one stage of up to 256 keys with two query tiles, at head dim 32)
inline bool mfma_dqr_gate_ok(int D, int N) { return D == 32 && N <= 256; }
int mfma_dqr_qrows(int D, int N);  // query rows per workgroup of the double-buffered dQ kernel (64 or 32), 0 where it is not built for such rows
int launch_mfma_dkdv(const EvoAttnParams &p, const Extra &e, hipStream_t st);
int launch_mfma_dqw(const EvoAttnParams &p, const Extra &e, hipStream_t st);  // dQ where no dBias is asked for
// dQ, dK and dV at once (head dims 32, 8): key tiles of 16 per wave
inline int mfma_fused_tiles(int N) {
    if (N <= 128) return 2;
    const int blocks = (N + 255) / 256;   // fewest blocks of at most 256 keys, as narrow as they can be
    return (N + blocks * 64 - 1) / (blocks * 64);
}
inline int mfma_fused8_tiles(int N) {
    if (N <= 128) return 2;
    const int blocks = (N + 383) / 384;   // (of at most 384 keys)
    return (N + blocks * 64 - 1) / (blocks * 64);
}
inline int mfma_fused_keys(const EvoAttnParams &p) { return 64 * (p.D == 8 ? mfma_fused8_tiles(p.N) : mfma_fused_tiles(p.N)); }   // of a block
inline int mfma_fused_blocks(const EvoAttnParams &p) { return (p.N + mfma_fused_keys(p) - 1) / mfma_fused_keys(p); }   // one after the other
// Workgroups.  With several blocks each has a scratch of a problem's dQ (N x D fp32) in the workspace and at most as many as are resident at a time,
// two on each CU, share the problems.
inline int64_t mfma_fused_wgs(const EvoAttnParams &p) {
    const int64_t problems = (int64_t)p.B * p.H * p.S;
    return mfma_fused_blocks(p) > 1 && problems > 512 ? 512 : problems;
}
int launch_stream_fwd8(const EvoAttnParams &p, const Extra &e, hipStream_t st);  // forward with a bias, head dim 8: two S rows per workgroup
int launch_mfma_fused8(const EvoAttnParams &p, const Extra &e, hipStream_t st);
int launch_mfma_fused(const EvoAttnParams &p, const Extra &e, hipStream_t st);
int launch_stream_bwd_one_d64(const EvoAttnParams &p, const Extra &e, hipStream_t st);   // dQ, dK, dV and dBias of one S row (mfma_stream.hip)
int launch_mfma_dbias(const EvoAttnParams &p, const Extra &e, hipStream_t st);  // dBias partials alone (reads delta)
int launch_column_reduce(const float *part, int blocks, int cols, void *out, int dtype, hipStream_t st);  // out[c] = sum of part[.][c], fixed order

}  // namespace evo
