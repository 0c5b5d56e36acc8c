// Host launcher of the multi-step forward kernels.
#include "neuron_fwd.h"

#include <cmath>

namespace sjhip {

namespace {

// Whether the [T, N] tensors of a call are together a third larger than the 256 MiB cache in front of the memory: what
// the kernel moves then passes through that cache anyway, and marking one side of it as streaming leaves the cache to
// the other side.  Which side was measured with both policies on one machine, forward plus replaying backward repeated on
// the same tensors, us (x tensor in MB; default -> streaming):
//   * fp32, stores streaming (x stays for the backward, which gains as well).  Spikes only, T = 8: 160 MB 133 -> 136,
//     192 MB 166 -> 162, 256 MB 226 -> 211, 320 MB 283 -> 261, 536 MB 471 -> 448; T = 128: 175 MB 190 -> 201, 320 MB
//     389 -> 363, 536 MB 580 -> 534.  With v_seq, T = 8: 110 MB 143 -> 146, 128 MB 160 -> 149, 320 MB 398 -> 365,
//     T = 16, 2.1 GB: 2617 -> 2563 (streaming the x loads instead: 2611 -> 2647).
//   * 16 bit with spikes only, x loads streaming (streaming the stores: 150 -> 167 in the forward of T = 32, N = 6.4 M).
//     fp16, T = 6: 140 MB 132 -> 131, 155 MB 144 -> 144, 170 MB 165 -> 160, 192 MB 187 -> 171, 400 MB 412 -> 410; T = 32,
//     300 MB: 470 -> 450.  (With v_seq and every op rounded it loses from 400 MB on: 576 -> 608.)
// Inside a network less is left of it: three inputs in turn, an elementwise operation that writes x before the neuron and one that
// reads the spikes after it, everything together, us:
//   * fp32, T = 8, inference: 192 MB 197 -> 186, 256 MB 266 -> 262, 320 MB 327 -> 321, 536 MB 548 -> 551; training: 422 -> 422,
//     570 -> 563, 691 -> 685, 1163 -> 1165.  With v_seq, inference 240 -> 220, 321 -> 309, 388 -> 381, 650 -> 652, training 468 -> 456,
//     624 -> 617, 752 -> 743, 1271 -> 1271; T = 4, 128 MB 174 -> 136.  It costs at T = 4 and 5 from 160 to 192 MB (258 -> 269,
//     206 -> 202; training 482 -> 496, 395 -> 406).
//   * fp16, T = 8: inference 211 -> 205, 279 -> 272, 429 -> 422, training 455 -> 445, 599 -> 593, 929 -> 923.
// A reader of the spikes finds less of them in the cache: forward and sum over T 106 -> 121 at 192 MB, 156 -> 153 at 256 MB.
// Below the bound either policy costs up to 10 %: the next reader of the spikes, or the backward, finds them in the cache.  16-bit
// sequences in pieces keep the default policy: neither was measured for them.
bool beyond_cache(const FwdArgs &a, int element_bytes) {
  constexpr int64_t kBytes = (int64_t)256 * 1024 * 1024 / 3 * 4;
  const int64_t tensors = 2 + (a.v_seq != nullptr) + (a.h != nullptr);
  return a.T > 1 && a.N > kBytes / (element_bytes * tensors) / a.T;
}

template <typename S, bool ROUND_EACH, bool PACKED = false>
int launch_typed(const FwdArgs &a, bool vector, hipStream_t stream) {
  int block = tuning().fwd_block;
  // (the block size changes only with the runs that answer a resonant row stride, not with the contiguous eighths)
  if (a.spread > 1 && tuning().column_spread == 2) block = spread_block(a.N * (int64_t)sizeof(S));
  const int V = vector ? Acc<S, true, true>::V : 1;
  const int64_t items = (a.N + V - 1) / V;
  const int64_t blocks = (items + block - 1) / block;
  if (blocks > 0x7fffffffLL) return fail(SJHIP_ERR_TOO_LARGE, "forward: N=%lld needs %lld blocks", (long long)a.N, (long long)blocks);
  // the residency cap pays for fp32 storage writing two or three [T, N] tensors (spikes plus v_seq and / or h_seq);
  // with spikes only, and with 16-bit storage (more wavefronts hide its conversions), uncapped is faster (measured)
  // A short sequence has few rows in flight per work-item and needs more resident blocks instead: twice the cap
  // below 16 steps, none below 4 (measured at T = 1, 2, 4, 8, 16).  ILIF's step is a longer dependent chain (a
  // quotient, a clamp and a rounding on top of the charge): with two resident blocks that latency shows, with four
  // it is hidden (measured 1.47 -> 1.24 ms at T = 16, N = 33.5 M).  The same holds for EIF's exp().
  const bool several_outputs = a.v_seq != nullptr || a.h != nullptr;
  int cap = tuning().fwd_blocks_per_cu;
  if (a.T < 4) cap = 0;
  else if (a.T < 16 || a.soft_reset == RESET_COUNT || a.charge == CH_EIF_DIV || a.charge == CH_EIF_MUL) cap *= 2;
  const unsigned lds = (sizeof(S) == 4 && several_outputs) ? occupancy_cap_lds(cap) : 0u;
  ProfileScope prof(KC_FORWARD, stream);
  const dim3 grid((unsigned)blocks), threads(block);
  // which accesses stream: see FwdOut and beyond_cache()
  const bool stream_x = sizeof(S) == 2 && a.T > 1 && (several_outputs ? !ROUND_EACH : beyond_cache(a, 2));
  const bool stream_out = sizeof(S) == 4 && beyond_cache(a, 4);
  if constexpr (PACKED) {
    if (vector) hipLaunchKernelGGL((forward_kernel<S, true, ROUND_EACH, FWD_OUT_PACKED>), grid, threads, lds, stream, a);
    else hipLaunchKernelGGL((forward_kernel<S, false, ROUND_EACH, FWD_OUT_PACKED>), grid, threads, lds, stream, a);
  } else if (stream_x) {
    if constexpr (sizeof(S) == 2) {
      if (vector) hipLaunchKernelGGL((forward_kernel<S, true, ROUND_EACH, FWD_OUT_DENSE_STREAM_X>), grid, threads, lds, stream, a);
      else hipLaunchKernelGGL((forward_kernel<S, false, ROUND_EACH, FWD_OUT_DENSE_STREAM_X>), grid, threads, lds, stream, a);
    }
  } else if (stream_out) {
    if constexpr (sizeof(S) == 4) {
      if (vector) hipLaunchKernelGGL((forward_kernel<S, true, ROUND_EACH, FWD_OUT_DENSE_STREAM_OUT>), grid, threads, lds, stream, a);
      else hipLaunchKernelGGL((forward_kernel<S, false, ROUND_EACH, FWD_OUT_DENSE_STREAM_OUT>), grid, threads, lds, stream, a);
    }
  } else if (a.T == 1) {
    if (vector) hipLaunchKernelGGL((forward_kernel<S, true, ROUND_EACH, FWD_OUT_DENSE | FWD_OUT_SHORT>), grid, threads, lds, stream, a);
    else hipLaunchKernelGGL((forward_kernel<S, false, ROUND_EACH, FWD_OUT_DENSE | FWD_OUT_SHORT>), grid, threads, lds, stream, a);
  } else {
    if (vector) hipLaunchKernelGGL((forward_kernel<S, true, ROUND_EACH, FWD_OUT_DENSE>), grid, threads, lds, stream, a);
    else hipLaunchKernelGGL((forward_kernel<S, false, ROUND_EACH, FWD_OUT_DENSE>), grid, threads, lds, stream, a);
  }
  return check_launch(PACKED ? "forward_packed" : "forward");
}

template <typename S, bool ROUND_EACH> int launch_pieces_typed(const FwdArgs &a, hipStream_t stream) {
  // From 64 steps on, one wavefront per block: the steady-state loop keeps a block's next rows in flight while it
  // computes, so half the resident work-items still fill the memory pipeline, and with a fixed number of neuron-steps
  // a longer sequence means fewer, longer blocks, whose last round leaves less of the chip idle when they are small
  // (2^29 neuron-steps, fp32, T = 64 / 128 / 512: 1.198 / 1.234 / 1.327 ms against 1.231 / 1.283 / 1.398 with 128
  // lanes; T = 48: 1.304 against 1.283).
  const int block = a.T >= 64 && tuning().fwd_block > 64 ? 64 : tuning().fwd_block;
  const int64_t items = (a.N + Acc<S, true, true>::V - 1) / Acc<S, true, true>::V;
  const int64_t blocks = (items + block - 1) / block;
  if (blocks > 0x7fffffffLL) return fail(SJHIP_ERR_TOO_LARGE, "forward(pieces): N=%lld", (long long)a.N);
  const unsigned lds = (sizeof(S) == 4 && a.v_seq != nullptr) ? occupancy_cap_lds(tuning().fwd_blocks_per_cu) : 0u;
  ProfileScope prof(KC_FORWARD, stream);
  if (sizeof(S) == 4 && beyond_cache(a, 4)) {
    if constexpr (sizeof(S) == 4)
      hipLaunchKernelGGL((forward_pieces_kernel<S, ROUND_EACH, FWD_OUT_DENSE_STREAM_OUT>), dim3((unsigned)blocks), dim3(block), lds, stream, a);
  } else {
    hipLaunchKernelGGL((forward_pieces_kernel<S, ROUND_EACH>), dim3((unsigned)blocks), dim3(block), lds, stream, a);
  }
  return check_launch("forward(pieces)");
}

}  // namespace

int launch_forward_pieces(int neuron, int dtype, const sjhip_neuron_params &p, int64_t T, int64_t N, int64_t chunk,
                          const void *x_seq, const void *v_init, const float *k_device, void *spike_seq, void *v_seq,
                          void *v_last, void *checkpoints, hipStream_t stream) {
  FwdArgs a;
  bool round_each = false;
  int rc = build_fwd_args(a, round_each, neuron, dtype, p, T, N, x_seq, v_init, k_device, spike_seq, v_seq, v_last, nullptr);
  if (rc != SJHIP_OK) return rc;
  const int V = dtype == SJHIP_F32 ? 4 : 8;
  if (N < V || !aligned16(x_seq) || !(a.v_init_broadcast || aligned16(v_init)) || !aligned16(spike_seq) || !aligned16(v_seq) ||
      !aligned16(v_last) || !aligned16(checkpoints))
    return fail(SJHIP_ERR_UNSUPPORTED, "forward(pieces): N=%lld must be at least %d and every tensor 16-byte aligned", (long long)N, V);
  const uint64_t row = (uint64_t)N * (16 / V), all = (uint64_t)T * row;
  const uint64_t kept = (uint64_t)(T > chunk ? (T + chunk - 1) / chunk - 1 : 0) * N * (checkpoints_are_f32(dtype, p.flags) ? 4 : 16 / V);
  if (N % V != 0 && any_overlap({{spike_seq, all}, {v_seq, all}, {v_last, row}, {checkpoints, kept}},
                                {{x_seq, all}, {v_init, a.v_init_broadcast ? 4 : row}}))
    return fail(SJHIP_ERR_UNSUPPORTED, "forward(pieces): N=%lld is not a multiple of %d: no output may overlap an input", (long long)N, V);
  a.checkpoints = checkpoints; a.chunk = chunk;
  switch (dtype) {
    case SJHIP_F32: return launch_pieces_typed<float, false>(a, stream);
    case SJHIP_F16: return round_each ? launch_pieces_typed<f16_t, true>(a, stream) : launch_pieces_typed<f16_t, false>(a, stream);
    case SJHIP_BF16: return round_each ? launch_pieces_typed<bf16_t, true>(a, stream) : launch_pieces_typed<bf16_t, false>(a, stream);
    default: return fail(SJHIP_ERR_INVALID, "forward(pieces): dtype %d", dtype);
  }
}

int launch_forward_packed(int neuron, int dtype, const sjhip_neuron_params &p, int64_t T, int64_t N,
                          const void *x_seq, const void *v_init, const float *k_device, uint8_t *spike_bits,
                          void *v_seq, void *v_last, hipStream_t stream) {
  if (N % 8 != 0)
    return fail(SJHIP_ERR_UNSUPPORTED, "forward_packed: N=%lld is not a multiple of 8 (rows must start on a byte)", (long long)N);
  FwdArgs a;
  bool round_each = false;
  int rc = build_fwd_args(a, round_each, neuron, dtype, p, T, N, x_seq, v_init, k_device, spike_bits, v_seq, v_last, nullptr);
  if (rc != SJHIP_OK) return rc;
  const bool vector = true;  // (N is a multiple of 8: no work-item is left with part of a group)
  switch (dtype) {
    case SJHIP_F32: return launch_typed<float, false, true>(a, vector, stream);
    case SJHIP_F16: return round_each ? launch_typed<f16_t, true, true>(a, vector, stream) : launch_typed<f16_t, false, true>(a, vector, stream);
    case SJHIP_BF16: return round_each ? launch_typed<bf16_t, true, true>(a, vector, stream) : launch_typed<bf16_t, false, true>(a, vector, stream);
    default: return fail(SJHIP_ERR_INVALID, "forward_packed: dtype %d", dtype);
  }
}

int launch_forward(int neuron, int dtype, const sjhip_neuron_params &p, int64_t T, int64_t N,
                   const void *x_seq, const void *v_init, const float *k_device, void *spike_seq,
                   void *v_seq, void *v_last, void *h_seq, hipStream_t stream) {
  FwdArgs a;
  bool round_each = false;
  int rc = build_fwd_args(a, round_each, neuron, dtype, p, T, N, x_seq, v_init, k_device, spike_seq, v_seq, v_last, h_seq);
  if (rc != SJHIP_OK) return rc;

  // any N and any alignment, but rows that V does not divide only apart from the inputs: see whole_group()
  const int V = dtype == SJHIP_F32 ? 4 : 8;
  const uint64_t row = (uint64_t)N * (16 / V), all = (uint64_t)T * row;
  const bool vector = N % V == 0 || (N >= V && !any_overlap({{spike_seq, all}, {v_seq, all}, {h_seq, all}, {v_last, row}},
                                                            {{x_seq, all}, {v_init, a.v_init_broadcast ? 4 : row}}));

  switch (dtype) {
    case SJHIP_F32: return launch_typed<float, false>(a, vector, stream);
    case SJHIP_F16: return round_each ? launch_typed<f16_t, true>(a, vector, stream) : launch_typed<f16_t, false>(a, vector, stream);
    case SJHIP_BF16: return round_each ? launch_typed<bf16_t, true>(a, vector, stream) : launch_typed<bf16_t, false>(a, vector, stream);
    default: return fail(SJHIP_ERR_INVALID, "forward: dtype %d", dtype);
  }
}

}  // namespace sjhip
