// Decode shrink and expand of the same projections in one launch.  A file of its own so that it
// compiles next to bgmv_decode.hip, whose device code it shares through bgmv_pages.hpp.
//
// Replaces the back-to-back dispatch_bgmv pairs of
// slora/models/peft/lora_unordered_batch_infer.py:267-273, 287-293, 307-313, 438-444.

#include "bgmv_pages.hpp"

namespace slora {
namespace {

// ---------------------------------------------------------------------------
// shrink and expand of the same projections in ONE launch
// ---------------------------------------------------------------------------
// The reference issues shrink and expand of a projection back to back
// (slora/models/peft/lora_unordered_batch_infer.py:267-273): two launches, the second of which cannot
// start before the first has drained, and both pay a launch, a record and the way of the first data.
// Here the grid holds the workgroups of both: first those of the shrink (an item's 8 rows of one
// projection each), then those of the expand (half of an item's 8 pages of
// B^T each).  Workgroups are handed out in that order and the first kind waits for nobody, so whatever a
// workgroup of the second kind waits for is running or done.  It has its pages and its y values on
// the way before it looks for the delta rows of its run.
//
// Hand-over: the value of a delta row's column travels in a word of its own behind the plan, (value | launch
// << 16), written with a device-scope store and read with device-scope loads; a reader repeats its loads until
// every word names this launch.  No counter, no wait for a store to be acknowledged and no second
// round trip stand between a producer's last product and the reader's arithmetic.  Which launch this is
// every workgroup knows from a word that nobody else writes (the launches it has taken part in; all of a run's take part
// in every one-launch call on the plan, so they agree), so the area is cleared by the plan build only and launches may be
// replayed.  Launches on one plan must not overlap.
//
// The wait is bounded: after spin_limit polls a wavefront computes the rows of its run itself (pages_recompute)
// and leaves a mark in the plan's status word.
//
// Both halves in one kernel cost 28 to 45 spilled scalar registers, depending on type and page width (lanes of
// vector registers, no memory); the shrink by itself spills none.
//
// What it took: a form whose every workgroup did both halves ran 44 us for q, k and v of S2's 256 tokens; this
// arrangement with the general paths inlined 62, without them 36, with one polling load per token and workgroup
// instead of every lane reading all its columns (the polls kept the shrink's own loads waiting) 33.
//
// Grid, two forms (see bgmv_expand_kernel): two-dimensional, x = item, y < nproj: shrink of projection y, else expand
// half y - nproj; one-dimensional (INTERLEAVE): the shrinks projection by projection, then the expand
// workgroups of an item one after the other.  LDS: the shrink's staging area, or a strip per wavefront
// and token and the delta rows.
template <typename T, int NV, bool INTERLEAVE>
__global__ __launch_bounds__(256, NV > 12 ? 2 : (NV > 8 ? 3 : 4)) void bgmv_lora_kernel(const PageArgs) {
  extern __shared__ u32x4 s_x[];  // [kTT][h_in / 8]
  const PageArgs& p = page_args();
  int unit = (int)blockIdx.x, sub = (int)blockIdx.y;
  if (INTERLEAVE) {
    if (unit < p.n_units * p.nproj) {
      sub = unit / p.n_units;
      unit -= sub * p.n_units;
    } else {
      const int S = 2 * p.nproj, id = unit - p.n_units * p.nproj, g = id >> 3;
      unit = (g / S) * 8 + (id & 7);
      sub = p.nproj + g % S;
    }
  }
  if (sub < p.nproj) {
    for (;;) {
      const int n_items = pages_shrink<T, NV, true>(p, unit, sub, s_x);
      // a launch sized for a fraction of the plan's capacity: the items beyond the grid, if the batch has that many
      unit += p.n_units;
      if (!p.strided || unit >= n_items) return;
      __syncthreads();  // the staging area of the item before is free
    }
  }
  sub -= p.nproj;
  uint16_t* s_strip = reinterpret_cast<uint16_t*>(s_x) + (threadIdx.x >> 6) * (kTT * ExpandPass<NV>::kStrip);
  uint32_t* s_delta = reinterpret_cast<uint32_t*>(reinterpret_cast<uint16_t*>(s_x) + 4 * kTT * ExpandPass<NV>::kStrip);
  for (;;) {
    const int n_items = pages_expand<T, NV, true>(p, unit, sub, s_strip, s_delta);
    unit += p.n_units;
    if (!p.strided || unit >= n_items) return;
    __syncthreads();  // the delta rows of the item before have been read
  }
}

template <typename T, int NV>
int launch_lora(const PageArgs& p, hipStream_t stream) {
  auto kernel = p.interleave ? bgmv_lora_kernel<T, NV, true> : bgmv_lora_kernel<T, NV, false>;
  constexpr size_t strips = 4 * kTT * ExpandPass<NV>::kStrip * sizeof(uint16_t) + kDeltaBytes;
  constexpr size_t staging = (size_t)kTT * ExpandPass<NV>::kElems * 2, lds = strips > staging ? strips : staging;
  static PerDeviceOnce once[2];
  if (!raise_dynamic_lds(reinterpret_cast<const void*>(kernel), (int)lds, once[p.interleave])) return SLORA_ERR_LAUNCH;
  dim3 grid((uint32_t)p.n_units, 3 * p.nproj);
  if (p.interleave) grid = dim3((uint32_t)(p.n_units * 3 * p.nproj), 1);
  hipLaunchKernelGGL(kernel, grid, dim3(256), lds, stream, p);
  return hipGetLastError() == hipSuccess ? SLORA_OK : SLORA_ERR_LAUNCH;
}

template <typename T>
int dispatch_lora(const PageArgs& p, int64_t page_elems, hipStream_t stream) {
  switch (page_elems / (8 * kWave)) {
    case 8: return launch_lora<T, 8>(p, stream);
    case 10: return launch_lora<T, 10>(p, stream);
    case 12: return launch_lora<T, 12>(p, stream);
    default: return launch_lora<T, 16>(p, stream);
  }
}

// Whether one launch serves the call (whole one-pass pages, delta as wide as the plan, and a plan with a hand-over area whose
// launches put the workgroups of an item on its XCD), and is the faster form.  `units`: items the grid is sized for, which
// is the batch's own number only if the caller knows it (`counted`), else the plan's capacity or a quarter of it.
//
// Both sides measured in graphs of cold layers, us one launch / two, shrink + expand of q, k and v and in brackets of o:
//   ranks up to 16, hidden 4096: 8 items 4.6 / 5.6 (4.4 / 6.0), 80 10.7 / 11.9 (7.4 / 9.0), 232 22.4 / 22.5 (10.0 / 12.2), 296 27.0 / 26.8
//   (13.1 / 15.0), 528 38.9 / 36.6 (16.4 / 18.1); 5120: 272 34.8 / 36.1 (17.1 / 19.6), 336 42.3 / 40.1; 8192: 128 20.4 / 20.9 (13.7 /
//   15.8), 216 29.9 / 27.8 (17.2 / 18.2), 448 57.8 / 48.0 (28.2 / 27.2);
//   rank 32, 4096: 32 5.7 / 7.1 (5.0 / 6.9), 64 8.4 / 9.0 (6.5 / 7.6), 160 15.8 / 15.5 (9.1 / 10.2), 256 19.7 / 20.4 (10.0 / 11.0), 416 29.1 /
//   28.1 (14.3 / 14.8), 896 56.8 / 51.0 (22.2 / 22.9);
//   ranks to 64, 4096: 16 5.1 / 6.6 (5.0 / 6.5), 80 9.0 / 8.3 (6.8 / 6.9), 96 13.6 / 11.9 (8.2 / 8.1), 128 13.4 / 12.2 (7.9 / 8.3), 224 18.7 /
//   18.6 (10.0 / 10.1), 368 27.0 / 25.5 (14.3 / 12.8), 512 33.3 / 31.9 (15.6 / 15.1), 832 51.3 / 46.6 (20.8 / 21.2); 5120: 80 11.2 / 10.3
//   (7.3 / 8.5), 256 24.3 / 24.2 (12.3 / 12.4), 464 43.2 / 40.2 (19.8 / 18.3); 8192: 80 14.0 / 13.2 (9.0 / 9.9), 328 45.0 / 41.5 (20.5 / 20.5);
//   k and v a quarter or an eighth of a page, 4096: 80 7.3 / 8.3, 144 11.2 / 12.5, 280 17.9 / 17.8, 512 27.7 / 26.4; 8192: 88 11.8 / 14.0,
//   128 16.1 / 17.2, 192 22.7 / 23.2, 328 35.7 / 32.9.
// A launch whose shrink workgroups fit the chip at once saves the second launch, record and first data.  From there on the
// expand's pages compete with the shrink's loads, and already from about forty items where ranks go beyond 32 and all of q, k and v
// have outputs as wide as a page: there a run waits for the slowest of eight workgroups.  Of a capacity-sized grid most
// workgroups find no item, and the items are at most what the capacity holds beside the padding of the eight queues:
// 23 tokens, grid of 256 for 96 items, 18.0 / 14.0 (8.1 / 8.8); 8 tokens, 136, 10.5 / 9.9 (6.9 / 6.9); 4 tokens, 104, 5.5 / 7.2 (4.9 / 6.6); rank 8, 512
// tokens, 136 for 168, 20.7 / 22.6 (13.2 / 15.8).
bool lora_one_launch(const ExpandArgs& e, int64_t h_in, int64_t batch, int64_t rank_cap, int64_t units, bool counted, int nproj) {
  // (delta as wide as the plan lists: a launch over fewer columns would leave the words and counters of the others behind,
  // and a later one over all of them would wait for rows that name an older launch)
  if (h_in != e.page_elems || e.x_cols != rank_cap || !pages_serve(e, nproj, rank_cap) || !plan_hand_over(batch, rank_cap) ||
      units % kXcds != 0)
    return false;
  const int64_t resident = 256 * (e.page_elems <= ExpandPass<8>::kElems ? 4 : (e.page_elems <= ExpandPass<12>::kElems ? 3 : 2));
  const bool narrow = nproj == 3 && e.pages_shift[1] >= 2 && e.pages_shift[2] >= 2;
  if (e.x_cols <= 32 || narrow) return units * nproj <= resident;
  const int64_t items = counted ? units : plan_max_items(batch, rank_cap) - plan_padding_items(rank_cap);
  return items * nproj <= (nproj == 3 ? 128 : 256);
}

bool overlap(const void* a, int64_t a_bytes, const void* b, int64_t b_bytes) {
  const uintptr_t pa = reinterpret_cast<uintptr_t>(a), pb = reinterpret_cast<uintptr_t>(b);
  return pa < pb + (uint64_t)b_bytes && pb < pa + (uint64_t)a_bytes;
}

int lora_common(const void* plan, int64_t n_items, int64_t rank_cap, void* const y[3], void* const delta[3],
                const int64_t h_out[3], int nproj, int qkvo0, const void* x, const void* wa, const void* wb,
                const slora_tables* tables, const int64_t* bins, const void* scales, int scales_dtype, int64_t batch,
                int64_t h_in, int64_t delta_cols, int64_t page_elems, int64_t n_pages, int dtype, void* stream) {
  ShrinkArgs s{};
  PageArgs p{};
  int64_t grid_s = 0, grid_e = 0;
  int rc = shrink_prepare(plan, n_items, rank_cap, delta, nproj, qkvo0, x, wa, tables, bins, batch, h_in, delta_cols,
                          page_elems, n_pages, dtype, s, grid_s);
  if (rc != SLORA_OK) return rc == kNothingToDo ? SLORA_OK : rc;
  const void* xs[3] = {delta[0], delta[1], delta[2]};
  rc = expand_prepare(plan, n_items, rank_cap, y, xs, h_out, nproj, qkvo0, wb, tables, bins, scales, scales_dtype,
                      batch, delta_cols, page_elems, n_pages, dtype, p.e, grid_e);
  const bool expands = rc != kNothingToDo;
  if (expands && rc != SLORA_OK) return rc;
  // whole 16-byte pieces of delta, where anything reads it: a call without outputs is the shrink alone
  if (expands && (delta_cols & 7) != 0) return SLORA_ERR_UNSUPPORTED;
  // an output that shares memory with the activations: two launches read all of those before the first output is written
  bool in_place = false;
  for (int i = 0; i < nproj; ++i) in_place = in_place || overlap(x, batch * h_in * 2, y[i], batch * h_out[i] * 2);
  if (!expands || in_place || !lora_one_launch(p.e, h_in, batch, rank_cap, grid_s, grid_s == n_items, nproj)) {
    rc = slora_bgmv_shrink_planned(plan, rank_cap, n_items, nproj, delta[0], delta[1], delta[2], x, wa, tables, bins, batch,
                                   h_in, delta_cols, page_elems, n_pages, qkvo0, dtype, stream);
    if (rc != SLORA_OK || !expands) return rc;
    return slora_bgmv_expand_planned(plan, rank_cap, n_items, nproj, y[0], y[1], y[2], xs[0], xs[1], xs[2], wb, tables, bins,
                                     scales, scales_dtype, batch, delta_cols, h_out[0], h_out[1], h_out[2], page_elems,
                                     n_pages, qkvo0, dtype, stream);
  }
  fill_pages_shrink(p, s, nproj);
  fill_pages_expand(p, p.e, nproj);
  p.epochs = const_cast<int*>(p.plan) + plan_hand_offset(batch, rank_cap);
  p.words = reinterpret_cast<uint32_t*>(p.epochs + plan_max_items(batch, rank_cap) * kEpochWords);
  p.pitch = (int)plan_hand_pitch(rank_cap);
  p.spin_limit = 1 << 14;
  p.n_units = (int)grid_s;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  return dtype == SLORA_DTYPE_F16 ? dispatch_lora<F16>(p, page_elems, st) : dispatch_lora<BF16>(p, page_elems, st);
}

}  // namespace
}  // namespace slora

extern "C" {

int slora_bgmv_lora_planned(void* plan, int64_t rank_cap, int64_t n_items, int nproj, void* y0, void* y1, void* y2,
                            void* delta0, void* delta1, void* delta2, const void* x, const void* w_a, const void* w_b,
                            const slora_tables* tables, const int64_t* bins, const void* scales, int scales_dtype,
                            int64_t batch, int64_t h_in, int64_t delta_cols, int64_t h_out0, int64_t h_out1,
                            int64_t h_out2, int64_t page_elems, int64_t n_pages, int qkvo, int dtype, void* stream) {
  if (plan == nullptr) return SLORA_ERR_NULL_POINTER;
  if (rank_cap <= 0 || rank_cap > SLORA_MAX_RANK) return SLORA_ERR_BAD_SHAPE;
  if (nproj != 1 && nproj != 3) return SLORA_ERR_BAD_SHAPE;
  if (nproj == 3 && qkvo != 0) return SLORA_ERR_BAD_SHAPE;
  if (nproj == 1 && (qkvo < 0 || qkvo > 3)) return SLORA_ERR_BAD_SHAPE;
  void* ys[3] = {y0, y1, y2};
  void* ds[3] = {delta0, delta1, delta2};
  const int64_t hs[3] = {h_out0, h_out1, h_out2};
  return slora::lora_common(plan, n_items, rank_cap, ys, ds, hs, nproj, qkvo, x, w_a, w_b, tables, bins, scales,
                            scales_dtype, batch, h_in, delta_cols, page_elems, n_pages, dtype, stream);
}

}  // extern "C"
