// Decode kernels' straight line: pages of exactly one pass (hidden 4096, 5120, 6144 or 8192), plans that list every
// row of delta.  The shrink and the expand of a planned launch, by themselves (bgmv_decode.hip) or both in one
// launch with the delta rows handed over inside it (bgmv_lora.hip).
//
// What a launch of a few tokens waits for is one wavefront's chain of round trips and instructions, so the code that a
// wavefront runs through holds no test it could do without, and what only other runs need is kept out of its registers
// (page_args_again): with the general paths inlined as they were, a one-token shrink took 7.5 us of a launch
// that now takes 5.0 for both halves.  The shrink kernels spill no register.  The expand kernels spill up to 4 scalar ones and,
// at pages of 6144 elements, 2 or 3 vector ones (12 to 16 bytes of scratch; the f16 form over full-width outputs none: 128
// registers are what four workgroups per compute unit allow).
#pragma once

#include "bgmv_device.hpp"

namespace slora {
namespace {

constexpr int kFastRank = 128;  // largest rank of the vector path
constexpr int kDeltaBytes = kTT * kFastRank * 2 + kTT * 4;  // LDS of the hand-over: the run's delta rows, a word per wavefront

struct PageArgs {
  // what the straight line reads
  const int* plan;
  int* epochs;      // hand-over: kEpochWords per item
  uint32_t* words;  // hand-over: pitch words per (token, projection)
  const void* x;
  const void* wa;
  const void* wb;
  const void* scales;
  void* delta[3];
  void* y[3];
  int h_out[3], pages_shift[3];
  int d_cols, pitch, batch, rank_cap, qkvo0, scales_dtype, y_aligned, spin_limit;
  int n_units, nproj, strided, interleave;
  // what the rest is served from (pages_general)
  ExpandArgs e;
};

typedef const PageArgs __attribute__((address_space(4))) * KernArgs;

// The arguments of a kernel whose only parameter they are, read through the argument segment itself ...
__device__ __forceinline__ const PageArgs& page_args() {
  return *(const PageArgs*)(KernArgs)__builtin_amdgcn_kernarg_segment_ptr();
}
// ... and once more, for a path that is hardly ever taken: the compiler may not load in front of it what only it needs
__device__ __forceinline__ const PageArgs& page_args_again(const PageArgs& p) {
  KernArgs q = (KernArgs)&p;
  asm volatile("" : "+s"(q));
  return *(const PageArgs*)q;
}

// The thread's number as a value of its own: what is computed from it stays inside the loop over items that a launch
// hardly ever takes a second turn of (in front of it, dozens of lane masks fill the scalar registers).
__device__ __forceinline__ int thread_here() {
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));
  return tid;
}

// What a workgroup of one kind and projection reads of the arguments, in one group of scalar loads that nothing waits in
// front of (left to themselves the loads follow each other where each is first used: 8.2 -> 9.1 us for the expand of
// 23 tokens).
struct ShrinkHot {
  const int* plan;
  const void* x;
  const void* wa;
  void* delta;
  int* epochs;
  uint32_t* words;
  int d_cols, batch, rank_cap, qkvo0, pitch;
  __device__ __forceinline__ ShrinkHot(const PageArgs& p, int proj)
      : plan(p.plan), x(p.x), wa(p.wa), delta(p.delta[proj]), epochs(p.epochs), words(p.words), d_cols(p.d_cols),
        batch(p.batch), rank_cap(p.rank_cap), qkvo0(p.qkvo0), pitch(p.pitch) {
    asm volatile("" ::"s"(plan), "s"(x), "s"(wa), "s"(delta), "s"(epochs), "s"(words), "s"(d_cols), "s"(batch), "s"(rank_cap),
                 "s"(qkvo0), "s"(pitch));
  }
};
struct ExpandHot {
  const int* plan;
  const void* wb;
  const void* scales;
  const void* delta;
  void* y;
  int* epochs;
  uint32_t* words;
  int h_out, pages_shift, d_cols, batch, rank_cap, qkvo0, pitch, scales_dtype, y_aligned, spin_limit;
  __device__ __forceinline__ ExpandHot(const PageArgs& p, int proj)
      : plan(p.plan), wb(p.wb), scales(p.scales), delta(p.delta[proj]), y(p.y[proj]), epochs(p.epochs), words(p.words),
        h_out(p.h_out[proj]), pages_shift(p.pages_shift[proj]), d_cols(p.d_cols), batch(p.batch), rank_cap(p.rank_cap),
        qkvo0(p.qkvo0), pitch(p.pitch), scales_dtype(p.scales_dtype), y_aligned(p.y_aligned), spin_limit(p.spin_limit) {
    asm volatile("" ::"s"(plan), "s"(wb), "s"(scales), "s"(delta), "s"(y), "s"(epochs), "s"(words), "s"(h_out), "s"(pages_shift),
                 "s"(d_cols), "s"(batch), "s"(rank_cap), "s"(qkvo0), "s"(pitch), "s"(scales_dtype), "s"(y_aligned), "s"(spin_limit));
  }
};

// Runs whose pages are all whole one-pass pages inside the output, on the vector path.  In a one-launch LoRA (HAND) their
// readers take delta from the tagged words; the others read delta itself, which their producers store, and wait for, in
// front of the words.  (Both sides of the hand-over decide this from the run alone.)
__device__ __forceinline__ bool page_fast(int r, int pages_shift, int h_out, int y_aligned) {
  // (one test: no branch between what the record says and the loads that follow from it)
  const int rest = (r & (r - 1)) | (h_out & 7) | (pages_shift > 0 ? r & ((1 << pages_shift) - 1) : 0);
  return (rest == 0) & (r >= 8) & (r <= kFastRank) & (y_aligned != 0);
}

// memory operations of this wavefront acknowledged (vmcnt(0)) before anything that follows
__device__ __forceinline__ void wait_own_stores() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0x0F70);
  asm volatile("" ::: "memory");
}

// One workgroup: rows j0 .. j0 + 7 of one projection of an item, as shrink_fast computes them; wavefront w has rows
// w and w + 4.  HAND: the rows are also handed over; one without a page passes on what delta holds (readers wait for
// every row of the rank).  s_x: [kTT][NV * 64] LDS words.
template <typename T, int NV, bool HAND>
__device__ __forceinline__ int pages_shrink(const PageArgs& args, int unit, int proj, u32x4* s_x) {
  constexpr int XS = (NV + 3) / 4;  // activation vectors a thread stages per token
  const int tid = thread_here(), lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const ShrinkHot p(args, proj);
  const int proj_abs = p.qkvo0 + proj;
  int* ep = HAND ? p.epochs + (int64_t)unit * kEpochWords + proj_abs * 3 : nullptr;
  const int epoch = HAND ? *ep : 0;  // (arrives in front of the activations, which every wavefront waits for before the barrier)
  Item it;
  int page[2];
  load_item<true>(p.plan, unit, proj_abs, wave, wave + 4, p.batch, p.rank_cap, it, page[0], page[1]);
  const int r_eff = it.r < p.d_cols ? it.r : p.d_cols;
  if (it.n_tok <= 0) return it.plan_items;
  if (it.j0 >= r_eff) return it.plan_items;  // uniform over the workgroup; nobody waits for it
  const u32x4* xg = reinterpret_cast<const u32x4*>(p.x);
  u32x4 xr[kTT][XS];
#pragma unroll
  for (int t = 0; t < kTT; ++t) {
    if (t >= it.n_tok) break;
    const u32x4* xrow = xg + (int64_t)it.tok[t] * (NV * kWave);
#pragma unroll
    for (int i = 0; i < XS; ++i) {
      const int v = i * 256 + tid;
      xr[t][i] = xrow[v < NV * kWave ? v : 0];
    }
  }
  __builtin_amdgcn_sched_barrier(0);  // keep the activation loads in front: the LDS stores wait for them only
  u32x4 wv[2][NV];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const u32x4* src = reinterpret_cast<const u32x4*>(reinterpret_cast<const uint16_t*>(p.wa) +
                                                      (int64_t)(page[i] >= 0 ? page[i] : 0) * ExpandPass<NV>::kElems);
#pragma unroll
    for (int c = 0; c < NV; ++c) wv[i][c] = ldg16_stream(src + c * kWave + lane);
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int t = 0; t < kTT; ++t)
#pragma unroll
    for (int i = 0; i < XS; ++i) {
      const int v = i * 256 + tid;
      if (t < it.n_tok && v < NV * kWave) s_x[t * NV * kWave + v] = xr[t][i];
    }
  __syncthreads();
  // lane 4 i + t of the wavefront files row i, token t
  const int my_t = lane & 3, my_i = lane >> 2, my_row = it.j0 + wave + 4 * my_i, my_tok = item_token(it, my_t);
  const bool files = lane < 2 * kTT && my_t < it.n_tok && my_row < r_eff;
  const bool fast = !HAND || page_fast(it.r, args.pages_shift[proj], args.h_out[proj], args.y_aligned), have = (my_i == 0 ? page[0] : page[1]) >= 0;
  uint16_t* dst = reinterpret_cast<uint16_t*>(p.delta) + (int64_t)my_tok * p.d_cols + my_row;
  uint32_t* word = HAND ? p.words + ((int64_t)my_tok * 4 + proj_abs) * p.pitch + my_row : nullptr;
  uint16_t old = 0;
  if (HAND && (page[0] < 0 || page[1] < 0) && files) old = *dst;
  float mine = 0.f;
#pragma unroll
  for (int t = 0; t < kTT; ++t) {
    if (t < it.n_tok) {
      // (no test of the column in between: the activations of a token are read back to back)
      float acc[2] = {0.f, 0.f};
#pragma unroll
      for (int c = 0; c < NV; ++c) {
        const u32x4 xv = s_x[(t * NV + c) * kWave + lane];
#pragma unroll
        for (int i = 0; i < 2; ++i) acc[i] = dot8<T>(wv[i][c], xv, acc[i]);
      }
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const float sum = wave_sum(acc[i]);
        if (lane == 4 * i + t) mine = sum;
      }
    }
  }
  if (files) {
    uint16_t v = T::from_float(mine);
    if (!HAND) {
      if (have) *dst = v;
    } else {
      if (!have) v = old;
      if (!fast) {
        st16_coherent(dst, v);
        wait_own_stores();
      }
      __hip_atomic_store(word, (uint32_t)v | ((uint32_t)(epoch + 1) << 16), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (fast) *dst = v;
    }
  }
  if (HAND && tid == 0) *ep = epoch + 1;
  return it.plan_items;
}

// After a wait that lasted too long: the delta rows of the run by one wavefront, summed as pages_shrink sums them (the
// same bits), left in delta.
template <typename T, int NV>
__device__ __forceinline__ void pages_recompute(const PageArgs& args, const Item& it, int proj) {
  const PageArgs& p = page_args_again(args);
  const int lane = threadIdx.x & 63;
  const int proj_abs = p.qkvo0 + proj;
  const int r_eff = it.r < p.d_cols ? it.r : p.d_cols;
  uint16_t* y = reinterpret_cast<uint16_t*>(p.delta[proj]);
#pragma unroll 1
  for (int row = 0; row < r_eff; ++row) {
    const int64_t page = lookup_page(p.e.t, it.base + (int64_t)it.r * proj_abs + row);
    if (page < 0) continue;
    const u32x4* w = reinterpret_cast<const u32x4*>(reinterpret_cast<const uint16_t*>(p.wa) + page * ExpandPass<NV>::kElems);
#pragma unroll 1
    for (int t = 0; t < it.n_tok; ++t) {
      const int64_t tk = item_token(it, t);
      const u32x4* x = reinterpret_cast<const u32x4*>(p.x) + tk * (NV * kWave);
      float acc = 0.f;
#pragma unroll 1
      for (int v = lane; v < NV * kWave; v += kWave) acc = dot8<T>(w[v], x[v], acc);
      const float sum = wave_sum(acc);
      if (lane == 0) st16_coherent(y + tk * p.d_cols + row, T::from_float(sum));
    }
  }
  if (lane == 0)
    __hip_atomic_fetch_or(const_cast<int*>(p.plan) + PH_STATUS, kPlanStatusTimeout, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  wait_own_stores();
}

// A wavefront's share of the expand of a run that is not page_fast, page k: element by element, with HAND from delta
// itself once every row of every token has been handed over.
template <typename T, int NV, bool HAND>
__device__ __forceinline__ void pages_general(const PageArgs& args, const Item& it, int proj, int k, int epoch) {
  const PageArgs& p = page_args_again(args);
  const int lane = threadIdx.x & 63;
  const int proj_abs = p.qkvo0 + proj;
  const int r_eff = it.r < p.d_cols ? it.r : p.d_cols;
  if (HAND) {
    const uint32_t tag = (uint32_t)(epoch + 1) << 16;
    const uint32_t* words = p.words + (int64_t)proj_abs * p.pitch;
#pragma unroll 1
    for (int spins = 0;; ++spins) {
      bool ok = true;
#pragma unroll 1
      for (int t = 0; t < it.n_tok; ++t)
#pragma unroll 1
        for (int d = lane; d < r_eff; d += kWave) {
          const uint32_t v = __hip_atomic_load(words + (int64_t)item_token(it, t) * 4 * p.pitch + d, __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_AGENT);
          ok = ok && (v & 0xffff0000u) == tag;
        }
      if (__ballot(!ok) == 0) break;
      if (spins >= p.spin_limit) {
        pages_recompute<T, NV>(p, it, proj);
        break;
      }
      __builtin_amdgcn_s_sleep(4);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  }
  if (r_eff <= 0) return;
  // page k, and on the run's last listed item the pages that no item lists
  const int n_pg = expand_pages(p.e, proj, it.r);
  const int64_t base_li = it.base + (int64_t)it.r * proj_abs;
  const float scale = load_scale(p.scales, p.scales_dtype, it.a);
#pragma unroll 1
  for (int kk = k; kk < n_pg; kk += kRB) {
    expand_scalar<T, HAND>(p.e, proj, it, r_eff, kk, base_li, scale);
    if (!it.more) break;
  }
}

// The arithmetic of a page for a run whose outputs are shared by LPO lanes each (see expand_update, which it is for
// a page in one pass).  s_strip: kTT strips of the wavefront.
template <typename T, int NV, int LPO>
__device__ __forceinline__ void page_update(const Item& it, uint16_t* y, int h_stride, const u32x4 (&wv)[NV],
                                            const u32x4 (&xv)[kTT], const u32x4 (&yv)[kTT], int n_page0, int n_end,
                                            float scale, int lane, uint16_t* s_strip) {
  constexpr int OPW = kWave / LPO, kOut = NV * OPW;  // outputs of a load, of the page
  const int n_mine = n_page0 + lane * 8;
  const bool y_ok = lane * 8 < kOut && n_mine < n_end;
  // every token's sums into a strip of its own, then every token's outputs: the way through LDS is paid once
#pragma unroll
  for (int t = 0; t < kTT; ++t) {
    if (t < it.n_tok) {
#pragma unroll
      for (int g8 = 0; g8 < ExpandPass<NV>::kGroups; ++g8) {
        float part[kVecPerPass];
#pragma unroll
        for (int c = 0; c < kVecPerPass; ++c)
          part[c] = g8 * kVecPerPass + c < NV ? dot8<T>(wv[g8 * kVecPerPass + c < NV ? g8 * kVecPerPass + c : 0], xv[t], 0.f) : 0.f;
        file_sums<T, LPO>(part, scale, lane, s_strip + t * ExpandPass<NV>::kStrip + g8 * kVecPerPass * OPW);
      }
    }
  }
  // the same wavefront wrote the strips: its LDS operations complete in order
#pragma unroll
  for (int t = 0; t < kTT; ++t) {
    if (t < it.n_tok) {
      uint16_t* yt = y + (int64_t)it.tok[t] * h_stride;
      const uint16_t* strip = s_strip + t * ExpandPass<NV>::kStrip;
      const u32x4 dv = *reinterpret_cast<const u32x4*>(strip + (y_ok ? lane * 8 : 0));
      if (y_ok) {
        u32x4 out;
#pragma unroll
        for (int q = 0; q < 4; ++q) out[q] = T::add2(yv[t][q], dv[q]);
        stg16_stream(yt + n_mine, out);
      }
      if (kOut > 8 * kWave) {
        // outputs 512.. of the page (rank 8 and wide pages only): y is loaded here, behind the sums
#pragma unroll 1
        for (int s0 = 8 * kWave; s0 < kOut; s0 += 8 * kWave) {
          const int n2 = n_mine + s0;
          if (s0 + lane * 8 < kOut && n2 < n_end) {
            const u32x4 y2 = ldg16_stream(yt + n2);
            const u32x4 d2 = *reinterpret_cast<const u32x4*>(strip + s0 + lane * 8);
            u32x4 out;
#pragma unroll
            for (int q = 0; q < 4; ++q) out[q] = T::add2(y2[q], d2[q]);
            stg16_stream(yt + n2, out);
          }
        }
      }
    }
  }
}

// One workgroup: pages 4 h .. 4 h + 3 of an item's block (h = sub % 2) of projection sub / 2, one a wavefront.
// s_strip: kTT strips of the wavefront; s_delta (HAND): kDeltaBytes.
template <typename T, int NV, bool HAND>
__device__ __forceinline__ int pages_expand(const PageArgs& args, int unit, int sub, uint16_t* s_strip, uint32_t* s_delta) {
  const int tid = thread_here(), lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int proj = sub >> 1;
  const ExpandHot p(args, proj);
  const int proj_abs = p.qkvo0 + proj;
  const int jr = (sub & 1) * 4 + wave;  // page inside the item's block
  int* ep = HAND ? p.epochs + (int64_t)unit * kEpochWords + proj_abs * 3 + 1 + (sub & 1) : nullptr;
  int epoch = HAND ? *ep : 0;
  Item it;
  int page = -1, page_unused = -1;
  load_item<true>(p.plan, unit, proj_abs, jr, jr, p.batch, p.rank_cap, it, page, page_unused);
  if (it.n_tok <= 0) return it.plan_items;
  if (HAND) {
    epoch = __builtin_amdgcn_readfirstlane(epoch);
    asm volatile("" : "+s"(epoch));
  }
  const int r = it.r, r_eff = r < p.d_cols ? r : p.d_cols;
  const int sh = p.pages_shift, n_pg = sh > 0 ? (r + (1 << sh) - 1) >> sh : r;
  int k = it.j0 + jr;
  const bool fast = page_fast(r, sh, p.h_out, p.y_aligned);
  if (!fast || (k - wave >= n_pg && !it.more)) {  // (uniform over the workgroup)
    if (HAND) {
      __builtin_amdgcn_s_barrier();  // all four wavefronts have read the word
      if (tid == 0) *ep = epoch + 1;
    }
    if (!fast && (k < n_pg || it.more)) pages_general<T, NV, HAND>(args, it, proj, k, epoch);
    return it.plan_items;
  }
  const int lg_r = __builtin_ctz((unsigned)r), lpo = r >> 3;
  const int h_stride = p.h_out;
  uint16_t* y = reinterpret_cast<uint16_t*>(p.y);
  const int outs = ExpandPass<NV>::kElems >> lg_r;
  const int d0 = (lane & (lpo - 1)) * 8;
  const uint32_t scale_bits = scale_word(p.scales, p.scales_dtype, it.a);
  bool wait = HAND;  // the rows of the run are still to be waited for
  for (;;) {
    const bool mine = k < n_pg && page >= 0;  // a wavefront without a page only helps with the hand-over
    if (wait || mine) {
      const uint16_t* wpage = reinterpret_cast<const uint16_t*>(p.wb) + (int64_t)(mine ? page : 0) * ExpandPass<NV>::kElems;
      const int n_page0 = mine ? k * outs : 0;
      const int n_end = h_stride < n_page0 + outs ? h_stride : n_page0 + outs;
      u32x4 wv[NV], yv[kTT], xv[kTT];
#pragma unroll
      for (int c = 0; c < NV; ++c) wv[c] = ldg16_stream(wpage + (c * kWave + lane) * 8);
      const int n_mine = lane * 8 < outs && n_page0 + lane * 8 < n_end ? n_page0 + lane * 8 : n_page0;
      // (a token the run does not have re-reads the first one's row: a test per token in between costs more, 19.8 -> 23.1
      // us for q, k and v of S2; lanes with no outputs re-read the page's first ones; neither value is used)
#pragma unroll
      for (int t = 0; t < kTT; ++t)
        yv[t] = ldg16_stream(y + (int64_t)(t < it.n_tok ? it.tok[t] : it.tok[0]) * h_stride + n_mine);
      const uint16_t* delta = reinterpret_cast<const uint16_t*>(p.delta) + (d0 < r_eff ? d0 : 0);
      if (!HAND) {
#pragma unroll
        for (int t = 0; t < kTT; ++t) xv[t] = ldg16(delta + (int64_t)(t < it.n_tok ? it.tok[t] : it.tok[0]) * p.d_cols);
      } else {
        if (wait) {
          // wavefront t waits for the delta row of token t, two columns a lane, and leaves it in LDS
          wait = false;
          uint32_t* s_row = s_delta + wave * (kFastRank / 2);
          int late = 0;
          if (wave < it.n_tok) {
            const uint32_t tag = (uint32_t)(epoch + 1) << 16;
            const bool reads = 2 * lane < r_eff;
            const uint64_t* pair =
                reinterpret_cast<const uint64_t*>(p.words + ((int64_t)item_token(it, wave) * 4 + proj_abs) * p.pitch) + (reads ? lane : 0);
#pragma unroll 1
            for (int spins = 0;; ++spins) {
              const uint64_t v = __hip_atomic_load(pair, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
              const uint32_t lo = (uint32_t)v, hi = (uint32_t)(v >> 32);
              if (__ballot((((lo ^ tag) | (hi ^ tag)) >> 16) != 0) == 0) {
                if (2 * lane < kFastRank) s_row[lane] = (lo & 0xffffu) | (hi << 16);
                break;
              }
              if (spins >= p.spin_limit) {
                late = 1;
                break;
              }
              __builtin_amdgcn_s_sleep(2);
            }
          }
          if (lane == 0) s_delta[kTT * kFastRank / 2 + wave] = (uint32_t)late;
          // LDS writes of this wavefront done (lgkmcnt(0); the loads above stay on their way), then meet
          asm volatile("" ::: "memory");
          __builtin_amdgcn_s_waitcnt(0xC07F);
          __builtin_amdgcn_s_barrier();
          asm volatile("" ::: "memory");
          if (tid == 0) *ep = epoch + 1;
        }
#pragma unroll
        for (int t = 0; t < kTT; ++t) xv[t] = *reinterpret_cast<const u32x4*>(s_delta + t * (kFastRank / 2) + d0 / 2);
        const u32x4 any_late = *reinterpret_cast<const u32x4*>(s_delta + kTT * kFastRank / 2);
        if (__builtin_amdgcn_readfirstlane((int)(any_late[0] | any_late[1] | any_late[2] | any_late[3])) != 0 && mine) {
          pages_recompute<T, NV>(args, it, proj);
#pragma unroll
          for (int t = 0; t < kTT; ++t)
            if (t < it.n_tok) xv[t] = ldg16_coherent(delta + (int64_t)it.tok[t] * p.d_cols);
        }
      }
      if (mine) {
        if (r_eff < r) {  // delta is narrower than the rank: the columns behind it count nothing
#pragma unroll
          for (int t = 0; t < kTT; ++t)
            if (d0 >= r_eff) xv[t] = zero16();
#pragma unroll
          for (int c = 0; c < NV; ++c)
            if (d0 >= r_eff) wv[c] = zero16();
        }
        const float scale = scale_of(scale_bits, p.scales, p.scales_dtype, it.a);
        switch (lpo) {
          case 1: page_update<T, NV, 1>(it, y, h_stride, wv, xv, yv, n_page0, n_end, scale, lane, s_strip); break;
          case 2: page_update<T, NV, 2>(it, y, h_stride, wv, xv, yv, n_page0, n_end, scale, lane, s_strip); break;
          case 4: page_update<T, NV, 4>(it, y, h_stride, wv, xv, yv, n_page0, n_end, scale, lane, s_strip); break;
          case 8: page_update<T, NV, 8>(it, y, h_stride, wv, xv, yv, n_page0, n_end, scale, lane, s_strip); break;
          default: page_update<T, NV, 16>(it, y, h_stride, wv, xv, yv, n_page0, n_end, scale, lane, s_strip); break;
        }
      }
    }
    // (a plan of less than the adapter's rank) the run's last listed item: the pages that no item lists
    if (!it.more) return it.plan_items;
    k += kRB;
    if (k >= n_pg) return it.plan_items;
    const PageArgs& q = page_args_again(args);
    page = (int)lookup_page(q.e.t, it.base + (int64_t)r * proj_abs + k);
  }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
bool whole_pages(int64_t page_elems) {
  return page_elems == ExpandPass<8>::kElems || page_elems == ExpandPass<10>::kElems ||
         page_elems == ExpandPass<12>::kElems || page_elems == ExpandPass<16>::kElems;
}

// Whether pages_expand serves an expand: pages of exactly one pass, outputs of whole pages (or an eighth of one: grouped-
// query k and v), every row of delta listed.
bool pages_serve(const ExpandArgs& e, int nproj, int64_t rank_cap) {
  for (int i = 0; i < nproj; ++i)
    if (e.pages_shift[i] != -1 && (e.pages_shift[i] < 1 || e.pages_shift[i] > 3)) return false;
  return whole_pages(e.page_elems) && e.x_cols <= rank_cap && (e.x_cols & 7) == 0;
}

void fill_pages_shrink(PageArgs& p, const ShrinkArgs& s, int nproj) {
  p.plan = s.plan;
  p.x = s.x;
  p.wa = s.w;
  p.d_cols = s.y_cols;
  p.batch = s.batch;
  p.rank_cap = s.rank_cap;
  p.qkvo0 = s.qkvo0;
  p.strided = s.strided;
  p.nproj = nproj;
  for (int i = 0; i < 3; ++i) p.delta[i] = s.y[i];
}

void fill_pages_expand(PageArgs& p, const ExpandArgs& e, int nproj) {
  p.plan = e.plan;
  p.wb = e.w;
  p.d_cols = e.x_cols;
  p.batch = e.batch;
  p.rank_cap = e.rank_cap;
  p.qkvo0 = e.qkvo0;
  p.strided = e.strided;
  p.nproj = nproj;
  p.scales = e.scales;
  p.scales_dtype = e.scales_dtype;
  p.y_aligned = e.y_aligned;
  p.interleave = 0;
  for (int i = 0; i < 3; ++i) {
    p.delta[i] = const_cast<void*>(e.x[i]);
    p.y[i] = e.y[i];
    p.h_out[i] = e.h_out[i];
    p.pages_shift[i] = e.pages_shift[i];
    if (i < nproj && p.pages_shift[i] > 0) p.interleave = 1;  // an output narrower than a page
  }
  p.e = e;
}

}  // namespace
}  // namespace slora
