// dispatch.hip — deterministic token->expert dispatch plan for gfx950.
//
// Replaces the host plan of MoELayer.decodeMany (Sources/FFAI/Models/
// MoELayer.swift:752-792: token-major (expert, token, slot) tuples, a stable
// sort by expert, inv_perm) and the host CSR offsets of the m1 path
// (:1035-1058), with no host round trip:
//   1. histogram of expert ids (LDS atomics: counts are order independent),
//   2. exclusive scan -> CSR offsets, plus the ascending list of used experts,
//   3. stable permute: entries are ranked inside each wave with ballots over
//      the expert-id bits, waves are ordered inside a tile, tiles in order, so
//      position = offsets[e] + (#earlier entries with expert e). The result is
//      the stable order (expert asc, token asc, slot asc) bit for bit.
//
// Small plans run in one workgroup, most others in one launch of a block per
// expert (plan_by_experts). The largest split the entries into chunks: a
// per-chunk histogram pass, a scan pass, and a scatter pass that starts every
// chunk at its own per-expert base.
#include <algorithm>

#include "moe_common.hpp"
#include "moe_internal.hpp"

namespace moe {

constexpr int kPlanThreads = 256;
constexpr int kPlanMaxE = 1024;
constexpr int kChunk = 1024;             // entries per chunk in the multi-block plan
constexpr int kSingleBlockMax = 1024;    // M at or below which one workgroup plans
// Whether a block per expert plans (plan_experts_kernel) rather than one
// workgroup (up to kSingleBlockMax entries) or the three passes over chunks. It
// holds the ids of a block in 32 registers per thread at most, reads E M ids, and
// one expert's entries are one block's to write, so it is kept to where it is the
// faster one (us of the plan, the other way / a block per expert; 10 to 40 % less
// with the GEMM's tiles in place of the used list):
//  - above 512 entries: 513 on 128 experts 4.8 / 3.4; with more than 512 experts
//    from 1024 (768 on 1024 experts 6.0 / 6.7, 1024 on 1024 7.0 / 6.7);
//  - to 32768 entries on up to 256 experts (12.1 / 8.7), 16384 above (512 experts
//    12.6 / 7.5, 1024 16.2 / 12.1; 32768 on 1024 20.8 / 28.3);
//  - to 8192 entries per expert on average (8192 on one 8.8 / 6.0, 16384 on one
//    8.9 / 10.1, 16384 on two 8.8 / 7.6, 32768 on two 9.7 / 13.3, on eight 10.3 /
//    8.5). Uneven loads move the line only at the far end: half of 16384 entries
//    on one of 128 experts 10.4 / 7.4, half of 32768 11.6 / 13.0.
constexpr int kPlanExpertsMin = 512, kPlanExpertsMax = 32768;
static bool plan_by_experts(int M, int E) {
  if (M <= kPlanExpertsMin || M > kPlanExpertsMax) return false;
  if (E > 512 && M < 1024) return false;
  if (E > 256 && M > kPlanExpertsMax / 2) return false;
  return M <= 8192 * E;
}

// Exclusive scan of cnt[0..E) over NT threads (4 experts per thread).
// Writes offsets[0..E], counts, the used list, and base[e] = offsets[e].
template <int NT = kPlanThreads>
__device__ void scan_experts(const uint32_t* cnt, int E, uint32_t* counts, uint32_t* offsets,
                             uint32_t* used, uint32_t* base) {
  __shared__ uint32_t wsum[NT / 64], wused[NT / 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  uint32_t c[4], f[4], tot = 0, ftot = 0;
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const int e = tid * 4 + j;
    c[j] = e < E ? cnt[e] : 0u;
    f[j] = c[j] > 0 ? 1u : 0u;
    tot += c[j];
    ftot += f[j];
  }
  // inclusive wave scan of (tot, ftot) by DPP (shuffles put an LDS round
  // trip per step on the plan's chain)
  const uint32_t s = wave_scan_u32(tot), fs = wave_scan_u32(ftot);
  if (lane == 63) {
    wsum[wave] = s;
    wused[wave] = fs;
  }
  __syncthreads();
  // the earlier waves' totals, all read at once
  uint32_t wb = 0, fb = 0;
#pragma unroll
  for (int w = 0; w < NT / 64; w++) {
    const uint32_t a = wsum[w], b = wused[w];
    wb += w < wave ? a : 0u;
    fb += w < wave ? b : 0u;
  }
  uint32_t run = wb + s - tot, frun = fb + fs - ftot;
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const int e = tid * 4 + j;
    if (e < E) {
      counts[e] = c[j];
      offsets[e] = run;
      base[e] = run;
      if (f[j]) used[1 + frun] = (uint32_t)e;
    }
    run += c[j];
    frun += f[j];
  }
  if (tid == NT - 1) {
    offsets[E] = run;
    used[0] = frun;
  }
  __syncthreads();
}

// Rank of this lane's entry among earlier lanes of the wave with the same
// expert, and the number of such lanes in the wave (valid lanes only).
__device__ __forceinline__ void wave_peers(uint32_t e, bool valid, int nbits, uint32_t* rank,
                                           uint32_t* count, bool* last) {
  const int lane = threadIdx.x & 63;
  uint64_t peers = __ballot(valid);
  for (int b = 0; b < nbits; b++) {
    const bool bit = (e >> b) & 1u;
    const uint64_t bal = __ballot(valid && bit);
    peers &= bit ? bal : ~bal;
  }
  const uint64_t below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  *rank = (uint32_t)__popcll(peers & below);
  *count = (uint32_t)__popcll(peers);
  *last = (peers >> lane) == 1ull;
}

// Ranks the entries [begin, end) in order and scatters them starting from
// cursor[e]; cursor ends advanced by the number of entries of each expert.
// NT threads; the waves take turns at the cursors, only those with entries.
template <int NT = kPlanThreads>
__device__ void stable_scatter(const uint32_t* __restrict__ idx, int begin, int end, int E,
                               int nbits, uint32_t* cursor, uint32_t* __restrict__ perm,
                               uint32_t* __restrict__ inv) {
  const int tid = threadIdx.x, wave = tid >> 6;
  for (int base = begin; base < end; base += NT) {
    const int m = base + tid;
    uint32_t e = m < end ? idx[m] : 0xffffffffu;
    const bool valid = m < end && e < (uint32_t)E;
    uint32_t rank, count;
    bool last;
    wave_peers(e, valid, nbits, &rank, &count, &last);
    const int nw = min(NT, end - base + 63) / 64;  // block-uniform
    for (int w = 0; w < nw; w++) {
      if (wave == w && valid) {
        const uint32_t pos = cursor[e] + rank;
        perm[pos] = (uint32_t)m;
        inv[m] = pos;
        if (last) cursor[e] += count;
      }
      __syncthreads();
    }
  }
}

// stable_scatter over entries [begin, begin + n) whose ids thread t already
// holds: ev[i] = the id of entry begin + t + NT i (n <= NT * PER), loaded
// all at once up front. Loading them tile by tile, after each tile's
// barriers, put one memory round trip per NT entries on the plan's
// critical path.
template <int NT, int PER>
__device__ void stable_scatter_held(const uint32_t (&ev)[PER], int begin, int n, int E, int nbits,
                                    uint32_t* cursor, uint32_t* __restrict__ perm,
                                    uint32_t* __restrict__ inv) {
  const int tid = threadIdx.x, wave = tid >> 6;
#pragma unroll
  for (int i = 0; i < PER; i++) {
    const int base = i * NT;
    if (base >= n) break;  // block-uniform
    const int o = base + tid, m = begin + o;
    const uint32_t e = o < n ? ev[i] : 0xffffffffu;
    const bool valid = o < n && e < (uint32_t)E;
    uint32_t rank, count;
    bool last;
    wave_peers(e, valid, nbits, &rank, &count, &last);
    const int nw = min(NT, n - base + 63) / 64;  // block-uniform
    for (int w = 0; w < nw; w++) {
      if (wave == w && valid) {
        const uint32_t pos = cursor[e] + rank;
        perm[pos] = (uint32_t)m;
        inv[m] = pos;
        if (last) cursor[e] += count;
      }
      __syncthreads();
    }
  }
}

__device__ __forceinline__ int id_bits(int E) {
  int nb = 0;
  while ((1 << nb) < E) nb++;
  return nb;
}

__global__ __launch_bounds__(kPlanThreads) void plan_single_kernel(
    const uint32_t* __restrict__ idx, int M, int E, uint32_t* counts, uint32_t* offsets,
    uint32_t* perm, uint32_t* inv, uint32_t* used) {
  __shared__ uint32_t cnt[kPlanMaxE], cursor[kPlanMaxE];
  constexpr int PER = kSingleBlockMax / kPlanThreads;
  const int tid = threadIdx.x;
  // every id of this thread's entries in flight at once, kept for the scatter
  uint32_t ev[PER];
#pragma unroll
  for (int i = 0; i < PER; i++) {
    const int m = tid + i * kPlanThreads;
    ev[i] = m < M ? idx[m] : 0xffffffffu;
  }
  for (int e = tid; e < E; e += kPlanThreads) cnt[e] = 0;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < PER; i++)
    if (ev[i] < (uint32_t)E) atomicAdd(&cnt[ev[i]], 1u);
  __syncthreads();
  scan_experts(cnt, E, counts, offsets, used, cursor);
  stable_scatter_held<kPlanThreads, PER>(ev, 0, M, E, id_bits(E), cursor, perm, inv);
}

// Routing and dispatch plan of a small batch in one launch: the NT / 64
// waves route tokens t = wave, wave + NT / 64, ... exactly as
// router_topk_kernel does (wave_topk, same results bit for bit), then the
// block plans the T * k entries as plan_single_kernel does, reading the ids
// from LDS. One wave per token past four tokens: the routing chain of a
// wave outlasts the launch it saves once a wave routes two tokens or more of
// a larger batch (Qwen3 shape, per layer step: 16 tokens on 4 waves 96.5 us
// against 90.7 us for the top-k and plan launches; 64 tokens on 16 waves
// 142.9 us against 133.6 us; 16 tokens on 16 waves 83.6 us against 84.4 us).
constexpr int kRoutePlanMaxT = 16;
constexpr int kRoutePlanMaxM = 1024;

template <typename XT, int EPL, int NT>
__global__ __launch_bounds__(NT) void route_plan_kernel(
    const XT* __restrict__ logits, int T, int E, int k, const RouteOpts ro, uint32_t* idx, float* w,
    uint32_t* counts, uint32_t* offsets, uint32_t* perm, uint32_t* inv, uint32_t* used) {
  __shared__ float sc[NT / 64][kTopkMaxE];
  __shared__ uint32_t sidx[kRoutePlanMaxM];
  __shared__ uint32_t cnt[kPlanMaxE], cursor[kPlanMaxE];
  const int tid = threadIdx.x, wv = tid >> 6, lane = tid & 63;
  const int M = T * k;
  for (int e = tid; e < E; e += NT) cnt[e] = 0;
  for (int t = wv; t < T; t += NT / 64) {  // wave-uniform
    int sel;
    float wt;
    wave_topk<XT, EPL>(logits + (size_t)t * E, E, k, ro, sc[wv], true, &sel, &wt);
    if (lane < k) {
      idx[t * k + lane] = (uint32_t)sel;
      w[t * k + lane] = wt;
      sidx[t * k + lane] = (uint32_t)sel;
    }
  }
  __syncthreads();
  for (int m = tid; m < M; m += NT) {
    const uint32_t e = sidx[m];
    if (e < (uint32_t)E) atomicAdd(&cnt[e], 1u);
  }
  __syncthreads();
  scan_experts<NT>(cnt, E, counts, offsets, used, cursor);
  stable_scatter<NT>(sidx, 0, M, E, id_bits(E), cursor, perm, inv);
}

hipError_t launch_route_plan(const void* logits, int dt, int T, int E, int k, const RouteOpts& ro,
                             uint32_t* idx, float* w, uint32_t* counts, uint32_t* offsets,
                             uint32_t* perm, uint32_t* inv, uint32_t* used, hipStream_t st) {
  if (T > kRoutePlanMaxT || T * k > kRoutePlanMaxM || E > kTopkMaxE || k > 64)
    return hipErrorInvalidValue;
#define MOE_RP(XT, EPL)                                                                          \
  if (T <= 4)                                                                                    \
    hipLaunchKernelGGL((route_plan_kernel<XT, EPL, kPlanThreads>), dim3(1), dim3(kPlanThreads),  \
                       0, st, (const XT*)logits, T, E, k, ro, idx, w, counts, offsets, perm, inv, \
                       used);                                                                    \
  else if (T <= 8)                                                                               \
    hipLaunchKernelGGL((route_plan_kernel<XT, EPL, 512>), dim3(1), dim3(512), 0, st,             \
                       (const XT*)logits, T, E, k, ro, idx, w, counts, offsets, perm, inv, used); \
  else                                                                                           \
    hipLaunchKernelGGL((route_plan_kernel<XT, EPL, 1024>), dim3(1), dim3(1024), 0, st,           \
                       (const XT*)logits, T, E, k, ro, idx, w, counts, offsets, perm, inv, used); \
  return hipGetLastError();
#define MOE_RP_E(XT)                  \
  if (E <= 64) { MOE_RP(XT, 1) }      \
  if (E <= 128) { MOE_RP(XT, 2) }     \
  if (E <= 256) { MOE_RP(XT, 4) }     \
  MOE_RP(XT, kTopkEPL)
  if (dt == DT_BF16) { MOE_RP_E(bf16_t) }
  if (dt == DT_F16) { MOE_RP_E(f16_t) }
  if (dt == DT_F32) { MOE_RP_E(float) }
#undef MOE_RP_E
#undef MOE_RP
  return hipErrorInvalidValue;
}

// The whole plan in one launch, a block per expert: every block reads all M ids
// (held in registers, 4 QUADS per thread; 1024 threads, each wave a contiguous
// share so that wave and lane order are token order), counts those below its
// expert (its offset) and its own, and writes its own entries in order. The
// E M id reads come from L2 (128 experts, 32768 ids: 16.8 MB) and cost less than
// the launches, the one-block scan and the waves' turns at the cursors that one
// workgroup or three passes over chunks take (us: 1998 ids 11.8 -> 5.0, 4000
// ids with the GEMM's row tiles 16.6 + 5.6 -> 5.5, 16384 ids on 256 experts
// 5.3 + 5.5 + 9.8 -> 6.3, 32768 on 128 experts 4.9 + 4.9 + 10.6 -> 9.0).
// items (nullable): also the GEMM's row tiles. Expert e's tiles start at slot
// offset / kGemmTileRows + e, which leaves room for every tile before them
// (ceil(c / R) <= floor((o + c) / R) - floor(o / R) + 1); a slot without a tile
// holds no rows (kGemmNoTile).
// used (nullable): the used list, which needs how many experts below e occur: a
// word per expert, set by plain stores (every store of a word writes the same
// value). With atomics on a bitmap, lanes of one word took turns: 32768 ids on 32
// experts 31.6 us, now 8.2; on 128 experts 14.9 -> 8.5.
template <int QUADS>
__global__ __launch_bounds__(1024) void plan_experts_kernel(
    const uint32_t* __restrict__ idx, int M, int E, uint32_t* __restrict__ counts,
    uint32_t* __restrict__ offsets, uint32_t* __restrict__ perm, uint32_t* __restrict__ inv,
    uint32_t* __restrict__ used, uint32_t* __restrict__ items) {
  __shared__ uint32_t wlt[16], weq[16];
  __shared__ uint32_t seen[kPlanMaxE];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t e = blockIdx.x;
  const rsrc_t iv = make_rsrc(idx, (uint32_t)M * 4u);
  // quad q of this lane: entries 4 ((wave QUADS + q) 64 + lane) + c
  u32x4_t id[QUADS];
#pragma unroll
  for (int q = 0; q < QUADS; q++) id[q] = bload128(iv, (uint32_t)((wave * QUADS + q) * 64 + lane) * 16u);
  if (used) seen[tid] = 0;  // kPlanMaxE threads
  uint32_t lt = 0, eq = 0;
#pragma unroll
  for (int q = 0; q < QUADS; q++)
#pragma unroll
    for (int c = 0; c < 4; c++) {
      const int m = 4 * ((wave * QUADS + q) * 64 + lane) + c;
      if (m >= M) id[q][c] = 0xFFFFFFFFu;  // past the end the view reads zeros
      lt += id[q][c] < e ? 1u : 0u;
      eq += id[q][c] == e ? 1u : 0u;
    }
  const uint32_t slt = wave_scan_u32(lt), seq = wave_scan_u32(eq);
  if (lane == 63) {
    wlt[wave] = slt;
    weq[wave] = seq;
  }
  __syncthreads();
  uint32_t off = 0, n = 0, at = 0;
#pragma unroll
  for (int w = 0; w < 16; w++) {
    const uint32_t a = wlt[w], b = weq[w];
    off += a;
    n += b;
    at += w < wave ? b : 0u;
  }
  if (used) {
#pragma unroll
    for (int q = 0; q < QUADS; q++)
#pragma unroll
      for (int c = 0; c < 4; c++)
        if (id[q][c] < e) seen[id[q][c]] = 1;
  }
  // this wave's entries of the expert, in order: quad by quad, lane by lane
  uint32_t run = off + at;
#pragma unroll
  for (int q = 0; q < QUADS; q++) {
    uint64_t b[4];
    uint32_t before = 0, all = 0;
#pragma unroll
    for (int c = 0; c < 4; c++) {
      b[c] = __ballot(id[q][c] == e);
      before += __builtin_amdgcn_mbcnt_hi((uint32_t)(b[c] >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)b[c], 0u));
      all += (uint32_t)__popcll(b[c]);
    }
    uint32_t p = run + before;
#pragma unroll
    for (int c = 0; c < 4; c++) {
      if (id[q][c] == e) {
        const uint32_t m = (uint32_t)(4 * ((wave * QUADS + q) * 64 + lane) + c);
        perm[p] = m;
        inv[m] = p;
        p++;
      }
    }
    run += all;
  }
  if (tid == 0) {
    counts[e] = n;
    offsets[e] = off;
    if (e == (uint32_t)E - 1u) offsets[E] = off + n;
  }
  if (items) {
    constexpr uint32_t R = kGemmTileRows;
    const uint32_t first = off / R + e, end = (off + n) / R + e + 1u;
    for (uint32_t t = (uint32_t)tid; t < end - first; t += 1024u) {
      const uint32_t r = t * R;
      const bool live = r < n;
      items[4 + 2 * (first + t)] = live ? e : kGemmNoTile;
      items[5 + 2 * (first + t)] = live ? (off + r) | ((min(n - r, R) - 1u) << kGemmRowShift) : 0u;
    }
    if (e == (uint32_t)E - 1u && tid == 0) items[0] = end;
  }
  if (used) {
    __syncthreads();
    if (wave == 0) {
      uint32_t rank = 0;
#pragma unroll
      for (int j = 0; j < kPlanMaxE / 64; j++) rank += (uint32_t)__popcll(__ballot(seen[64 * j + lane] != 0));
      if (lane == 0) {
        if (n) used[1 + rank] = e;
        if (e == (uint32_t)E - 1u) used[0] = rank + (n ? 1u : 0u);
      }
    }
  }
}

// Multi-block pass 1: per-chunk histograms, hist[c * E + e].
__global__ __launch_bounds__(kPlanThreads) void plan_hist_kernel(const uint32_t* __restrict__ idx,
                                                                 int M, int E,
                                                                 uint32_t* __restrict__ hist) {
  __shared__ uint32_t cnt[kPlanMaxE];
  const int tid = threadIdx.x, c = blockIdx.x;
  for (int e = tid; e < E; e += kPlanThreads) cnt[e] = 0;
  __syncthreads();
  const int begin = c * kChunk, end = min(M, begin + kChunk);
  for (int m = begin + tid; m < end; m += kPlanThreads) {
    const uint32_t e = idx[m];
    if (e < (uint32_t)E) atomicAdd(&cnt[e], 1u);
  }
  __syncthreads();
  for (int e = tid; e < E; e += kPlanThreads) hist[(size_t)c * E + e] = cnt[e];
}

// Multi-block pass 2 (one block): totals, scan, and each chunk's starting
// position per expert, written back over hist.
__global__ __launch_bounds__(kPlanThreads) void plan_scan_kernel(int nchunks, int E,
                                                                 uint32_t* __restrict__ hist,
                                                                 uint32_t* counts, uint32_t* offsets,
                                                                 uint32_t* used) {
  __shared__ uint32_t cnt[kPlanMaxE], base[kPlanMaxE];
  const int tid = threadIdx.x;
  // chunks in batches of kScanBatch: a batch's loads are all in flight
  // before the first add (one round trip per batch, not per chunk)
  constexpr int kScanBatch = 16;
  for (int e = tid; e < E; e += kPlanThreads) {
    uint32_t s = 0;
    for (int c0 = 0; c0 < nchunks; c0 += kScanBatch) {
      uint32_t h[kScanBatch];
#pragma unroll
      for (int j = 0; j < kScanBatch; j++)
        h[j] = (c0 + j < nchunks) ? hist[(size_t)(c0 + j) * E + e] : 0u;
#pragma unroll
      for (int j = 0; j < kScanBatch; j++) s += h[j];
    }
    cnt[e] = s;
  }
  __syncthreads();
  scan_experts(cnt, E, counts, offsets, used, base);
  for (int e = tid; e < E; e += kPlanThreads) {
    uint32_t run = base[e];
    for (int c0 = 0; c0 < nchunks; c0 += kScanBatch) {
      uint32_t h[kScanBatch];
#pragma unroll
      for (int j = 0; j < kScanBatch; j++)
        h[j] = (c0 + j < nchunks) ? hist[(size_t)(c0 + j) * E + e] : 0u;
#pragma unroll
      for (int j = 0; j < kScanBatch; j++) {
        if (c0 + j < nchunks) hist[(size_t)(c0 + j) * E + e] = run;
        run += h[j];
      }
    }
  }
}

// Multi-block pass 3: stable scatter of each chunk from its own bases.
__global__ __launch_bounds__(kPlanThreads) void plan_scatter_kernel(
    const uint32_t* __restrict__ idx, int M, int E, const uint32_t* __restrict__ hist,
    uint32_t* perm, uint32_t* inv) {
  __shared__ uint32_t cursor[kPlanMaxE];
  constexpr int PER = kChunk / kPlanThreads;
  const int tid = threadIdx.x, c = blockIdx.x;
  const int begin = c * kChunk, end = min(M, begin + kChunk);
  uint32_t ev[PER];  // the chunk's ids, all loads in flight at once
#pragma unroll
  for (int i = 0; i < PER; i++) {
    const int m = begin + tid + i * kPlanThreads;
    ev[i] = m < end ? idx[m] : 0xffffffffu;
  }
  for (int e = tid; e < E; e += kPlanThreads) cursor[e] = hist[(size_t)c * E + e];
  __syncthreads();
  stable_scatter_held<kPlanThreads, PER>(ev, begin, end - begin, E, id_bits(E), cursor, perm, inv);
}

__global__ void identity_plan_kernel(uint32_t* offsets, uint32_t* used, int M) {
  if (threadIdx.x == 0) {
    offsets[0] = 0;
    offsets[1] = (uint32_t)M;
    used[0] = 1;
    used[1] = 0;
  }
}

__global__ __launch_bounds__(kPlanThreads) void used_from_offsets_kernel(const uint32_t* offsets,
                                                                         int E, uint32_t* used) {
  __shared__ uint32_t cnt[kPlanMaxE], dummy_off[kPlanMaxE + 1], dummy_cnt[kPlanMaxE],
      dummy_base[kPlanMaxE];
  for (int e = threadIdx.x; e < E; e += kPlanThreads) cnt[e] = offsets[e + 1] - offsets[e];
  __syncthreads();
  scan_experts(cnt, E, dummy_cnt, dummy_off, used, dummy_base);
}

size_t dispatch_scratch_bytes(int T, int k, int E) {
  const long M = (long)T * k;
  if (M <= 4096) return 0;  // planned in one launch: the passes over chunks start above 8192
  const long nchunks = (M + kChunk - 1) / kChunk;
  return (size_t)(nchunks * E * 4);
}

// Row tiles of the grouped GEMM over an expert-sorted plan (the list format is
// described at launch_gemm_items), by block `blk` of `nblk`: every block counts
// each expert's tiles and scans the counts for its first one (thread t: experts
// t * EPT .. + EPT), then a wave per expert writes its tiles. With one thread per
// expert, a single expert's list was a chain of stores that grew with its rows (us
// of list and product at N 512, K 2048, 4 bits: 8192 rows 48.1 -> 44.9, 32768
// rows 139.9 -> 126.1). Without the scan, each expert from a slot its offset
// gives, the list's empty slots leave the XCDs with unequal shares of the tiles:
// for 256-row tiles up to a tenth of a layer step (8-bit, 32 experts of 2880 x
// 2880, 1800 tokens 655 -> 596).
__device__ __forceinline__ void gemm_items_body(const uint32_t* __restrict__ offsets, int E, int blk, int nblk,
                                                bool tall, uint32_t* __restrict__ items) {
  __shared__ uint32_t wsum[kPlanThreads / 64], start[kPlanMaxE];
  constexpr int EPT = kPlanMaxE / kPlanThreads;  // experts per thread
  const uint32_t R = tall ? kTallTileRows : kGemmTileRows;
  const int shift = tall ? kTallRowShift : kGemmRowShift;
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  uint32_t tiles[EPT], tot = 0;
#pragma unroll
  for (int j = 0; j < EPT; j++) {
    const int e = t * EPT + j;
    const uint32_t rows = e < E ? offsets[e + 1] - offsets[e] : 0u;
    tiles[j] = tall ? (rows + (uint32_t)kTallTileRows - 1u) / (uint32_t)kTallTileRows
                    : (rows + (uint32_t)kGemmTileRows - 1u) / (uint32_t)kGemmTileRows;  // constant divisors
    tot += tiles[j];
  }
  const uint32_t s = wave_scan_u32(tot);
  if (lane == 63) wsum[wave] = s;
  __syncthreads();
  uint32_t at = s - tot, all = 0;
#pragma unroll
  for (int w = 0; w < kPlanThreads / 64; w++) {
    at += w < wave ? wsum[w] : 0u;
    all += wsum[w];
  }
  if (blk == 0 && t == 0) items[0] = all;
#pragma unroll
  for (int j = 0; j < EPT; j++) {
    const int e = t * EPT + j;
    if (e < E) start[e] = at;
    at += tiles[j];
  }
  __syncthreads();
  for (int e = blk * (kPlanThreads / 64) + wave; e < E; e += nblk * (kPlanThreads / 64)) {
    const uint32_t off = offsets[e], n = offsets[e + 1] - off, first = start[e];
    for (uint32_t i = (uint32_t)lane; i * R < n; i += 64u) {
      const uint32_t r = i * R;
      items[4 + 2 * (first + i)] = (uint32_t)e;
      items[5 + 2 * (first + i)] = (off + r) | ((min(n - r, R) - 1u) << shift);
    }
  }
}
// Blocks of the list: a wave per expert, up to 32 blocks.
static int item_blocks(int E) { return std::min((E + kPlanThreads / 64 - 1) / (kPlanThreads / 64), 32); }

__global__ __launch_bounds__(kPlanThreads) void gemm_items_kernel(
    const uint32_t* __restrict__ offsets, int E, uint32_t* __restrict__ items, bool tall) {
  gemm_items_body(offsets, E, (int)blockIdx.x, (int)gridDim.x, tall, items);
}

// Multi-block pass 3 with the grouped GEMM's row tiles: each block scatters
// its chunk as plan_scatter_kernel does, and the blocks past the chunks write
// the tiles (they need only the offsets, which the scan pass wrote). One launch
// fewer per prefill step.
__global__ __launch_bounds__(kPlanThreads) void plan_scatter_items_kernel(
    const uint32_t* __restrict__ idx, int M, int E, const uint32_t* __restrict__ hist,
    uint32_t* perm, uint32_t* inv, const uint32_t* __restrict__ offsets,
    uint32_t* __restrict__ items, bool tall) {
  __shared__ uint32_t cursor[kPlanMaxE];
  constexpr int PER = kChunk / kPlanThreads;
  const int tid = threadIdx.x, c = blockIdx.x;
  const int nchunks = (M + kChunk - 1) / kChunk;
  if (c >= nchunks) {  // block-uniform, before any barrier
    gemm_items_body(offsets, E, c - nchunks, (int)gridDim.x - nchunks, tall, items);
    return;
  }
  const int begin = c * kChunk, end = min(M, begin + kChunk);
  uint32_t ev[PER];  // the chunk's ids, all loads in flight at once
#pragma unroll
  for (int i = 0; i < PER; i++) {
    const int m = begin + tid + i * kPlanThreads;
    ev[i] = m < end ? idx[m] : 0xffffffffu;
  }
  for (int e = tid; e < E; e += kPlanThreads) cursor[e] = hist[(size_t)c * E + e];
  __syncthreads();
  stable_scatter_held<kPlanThreads, PER>(ev, begin, end - begin, E, id_bits(E), cursor, perm, inv);
}

hipError_t launch_dispatch_plan(const uint32_t* idx, int T, int k, int E, uint32_t* counts,
                                uint32_t* offsets, uint32_t* perm, uint32_t* inv_perm,
                                uint32_t* used, void* scratch, size_t scratch_bytes,
                                hipStream_t st, uint32_t* items, bool tall, bool* items_done) {
  if (items_done) *items_done = false;
  const int M = T * k;
  if (E > kPlanMaxE) return hipErrorInvalidValue;
  if (plan_by_experts(M, E)) {
    if (tall) items = nullptr;  // a list without empty slots (launch_gemm_items)
#define MOE_PE(QUADS)                                                                              \
  hipLaunchKernelGGL((plan_experts_kernel<QUADS>), dim3(E), dim3(1024), 0, st, idx, M, E, counts,   \
                     offsets, perm, inv_perm, items ? nullptr : used, items)
    if (M <= 4096) MOE_PE(1);
    else if (M <= 8192) MOE_PE(2);
    else if (M <= 16384) MOE_PE(4);
    else MOE_PE(8);
#undef MOE_PE
    if (items_done) *items_done = items != nullptr;
    return hipGetLastError();
  }
  if (M <= kSingleBlockMax) {
    hipLaunchKernelGGL(plan_single_kernel, dim3(1), dim3(kPlanThreads), 0, st, idx, M, E, counts,
                       offsets, perm, inv_perm, used);
    return hipGetLastError();
  }
  const int nchunks = (M + kChunk - 1) / kChunk;
  if (scratch == nullptr || scratch_bytes < (size_t)nchunks * E * 4) return hipErrorInvalidValue;
  uint32_t* hist = reinterpret_cast<uint32_t*>(scratch);
  hipLaunchKernelGGL(plan_hist_kernel, dim3(nchunks), dim3(kPlanThreads), 0, st, idx, M, E, hist);
  hipLaunchKernelGGL(plan_scan_kernel, dim3(1), dim3(kPlanThreads), 0, st, nchunks, E, hist,
                     counts, offsets, used);
  if (items) {
    hipLaunchKernelGGL(plan_scatter_items_kernel, dim3(nchunks + item_blocks(E)), dim3(kPlanThreads), 0, st, idx,
                       M, E, hist, perm, inv_perm, offsets, items, tall);
    if (items_done) *items_done = true;
  } else {
    hipLaunchKernelGGL(plan_scatter_kernel, dim3(nchunks), dim3(kPlanThreads), 0, st, idx, M, E,
                       hist, perm, inv_perm);
  }
  return hipGetLastError();
}

hipError_t launch_gemm_items(const uint32_t* offsets, int E, uint32_t* items, bool tall, hipStream_t st) {
  if (E > kPlanMaxE) return hipErrorInvalidValue;
  hipLaunchKernelGGL(gemm_items_kernel, dim3(item_blocks(E)), dim3(kPlanThreads), 0, st, offsets, E, items, tall);
  return hipGetLastError();
}

hipError_t launch_identity_plan(uint32_t* offsets, uint32_t* used, int M, hipStream_t st) {
  hipLaunchKernelGGL(identity_plan_kernel, dim3(1), dim3(64), 0, st, offsets, used, M);
  return hipGetLastError();
}

hipError_t launch_used_from_offsets(const uint32_t* offsets, int E, uint32_t* used,
                                    hipStream_t st) {
  if (E > kPlanMaxE) return hipErrorInvalidValue;
  hipLaunchKernelGGL(used_from_offsets_kernel, dim3(1), dim3(kPlanThreads), 0, st, offsets, E,
                     used);
  return hipGetLastError();
}

}  // namespace moe
