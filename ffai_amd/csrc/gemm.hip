// gemm.hip — prefill-side grouped dequant GEMM on the gfx950 matrix cores.
//
// Replaces Ops.moeGatherDequantGemmInt4 bm8/bm16/bm64/m1
// (Sources/FFAI/Ops/Ops.swift:4553-5201, 6499-6585) with the tile choice of
// MoELayer.swift:855-882, generalised to 2/3/4/5/6/8-bit weights, group sizes
// 32/64/128 and scale dtypes independent of the activation dtype:
//   gate/up:  act[p, n] = act_fn(round(Wg[e(p)][n] . x[row(p)]),
//                                round(Wu[e(p)][n] . x[row(p)]))
//   single:   out[p, n] = round(W[e(p)][n] . a[p])
// over the expert-sorted positions p of a dispatch plan.
//
// Operands are f16 on v_mfma_f32_16x16x32_f16 (weights as A, activations as B,
// so that a lane's accumulators are consecutive output columns of one row):
//  - weights are dequantised exactly to s * q + b rounded once to f16
//    (2^-12 relative; bf16 operands would round them to 2^-9): 4-bit codes
//    become f16 q through the scaled fp8 conversion, other widths enter as
//    1024 + q (exact in f16) less 1024; one packed fma gives s * q + b;
//  - activations of an f16 layer are used as they are; those of a bf16 layer
//    are scaled by 2^-8 into f16 range (exact for magnitudes 2^-6 .. 1.6e7,
//    saturating beyond) beforehand (launch_to_a16, and the gate/up epilogue
//    writes its activation in that form for the down GEMM); the epilogue
//    multiplies the fp32 sums by 2^8.
//
// Work: row tiles of up to 96 rows of an expert, listed on the device from the
// CSR offsets (launch_gemm_items), times column blocks of 128 weight rows (64
// gate and 64 up rows for a pair). A block is four waves side by side over the
// weight rows, two 16-row weight tiles each, over 2, 4 or 6 16-row activation
// tiles (32-row steps, a compile-time loop each). Blocks b, b + 8, ... run on
// one XCD: the (tile, column block) pairs are split into 8 contiguous ranges,
// so neighbouring column blocks of a row tile share its L2.
//
// The split: at 64 to 128 rows per expert neither the matrix cores nor HBM
// bind; what did was one large block per CU waiting on its own chunk (two
// waves per SIMD in lockstep, weights through LDS) and bytes through the CU's
// L1: about 33 bytes per clock arrive from L2. So blocks are small (53 KB of
// LDS, 168 VGPRs: three per CU), weights go from memory straight to the
// operand registers of the one wave that uses them, and every byte fetched is
// used: K is permuted so that lane (n, kb) holds whole 32-value units (unit
// 4 c + kb of weight row n in chunk c; the MFMA's k index is free as long as
// both operands agree), two chunks of codes are loaded together (one 128-byte
// line of a row at 4 bits), and scales pass through a wave-private LDS table 8
// groups at a time (loaded per chunk, each word cost a line visit per row).
// Per 128-value chunk the activation rows are copied from memory into one of
// two LDS stages (buffer loads with the LDS flag) under the products of the
// chunk before; one block barrier per chunk.
// Measured against 256- and 128-row tiles of 512 threads, one block per CU,
// with the weights through LDS (us per layer step): 2048 tokens on 256 3/6-bit
// experts 347 -> 289 (gate/up launch 189 -> 153, down 119 -> 99), 1000 tokens
// on 32 experts of 2880 x 2880 at 4 bits 393 -> 358, 4096 tokens on 128 experts
// with Zipf loads 460-494 -> 461-478 by box and run (gate/up launch 270 -> 261,
// down 150 -> 154). From some hundreds of rows per expert on, tall tiles share a
// weight fetch better: gemm_tall.hip (gemm_tall in api.cpp has the line).
// Storing the tile through LDS, whole row segments at a time, changed nothing
// (470 / 286 / 357 us against 470 / 288 / 355 for the last, first and second case).
// Not kept: 256 weight rows per block (four 16-row tiles per wave, 2 waves per
// SIMD; the three cases 333 / 429 / 479 us), scales loaded per chunk and one
// chunk of codes at a time (314 / 382 / 489).
#include <hip/hip_ext.h>

#include <type_traits>

#include "gemm_units.hpp"

#ifndef MOE_BITS
#define MOE_BITS 4
#endif

namespace moe {

typedef float f32x4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4_t mma16(u32x4_t a, u32x4_t b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a),
                                                __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
}

constexpr int kGBK = 128;  // values per K chunk (256 bytes of an LDS row)

// A stage row is 256 bytes (one chunk), the banks repeat every 256 bytes, and a
// 16-byte read serves 16 lanes per cycle: not 16 neighbours, but lanes 0-3,
// 12-15, 20-27 of 32 and then the rest. The 16-byte piece q of row r sits at
// slot q ^ p(r), p a permutation of r & 15 whose upper bits make the rows
// {0-3, 12-15} and {4-11} each fill a pair of quarters that kb ^ 1 swaps: the
// lanes (n, kb) of a fragment read (piece 4 kb + s) then cover every bank under
// that order and under plain neighbours; with p(r) = r half of them met (3.4
// conflict cycles per read counted; 362 -> 357 us at 1000 tokens on 32 experts,
// 475 -> 472 at 4096 on 128). Four neighbouring slots stay four neighbouring
// pieces, so a row's copy from memory is 64 bytes at a time.
__host__ __device__ constexpr uint32_t stage_perm(uint32_t r) {
  return (r & 3u) | (((r >> 2) ^ (r >> 3)) & 1u) << 3 | ((r >> 3) & 1u) << 2;
}
__device__ __forceinline__ uint32_t stage_slot(uint32_t q, uint32_t r) { return q ^ stage_perm(r & 15u); }

// A unit's 16-bit scale and bias (bf16 or f16 storage) as an f16 pair. Both
// conversions are computed and one is selected (a branch on the storage type
// here split every chunk of the main loop into a dozen basic blocks).
__device__ __forceinline__ h2_t sb_h2(uint32_t raw, bool bf16) {
  // bf16: exact inside f16's range
  const h2_t from_bf{(_Float16)__uint_as_float(raw << 16), (_Float16)__uint_as_float(raw & 0xFFFF0000u)};
  return bf16 ? from_bf : __builtin_bit_cast(h2_t, raw);
}

// LDS of a block: six 8 KB objects (two 16-row tiles of a chunk each), so that
// the compiler tracks the memory-to-LDS copies into each on their own.
constexpr int kGemmObjBytes = 32 * 256;
struct GemmLds {
  unsigned char *a0, *a1, *a2, *a3, *a4, *a5;
  uint32_t* sb;  // [4 waves][2 tiles][8 groups][16 rows] scale and bias pairs
};

// Register sets of weight codes, one per chunk. Up to 4 bits a chunk is at
// most half a 128-byte line of a weight row: two chunks' loads go out
// together, so that both come from one fetch of the line.
template <int BITS> struct GemmDepth {
  static constexpr int NSET = BITS > 4 ? 2 : 4;
};

template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (N > 0) {
    static_for<N - 1>(f);
    f(std::integral_constant<int, N - 1>{});
  }
}

// One block's tile: MT 16-row tiles of activation rows from m0 (`rows` of the
// rows hold positions of expert e), weight rows of column block bn.
template <int MT, int BITS, typename XT, bool GATEUP>
__device__ __forceinline__ void gemm_tile(const GemmArgs& a, const GemmLds L, uint32_t e, uint32_t m0,
                                          int bn, uint32_t rows) {
  constexpr int NT = 2;              // 16-row weight tiles per wave (a pair: gate and up)
  constexpr int NSET = GemmDepth<BITS>::NSET, TRIP = 4;  // chunks per loop trip
  constexpr float OSCALE = __is_same(XT, bf16_t) ? (float)(1 << kA16Shift) : 1.0f;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n16 = lane & 15, kb = lane >> 4;
  const int N = a.N, K = a.K, CU = K >> 5, groups = CU >> a.gsh, row_words = CU * BITS;
  const int nchunks = (K + kGBK - 1) / kGBK;  // the last may hold two units only
  const bool half_tail = K % kGBK != 0;
  const bool sb_bf16 = a.sb_bf16 != 0;
  // row tile I of stage ST: 4 KB in object (ST MT + I) / 2
  auto tile_lds = [&](auto st, auto it) -> unsigned char* {
    constexpr int T = decltype(st)::value * MT + decltype(it)::value, O = T / 2;
    return (O == 0 ? L.a0 : O == 1 ? L.a1 : O == 2 ? L.a2 : O == 3 ? L.a3 : O == 4 ? L.a4 : L.a5) +
           (T & 1) * 4096;
  };

  // ---- activations: this lane copies, of each row tile, slot n16 of row arow
  const rsrc_t xr = make_rsrc(a.x, (uint32_t)min((size_t)a.x_rows * K * 2u, (size_t)0xFFFFFFFFu));
  const rsrc_t permv = make_rsrc(a.perm, (uint32_t)__builtin_amdgcn_readfirstlane(a.perm ? -1 : 0));
  const uint32_t arow = (uint32_t)(4 * wave + kb);
  uint32_t xpos[MT], praw[MT], xoff[MT];
#pragma unroll
  for (int i = 0; i < MT; i++) {
    xpos[i] = m0 + min(16u * i + arow, rows - 1u);
    praw[i] = bload32(permv, xpos[i] * 4u);
  }
  auto set_xoff = [&]() -> void {
    const uint32_t piece = stage_slot((uint32_t)n16, arow);
#pragma unroll
    for (int i = 0; i < MT; i++) {
      const uint32_t xrow = a.perm ? praw[i] / (uint32_t)a.topk : xpos[i];
      xoff[i] = (xrow * (uint32_t)K + 8u * piece) * 2u;
    }
  };
  // chunk's rows into stage st (past the last chunk: offsets past the view's
  // end or never read)
  auto dma_a = [&](int chunk, auto st) -> void {
    const uint32_t coff = chunk < nchunks ? (uint32_t)(chunk * kGBK * 2) : 0x80000000u;
    static_for<MT>([&](auto it) -> void {
      unsigned char* dst = tile_lds(st, it) + wave * 1024;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, (__attribute__((address_space(3))) void*)dst, 16,
                                               xoff[decltype(it)::value] + coff, 0, 0, 0);
    });
  };

  // ---- weights: lane (n16, kb) holds unit 4 c + kb of weight row n16 of both
  // tiles. The two tiles of a single projection interleave their rows in
  // fours so that a lane's outputs are 8 consecutive columns. Rows past N
  // read zeros through the expert's view.
  const int r0 = GATEUP ? bn * 64 + 16 * wave + n16 : bn * 128 + 32 * wave + 8 * (n16 >> 2) + (n16 & 3);
  constexpr int kTileRow = GATEUP ? 0 : 4;  // the second tile's rows
  const size_t erows = (size_t)e * (size_t)N;
  const uint32_t row_bytes = (uint32_t)row_words * 4u;
  const rsrc_t w0 = make_rsrc(a.p0.w + erows * row_words, (uint32_t)N * row_bytes);
  const rsrc_t w1 = make_rsrc((GATEUP ? a.p1.w : a.p0.w) + erows * row_words, (uint32_t)N * row_bytes);
  const uint32_t woff = (uint32_t)r0 * row_bytes + (uint32_t)(kb * BITS * 4);
  struct WSet {
    uint32_t w[NT][BITS];
  };
  auto load_set = [&](int chunk, WSet& u) -> void {
    const uint32_t coff = chunk < nchunks ? (uint32_t)(chunk * 4 * BITS * 4) : 0x80000000u;
#pragma unroll
    for (int j = 0; j < NT; j++)
      bload_unit<BITS>((GATEUP && j == 1) ? w1 : w0, woff + (coff + (uint32_t)(j * kTileRow) * row_bytes), u.w[j]);
  };
  // Scales and biases pass through a wave-private LDS table, a segment of
  // 8 groups (4 at 128 values) of the wave's 32 rows at a time, converted once:
  // lane (n16, kb) loads the words of groups 2 kb, 2 kb + 1 and stores the two
  // (scale, bias) f16 pairs. Loaded per chunk, each word cost a visit to a
  // line per row. Rows with an odd number of groups may start in a word's
  // upper half: a second word supplies the rest.
  const uint32_t sbytes = (uint32_t)N * (uint32_t)groups * 2u;
  auto sb_view = [&](const void* p) -> rsrc_t {
    return make_rsrc(reinterpret_cast<const uint16_t*>(p) + erows * groups, sbytes);
  };
  const rsrc_t sv[NT] = {sb_view(a.p0.s), sb_view(GATEUP ? a.p1.s : a.p0.s)};
  const rsrc_t bv[NT] = {sb_view(a.p0.b), sb_view(GATEUP ? a.p1.b : a.p0.b)};
  const bool odd_groups = (groups & 1) != 0;
  struct Seg {
    uint32_t s[NT], b[NT], s2[NT], b2[NT];
  };
  auto load_seg = [&](int chunk, Seg& g) -> void {  // the segment starting at chunk
    const uint32_t g0 = (uint32_t)((4 * chunk) >> a.gsh) + 2u * kb;
#pragma unroll
    for (int j = 0; j < NT; j++) {
      const uint32_t el = (uint32_t)(r0 + j * kTileRow) * (uint32_t)groups + g0;
      g.s[j] = bload32(sv[j], (el >> 1) * 4u);
      g.b[j] = bload32(bv[j], (el >> 1) * 4u);
    }
    if (odd_groups) {
#pragma unroll
      for (int j = 0; j < NT; j++) {
        const uint32_t el = (uint32_t)(r0 + j * kTileRow) * (uint32_t)groups + g0 + 1u;
        g.s2[j] = bload32(sv[j], (el >> 1) * 4u);
        g.b2[j] = bload32(bv[j], (el >> 1) * 4u);
      }
    }
  };
  uint32_t* sbt = L.sb + wave * (NT * 128);
  auto store_seg = [&](int chunk, const Seg& g) -> void {
    uint32_t sw[NT], bw[NT];
#pragma unroll
    for (int j = 0; j < NT; j++) {
      sw[j] = g.s[j];
      bw[j] = g.b[j];
    }
    if (odd_groups) {
      const uint32_t sh = 16u * (((uint32_t)n16 + (uint32_t)((4 * chunk) >> a.gsh)) & 1u);  // rows: parity of n16
#pragma unroll
      for (int j = 0; j < NT; j++) {
        sw[j] = __builtin_amdgcn_alignbit(g.s2[j], g.s[j], sh);
        bw[j] = __builtin_amdgcn_alignbit(g.b2[j], g.b[j], sh);
      }
    }
#pragma unroll
    for (int j = 0; j < NT; j++) {
      const h2_t lo = sb_h2(__builtin_amdgcn_perm(bw[j], sw[j], 0x05040100u), sb_bf16);
      const h2_t hi = sb_h2(__builtin_amdgcn_perm(bw[j], sw[j], 0x07060302u), sb_bf16);
      sbt[j * 128 + 32 * kb + n16] = __builtin_bit_cast(uint32_t, lo);
      sbt[j * 128 + 32 * kb + 16 + n16] = __builtin_bit_cast(uint32_t, hi);
    }
    __atomic_signal_fence(__ATOMIC_SEQ_CST);  // other lanes of the wave read them (LDS runs in order)
  };
  // chunks of a segment: 2 at 32-value groups, else 4
  const bool g32 = a.gsh == 0;
  // tile j's pair of the lane's unit in a chunk (dead units of a half chunk
  // read the last group's, which chunk_step masks)
  auto read_sb = [&](int chunk, bool tail, int j) -> h2_t {
    const int seg0 = g32 ? (chunk & ~1) : (chunk & ~3);
    int unit = 4 * (chunk - seg0) + kb;
    if (tail) unit = min(unit, CU - 1 - 4 * seg0);
    return __builtin_bit_cast(h2_t, sbt[j * 128 + ((unit >> a.gsh) << 4) + n16]);
  };
  struct SB {
    h2_t v[NT];  // scale, bias
  };
  // values [8 s, 8 s + 8) of tile j's unit
  auto dequant = [&](const WSet& u, const SB& q, int j, int s) -> u32x4_t {
    h2_t c[4];
    quarter_codes<BITS>(u.w[j], s, c);
    const h2_t sc = __builtin_shufflevector(q.v[j], q.v[j], 0, 0), bi = __builtin_shufflevector(q.v[j], q.v[j], 1, 1);
    u32x4_t v;
#pragma unroll
    for (int p = 0; p < 4; p++) v[p] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(c[p], sc, bi));
    return v;
  };

  f32x4_t acc[NT][MT];
#pragma unroll
  for (int j = 0; j < NT; j++)
#pragma unroll
    for (int i = 0; i < MT; i++) acc[j][i] = f32x4_t{};

  const uint32_t abase = (uint32_t)n16 * 256u + (stage_slot((uint32_t)(4 * kb), (uint32_t)n16) << 4);
  // Activation fragments of a 32-value step. Up to 4 row tiles double-buffer
  // them (the next step's are read during this step's first tile), more read
  // the next step's into the same registers right after their last use.
  constexpr int AB = MT > 4 ? 1 : 2, JR = AB == 2 ? 0 : NT - 1;
  struct Frags {
    u32x4_t f[AB][MT];
  };
  auto read_frag = [&](auto st, auto it, int s, bool mask, Frags& F) -> void {
    u32x4_t av = *reinterpret_cast<const u32x4_t*>(tile_lds(st, it) + (abase ^ (uint32_t)(s << 4)));
    if (mask) {
#pragma unroll
      for (int q = 0; q < 4; q++) av[q] = kb >= 2 ? 0u : av[q];
    }
    F.f[s & (AB - 1)][decltype(it)::value] = av;
  };
  // Chunk c in stage st (the next one's is nst): its set is u[U % NSET], its
  // first fragments are in F and the first tile's first quarter in wa. The
  // next chunk's activations are copied into the other stage, which every
  // wave has left since the last barrier, then weights are loaded into the
  // sets that have become free; at the chunk's end only those loads may still
  // be in flight. LAST: one of the chunks after the loop, the last of which
  // may hold two units only.
  WSet u[NSET];
  Seg seg;
  SB q;
  u32x4_t wa;
  Frags F;
  auto chunk_step = [&](auto uu, auto st, auto nst, auto last, int c) -> void {
    constexpr int U = decltype(uu)::value;
    constexpr bool LAST = decltype(last)::value;
    // this chunk loads weights (the trip after the loop: only for its own chunks)
    constexpr bool kLoads = NSET == 2 ? !(LAST && U == 3) : ((U & 1) == 0 && !(LAST && U == 2));
    constexpr int kNew = kLoads ? (NSET == 2 ? 1 : 2) * NT * kUnitLoads<BITS> : 0;
    const bool tail = LAST && half_tail && c == nchunks - 1, ntail = half_tail && c + 1 == nchunks - 1;
    // the table's segment is read for the last time at the end of the chunk
    // before its last one
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    if (U == 3 || (U == 1 && g32)) store_seg(c + 1, seg);
    if (U == 0 || (U == 2 && g32)) load_seg(g32 ? c + 2 : c + 4, seg);
    dma_a(c + 1, nst);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (kLoads) {
      if constexpr (NSET == 2) {
        load_set(c + 1, u[(U + 1) % NSET]);
      } else {
        load_set(c + 2, u[(U + 2) % NSET]);
        load_set(c + 3, u[(U + 3) % NSET]);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    // A half chunk's dead units get a zero scale and bias, and zero weights in
    // the quarter at hand: the codes that follow the row, with the row's last
    // scale, could overflow f16, and infinity times a masked activation is not zero.
    if (LAST && tail) {
      const uint32_t live = kb >= 2 ? 0u : ~0u;
#pragma unroll
      for (int j = 0; j < NT; j++)
        q.v[j] = __builtin_bit_cast(h2_t, __builtin_bit_cast(uint32_t, q.v[j]) & live);
      wa &= live;
    }
    const WSet &cu = u[U % NSET], &nu = u[(U + 1) % NSET];
    u32x4_t wb;
#pragma unroll
    for (int s = 0; s < 4; s++) {
#pragma unroll
      for (int j = 0; j < NT; j++) {
        u32x4_t& wf = (j & 1) ? wb : wa;
        u32x4_t& wn = (j & 1) ? wa : wb;
        if (s == 3 && j == JR) {
          // every read of this chunk's stage has returned; the next chunk's
          // copies are waited for, its first fragments read behind the
          // barrier under this chunk's last products
          vmcnt_wait<kNew>();
          lds_barrier_copies_in_flight();
        }
        if (s == 3) {
          if (j == 0) q.v[0] = read_sb(c + 1, ntail, 0);
          if (j == NT - 1) q.v[1] = read_sb(c + 1, ntail, 1);
        }
        static_for<MT>([&](auto it) -> void {
          constexpr int I = decltype(it)::value;
          acc[j][I] = mma16(wf, F.f[s & (AB - 1)][I], acc[j][I]);
          if (j == JR) {
            if (s < 3) read_frag(st, it, s + 1, tail, F);
            else read_frag(nst, it, 0, (LAST || U == 3) && ntail, F);
          }
        });
        if (j < NT - 1) wn = dequant(cu, q, j + 1, s);
        else if (s < 3) wn = dequant(cu, q, 0, s + 1);
        else wn = dequant(nu, q, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };

  load_seg(0, seg);
#pragma unroll
  for (int i = 0; i < (NSET == 2 ? 1 : 2); i++) load_set(i, u[i]);
  __builtin_amdgcn_sched_barrier(0);
  set_xoff();
  dma_a(0, std::integral_constant<int, 0>{});
  __builtin_amdgcn_sched_barrier(0);
  store_seg(0, seg);
#pragma unroll
  for (int j = 0; j < NT; j++) q.v[j] = read_sb(0, half_tail && nchunks == 1, j);
  wa = dequant(u[0], q, 0, 0);
  vmcnt_wait<0>();
  lds_barrier_copies_in_flight();
  static_for<MT>([&](auto it) -> void {
    read_frag(std::integral_constant<int, 0>{}, it, 0, half_tail && nchunks == 1, F);
  });

  // whole trips, then the chunks left over (a condition inside the loop would
  // make its head wait for every load)
  int c = 0;
  auto trip = [&](auto last) -> void {
    static_for<TRIP>([&](auto uu) -> void {
      constexpr int U = decltype(uu)::value, ST = U & 1;
      if (!decltype(last)::value || c + U < nchunks)
        chunk_step(uu, std::integral_constant<int, ST>{}, std::integral_constant<int, 1 - ST>{}, last, c + U);
    });
  };
  for (; c + TRIP < nchunks; c += TRIP) trip(std::false_type{});
  trip(std::true_type{});
  // copies may still be in flight: they must land before the LDS is another block's
  vmcnt_wait<0>();
  // every load counts in the waits above, also one of a chunk that did not
  // run: a use of each set keeps the compiler from dropping any
#pragma unroll
  for (int i = 0; i < NSET; i++)
#pragma unroll
    for (int j = 0; j < NT; j++)
#pragma unroll
      for (int k = 0; k < BITS; k++) asm volatile("" ::"v"(u[i].w[j][k]));

  // ---- epilogue: lane (n16, kb) holds activation row 16 i + n16 and 4 (gate/up)
  // or 8 consecutive output columns
  constexpr int OC = GATEUP ? 4 : 8;
  const int cn0 = GATEUP ? bn * 64 + 16 * wave + 4 * kb : bn * 128 + 32 * wave + 8 * kb;
  uint16_t* out = reinterpret_cast<uint16_t*>(a.out);
  const XT* ob0 = reinterpret_cast<const XT*>(a.p0.ob);
  const XT* ob1 = reinterpret_cast<const XT*>(GATEUP ? a.p1.ob : a.p0.ob);
  auto epilogue = [&](auto actc, auto biasc, auto xtc) -> void {
    constexpr int ACT = decltype(actc)::value;
    constexpr bool BIAS = decltype(biasc)::value, XT_ONLY = decltype(xtc)::value;
    float obg[OC], obu[OC];
#pragma unroll
    for (int t = 0; t < OC; t++) {
      obg[t] = (BIAS && ob0) ? to_f<XT>(ob0[erows + cn0 + t]) : -0.0f;
      obu[t] = (BIAS && GATEUP && ob1) ? to_f<XT>(ob1[erows + cn0 + t]) : -0.0f;
    }
#pragma unroll
    for (int i = 0; i < MT; i++) {
      uint32_t o[OC / 2];
#pragma unroll
      for (int h = 0; h < OC / 2; h++) {
        uint32_t pk = 0;
#pragma unroll
        for (int t2 = 0; t2 < 2; t2++) {
          const int t = 2 * h + t2;
          float v = acc[t >> 2][i][t & 3] * OSCALE;
          uint16_t bits;
          if constexpr (!GATEUP && !BIAS && XT_ONLY && ACT != ACT_RELU2) {
            // the stored value is the sum rounded once: one conversion
            bits = __builtin_bit_cast(uint16_t, from_f<XT>(v));
          } else {
            v = round_to<XT>(v);
            if constexpr (BIAS) v = round_to<XT>(v + obg[t]);
            if constexpr (GATEUP) {
              float up = round_to<XT>(acc[1][i][t & 3] * OSCALE);
              if constexpr (BIAS) up = round_to<XT>(up + obu[t]);
              bits = __builtin_bit_cast(uint16_t, to_a16<XT>(apply_act<XT>(v, up, ACT, a.alpha, a.limit)));
            } else {
              // single projections: squared ReLU only
              const float y = ACT == ACT_RELU2 ? apply_act<XT>(0.f, v, ACT_RELU2, 0.f, 0.f) : v;
              const uint16_t as_xt = __builtin_bit_cast(uint16_t, from_f<XT>(y));
              if constexpr (XT_ONLY) {
                bits = as_xt;
              } else {
                const uint16_t as_a16 = __builtin_bit_cast(uint16_t, to_a16<XT>(y));
                bits = a.out_a16 ? as_a16 : as_xt;
              }
            }
          }
          pk |= (uint32_t)bits << (16 * t2);
        }
        o[h] = pk;
      }
      const uint32_t r = (uint32_t)(16 * i + n16);
      if (r < rows) {
        uint16_t* dst = out + (size_t)(m0 + r) * N + cn0;
        if constexpr (GATEUP) *reinterpret_cast<u32x2_t*>(dst) = u32x2_t{o[0], o[1]};
        else *reinterpret_cast<u32x4_t*>(dst) = u32x4_t{o[0], o[1], o[2], o[3]};
      }
    }
  };
  if (cn0 >= N) return;  // N % 8 == 0 (host check): whole groups of columns
  using kNo = std::false_type;
  using kYes = std::true_type;
  const bool has_bias = ob0 != nullptr || (GATEUP && ob1 != nullptr);
  // Straight-line per activation kind, per presence of an output bias (without
  // one the sum is rounded once) and per output form
  auto by_bias = [&](auto actc, auto xtc) -> void {
    if (has_bias) epilogue(actc, kYes{}, xtc);
    else epilogue(actc, kNo{}, xtc);
  };
  if constexpr (GATEUP) {
    if (a.act == ACT_GPTOSS) by_bias(std::integral_constant<int, ACT_GPTOSS>{}, kNo{});
    else if (a.act == ACT_GEGLU) by_bias(std::integral_constant<int, ACT_GEGLU>{}, kNo{});
    else by_bias(std::integral_constant<int, ACT_SWIGLU>{}, kNo{});
  } else {
    auto by_out = [&](auto actc) -> void {
      if (a.out_a16) by_bias(actc, kNo{});
      else by_bias(actc, kYes{});
    };
    if (a.act == ACT_RELU2) by_out(std::integral_constant<int, ACT_RELU2>{});
    else by_out(std::integral_constant<int, ACT_SWIGLU>{});
  }
}

template <int BITS, typename XT, bool GATEUP>
__global__ __launch_bounds__(256, 3) void gemm_grouped_kernel(const GemmArgs a) {
  __shared__ __align__(16) unsigned char a0[kGemmObjBytes], a1[kGemmObjBytes], a2[kGemmObjBytes],
      a3[kGemmObjBytes], a4[kGemmObjBytes], a5[kGemmObjBytes];
  __shared__ uint32_t sb[4 * 2 * 128];
  // (tile, column block) pairs, column blocks of a tile together, split into
  // 8 contiguous ranges, one per XCD (blocks b, b + 8, ... share an XCD)
  const uint32_t nb = (uint32_t)a.col_blocks;
  const uint32_t n = __builtin_amdgcn_readfirstlane(a.items[0]) * nb;
  const uint32_t per = (n + 7u) >> 3;
  const uint32_t j = blockIdx.x >> 3;
  if (j >= per) return;
  const uint32_t wi = (blockIdx.x & 7u) * per + j;
  if (wi >= n) return;
  const uint32_t t = wi / nb;
  const uint32_t e = __builtin_amdgcn_readfirstlane(a.items[4 + 2 * t]);
  if (e == kGemmNoTile) return;
  const uint32_t x1 = __builtin_amdgcn_readfirstlane(a.items[5 + 2 * t]);
  const uint32_t m0 = x1 & ((1u << kGemmRowShift) - 1u), rows = (x1 >> kGemmRowShift) + 1u;
  const int bn = (int)(wi - t * nb);
  const GemmLds L{a0, a1, a2, a3, a4, a5, sb};
  if (rows > 64) gemm_tile<6, BITS, XT, GATEUP>(a, L, e, m0, bn, rows);
  else if (rows > 32) gemm_tile<4, BITS, XT, GATEUP>(a, L, e, m0, bn, rows);
  else gemm_tile<2, BITS, XT, GATEUP>(a, L, e, m0, bn, rows);
}

template <int BITS, typename XT, bool GATEUP>
static hipError_t launch_gemm_v(const GemmArgs& a, int grid, hipStream_t st, KEvents ev) {
  hipExtLaunchKernelGGL((gemm_grouped_kernel<BITS, XT, GATEUP>), dim3(grid), dim3(256), 0, st,
                        ev.start, ev.stop, 0, a);
  return hipGetLastError();
}

#define MOE_CAT2(a, b) a##b
#define MOE_CAT(a, b) MOE_CAT2(a, b)

// A rows are f16 operands (A16 for a bf16 layer) in every case.
hipError_t MOE_CAT(launch_gemm_b, MOE_BITS)(int xdt, bool gateup, const GemmArgs& a, int grid,
                                             hipStream_t st, KEvents ev) {
  if (xdt == DT_BF16)
    return gateup ? launch_gemm_v<MOE_BITS, bf16_t, true>(a, grid, st, ev)
                  : launch_gemm_v<MOE_BITS, bf16_t, false>(a, grid, st, ev);
  if (xdt == DT_F16)
    return gateup ? launch_gemm_v<MOE_BITS, f16_t, true>(a, grid, st, ev)
                  : launch_gemm_v<MOE_BITS, f16_t, false>(a, grid, st, ev);
  return hipErrorInvalidValue;
}

}  // namespace moe
