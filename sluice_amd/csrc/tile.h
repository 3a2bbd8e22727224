// Tiled expert product for calls with many tokens per expert (gfx950, wave64).
//
// The decode kernels stream an expert's weights once per 16 token columns: at
// prefill sizes every further 16 tokens of an expert read its weights again
// and the matrix cores wait for them.  Here a workgroup owns CH weight rows
// of one expert and BM of its tokens, keeps the product in registers over the
// whole of K, and loads both operands to LDS by DMA (global_load_lds, 16
// bytes per lane, no registers in between), ST - 1 stages ahead.
//
//   * sort: one workgroup groups the call's pairs by slot (order[]) and cuts
//     each slot's run into tiles of <= BM pairs; the shared experts' pairs
//     follow, every token in order.
//   * gemm1: act[pos] = bf16(silu(g) * u), rows in sorted order, so that
//     gemm2 reads them without a gather; a wave holds gate and up rows of the
//     same channels.
//   * gemm2: partial[pair] = W2 . act[pos] (fp32), which the combine weights
//     and sums.
//
// A pair's sums have the decode kernels' order, so its bits depend neither on
// the size of its call nor on the slot its expert sits in: the products of a
// chunk meet in the same MFMAs, and K is summed in the decode kernels' parts
// (their waves), whose sums are added in part order.  The second set of
// accumulators costs no time; what the order rules out is to start K at an
// offset of the slot's own, so that workgroups do not meet in the same memory
// channels (217 against 229, 574 against 594 and 696 against 703 us for the
// calls below).
//
// Bound: HBM while the experts have few tokens (the weights are read once;
// 4.2 TB/s in gemm1 of the V2-Lite call below, the DMA stream alone reaches
// 6.2), the operand traffic out of L2 beyond (a 4096-token call runs no faster
// with the LDS reads scheduled between the products).  Whole calls, timed in
// turn with the decode kernels, same bits: Qwen3 shape, 4096 tokens, 4076 ->
// 593 us; V2-Lite shape, 509 tokens over 48 slots, 562 -> 225 us; V3 fp8, 384
// tokens over 64 of 256 experts, 1438 -> 700 us (before rows past a tile's
// pairs were left out and fp8 went to bf16 by one instruction per pair, 27 us
// more).
//
// LDS rows are 128 bytes (64 bf16 or 128 fp8 of K) in eight 16-byte segments,
// the segment at place p of row r stored at p ^ (r & 7); places and swizzle
// are in the lanes' global addresses, since a DMA writes its lanes
// consecutively.  A 16-byte LDS read serves 16 lanes at a time over 64 banks,
// and the lanes that meet come from two neighbouring K groups (lanes 0-3,
// 12-15 and 20-27, ...).  Read m of K group kb takes segment 2kb + m (the
// decode kernels' order), which sits at place 4m + kb: the two groups then
// fall on even and odd places (at place 2kb + m half of the LDS cycles were
// conflicts).  An fp8 chunk's tokens are two rows of 64: half h of weight
// segment 2kb + i meets token segment 4kb + 2i + h, place 4i + 2h + (kb & 1)
// of row kb >> 1.
//
// (Internal to moe.hip, which includes it inside its anonymous namespace.)
#pragma once

// One tile: pairs order[pos0 .. pos0 + count) of one slot.  ft, nt: the
// slot's first tile and its number of tiles.
struct TileRec {
  int32_t slot_field;
  int32_t pos0;
  int32_t count;
  uint32_t ft_nt;  // ft | nt << 16
};
static_assert(sizeof(TileRec) == 16, "TileRec");

// The sorted call: header {tiles, 0, 0, 0}, then the tile records.
struct TilePlan {
  int32_t* hdr;    // {tiles, routed tiles, 0, 0}
  TileRec* tiles;
  uint16_t* order;  // [P2] pair of a sorted position
  int32_t* valid;   // [P]
};
static_assert(SLUICE_MAX_PREFILL_PAIRS <= 65536, "pairs are 16-bit");

constexpr int kSortThreads = 1024;
constexpr int kSortWaves = kSortThreads / SLUICE_WAVE;

// Pairs per tile of a slot with n > 0 of them.
__host__ __device__ inline int tile_size(int n, int bm) {
  const int nt = (n + bm - 1) / bm;
  return ((n + nt - 1) / nt + 15) & ~15;
}

// Upper bound of the tiles of a call over at most `slots` slots.
inline long tile_bound(int P, int slots, int T, int n_sh, int bm) {
  return (long)P / bm + std::min(P, slots) + (long)n_sh * ((T + bm - 1) / bm);
}

// Pairs grouped by slot (resident slots ascending, then those whose rows may
// still stream), cut into tiles of at most bm pairs.  The order of the pairs
// inside a slot is whatever the LDS atomics make it: a pair's product does
// not depend on its column.  One workgroup, latency-bound: a thread keeps its
// U pairs' slots and ranks in registers between counting and placing (at U = 64
// 84 bytes per lane go to scratch, at 32 32), and the pairs are placed in LDS and
// written out whole (scattered global stores, one line each, took most of the
// kernel).  P <= U * kSortThreads.
template <int U>
__global__ __launch_bounds__(kSortThreads) void moe_sort_kernel(
    const int32_t* __restrict__ ids, int P, const int32_t* __restrict__ map, int E, int S,
    const int32_t* __restrict__ pending, int T, int n_sh, int bm, TilePlan pl) {
  __shared__ int slot_of[SLUICE_MAX_EXPERTS];
  __shared__ int cnt[SLUICE_MAX_SLOTS];
  __shared__ int wsum[4][kSortWaves];
  __shared__ __align__(16) uint16_t placed[U * kSortThreads];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  constexpr int B = 8;  // ids in flight per thread
  static_assert(U % B == 0, "sort batches");
  int at[U];  // slot | rank << 10, -1 = not resident
#pragma unroll
  for (int u = 0; u < B; ++u) at[u] = tid + u * kSortThreads < P ? ids[tid + u * kSortThreads] : -1;
  for (int e = tid; e < E; e += kSortThreads) {
    const int s = map != nullptr ? map[e] : e;
    slot_of[e] = (unsigned)s < (unsigned)S ? s : -1;
  }
  for (int s = tid; s < S; s += kSortThreads) cnt[s] = 0;
  const int pend = tid < S && pending != nullptr && pending[tid] != 0 ? 1 : 0;
  __syncthreads();
#pragma unroll
  for (int b = 0; b < U; b += B) {
    if (b * kSortThreads >= P) break;
    if (b + B < U) {
#pragma unroll
      for (int u = b + B; u < b + 2 * B; ++u)
        at[u] = tid + u * kSortThreads < P ? ids[tid + u * kSortThreads] : -1;
    }
#pragma unroll
    for (int u = b; u < b + B; ++u) {
      const int p = tid + u * kSortThreads;
      const int s = (unsigned)at[u] < (unsigned)E ? slot_of[at[u]] : -1;
      at[u] = s >= 0 ? s | atomicAdd(&cnt[s], 1) << 10 : -1;
      if (p < P) pl.valid[p] = s >= 0 ? 1 : 0;
    }
  }
  __syncthreads();
  // Exclusive scans over the slots (thread s owns slot s): pairs and tiles,
  // the resident slots' and the pending ones'.
  const int n = tid < S ? cnt[tid] : 0;
  // Equal tiles, whole fragments of 16: ceil(n / bm) of them, or fewer.
  const int size = n > 0 ? tile_size(n, bm) : 16, nt = (n + size - 1) / size;
  int v[4] = {pend ? 0 : n, pend ? 0 : nt, pend ? n : 0, pend ? nt : 0}, in[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    in[c] = v[c];
#pragma unroll
    for (int off = 1; off < SLUICE_WAVE; off <<= 1) {
      const int o = __shfl_up(in[c], off, SLUICE_WAVE);
      if (lane >= off) in[c] += o;
    }
    if (lane == SLUICE_WAVE - 1) wsum[c][wave] = in[c];
  }
  __syncthreads();
  int base[4] = {0, 0, 0, 0}, tot[4] = {0, 0, 0, 0};
  for (int w = 0; w < kSortWaves; ++w)
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      if (w < wave) base[c] += wsum[c][w];
      tot[c] += wsum[c][w];
    }
  const int o = pend ? 2 : 0;
  const int pos = (pend ? tot[0] : 0) + base[o] + in[o] - v[o];
  const int ft = (pend ? tot[1] : 0) + base[o + 1] + in[o + 1] - v[o + 1];
  if (tid < S) cnt[tid] = pos;
  __syncthreads();
#pragma unroll
  for (int u = 0; u < U; ++u) {
    if (u * kSortThreads >= P) break;
    if (tid + u * kSortThreads < P && at[u] >= 0)
      placed[cnt[at[u] & 1023] + (at[u] >> 10)] = (uint16_t)(tid + u * kSortThreads);
  }
  for (int i = 0; i < nt; ++i)  // 0 beyond the slots
    pl.tiles[ft + i] = TileRec{tid | (pend ? kPendingBit : 0), pos + i * size,
                               min(size, n - i * size), (uint32_t)ft | ((uint32_t)nt << 16)};
  const int routed = tot[1] + tot[3], ssize = tile_size(T, bm), per = (T + ssize - 1) / ssize;
  for (int i = tid; i < n_sh * per; i += kSortThreads) {
    const int g = i / per, c = i - g * per;
    pl.tiles[routed + i] = TileRec{S + g, P + g * T + c * ssize, min(ssize, T - c * ssize),
                                   (uint32_t)(routed + g * per) | ((uint32_t)per << 16)};
  }
  for (int i = tid; i < n_sh * T; i += kSortThreads) pl.order[P + i] = (uint16_t)(P + i);
  if (tid == 0) {
    pl.hdr[0] = routed + n_sh * per;
    pl.hdr[1] = routed;
  }
  __syncthreads();
  const int used = tot[0] + tot[2];
  for (int i = tid; i < used / 8; i += kSortThreads)
    reinterpret_cast<u32x4_t*>(pl.order)[i] = reinterpret_cast<const u32x4_t*>(placed)[i];
  if (tid < used % 8) pl.order[used / 8 * 8 + tid] = placed[used / 8 * 8 + tid];
}

// 16 bytes per lane from base + voff into LDS at lds + 16 * lane.  No
// register is written, so the compiler has nothing to reuse early; the
// matching wait is dma_wait.  (With the builtin the compiler waits for every
// DMA in flight at each LDS read.)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"  // m0 is reserved; its own uses see the clobber
__device__ __forceinline__ void dma16(uint32_t lds, const void* base, uint32_t voff) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
               ::"s"(lds), "v"(voff), "s"(base)
               : "memory", "m0");
}
#pragma clang diagnostic pop

// Waits until at most N of this wave's DMAs are in flight and its LDS reads
// are done, then for the whole workgroup.
template <int N>
__device__ __forceinline__ void dma_wait() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

struct TileArgs {
  const uint16_t* x;
  ExpertW W;
  TilePlan plan;
  CallShape cs;
  uint16_t* act;
  float* partial;
};

// A uniform load of what an earlier kernel wrote, through the scalar cache
// (the compiler takes a vector load past the DMA's memory clobbers).
template <typename T>
__device__ __forceinline__ T ldu(const T* p) {
  static_assert(sizeof(T) % 4 == 0, "whole words");
  struct Words {
    uint32_t w[sizeof(T) / 4];
  } r;
#pragma unroll
  for (size_t i = 0; i < sizeof(T) / 4; ++i)
    r.w[i] = ((const __attribute__((address_space(4))) uint32_t*)(uintptr_t)p)[i];
  return __builtin_bit_cast(T, r);
}

// CH weight rows x BM pairs per item, WC x WP waves, ST stages.
template <bool FP8_, bool G1_, int CH_, int BM_, int WC_, int WP_, int ST_>
struct TileCfg {
  static constexpr bool FP8 = FP8_, G1 = G1_;
  static constexpr int CH = CH_, BM = BM_, WC = WC_, WP = WP_, ST = ST_;
  static constexpr int NW = WC * WP, ESZ = FP8 ? 1 : 2;
  static constexpr int KS = FP8 ? 128 : 64;       // K per stage
  static constexpr int SUB = KS / 64;             // 128-byte token sub-tiles per stage
  static constexpr int KP = G1 ? kKS : G2Shape<FP8>::K;  // K parts, as the decode kernels have
  static constexpr int CW = CH / WC, PW = BM / WP;
  static constexpr int FM = CW / 16, FN = PW / 16;
  static constexpr int kStage = CH * 128 + BM * KS * 2;
  static constexpr int NA = CH / 8 / NW, NB = BM / 8 * SUB / NW;  // DMAs per wave and stage
  static constexpr int kOut = G1 ? CH / 2 : CH;   // output channels per item
  // DMAs of a stage that load the rows of ng fragments per wave column.
  static constexpr int loads(int ng) { return (2 * ng * WP * SUB + NW - 1) / NW; }
  static_assert(NA * NW * 8 == CH && NB * NW * 8 == BM * SUB && FM % 2 == 0, "tile split");
};

// Persistent workgroups.  While an item's last products run, nothing of the
// next one is known to the memory system, and its first stage is three
// dependent loads away (record, tokens, operands): so the next item's record
// and tokens are loaded behind the current item's first stages, and its first
// stages are issued before the current item's epilogue.
template <typename C>
__global__ __launch_bounds__(64 * C::NW) void moe_tile_kernel(TileArgs a) {
  constexpr int CH = C::CH, BM = C::BM, NW = C::NW, FM = C::FM, FN = C::FN, ST = C::ST;
  constexpr bool FP8 = C::FP8, G1 = C::G1;
  __shared__ __align__(1024) uint8_t lds[ST * C::kStage];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int wc = wave % C::WC, wp = wave / C::WC;
  const int R = lane & 15, kb = lane >> 4;
  const int H = a.cs.H, I = a.cs.I;
  const int n_out = G1 ? I : H, K = G1 ? H : I;
  const int n_cb = (n_out + C::kOut - 1) / C::kOut;
  const int nk = K / C::KS;
  const uint32_t by_k = 0xffffffffu / (uint32_t)a.cs.k + 1;
  const uint32_t lds0 =
      (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)lds;
  // XCD x (workgroups are dealt to the 8 XCDs in turn) takes a contiguous
  // eighth of the routed items, so the tiles and channel blocks of an expert
  // meet in one L2, and an eighth of the shared ones, whose weights serve
  // many tiles: each XCD reads its share of the weights.
  const int routed = ldu(a.plan.hdr + 1) * n_cb, shared = ldu(a.plan.hdr) * n_cb - routed;
  const int xcds = (int)gridDim.x % 8 == 0 ? 8 : 1;
  const int xcd = (int)blockIdx.x % xcds, rank = (int)blockIdx.x / xcds;
  const int per_xcd = (int)gridDim.x / xcds;
  const int r0 = (int)((long)routed * xcd / xcds), rn = (int)((long)routed * (xcd + 1) / xcds) - r0;
  const int s0 = (int)((long)shared * xcd / xcds), sn = (int)((long)shared * (xcd + 1) / xcds) - s0;
  const int sp = (lane & 7) ^ (lane >> 3);            // LDS place of this lane's segment
  const int aseg = 2 * (sp & 3) + (sp >> 2);          // weight segment there
  const int bseg = FP8 ? (sp >> 1) + 4 * (sp & 1) : aseg;  // token segment

  struct Item {
    int slot_field, pos0, count, cb;
  };
  // The n-th item of this XCD (the caller checks n < rn + sn).
  auto item_at = [&](int n) {
    const int item = n < rn ? r0 + n : routed + s0 + (n - rn);
    const TileRec t = ldu(a.plan.tiles + item / n_cb);
    const int ft = (int)(t.ft_nt & 0xffff), nt = (int)(t.ft_nt >> 16);
    const int local = item - ft * n_cb, cb = local / nt;
    const TileRec rec = ldu(a.plan.tiles + ft + (local - cb * nt));
    return Item{rec.slot_field, rec.pos0, rec.count, cb};
  };
  // This wave's i-th token DMA of a stage: 8 rows of sub-tile token_sub(i),
  // lower rows first, so that a tile with few pairs loads few rows.
  auto token_sub = [&](int i) { return (wave + i * NW) % C::SUB; };
  auto token_group = [&](int i) { return (wave + i * NW) / C::SUB; };
  // The fragments per wave column that hold an item's pairs, rounded up to
  // the K loops there are.
  auto fragments = [&](int count) {
    const int n = (((count + 15) >> 4) + C::WP - 1) / C::WP;
    constexpr int kUnit = FN >= 4 ? FN / 4 : FN / 2;
    return (n + kUnit - 1) / kUnit * kUnit;
  };
  // The rows this lane loads of an item: pairs (gemm1; turned into tokens when
  // they are used, so that nothing waits for them here) or sorted positions.
  auto rows_of = [&](const Item& it, int (&rows)[C::NB]) {
#pragma unroll
    for (int i = 0; i < C::NB; ++i) {
      const int row = min(token_group(i) * 8 + (lane >> 3), it.count - 1);
      rows[i] = G1 ? (int)a.plan.order[it.pos0 + row] : row;
    }
  };

  // The wave's fp8 block scales of an item, the 64 chunks of window w, chunk
  // c in lane c & 63 (a load per chunk would wait for every DMA in flight):
  // of its gate and up rows, or of its hidden rows.
  struct Scales {
    float a, b;
  };
  auto scales_of = [&](const Item& t, int w) {
    const int slot = t.slot_field & kSlotMask;
    // a channel of the wave's 128-row blocks
    const int ch = min(t.cb * C::kOut + wc * (G1 ? C::CW / 2 : C::CW), n_out - 1);
    const int c = min(w * 64 + lane, nk - 1);
    if (G1) {
      const G1Src src = g1_src<1>(a.W, a.cs, slot, ch / 16);
      return Scales{src.sg[c], src.su[c]};
    }
    const float v = g2_src<1>(a.W, a.cs, slot, ch / 32).sr[c];
    return Scales{v, v};
  };

  // Operand addresses of the item being loaded.
  const uint8_t *abase = nullptr, *bbase = nullptr;
  uint32_t va[C::NA], vb[C::NB];
  auto address = [&](const Item& it, const int (&rows)[C::NB]) {
    const int slot = it.slot_field & kSlotMask, ch0 = it.cb * C::kOut;
    uint32_t ald;
    if (G1) {
      const bool rt = slot < a.W.S;
      const size_t v = (size_t)(rt ? 0 : slot - a.W.S) * I;
      abase = rt ? a.W.w13 + (size_t)slot * 2 * I * H * C::ESZ : a.W.sh_w13 + v * H * C::ESZ;
      ald = (uint32_t)H * C::ESZ;
      bbase = (const uint8_t*)a.x;
    } else {
      const G2Src src = g2_src<C::ESZ>(a.W, a.cs, slot, 0);
      abase = src.a0;
      ald = (uint32_t)src.ld * C::ESZ;
      bbase = (const uint8_t*)(a.act + (size_t)it.pos0 * I);
    }
    const uint32_t up = (uint32_t)(slot < a.W.S ? I : a.W.I_s);  // first up row after the gate's
#pragma unroll
    for (int i = 0; i < C::NA; ++i) {
      const int l = (wave + i * NW) * 8 + (lane >> 3);  // LDS row
      uint32_t row;
      if (G1) {
        const int w = l / C::CW, h = l % C::CW / (C::CW / 2), j = l % (C::CW / 2);
        row = (uint32_t)min(ch0 + w * (C::CW / 2) + j, I - 1) + (h ? up : 0u);
      } else {
        row = (uint32_t)min(ch0 + l, H - 1);
      }
      va[i] = row * ald + (uint32_t)aseg * 16;
    }
#pragma unroll
    for (int i = 0; i < C::NB; ++i) {
      uint32_t row = (uint32_t)rows[i];
      if (G1)  // pair / k is exact: pairs are below 2^16
        row = slot >= a.W.S      ? row - (uint32_t)(a.cs.T * a.cs.k + (slot - a.W.S) * a.cs.T)
              : a.cs.k > 1 ? __umulhi(row, by_k)
                           : row;
      vb[i] = row * (uint32_t)(K * 2) + (uint32_t)(token_sub(i) * 128 + bseg * 16);
    }
  };
  // Chunk k of the item goes to stage buffer buf.
  auto issue = [&](int k, int buf, int nb) {
    const uint8_t* ap = abase + (size_t)k * 128;
    const uint8_t* bp = bbase + (size_t)k * (C::KS * 2);
    const uint32_t d = lds0 + (uint32_t)(buf * C::kStage);
#pragma unroll
    for (int i = 0; i < C::NA; ++i) dma16(d + (wave + i * NW) * 1024, ap, va[i]);
#pragma unroll
    for (int i = 0; i < C::NB; ++i)
      if (i < nb)
        dma16(d + CH * 128 + token_sub(i) * (BM * 128) + token_group(i) * 1024, bp, vb[i]);
  };
  auto issue_first = [&](int count) {
    const int nb = C::loads(fragments(count));
#pragma unroll
    for (int s = 0; s < ST - 1; ++s)
      if (s < nk) issue(s, s, nb);
  };

  int n = rank;
  if (n >= rn + sn) return;
  Item it = item_at(n);
  int rows[C::NB];
  rows_of(it, rows);
  // The first scales of the item loaded next: ahead of its weights, or, where
  // the slot's rows may still stream, behind the wait like every other read
  // of them (the gap kernel itself copies scale rows only up to 32 KB and in
  // whole 16-byte vectors; others arrive with the weights).
  Scales nsc = {0.f, 0.f};
  auto scales_early = [&](const Item& t) {
    if (FP8 && (t.slot_field & kPendingBit) == 0) nsc = scales_of(t, 0);
  };
  auto await_item = [&](const Item& t) {
    await_slot(a.W.wait, t.slot_field);
    if (FP8 && (t.slot_field & kPendingBit) != 0) nsc = scales_of(t, 0);
  };
  scales_early(it);
  await_item(it);
  address(it, rows);
  issue_first(it.count);
  for (;;) {
    const int next = n + per_xcd;
    const bool more = next < rn + sn;
    const Item nit = more ? item_at(next) : it;
    rows_of(nit, rows);
    Scales sc = nsc;
    scales_early(nit);
    const int count = it.count, pos0 = it.pos0, ch0 = it.cb * C::kOut;
    const int wrow = G1 ? ch0 + wc * (C::CW / 2) : ch0 + wc * C::CW;  // the wave's first channel
    int pair[FN];  // this lane's (gemm2), for the epilogue
    if (!G1) {
#pragma unroll
      for (int g = 0; g < FN; ++g)
        pair[g] = a.plan.order[pos0 + min((g * C::WP + wp) * 16 + R, count - 1)];
    }
    // tot: the sums of the K parts done, acc: the part being summed.
    f32x4_t acc[FM][FN], tot[FM][FN];
#pragma unroll
    for (int f = 0; f < FM; ++f)
#pragma unroll
      for (int g = 0; g < FN; ++g) tot[f][g] = acc[f][g] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    // The K loop over NG of the wave's FN token fragments: the fragments past
    // the tile's pairs are left out.
    const auto k_loop = [&](auto ng) {
      constexpr int NG = decltype(ng)::value;
      int buf = 0, part = 1, cut = nk / C::KP;  // the next part and its first chunk
      for (int k = 0; k < nk; ++k) {
        if (k == cut) {
#pragma unroll
          for (int f = 0; f < FM; ++f)
#pragma unroll
            for (int g = 0; g < NG; ++g) {
              tot[f][g] += acc[f][g];
              acc[f][g] = f32x4_t{0.f, 0.f, 0.f, 0.f};
            }
          while (cut <= k) cut = ++part * nk / C::KP;
        }
        constexpr int nb = C::loads(NG), L = C::NA + nb;
        const int ahead = min(ST - 2, nk - 1 - k);  // stages after k in flight
        if (ST >= 4 && ahead >= 2)
          dma_wait<(ST >= 4 ? 2 * L : 0)>();
        else if (ST >= 3 && ahead >= 1)
          dma_wait<(ST >= 3 ? L : 0)>();
        else
          dma_wait<0>();
        if (k + ST - 1 < nk) issue(k + ST - 1, buf == 0 ? ST - 1 : buf - 1, nb);
        const uint8_t* sa = lds + buf * C::kStage + (wc * C::CW + R) * 128;
        const uint8_t* sb = lds + buf * C::kStage + CH * 128 + (wp * 16 + R) * 128;
        auto ldl = [](const uint8_t* p) { return *reinterpret_cast<const u32x4_t*>(p); };
        if constexpr (!FP8) {
#pragma unroll
          for (int m = 0; m < 2; ++m) {
            const int o = ((4 * m + kb) ^ (R & 7)) * 16;
            u32x4_t av[FM], bv[NG];
#pragma unroll
            for (int f = 0; f < FM; ++f) av[f] = ldl(sa + f * 2048 + o);
#pragma unroll
            for (int g = 0; g < NG; ++g) bv[g] = ldl(sb + g * C::WP * 2048 + o);
#pragma unroll
            for (int f = 0; f < FM; ++f)
#pragma unroll
              for (int g = 0; g < NG; ++g) acc[f][g] = mfma16x16x32_bf16(av[f], bv[g], acc[f][g]);
          }
        } else {
          if (k != 0 && (k & 63) == 0) sc = scales_of(it, k >> 6);
          const float c0 = __uint_as_float(
              (uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(sc.a), k & 63));
          const float c1 = __uint_as_float(
              (uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(sc.b), k & 63));
          f32x4_t t[FM][NG];
#pragma unroll
          for (int f = 0; f < FM; ++f)
#pragma unroll
            for (int g = 0; g < NG; ++g) t[f][g] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            const int oa = ((4 * i + kb) ^ (R & 7)) * 16;
            u32x4_t av[FM][2];
#pragma unroll
            for (int f = 0; f < FM; ++f)
              fp8x16_to_bf16(ldl(sa + f * 2048 + oa), av[f][0], av[f][1]);
#pragma unroll
            for (int h = 0; h < 2; ++h) {
              const int ob =
                  ((4 * i + 2 * h + (kb & 1)) ^ (R & 7)) * 16 + (kb >> 1) * (BM * 128);
              u32x4_t bv[NG];
#pragma unroll
              for (int g = 0; g < NG; ++g) bv[g] = ldl(sb + g * C::WP * 2048 + ob);
#pragma unroll
              for (int f = 0; f < FM; ++f)
#pragma unroll
                for (int g = 0; g < NG; ++g)
                  t[f][g] = mfma16x16x32_bf16(av[f][h], bv[g], t[f][g]);
            }
          }
#pragma unroll
          for (int f = 0; f < FM; ++f)
#pragma unroll
            for (int g = 0; g < NG; ++g) acc[f][g] += (G1 && f >= FM / 2 ? c1 : c0) * t[f][g];
        }
        buf = buf + 1 == ST ? 0 : buf + 1;
      }
    };
    const int ng = fragments(count);
    if (FN >= 4 && ng == FN / 4)
      k_loop(std::integral_constant<int, (FN >= 4 ? FN / 4 : FN)>{});
    else if (ng == FN / 2)
      k_loop(std::integral_constant<int, FN / 2>{});
    else if (FN >= 4 && ng == FN * 3 / 4)
      k_loop(std::integral_constant<int, (FN >= 4 ? FN * 3 / 4 : FN)>{});
    else
      k_loop(std::integral_constant<int, FN>{});
    if (more) {
      dma_wait<0>();  // every wave has read its last stage
      await_item(nit);
      address(nit, rows);
      issue_first(nit.count);
    }
    // Epilogue: column R of fragment g is pair pos0 + 16 (g WP + wp) + R, rows
    // 4 kb .. +4 of fragment f its channels.
#pragma unroll
    for (int g = 0; g < FN; ++g) {
      const int row = (g * C::WP + wp) * 16 + R;
      if (row >= count) continue;
      if (G1) {
#pragma unroll
        for (int f = 0; f < FM / 2; ++f) {
          const int ch = wrow + f * 16 + kb * 4;
          const f32x4_t gt = tot[f][g] + acc[f][g], u = tot[f + FM / 2][g] + acc[f + FM / 2][g];
          float o[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) o[r] = gt[r] / (1.0f + expf(-gt[r])) * u[r];
          if (ch < I)
            *reinterpret_cast<u32x2_t*>(a.act + (size_t)(pos0 + row) * I + ch) =
                u32x2_t{pack2_bf16(o[0], o[1]), pack2_bf16(o[2], o[3])};
        }
      } else {
#pragma unroll
        for (int f = 0; f < FM; ++f) {
          const int ch = wrow + f * 16 + kb * 4;
          if (ch < H)
            *reinterpret_cast<f32x4_t*>(a.partial + (size_t)pair[g] * H + ch) =
                tot[f][g] + acc[f][g];
        }
      }
    }
    if (!more) return;
    n = next;
    it = nit;
  }
}
