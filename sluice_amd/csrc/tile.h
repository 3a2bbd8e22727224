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
//   * gemm2: partial[pair] = w * W2 . act[pos] (fp32), which the combine sums
//     as it does for the decode kernels.
//
// Bound: HBM while the experts have few tokens (the weights are read once),
// the matrix cores and the LDS operand reads beyond.  Whole calls against the
// decode kernels: Qwen3 shape, 4096 tokens, 4084 -> 618 us; V2-Lite shape,
// 509 tokens over 48 slots, 628 -> 233 us; V3 fp8, 384 tokens over 64 of 256
// experts, 1364 -> 794 us.
//
// LDS rows are 128 bytes (64 bf16 or 128 fp8 of K) in eight 16-byte
// segments, segment s of row r at s ^ (r & 7), so the row-major DMA writes
// and the MFMA-order reads are both free of bank conflicts; the swizzle is
// in the lanes' global addresses, since a DMA writes its lanes consecutively.
// The K order inside a chunk is the same permutation for both operands.
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
  int32_t* hdr;
  TileRec* tiles;
  int32_t* order;  // [P2]
  int32_t* valid;  // [P]
};

constexpr int kSortThreads = 1024;
constexpr int kSortWaves = kSortThreads / SLUICE_WAVE;

// Upper bound of the tiles of a call over at most `slots` slots.
inline long tile_bound(int P, int slots, int T, int n_sh, int bm) {
  return (long)P / bm + std::min(P, slots) + (long)n_sh * ((T + bm - 1) / bm);
}

// Pairs grouped by slot (resident slots ascending, then those whose rows may
// still stream), cut into tiles of bm pairs.  The order of the pairs inside a
// slot is whatever the LDS atomics make it: a pair's product does not depend
// on its column.
__global__ __launch_bounds__(kSortThreads) void moe_sort_kernel(
    const int32_t* __restrict__ ids, int P, const int32_t* __restrict__ map, int E, int S,
    const int32_t* __restrict__ pending, int T, int n_sh, int bm, TilePlan pl) {
  __shared__ int slot_of[SLUICE_MAX_EXPERTS];
  __shared__ int cnt[SLUICE_MAX_SLOTS], cur[SLUICE_MAX_SLOTS];
  __shared__ int wsum[4][kSortWaves];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int e = tid; e < E; e += kSortThreads) {
    const int s = map != nullptr ? map[e] : e;
    slot_of[e] = (unsigned)s < (unsigned)S ? s : -1;
  }
  for (int s = tid; s < S; s += kSortThreads) cnt[s] = 0;
  const int pend = tid < S && pending != nullptr && pending[tid] != 0 ? 1 : 0;
  __syncthreads();
  constexpr int U = 8;  // ids in flight per thread
  for (int p0 = tid; p0 < P; p0 += U * kSortThreads) {
    int g[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int p = p0 + u * kSortThreads;
      g[u] = p < P ? ids[p] : -1;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int p = p0 + u * kSortThreads;
      const int s = (unsigned)g[u] < (unsigned)E ? slot_of[g[u]] : -1;
      if (s >= 0) atomicAdd(&cnt[s], 1);
      if (p < P) pl.valid[p] = s >= 0 ? 1 : 0;
    }
  }
  __syncthreads();
  // Exclusive scans over the slots (thread s owns slot s): pairs and tiles,
  // the resident slots' and the pending ones'.
  const int n = tid < S ? cnt[tid] : 0, nt = (n + bm - 1) / bm;
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
  if (tid < S) {
    cur[tid] = pos;
    for (int i = 0; i < nt; ++i)
      pl.tiles[ft + i] = TileRec{tid | (pend ? kPendingBit : 0), pos + i * bm,
                                 min(bm, n - i * bm), (uint32_t)ft | ((uint32_t)nt << 16)};
  }
  const int routed = tot[1] + tot[3], per = (T + bm - 1) / bm;
  for (int i = tid; i < n_sh * per; i += kSortThreads) {
    const int g = i / per, c = i - g * per;
    pl.tiles[routed + i] = TileRec{S + g, P + g * T + c * bm, min(bm, T - c * bm),
                                   (uint32_t)(routed + g * per) | ((uint32_t)per << 16)};
  }
  for (int i = tid; i < n_sh * T; i += kSortThreads) pl.order[P + i] = P + i;
  if (tid == 0) pl.hdr[0] = routed + n_sh * per;
  __syncthreads();
  for (int p0 = tid; p0 < P; p0 += U * kSortThreads) {
    int g[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int p = p0 + u * kSortThreads;
      g[u] = p < P ? ids[p] : -1;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int s = (unsigned)g[u] < (unsigned)E ? slot_of[g[u]] : -1;
      if (s >= 0) pl.order[atomicAdd(&cur[s], 1)] = p0 + u * kSortThreads;
    }
  }
}

// 16 bytes per lane from base + voff into LDS at lds + 16 * lane.  No
// register is written, so the compiler has nothing to reuse early; the
// matching wait is dma_wait.  (With the builtin the compiler waits for every
// DMA in flight at each LDS read.)
__device__ __forceinline__ void dma16(uint32_t lds, const void* base, uint32_t voff) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
               ::"s"(lds), "v"(voff), "s"(base)
               : "memory");
}

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
  const float* topk_w;
  uint16_t* act;
  float* partial;
};

// CH weight rows x BM pairs per item, WC x WP waves, ST stages.
template <bool FP8_, bool G1_, int CH_, int BM_, int WC_, int WP_, int ST_>
struct TileCfg {
  static constexpr bool FP8 = FP8_, G1 = G1_;
  static constexpr int CH = CH_, BM = BM_, WC = WC_, WP = WP_, ST = ST_;
  static constexpr int NW = WC * WP, ESZ = FP8 ? 1 : 2;
  static constexpr int KS = FP8 ? 128 : 64;       // K per stage
  static constexpr int SUB = KS / 64;             // 128-byte token sub-tiles per stage
  static constexpr int CW = CH / WC, PW = BM / WP;
  static constexpr int FM = CW / 16, FN = PW / 16;
  static constexpr int kStage = CH * 128 + BM * KS * 2;
  static constexpr int NA = CH / 8 / NW, NB = BM / 8 * SUB / NW;  // DMAs per wave and stage
  static constexpr int kOut = G1 ? CH / 2 : CH;   // output channels per item
  static_assert(NA * NW * 8 == CH && NB * NW * 8 == BM * SUB && FM % 2 == 0, "tile split");
};

template <typename C>
__global__ __launch_bounds__(64 * C::NW) void moe_tile_kernel(TileArgs a) {
  constexpr int CH = C::CH, BM = C::BM, NW = C::NW, FM = C::FM, FN = C::FN, ST = C::ST;
  constexpr bool FP8 = C::FP8, G1 = C::G1;
  __shared__ __align__(1024) uint8_t lds[ST * C::kStage];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int wc = wave % C::WC, wp = wave / C::WC;
  const int R = lane & 15, kb = lane >> 4;
  const int H = a.cs.H, I = a.cs.I, P = a.cs.T * a.cs.k;
  const int n_out = G1 ? I : H, K = G1 ? H : I;
  const int n_cb = (n_out + C::kOut - 1) / C::kOut;
  const int nk = K / C::KS;
  const int total = a.plan.hdr[0] * n_cb;
  const uint32_t lds0 =
      (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)lds;
  // XCD x (workgroups are dealt to the 8 XCDs in turn) takes a contiguous
  // eighth of the items, so the tiles and channel blocks of an expert meet
  // in one L2.
  const int xcds = (int)gridDim.x % 8 == 0 ? 8 : 1;
  const int xcd = (int)blockIdx.x % xcds, rank = (int)blockIdx.x / xcds;
  const int per_xcd = (int)gridDim.x / xcds;
  const int i_end = (int)((long)total * (xcd + 1) / xcds);
  const int seg = (lane & 7) ^ (lane >> 3);
  for (int item = (int)((long)total * xcd / xcds) + rank; item < i_end; item += per_xcd) {
    const TileRec r0 = a.plan.tiles[item / n_cb];
    const int ft = (int)(r0.ft_nt & 0xffff), nt = (int)(r0.ft_nt >> 16);
    const int local = item - ft * n_cb;
    const int cb = local / nt;
    const TileRec rec = a.plan.tiles[ft + local - cb * nt];
    const int slot = __builtin_amdgcn_readfirstlane(rec.slot_field) & kSlotMask;
    const int pos0 = __builtin_amdgcn_readfirstlane(rec.pos0);
    const int count = __builtin_amdgcn_readfirstlane(rec.count);
    const int ch0 = cb * C::kOut;
    await_slot(a.W.wait, rec.slot_field);
    // Operand addresses of this lane.
    const uint8_t *abase, *bbase;
    uint32_t ald;
    const float *sc0 = nullptr, *sc1 = nullptr;  // fp8 scale rows (chunk c at [c])
    const int wrow = G1 ? ch0 + wc * (C::CW / 2) : ch0 + wc * C::CW;  // the wave's first channel
    const int srow = min(wrow, n_out - 1);
    if (G1) {
      const bool routed = slot < a.W.S;
      const size_t v = (size_t)(routed ? 0 : slot - a.W.S) * I;
      abase = routed ? a.W.w13 + (size_t)slot * 2 * I * H * C::ESZ : a.W.sh_w13 + v * H * C::ESZ;
      ald = (uint32_t)H * C::ESZ;
      bbase = (const uint8_t*)a.x;
      if (FP8) {
        const G1Src src = g1_src<1>(a.W, a.cs, slot, srow / 16);
        sc0 = src.sg;
        sc1 = src.su;
      }
    } else {
      const G2Src src = g2_src<C::ESZ>(a.W, a.cs, slot, 0);
      abase = src.a0;
      ald = (uint32_t)src.ld * C::ESZ;
      bbase = (const uint8_t*)(a.act + (size_t)pos0 * I);
      if (FP8) sc0 = sc1 = g2_src<1>(a.W, a.cs, slot, srow / 32).sr;
    }
    const uint32_t up = (uint32_t)(slot < a.W.S ? I : a.W.I_s);  // first up row after the gate's
    uint32_t va[C::NA], vb[C::NB];
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
      va[i] = row * ald + (uint32_t)seg * 16;
    }
#pragma unroll
    for (int i = 0; i < C::NB; ++i) {
      const int q = wave + i * NW, sub = q / (BM / 8), g = q % (BM / 8);
      const int row = min(g * 8 + (lane >> 3), count - 1);
      const uint32_t t =
          G1 ? (uint32_t)pair_token(a.cs, a.plan.order[pos0 + row]) : (uint32_t)row;
      vb[i] = t * (uint32_t)(K * 2) + (uint32_t)(sub * 128 + seg * 16);
    }
    auto issue = [&](int k, int buf) {
      const uint8_t* ap = abase + (size_t)k * 128;
      const uint8_t* bp = bbase + (size_t)k * (C::KS * 2);
      const uint32_t d = lds0 + (uint32_t)(buf * C::kStage) + (uint32_t)wave * 1024;
#pragma unroll
      for (int i = 0; i < C::NA; ++i) dma16(d + i * NW * 1024, ap, va[i]);
#pragma unroll
      for (int i = 0; i < C::NB; ++i) dma16(d + CH * 128 + i * NW * 1024, bp, vb[i]);
    };
    // The wave's block scales, 64 chunks at a time, chunk k in lane k & 63: a
    // load per chunk would wait for every DMA in flight.
    float scv0 = 0.f, scv1 = 0.f;
    auto load_scales = [&](int k) {
      const int c = min(k + lane, nk - 1);
      scv0 = sc0[c];
      scv1 = G1 ? sc1[c] : scv0;
    };
    if (FP8) load_scales(0);
    f32x4_t acc[FM][FN];
#pragma unroll
    for (int f = 0; f < FM; ++f)
#pragma unroll
      for (int g = 0; g < FN; ++g) acc[f][g] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    dma_wait<0>();  // the previous item's readers of the stages and its stores are done
#pragma unroll
    for (int s = 0; s < ST - 1; ++s)
      if (s < nk) issue(s, s);
    int buf = 0;
    for (int k = 0; k < nk; ++k) {
      constexpr int L = C::NA + C::NB;
      const int ahead = min(ST - 2, nk - 1 - k);  // stages after k in flight
      if (ST >= 4 && ahead >= 2)
        dma_wait<(ST >= 4 ? 2 * L : 0)>();
      else if (ST >= 3 && ahead >= 1)
        dma_wait<(ST >= 3 ? L : 0)>();
      else
        dma_wait<0>();
      if (k + ST - 1 < nk) issue(k + ST - 1, buf == 0 ? ST - 1 : buf - 1);
      const uint8_t* sa = lds + buf * C::kStage + (wc * C::CW + R) * 128;
      const uint8_t* sb = lds + buf * C::kStage + CH * 128 + (wp * C::PW + R) * 128;
      auto ldl = [](const uint8_t* p) { return *reinterpret_cast<const u32x4_t*>(p); };
      if constexpr (!FP8) {
#pragma unroll
        for (int m = 0; m < 2; ++m) {
          const int o = ((2 * kb + m) ^ (R & 7)) * 16;
          u32x4_t av[FM], bv[FN];
#pragma unroll
          for (int f = 0; f < FM; ++f) av[f] = ldl(sa + f * 2048 + o);
#pragma unroll
          for (int g = 0; g < FN; ++g) bv[g] = ldl(sb + g * 2048 + o);
#pragma unroll
          for (int f = 0; f < FM; ++f)
#pragma unroll
            for (int g = 0; g < FN; ++g) acc[f][g] = mfma16x16x32_bf16(av[f], bv[g], acc[f][g]);
        }
      } else {
        if ((k & 63) == 0 && k != 0) load_scales(k);
        const float s0 = __uint_as_float(
            (uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(scv0), k & 63));
        const float s1 = __uint_as_float(
            (uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(scv1), k & 63));
        f32x4_t t[FM][FN];
#pragma unroll
        for (int f = 0; f < FM; ++f)
#pragma unroll
          for (int g = 0; g < FN; ++g) t[f][g] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const int oa = ((kb + 4 * i) ^ (R & 7)) * 16;
          u32x4_t av[FM][2];
#pragma unroll
          for (int f = 0; f < FM; ++f) fp8x16_to_bf16(ldl(sa + f * 2048 + oa), av[f][0], av[f][1]);
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const int ob = ((2 * kb + h) ^ (R & 7)) * 16 + i * BM * 128;
            u32x4_t bv[FN];
#pragma unroll
            for (int g = 0; g < FN; ++g) bv[g] = ldl(sb + g * 2048 + ob);
#pragma unroll
            for (int f = 0; f < FM; ++f)
#pragma unroll
              for (int g = 0; g < FN; ++g) t[f][g] = mfma16x16x32_bf16(av[f][h], bv[g], t[f][g]);
          }
        }
#pragma unroll
        for (int f = 0; f < FM; ++f)
#pragma unroll
          for (int g = 0; g < FN; ++g) acc[f][g] += (G1 && f >= FM / 2 ? s1 : s0) * t[f][g];
      }
      buf = buf + 1 == ST ? 0 : buf + 1;
    }
    // Epilogue: column R of fragment g is pair pos0 + wp * PW + 16 g + R, rows
    // 4 kb .. +4 of fragment f its channels.
#pragma unroll
    for (int g = 0; g < FN; ++g) {
      const int row = wp * C::PW + g * 16 + R;
      if (row >= count) continue;
      if (G1) {
#pragma unroll
        for (int f = 0; f < FM / 2; ++f) {
          const int ch = wrow + f * 16 + kb * 4;
          const f32x4_t gt = acc[f][g], u = acc[f + FM / 2][g];
          float o[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) o[r] = gt[r] / (1.0f + expf(-gt[r])) * u[r];
          if (ch < I)
            *reinterpret_cast<u32x2_t*>(a.act + (size_t)(pos0 + row) * I + ch) =
                u32x2_t{pack2_bf16(o[0], o[1]), pack2_bf16(o[2], o[3])};
        }
      } else {
        const int pair = a.plan.order[pos0 + row];
        const float w = pair < P ? a.topk_w[pair] : 1.0f;
#pragma unroll
        for (int f = 0; f < FM; ++f) {
          const int ch = wrow + f * 16 + kb * 4;
          const f32x4_t v = acc[f][g];
          if (ch < H)
            *reinterpret_cast<f32x4_t*>(a.partial + (size_t)pair * H + ch) =
                f32x4_t{w * v[0], w * v[1], w * v[2], w * v[3]};
        }
      }
    }
  }
}
