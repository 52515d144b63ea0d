// Thin tiles of the grouped forward: 128 P rows (weight rows) x 64 Q rows
// (tokens), for experts that hold at most 64 tokens.  Included by gemm.hip
// inside its namespace.
//
// Such an expert still streams its whole weight, so a thin tile is bound by how
// fast weight bytes come out of HBM, not by the matrix cores.  A kernel that
// does nothing but LDS-DMA of a weight reads 6.2 TB/s on MI355X; the 256 x 256
// tile reached 5.1 (K 7168) and 4.2 TB/s (K 2048) on it.  Four things differ
// from that tile:
//   * six ring stages of 25 KB instead of two of 66 KB: at 25 KB per us and CU
//     and 3 to 4 us of loaded latency about 100 KB must be on the way, and the
//     stages being read and refilled come on top;
//   * one barrier per stage: it publishes the next stage, whose fragments are
//     read under this stage's MFMAs, and frees this stage's slot for the loads
//     of the stage six further on;
//   * the load stream runs on across tiles: the stages issued during a tile's
//     last six belong to the workgroup's next tile, so the memory pipe never
//     drains between tiles;
//   * the output leaves straight from the accumulators (16 consecutive P
//     indices per lane), which leaves the ring to the next tile's stages.
// Every wave holds all 128 P rows (with the gate rows first, the gate and the
// up values of the same features) against Q rows 4m + w, m = 0..15.  Every
// output element is the same chain of 128-deep MFMAs as in a 256-row tile, so
// the bits do not depend on the tile that computed it.
// Measured, 32 experts, bf16 out, against 256-row tiles: N 4096, K 7168 with 4 /
// 32 / 64 rows per expert 205 -> 168, 200 -> 173, 190 -> 179 us; N 7168, K 2048
// 109 -> 86, 112 -> 94, 114 -> 105 us (5.8 and 5.6 TB/s at 4 rows).
#pragma once

constexpr uint32_t kThinP = 128;
constexpr uint32_t kThinQ = 64;
constexpr int kThinStages = 6;
// A stage: P rows, Q rows, four P scale blocks of 128 bytes, four Q scale
// blocks of 64, and 256 bytes that wave 3's scale load zeroes.
constexpr uint32_t kThinQOff = kThinP * kStageK;
constexpr uint32_t kThinScaleOff = kThinQOff + kThinQ * kStageK;
constexpr uint32_t kThinStageBytes = kThinScaleOff + 1024u;
constexpr uint32_t kThinRingBytes = kThinStages * kThinStageBytes;
static_assert(kThinRingBytes >= 2u * kStageBytes, "the ring also holds two stages of a wide tile");

// LDS of k_grouped_fwd_thin: the ring holds six stages of a thin tile or two
// of a wide one.
struct __align__(16) SmemThin {
  uint8_t ring[2][kThinRingBytes / 2];  // wide stages at ring[0], ring[1]; thin ones end to end
  int32_t order[kMaxGroups];  // first m-tile and group of every rank (order_tiles)
  int32_t gend[kMaxGroups];
  uint64_t scan_tmp[kWaves];
};
static_assert(sizeof(SmemThin) <= 160 * 1024, "LDS of one compute unit");

// Rows of group [gb, ge) are tiled by 256 from its first row rounded down to 4.
__device__ __forceinline__ uint32_t tiled_rows(int32_t gb, int32_t ge) {
  return ge > gb ? (uint32_t)(ge - (gb & ~3)) : 0u;
}

// A group of at most 64 rows fits a thin tile.  The last, partial tile of a
// larger group stays 256 rows high: it shares its weight tile in L2 with the
// group's other tiles, which run beside it, and tiles of different heights in
// the same rounds leave the workgroups with the short ones waiting (32 experts
// of 320 rows, N 4096, K 7168: 350 us, with 64-row last tiles 403).  Groups of
// 65 to 128 rows gained nothing from a 128-row form (198 us either way).
__device__ __forceinline__ bool is_thin(int32_t gb, int32_t ge) {
  return tiled_rows(gb, ge) <= kThinQ;
}

// The order of the groups' m-tiles: groups of 256-row tiles first, then thin and
// empty ones, each kind in index order.  Thin tiles draw more bandwidth per CU
// than 256-row ones, so a 256-row tile that starts beside them late is what the
// launch waits for: 32 experts of multinomial sizes around 56, N 7168, K 2048,
// 119 us in index order, 111 like this, 115 with 256-row tiles only.
// order[r] of rank r is its first m-tile << kRankBits | its group; returns the
// number of m-tiles.  Each thread owns 4 consecutive groups; a wave scans its
// threads' sums with lane shifts and the wave totals meet in tmp.  Three counts
// (wide groups, their tiles, all tiles) are 21-bit fields of one sum: a launch
// has at most 2^26 rows (operands are below 2 GiB, rows at least 32 bytes).
constexpr int kRankBits = 10;
constexpr uint32_t kRankGroup = (1u << kRankBits) - 1;
static_assert(kMaxGroups <= 1 << kRankBits, "a group index fits the low bits of a rank");

__device__ __forceinline__ uint32_t order_tiles(const int32_t* gend, int32_t* order, int E,
                                                uint64_t* tmp, uint32_t& wide_groups) {
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  uint64_t loc[4], sum = 0;
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int g = 4 * t + u;
    loc[u] = 0;
    if (g < E) {
      int32_t b, e;
      group_range(gend, g, b, e);
      const uint64_t tiles = (tiled_rows(b, e) + kTileQ - 1) / kTileQ;
      loc[u] = tiles << 42 | (is_thin(b, e) ? 0u : tiles << 21 | 1u);
    }
    sum += loc[u];
  }
  uint64_t inc = sum;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const uint64_t below = __shfl_up((unsigned long long)inc, off);
    inc += lane >= off ? below : 0;
  }
  if (lane == 63) tmp[wave] = inc;
  __syncthreads();
  uint64_t run = inc - sum, all = 0;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    if (w < wave) run += tmp[w];
    all += tmp[w];
  }
  constexpr uint32_t kField = (1u << 21) - 1;
  const uint32_t wide = (uint32_t)all & kField, wide_tiles = (uint32_t)(all >> 21) & kField;
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int g = 4 * t + u;
    const uint32_t wg = (uint32_t)run & kField, wt = (uint32_t)(run >> 21) & kField;
    const uint32_t at = (uint32_t)(run >> 42);
    const bool w = ((uint32_t)loc[u] & 1u) != 0;
    if (g < E)
      order[w ? wg : wide + (uint32_t)g - wg] =
          (int32_t)((w ? wt : wide_tiles + at - wt) << kRankBits | (uint32_t)g);
    run += loc[u];
  }
  __syncthreads();
  wide_groups = (uint32_t)uniform((int32_t)wide);
  return (uint32_t)uniform((int32_t)(all >> 42));
}

// The work of one launch, the same for every workgroup.
struct FwdPlan {
  uint32_t n_tiles, m_tiles;    // P tiles; m-tiles over all groups
  uint32_t pieces;              // thin P tiles per P tile: 2, or 1 if all tiles are thin
  uint32_t total, full;         // tiles; those in full rounds of the grid
  uint32_t S, chunk;            // K-ranges of a tile past `full`, stages per range
  uint32_t thin_rows;           // groups of at most this many rows take thin tiles
  uint32_t items;               // work items: full tiles, then (tile, range) pairs
};

// One work item: a tile and its range of the contraction.
struct FwdItem {
  uint32_t g, q0, p0, klo, kend;
  int32_t gb, ge;
  uint32_t tail, split;         // tile index past `full` and K-range (split tiles)
  bool part;
};

// Item index handled by this workgroup in the round starting at `base`
// (0xFFFFFFFF: none): each XCD takes a contiguous slice of the round.  A last,
// partial round is spread over all XCDs, and after a full round over the other
// end of each one's workgroups: the first ones may have had a 256-row tile
// (40 experts, one of 984 rows, the others of 24, N 3072, K 3072: 105 -> 95 us).
__device__ __forceinline__ uint32_t fwd_lid(uint32_t base, uint32_t items) {
  const uint32_t xcd = blockIdx.x & 7u;
  uint32_t per = gridDim.x >> 3, slot = blockIdx.x >> 3;
  if (items - base < gridDim.x) {
    if (base != 0) slot = per - 1u - slot;
    per = (items - base + 7u) >> 3;
    if (slot >= per) return 0xFFFFFFFFu;
  }
  return base + xcd * per + slot;
}

template <bool SWIGLU>
__device__ __forceinline__ void fwd_item(const SmemThin& sm, const FwdPlan& pl, int E, uint32_t K,
                                         uint32_t gm, uint32_t lid, FwdItem& it) {
  uint32_t tile = lid;
  it.part = pl.S > 1u && lid >= pl.full;
  it.tail = it.split = 0;
  it.klo = 0;
  it.kend = K;
  if (it.part) {
    it.tail = (lid - pl.full) / pl.S;
    it.split = (lid - pl.full) % pl.S;
    tile = pl.full + it.tail;
    it.klo = it.split * pl.chunk * kStageK;
    it.kend = min(K, it.klo + pl.chunk * kStageK);
  }
  uint32_t mt, nt;
  band_decode(tile, pl.m_tiles, pl.n_tiles, gm, mt, nt);
  // group of m-tile mt: the last rank whose first m-tile is <= mt
  const int at = last_le(sm.order, E, mt << kRankBits | kRankGroup);
  const uint32_t rank = (uint32_t)uniform(sm.order[at]);
  it.g = rank & kRankGroup;
  group_range(sm.gend, (int)it.g, it.gb, it.ge);
  it.gb = uniform(it.gb);
  it.ge = uniform(it.ge);
  it.q0 = (uint32_t)(it.gb & ~3) + (mt - (rank >> kRankBits)) * kTileQ;
  it.p0 = nt * pl.pieces * (SWIGLU ? kThinP / 2u : kThinP);
}

// THIN: the second half of the tile's P rows starts at tile row 64.
template <bool SCALED, bool SWIGLU, bool THIN>
__device__ __forceinline__ void fwd_operands(const FwdArgs& args, const FwdItem& it, Operand& P,
                                             Operand& Q) {
  const uint32_t K = (uint32_t)args.K;
  const uint8_t* wg = args.w + (int64_t)it.g * args.w_gstride;
  P.data = make_desc(wg, (uint32_t)((int64_t)(args.N - 1) * args.ldw + K));
  P.ld = (uint32_t)args.ldw;
  P.row0 = it.p0;
  P.hi = SWIGLU ? (uint32_t)args.N / 2u : (THIN ? kThinP / 2u : 128u);
  // The A range ends at the group's last row (ge >= 1: empty groups have no
  // tiles), so the rows of a partial m-tile past the group end load as zeros
  // instead of the next expert's rows: no fetch, and the matrix cores run
  // on zeros there (C2 +2%, C3 +1%; those rows are never stored).
  Q.data = make_desc(args.a, (uint32_t)((int64_t)(it.ge - 1) * args.lda + K));
  Q.ld = (uint32_t)args.lda;
  Q.row0 = it.q0;
  Q.hi = 128u;
  if (SCALED) {
    const uint8_t* wsg = args.ws + (int64_t)it.g * args.ws_gstride;
    P.scale = make_desc(wsg, scale_extent(K / 32, args.ldws, args.N));
    P.lds = (uint32_t)args.ldws;
    Q.scale = make_desc(args.as, scale_extent(K / 32, args.ldas, args.M));
    Q.lds = (uint32_t)args.ldas;
  }
}

// Header entry of a split tile of at most `rows` rows, and the slot of its
// partial for this K-range.
__device__ __forceinline__ char* split_slot(const FwdArgs& args, const FwdPlan& pl,
                                            const FwdItem& it, uint32_t rows, uint32_t piece) {
  if (it.split == 0 && piece == 0 && threadIdx.x == 0) {
    int32_t* hdr = reinterpret_cast<int32_t*>(args.split_ws) + 4 + 4 * it.tail;
    hdr[0] = (int32_t)it.q0;
    hdr[1] = (int32_t)it.p0;
    hdr[2] = it.gb;
    hdr[3] = min(it.ge, (int32_t)(it.q0 + rows));
  }
  return reinterpret_cast<char*>(args.split_ws) + kSplitHdrBytes +
         (int64_t)(it.tail * pl.S + it.split) * kPartialBytes;
}

template <int I, int N, class F>
__device__ __forceinline__ void unroll(const F& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    unroll<I + 1, N>(f);
  }
}

// The stream of ring stages of a workgroup's thin tiles, six stages ahead of the
// matrix cores.  A stage is 7 loads per wave: 4 of P and 2 of Q (load i of wave
// w fills slots 32i + 8w + l/8 of its operand; slot 64a + 16b + c holds row
// 64a + 4c + b, so a 16-row fragment is 16 slots in a row), then scales: waves 0
// and 1 two P blocks each, wave 2 the four Q blocks, wave 3 zeros (every wave
// issues the same number of loads, which the wait counts rely on).
template <bool SCALED>
struct ThinFeed {
  static constexpr int kLoads = 6 + (SCALED ? 1 : 0);
  Operand P, Q;
  desc_t S;             // this wave's scale operand
  uint32_t vp, vq, vs;  // lane offsets of load 0 without k
  uint32_t kcol;        // lane's chunk column within a stage (bytes)
  uint32_t lds, blk;    // bytes per scale block-row; lane's block within a stage
  uint32_t k, kend;     // next stage's first contraction byte, end of the item
  uint32_t left;        // stages of the tile not yet issued (past the last tile: no end)
  uint32_t bp, bq, bs;  // lane offsets of the stage being issued
  bool live;

  __device__ __forceinline__ void start(uint32_t klo, uint32_t khi) {
    const uint32_t lane = threadIdx.x & 63u, wave = wave_id();
    kcol = 16u * ((lane & 7u) ^ ((4u * wave + (lane >> 4)) & 7u));
    k = klo;
    kend = khi;
    left = (khi - klo + kStageK - 1) / kStageK;
    const uint32_t r = 4u * (8u * (wave & 1u) + (lane >> 3)) + (wave >> 1);
    vp = (P.row0 + r) * P.ld + kcol;
    vq = (Q.row0 + r) * Q.ld + kcol;
    if (SCALED) {
      const bool p = wave < 2u;
      S = p ? P.scale : Q.scale;
      lds = p ? P.lds : Q.lds;
      blk = p ? 2u * wave + (lane >> 5) : lane >> 4;
      vs = blk * lds + (p ? P.row0 + 4u * (lane & 31u) + ((lane & 16u) ? P.hi - 64u : 0u)
                          : Q.row0 + 4u * (lane & 15u));
      if (wave == 3u) blk = 0x80000000u;  // never inside a tile
    }
  }
  __device__ __forceinline__ void begin_stage() {
    const bool ok = live && k + kcol < kend;
    bp = ok ? vp + k : kOobOffset;
    bq = ok ? vq + k : kOobOffset;
    if (SCALED) bs = live && (k >> 5) + blk < (kend >> 5) ? vs : kOobOffset;
  }
  template <int I>
  __device__ __forceinline__ void load(uint8_t* stage) const {
    const uint32_t at = lds_offset(stage) + 1024u * wave_id();
    if constexpr (I < 4)
      dma_x4(P.data, at + 4096u * I, bp, ((I >> 1) * P.hi + 2u * (I & 1)) * P.ld);
    else if constexpr (I < 6)
      dma_x4(Q.data, at + kThinQOff + 4096u * (I - 4), bq, 2u * (I - 4) * Q.ld);
    else
      dma_x1(S, lds_offset(stage) + kThinScaleOff + 256u * wave_id(), bs, (k >> 5) * lds);
  }
};

// Output of a thin tile.  acc[4G + i] register r of lane c + 16g of wave w is the
// value of P index 64G + 16g + 4r + i and Q row 4c + w: per G a lane holds 16
// consecutive P values of one row.
__device__ __forceinline__ uint32_t thin_q_row() {
  return 4u * (threadIdx.x & 15u) + (threadIdx.x >> 6);
}
__device__ __forceinline__ uint32_t thin_p_col() { return 16u * ((threadIdx.x & 63u) >> 4); }

// The 16 values of half G as packed bf16: two 16-byte chunks.
__device__ __forceinline__ void thin_bf16(const v4f (&acc)[8], int G, uint4 (&v)[2]) {
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int r = 2 * h;
    v[h] = make_uint4(pack_bf16x2(acc[4 * G][r], acc[4 * G + 1][r]),
                      pack_bf16x2(acc[4 * G + 2][r], acc[4 * G + 3][r]),
                      pack_bf16x2(acc[4 * G][r + 1], acc[4 * G + 1][r + 1]),
                      pack_bf16x2(acc[4 * G + 2][r + 1], acc[4 * G + 3][r + 1]));
  }
}

template <bool F32>
__device__ __forceinline__ void thin_store(const v4f (&acc)[8], char* out, int64_t ldo_bytes,
                                           uint32_t q0, uint32_t qbeg, uint32_t qend, uint32_t p0,
                                           uint32_t pend) {
  const uint32_t q = q0 + thin_q_row();
  if (q < qbeg || q >= qend) return;
  char* row = out + (int64_t)q * ldo_bytes;
#pragma unroll
  for (int G = 0; G < 2; ++G) {
    const uint32_t p = p0 + 64u * (uint32_t)G + thin_p_col();
    if constexpr (F32) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float* dst = reinterpret_cast<float*>(row) + p + 4 * r;
        const v4f v = {acc[4 * G][r], acc[4 * G + 1][r], acc[4 * G + 2][r], acc[4 * G + 3][r]};
        if (p + 4u * r + 4u <= pend) {
          *reinterpret_cast<v4f*>(dst) = v;  // the ABI aligns rows to 4 elements
        } else {
#pragma unroll
          for (uint32_t e = 0; e < 4u; ++e)
            if (p + 4u * r + e < pend) dst[e] = v[e];
        }
      }
    } else {
      uint4 v[2];
      thin_bf16(acc, G, v);
#pragma unroll
      for (uint32_t h = 0; h < 2; ++h) {
        uint16_t* dst = reinterpret_cast<uint16_t*>(row) + p + 8u * h;
        if (p + 8u * h + 8u <= pend && (reinterpret_cast<uintptr_t>(dst) & 15u) == 0) {
          *reinterpret_cast<uint4*>(dst) = v[h];
        } else {
          const uint32_t w[4] = {v[h].x, v[h].y, v[h].z, v[h].w};
#pragma unroll
          for (uint32_t e = 0; e < 8u; ++e)
            if (p + 8u * h + e < pend) dst[e] = (uint16_t)(w[e >> 1] >> (16u * (e & 1u)));
        }
      }
    }
  }
}

// SiLU(gate) * up and its row-wise MXFP8 cast: half 0 holds 16 gate values of a
// token, half 1 the up values of the same features.  A 32-feature block is the
// lanes g, g ^ 1.  The arithmetic is epilogue_swiglu's, chunk by chunk.
template <int MODE, bool KEEP>
__device__ __forceinline__ void thin_swiglu(const v4f (&acc)[8], const FwdArgs& args, uint32_t q0,
                                            uint32_t qbeg, uint32_t qend, uint32_t p0) {
  const uint32_t f = p0 + thin_p_col();
  const int64_t F = args.N / 2;
  const uint32_t tok = q0 + thin_q_row();
  const bool in = tok >= qbeg && tok < qend;
  uint4 g[2], u[2];
  thin_bf16(acc, 0, g);
  thin_bf16(acc, 1, u);
  if (KEEP && in) {
    uint16_t* h = static_cast<uint16_t*>(args.out) + (int64_t)tok * args.ldo + f;
    *reinterpret_cast<uint4*>(h) = g[0];
    *reinterpret_cast<uint4*>(h + 8) = g[1];
    *reinterpret_cast<uint4*>(h + F) = u[0];
    *reinterpret_cast<uint4*>(h + F + 8) = u[1];
  }
  const uint4 a0 = swiglu_a_chunk(g[0], u[0]), a1 = swiglu_a_chunk(g[1], u[1]);
  uint32_t am = max(amax16_of_chunk(a0), amax16_of_chunk(a1));
  am = max(am, (uint32_t)__shfl_xor((int)am, 16));
  const uint32_t b = e8m0_from_amax16<MODE>(am);
  const bool any = __any(needs_full_encoder<MODE, false>(b));
  const uint2 o0 = any ? encode_chunk8<MODE, false, true>(a0, b)
                       : encode_chunk8<MODE, false, false>(a0, b);
  const uint2 o1 = any ? encode_chunk8<MODE, false, true>(a1, b)
                       : encode_chunk8<MODE, false, false>(a1, b);
  if (in) {
    uint8_t* dst = args.aq + (int64_t)tok * args.ldaq + f;  // 8-byte aligned
    *reinterpret_cast<uint2*>(dst) = o0;
    *reinterpret_cast<uint2*>(dst + 8) = o1;
    if ((threadIdx.x & 16u) == 0)
      args.as_out[(int64_t)tok * args.as_row + (int64_t)(f >> 5) * args.as_blk] = (uint8_t)b;
  }
}

// This workgroup's items from round `base` (item `it`) on, as long as their
// tiles are thin.  `base` advances past them.
template <bool SCALED, int OUT>
__device__ __forceinline__ void thin_run(SmemThin& sm, const FwdArgs& args, const FwdPlan& pl,
                                         int E, uint32_t gm, uint32_t& base, FwdItem& it) {
  constexpr bool F32 = OUT == kOutF32;
  constexpr bool SWIGLU = OUT >= kOutSwigluRceil;
  constexpr uint32_t kStep = SWIGLU ? kThinP / 2u : kThinP;  // output columns of a tile
  using Feed = ThinFeed<SCALED>;
  const uint32_t G = gridDim.x, K = (uint32_t)args.K;
  const uint32_t cols = SWIGLU ? (uint32_t)args.N / 2u : (uint32_t)args.N;
  // the workgroup's next thin tile after (b, x, piece); false if there is none
  auto advance = [&](uint32_t& b, FwdItem& x, uint32_t& piece) {
    if (++piece < pl.pieces && x.p0 + kStep < cols) {
      x.p0 += kStep;
      return true;
    }
    piece = 0;
    b += G;
    if (b >= pl.items) return false;
    const uint32_t lid = fwd_lid(b, pl.items);
    if (lid >= pl.items) return false;
    fwd_item<SWIGLU>(sm, pl, E, K, gm, lid, x);
    return tiled_rows(x.gb, x.ge) <= pl.thin_rows;
  };

  uint8_t* const ring = &sm.ring[0][0];
  Feed feed;
  FwdItem fit = it;  // the tile being loaded
  uint32_t fbase = base, fpiece = 0;
  auto feed_tile = [&]() {
    fwd_operands<SCALED, SWIGLU, true>(args, fit, feed.P, feed.Q);
    feed.start(fit.klo, fit.kend);
  };
  auto feed_next = [&]() {
    feed.live = advance(fbase, fit, fpiece);
    if (feed.live)
      feed_tile();
    else
      feed.left = 0xFFFFFFFFu;
  };
  feed.live = true;
  feed_tile();
#pragma unroll 1
  for (uint32_t d = 0; d < kThinStages; ++d) {
    feed.begin_stage();
    unroll<0, Feed::kLoads>([&](auto i) { feed.template load<i>(ring + d * kThinStageBytes); });
    feed.k += kStageK;
    if (--feed.left == 0) feed_next();
  }

  // LDS offsets of the lane's fragments and scale dwords within a stage
  const uint32_t lane = threadIdx.x & 63u, w = wave_id();
  const uint32_t m = lane & 15u, g = lane >> 4, sw = swz(m);
  const uint32_t clo = m * kStageK + ((g ^ sw) << 4), chi = m * kStageK + (((g + 4u) ^ sw) << 4);
  const uint32_t qr = kThinQOff + 2048u * w;
  const uint32_t ps = kThinScaleOff + 128u * g + 4u * m;
  const uint32_t qs = kThinScaleOff + 512u + 64u * g + 4u * m;

  // fragments and scale dwords of the stage in the matrix cores
  v8i a[8], b;
  uint32_t sa[2], sb;
  auto read_a = [&](const uint8_t* st, uint32_t p) {
    return lds_v8i(st + 2048u * p + clo, st + 2048u * p + chi);
  };
  auto read_b = [&](const uint8_t* st) { return lds_v8i(st + qr + clo, st + qr + chi); };
  // unscaled: scale byte 127 (2^0) everywhere
  auto read_sa = [&](const uint8_t* st, uint32_t G) {
    return SCALED ? *reinterpret_cast<const uint32_t*>(st + ps + 64u * G) : 0x7F7F7F7Fu;
  };
  auto read_sb = [&](const uint8_t* st) {  // Q row 4m + w: byte w
    return SCALED ? *reinterpret_cast<const uint32_t*>(st + qs) >> (8u * w) : 0x7F7F7F7Fu;
  };
  wait_barrier<(kThinStages - 1) * Feed::kLoads>();
  __builtin_amdgcn_sched_barrier(0);
  b = read_b(ring);
#pragma unroll
  for (uint32_t p = 0; p < 8; ++p) a[p] = read_a(ring, p);
  sa[0] = read_sa(ring, 0);
  sa[1] = read_sa(ring, 1);
  sb = read_sb(ring);

  uint32_t cur = 0;  // ring offset of the stage in the registers
  uint32_t piece = 0;
  do {
    uint32_t todo = (it.kend - it.klo + kStageK - 1) / kStageK;  // >= 1
    v4f acc[8];
#pragma unroll
    for (int p = 0; p < 8; ++p) acc[p] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    do {
      // Stages until this tile or the feed's tile ends; the loop over them has
      // no branch (MFMAs have no side effects, the compiler would move them
      // behind one).
      uint32_t n = min(todo, feed.left);
      todo -= n;
      feed.left -= n;
      do {
        // The next stage has landed (the four newer ones may be out; an
        // epilogue's stores only make the count stricter), and every wave
        // holds this stage in registers, so its slot takes the loads issued
        // below.
        wait_barrier<(kThinStages - 2) * Feed::kLoads>();
        __builtin_amdgcn_sched_barrier(0);
        uint8_t* dst = ring + cur;
        cur = cur == (kThinStages - 1) * kThinStageBytes ? 0u : cur + kThinStageBytes;
        const uint8_t* nx = ring + cur;
        feed.begin_stage();
        // The matrix work on this stage; each fragment register is refilled
        // from the next stage right after its last use, and the loads are
        // spread over it: a wave's issue stalls at a load until the address
        // unit takes it.
        unroll<0, 8>([&](auto i) {
          constexpr int p = decltype(i)::value;
          acc[p] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(
              a[p], b, acc[p], 0, 0, p & 3, (int)sa[p >> 2], 0, (int)sb);
          a[p] = read_a(nx, p);
          if constexpr (p == 3) sa[0] = read_sa(nx, 0);
          if constexpr (p == 7) {
            b = read_b(nx);
            sa[1] = read_sa(nx, 1);
            sb = read_sb(nx);
          }
          if constexpr (p < Feed::kLoads) feed.template load<p>(dst);
          __builtin_amdgcn_sched_barrier(0);
        });
        feed.k += kStageK;
      } while (--n != 0);
      if (feed.left == 0) feed_next();
    } while (todo != 0);
    const uint32_t gb = (uint32_t)it.gb, ge = (uint32_t)it.ge;
    if (it.part) {
      thin_store<true>(acc, split_slot(args, pl, it, kThinQ, piece), 1024, 0u, 0u, kThinQ,
                       piece * kThinP, 256u);
    } else if constexpr (SWIGLU) {
      constexpr int MODE =
          (OUT == kOutSwigluRceil || OUT == kOutSwigluKeepRceil) ? kModeRceil : kModeFloor;
      thin_swiglu<MODE, (OUT >= kOutSwigluKeepRceil)>(acc, args, it.q0, gb, ge, it.p0);
    } else {
      thin_store<F32>(acc, static_cast<char*>(args.out), args.ldo * (F32 ? 4 : 2), it.q0, gb, ge,
                      it.p0, (uint32_t)args.N);
    }
  } while (advance(base, it, piece));
  // the loads past the end have landed before anything else uses the ring
  wait_barrier<0>();
}

// The kernel's first argument, read again from the kernel-argument segment.
// Kept in registers over the tile loop, the 46 argument words of two kinds of
// tile outnumber the scalar registers (115 spilled to vector lanes in the fp32
// form, 73 in bf16; read per tile 38 and 39), and the 256-row tiles paid for it:
// 32 experts of 100 rows, N 7168, K 2048, 140.3 -> 139.4 us (k_grouped_fwd
// 138.2), with SwiGLU 150.6 -> 148.1 (148.3).
__device__ __forceinline__ FwdArgs reread_args() {
  typedef const FwdArgs __attribute__((address_space(4))) * KernArgs;
  KernArgs p = (KernArgs)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));  // opaque: the loads stay where they are
  return *(const FwdArgs*)p;
}

// ---------------------------------------------------------------------------
// The grouped forward for launches whose experts hold few rows: the tile order
// and the split of k_grouped_fwd, with thin tiles for the groups that fit one.
// `args` is the first parameter (reread_args).
// ---------------------------------------------------------------------------
template <bool SCALED, int OUT>
__global__ __launch_bounds__(kThreads, 1) void k_grouped_fwd_thin(FwdArgs args, uint32_t gm) {
  constexpr bool F32 = OUT == kOutF32;
  constexpr bool SWIGLU = OUT >= kOutSwigluRceil;
  constexpr bool KEEP = OUT >= kOutSwigluKeepRceil;
  constexpr int SW_MODE =
      (OUT == kOutSwigluRceil || OUT == kOutSwigluKeepRceil) ? kModeRceil : kModeFloor;
  __shared__ SmemThin sm;
  const int E = args.group_ends ? args.E : 1;
  const int32_t M = args.M;
  if (args.group_ends)
    monotone_ends_to_lds(args.group_ends, E, M, sm.gend);
  else if (threadIdx.x == 0)
    sm.gend[0] = M;
  __syncthreads();
  FwdPlan pl;
  uint32_t wide;  // groups of more rows than a thin tile
  pl.m_tiles = order_tiles(sm.gend, sm.order, E, sm.scan_tmp, wide);
  // SWIGLU: N = 2F weight rows; a tile covers 128 features of a (F % 128 == 0)
  pl.n_tiles = SWIGLU ? (uint32_t)args.N / 256u : ((uint32_t)args.N + kTileP - 1) / kTileP;
  pl.total = pl.m_tiles * pl.n_tiles;
  const uint32_t K = (uint32_t)args.K;
  // With a workspace, a last round of tiles that would leave at least half of
  // the workgroups idle is cut along K into S ranges (whole stages), one work
  // item each; k_fwd_split_reduce adds the S partials in a fixed order.
  const uint32_t G = gridDim.x;
  pl.full = pl.total / G * G;
  const uint32_t rem = pl.total - pl.full;
  const uint32_t nst = (K + kStageK - 1) / kStageK;
  pl.S = 1;
  pl.chunk = nst;
  if (args.split_ws != nullptr && rem > 0 && rem <= G / 2 && nst > 1) {
    pl.S = min(min(G / rem, nst), pl.full > 0 ? kMaxSplitTail : kMaxSplit);
    pl.chunk = (nst + pl.S - 1) / pl.S;
    pl.S = (nst + pl.chunk - 1) / pl.chunk;
  }
  int32_t* hdr = reinterpret_cast<int32_t*>(args.split_ws);
  if (hdr != nullptr && blockIdx.x == 0 && threadIdx.x == 0) {
    hdr[0] = pl.S > 1 ? (int32_t)rem : 0;
    hdr[1] = (int32_t)pl.S;
  }
  pl.items = pl.S > 1 ? pl.full + rem * pl.S : pl.total;
  pl.pieces = 2;
  // No thin tiles where they share a last round that is nearly full with 256-row
  // ones and the contraction is long, or the only round is nearly full: there
  // the 256-row tiles decide when the launch ends, and beside thin ones they
  // take longer (two rounds of 32 experts, N 4096, K 7168: multinomial sizes
  // around 56 180 us, with thin tiles 185; two experts of more than 64 rows 171
  // and 184; one round of 8 experts, N 7168, K 2048: 28.0 and 30.5).  The SwiGLU
  // forms gain from thin tiles there too (64 experts of Zipf sizes around 16,
  // N 2048, K 2048: 67 -> 56): their 256-row epilogue is the longer one.
  pl.thin_rows = kThinQ;
  const bool full_round = rem == 0 || 5 * rem > 4 * G;
  if (!SWIGLU && wide != 0 && pl.S == 1 && full_round &&
      (nst > 40 || (nst >= 16 && pl.total <= G)))
    pl.thin_rows = 0;
  // Nothing split and every tile thin (decode): the thin P tiles are the work
  // items, so that the last round is a finer share of the whole.
  if (wide == 0 && pl.S == 1) {
    pl.pieces = 1;
    pl.n_tiles = ((uint32_t)args.N + kThinP - 1) / kThinP;
    pl.items = pl.total = pl.full = pl.m_tiles * pl.n_tiles;
  }

  uint32_t base = 0;
  while (base < pl.items) {
    const uint32_t lid = fwd_lid(base, pl.items);
    if (lid >= pl.items) break;
    FwdItem it;
    fwd_item<SWIGLU>(sm, pl, E, K, gm, lid, it);
    if (tiled_rows(it.gb, it.ge) <= pl.thin_rows) {  // this item and the thin ones after it
      thin_run<SCALED, OUT>(sm, reread_args(), pl, E, gm, base, it);
      continue;
    }
    const FwdArgs args = reread_args();
    Operand P, Q;
    fwd_operands<SCALED, SWIGLU, false>(args, it, P, Q);
    const uint32_t q0 = it.q0, p0 = it.p0;
    v4f acc[64];
    if (it.part) {
      mainloop<SCALED>(sm, P, Q, it.klo, it.kend, acc);
      // the whole 256x256 fp32 partial, rows and columns unmasked
      epilogue<true>(sm, acc, split_slot(args, pl, it, kTileQ, 0), 1024, 0u, 0u, 256u, 0u, 256u);
    } else if constexpr (SWIGLU) {
      mainloop<SCALED>(sm, P, Q, 0u, K, acc);
      epilogue_swiglu<SW_MODE, KEEP>(sm, acc, args.aq, args.ldaq, args.as_out, args.as_row,
                                     args.as_blk, q0, (uint32_t)it.gb, (uint32_t)it.ge, p0,
                                     static_cast<uint16_t*>(args.out), args.ldo,
                                     (uint32_t)args.N / 2u);
    } else {
      mainloop<SCALED>(sm, P, Q, 0u, K, acc);
      const int64_t ldo_bytes = args.ldo * (F32 ? 4 : 2);
      if constexpr (F32)
        epilogue<true>(sm, acc, reinterpret_cast<char*>(args.out), ldo_bytes, q0, (uint32_t)it.gb,
                       (uint32_t)it.ge, p0, (uint32_t)args.N);
      else
        epilogue_bf16(sm, acc, reinterpret_cast<char*>(args.out), ldo_bytes, q0, (uint32_t)it.gb,
                      (uint32_t)it.ge, p0, (uint32_t)args.N);
    }
    base += G;
  }
}
