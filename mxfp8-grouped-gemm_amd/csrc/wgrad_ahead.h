// Weight gradient over few tokens per expert, bf16 dW, scaled operands
// (included by gemm.hip inside its namespace).
//
// With few tokens a tile is two to eight stages of MFMAs (1 us each) and a
// 128 KB store, and the loop of k_grouped_wgrad runs them one after the other:
// vmcnt counts stores and loads together, so the first stage of a tile waits
// until the stores of the tile before have left.  Here the next tile's first
// two stages are loaded before the stores are issued (they retire in that
// order), and the waits of those stages leave the stores in flight.  For that
// the ring has to be free during the stores: the tile is stored straight from
// the accumulators, whole 128-byte lines per instruction.  What is left is the
// store itself: 32 experts x 128 tokens, N 4096, K 7168 write 1.88 GB in
// 324 us, 5.8 TB/s (431 us, 4.4 TB/s, with the stores waited for), where a
// plain fill of such a buffer reaches 6.9.

// The tile straight from the accumulators.  Lane c + 16g holds, for P half G
// and Q fragment 4H + j, columns 64G + 16g .. +15 of row 64H + 4c + j (of the
// wave's 128 x 128): two 16-byte chunks.  Lanes c and c ^ 1 swap one chunk, so
// that one instruction writes the even lane's row and the next the odd lane's:
// 8 rows x 128 bytes each.  Issues exactly kAheadStores stores, or returns with
// none in flight where the wave's block is not wholly inside dW (the guarded
// stores' number varies).
__device__ __forceinline__ void store_bf16_direct(const v4f (&acc)[64], char* out,
                                                  int64_t ldo_bytes, uint32_t q0, uint32_t qend,
                                                  uint32_t p0, uint32_t pend) {
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t wave = wave_id();
  const uint32_t c = lane & 15u, g = lane >> 4;
  const bool odd = (c & 1u) != 0;
  const uint32_t qw = q0 + 128u * (wave >> 1), pw = p0 + 128u * (wave & 1u);
  const bool interior = qw + 128u <= qend && pw + 128u <= pend &&
                        ((reinterpret_cast<uintptr_t>(out) | (uintptr_t)ldo_bytes) & 15u) == 0 &&
                        ldo_bytes < (int64_t)1 << 24;
  const uint32_t row = 4u * (c & ~1u), col = 16u * g + (odd ? 8u : 0u);
  const __amdgpu_buffer_rsrc_t dst = __builtin_amdgcn_make_buffer_rsrc(
      out + (int64_t)qw * ldo_bytes + 2 * (int64_t)pw, (short)0,
      (int)(127u * (uint32_t)ldo_bytes + 256u), 0x00020000);
  const uint32_t voff = row * (uint32_t)ldo_bytes + 2u * col;
#pragma unroll
  for (uint32_t qj = 0; qj < kDirectFrags; ++qj)
#pragma unroll
    for (uint32_t G = 0; G < kDirectHalves; ++G) {
      const uint32_t a0 = 32u * G + qj;
      uint32_t x[2][4];
#pragma unroll
      for (uint32_t b = 0; b < 2; ++b)
#pragma unroll
        for (uint32_t d = 0; d < 4; ++d) {
          // chunk b: P fragments 4G .. 4G+3 of register 2b, then of 2b + 1
          const uint32_t r = 2u * b + (d >> 1), f = a0 + 16u * (d & 1u);
          x[b][d] = pack_bf16x2(acc[f][r], acc[f + 8u][r]);
        }
      u32x4 even, other;
#pragma unroll
      for (uint32_t d = 0; d < 4; ++d) {
        const uint32_t recv = swap_lane_pair(odd ? x[0][d] : x[1][d]);
        even[d] = odd ? recv : x[0][d];
        other[d] = odd ? x[1][d] : recv;
      }
      const uint32_t r0 = 64u * (qj >> 2) + (qj & 3u);
      if (interior) {
        static_assert(kDirectRows == 2, "the two stores below");
        const uint32_t soff = r0 * (uint32_t)ldo_bytes + 128u * G;
        __builtin_amdgcn_raw_buffer_store_b128(even, dst, voff, soff, kCacheNT);
        __builtin_amdgcn_raw_buffer_store_b128(other, dst, voff, soff + 4u * (uint32_t)ldo_bytes,
                                               kCacheNT);
        continue;
      }
#pragma unroll
      for (uint32_t k = 0; k < kDirectRows; ++k) {
        const u32x4 v = k ? other : even;
        const uint32_t q = qw + r0 + row + 4u * k, p = pw + 64u * G + col;
        if (q >= qend || p >= pend) continue;
        uint16_t* o = reinterpret_cast<uint16_t*>(out + (int64_t)q * ldo_bytes) + p;
        if (p + 8u <= pend && (reinterpret_cast<uintptr_t>(o) & 15u) == 0) {
          __builtin_nontemporal_store(v, reinterpret_cast<u32x4*>(o));
        } else {
          for (uint32_t e = 0; e < 8u && p + e < pend; ++e)
            o[e] = (uint16_t)(v[e >> 1] >> (16u * (e & 1u)));
        }
      }
    }
  if (!interior) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// A tile of one value (two bf16 in v: an expert without tokens, or NaN) that lies
// inside dW: wave w writes rows 64w .. 64w+63, two whole 512-byte rows per store,
// kAheadStores stores.  False, with nothing written, for any other tile.  Whole
// rows leave faster than the 128-byte lines above: 4 tokens per expert, all in
// one of 32, N 7168, K 2048, 175 -> 172 us (170 in k_grouped_wgrad, whose other
// routings take 210 to 220 where this kernel takes 157 to 173).
__device__ __forceinline__ bool store_bf16_value(uint32_t v, char* out, int64_t ldo_bytes,
                                                 uint32_t q0, uint32_t qend, uint32_t p0,
                                                 uint32_t pend) {
  if (q0 + kTileQ > qend || p0 + kTileP > pend ||
      ((reinterpret_cast<uintptr_t>(out) | (uintptr_t)ldo_bytes) & 15u) != 0 ||
      ldo_bytes >= (int64_t)1 << 24)
    return false;
  constexpr uint32_t kRows = 2u * kAheadStores;
  static_assert(kRows * kWaves == kTileQ, "the waves' rows make the tile");
  const uint32_t lane = threadIdx.x & 63u;
  const __amdgpu_buffer_rsrc_t dst = __builtin_amdgcn_make_buffer_rsrc(
      out + (int64_t)(q0 + kRows * wave_id()) * ldo_bytes + 2 * (int64_t)p0, (short)0,
      (int)((kRows - 1u) * (uint32_t)ldo_bytes + 512u), 0x00020000);
  const uint32_t voff = (lane >> 5) * (uint32_t)ldo_bytes + 16u * (lane & 31u);
  const u32x4 x = {v, v, v, v};
#pragma unroll
  for (uint32_t i = 0; i < (uint32_t)kAheadStores; ++i)
    __builtin_amdgcn_raw_buffer_store_b128(x, dst, voff, 2u * i * (uint32_t)ldo_bytes, kCacheNT);
  return true;
}

// One dW tile: its expert, token range and place.
struct AheadTile {
  int32_t g, tb, te;
  uint32_t q0, p0;
  bool nan;   // a group boundary inside a 32-token block: written as NaN

  __device__ __forceinline__ bool loads() const { return !nan && te > tb; }
  __device__ __forceinline__ void operands(const WgradArgs& args, Operand& P, Operand& Q) const {
    P.data = make_desc(args.ia, (uint32_t)((int64_t)(args.K - 1) * args.ldia + args.M));
    P.ld = (uint32_t)args.ldia;
    P.row0 = p0;
    P.hi = 128u;
    P.scale = make_desc(args.ias, scale_extent(args.M / 32, args.ldias, args.K));
    P.lds = (uint32_t)args.ldias;
    Q.data = make_desc(args.go, (uint32_t)((int64_t)(args.N - 1) * args.ldgo + args.M));
    Q.ld = (uint32_t)args.ldgo;
    Q.row0 = q0;
    Q.hi = 128u;
    Q.scale = make_desc(args.gos, scale_extent(args.M / 32, args.ldgos, args.N));
    Q.lds = (uint32_t)args.ldgos;
    // Opaque per use: hoisted out of the tile loop, the row steps of all loads
    // outnumber the scalar registers.
    asm volatile("" : "+s"(P.ld), "+s"(Q.ld), "+s"(P.lds), "+s"(Q.lds));
  }
};

__global__ __launch_bounds__(kThreads, 1) void k_grouped_wgrad_ahead(WgradArgs args, uint32_t gm) {
  __shared__ Smem sm;
  const int E = args.E;
  const int32_t M = args.M;
  monotone_ends_to_lds(args.group_ends, E, M, sm.gend);
  for (int g = threadIdx.x; g < E; g += kThreads) {
    int32_t b, e;
    group_range(sm.gend, g, b, e);
    sm.sched[g] = e - b;
  }
  __syncthreads();
  // largest expert first, as in k_grouped_wgrad
  for (int g = threadIdx.x; g < E; g += kThreads) {
    const int32_t sg = sm.sched[g];
    int rank = 0;
    for (int j = 0; j < E; ++j) {
      const int32_t sj = sm.sched[j];
      rank += (sj > sg) || (sj == sg && j < g);
    }
    sm.order[rank] = g;
  }
  __syncthreads();
  const uint32_t n_tiles = ((uint32_t)args.N + kTileQ - 1) / kTileQ;
  const uint32_t k_tiles = ((uint32_t)args.K + kTileP - 1) / kTileP;
  const uint32_t per_expert = n_tiles * k_tiles;
  const uint32_t total = per_expert * (uint32_t)E;

  AheadTile t;
  // Tile `lid` and the loads of its first two stages.
  auto open = [&](uint32_t lid) __attribute__((always_inline)) {
    const uint32_t rank = lid / per_expert;
    t.g = uniform(sm.order[rank]);
    uint32_t nt, kt;
    band_decode(lid - rank * per_expert, n_tiles, k_tiles, gm, nt, kt);
    int32_t tb, te;
    group_range(sm.gend, t.g, tb, te);
    t.tb = uniform(tb);
    t.te = uniform(te);
    t.nan = ((t.tb | t.te) & 31) != 0;
    t.q0 = nt * kTileQ;
    t.p0 = kt * kTileP;
    if (!t.loads()) return;
    Operand P, Q;
    t.operands(args, P, Q);
    Stream<true> st;
    st.init(P, Q, (uint32_t)t.tb, (uint32_t)t.te);
    const uint32_t kbeg = (uint32_t)t.tb & ~(uint32_t)(kStageK - 1);
    st.prologue(sm.ring[0], sm.ring[1], P, Q, kbeg,
                ((uint32_t)t.te - kbeg + kStageK - 1) / kStageK);
  };
  uint32_t lid = xcd_slice(0);
  if (lid >= total) return;
  open(lid);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  for (uint32_t base = gridDim.x;; base += gridDim.x) {
    v4f acc[64];
    if (t.loads()) {
      Operand P, Q;
      t.operands(args, P, Q);
      mainloop<true, false, true>(sm, P, Q, (uint32_t)t.tb, (uint32_t)t.te, acc);
    } else {
      const float v = t.nan ? __builtin_nanf("") : 0.0f;
#pragma unroll
      for (int i = 0; i < 64; ++i) acc[i] = v4f{v, v, v, v};
    }
    char* out = reinterpret_cast<char*>(args.dw) + (int64_t)t.g * args.ldw_e * 2;
    const uint32_t q0 = t.q0, p0 = t.p0;
    const bool value = !t.loads();
    const uint32_t v = t.nan ? 0x7FC07FC0u : 0u;  // what acc rounds to
    lid = xcd_slice(base);
    const bool more = lid < total;
    if (more) open(lid);
    if (!value || !store_bf16_value(v, out, args.ldw_n * 2, q0, (uint32_t)args.N, p0,
                                    (uint32_t)args.K))
      store_bf16_direct(acc, out, args.ldw_n * 2, q0, (uint32_t)args.N, p0, (uint32_t)args.K);
    if (!more) break;
  }
}
