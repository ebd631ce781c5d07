// The D = 576 latent attention kernel (attention.hip includes this inside its namespace,
// after AttnParams, Layout and RowPlan).
//
// One workgroup = one (row, split, 64 heads): 4 waves, one per SIMD with the whole register
// file (512 VGPRs per lane), over tiles of 32 entries held as bf16 in LDS.
//   S^T  wave (eh, hh): entries 16 eh .. + 15 of the tile x heads 32 hh .. + 31 over all 576
//        channels (18 K-steps of v_mfma_f32_16x16x32_bf16, two heads groups per K operand read),
//        so a score is whole in the lane that has it: no partial sums to exchange;
//   P^T  goes to LDS in bf16 (4 KB a tile, two of them);
//   O^T  wave w: the 16-channel blocks w, w + 4, .. w + 32 for all 64 heads, one V^T operand
//        read for four head groups.
// One barrier per tile: in iteration u the workgroup runs S(u+1), PV(u) -- whose matrix work
// covers the softmax of u+1 -- and writes tile u+2 to LDS, so three tiles are live.
// What bounds it: the matrix units (72 MFMA of 16 cycles per wave and tile = 1152 cycles) and,
// close behind, the LDS: K read twice (256 B a cycle), V^T once through the transposing reads
// (128), the tile's store and P, about 960 cycles a tile.  8 waves of 32 heads over quarters
// of D read K and V twice as often and exchanged partial scores: about 2100 cycles of LDS.
// Measured, against that kernel: a causal prompt of 8192 rows x 128 heads, top-2048 of 2048
// entries, 4.14 -> 2.94 ms (671 -> 947 TFLOP/s; a bf16 product of 16384^3 reaches 1360 on the
// same card); the decode step of 32 rows over 8192 keys 68.4 -> 61.5 us.  A tile takes about
// 2050 cycles (bf16; fp8 2280): one wave per SIMD issues an instruction every 5 cycles or so,
// 250 of them a tile, and the barrier adds 180; deeper operand prefetch changed nothing.
//
// Softmax: the exponent's reference is fixed at the first tile's maximum: softmax is exact for
// any reference as long as nothing overflows or underflows.  The weights that count are then
// 1 or more (the true maximum is no lower), so no value of an entry is lost at the low
// end.  At the high end a weight reaches 2^(rise of the scores above the first tile), which
// multiplies an entry's value: up to 2^kRoomNear that is the range of a softmax rescaled as it goes;
// above, the accumulators are looked at after the pass, and above 2^kRoomAbove the row sum itself
// would overflow.  Where either overflowed, the workgroup starts again from the true maxima of
// a pass over the scores alone (weights at most 1).  So no tile waits for the other waves'
// maxima, and O^T is never rescaled.

// An entry's table code: its source in the top two bits, its index below them.
constexpr uint32_t kEmptyEntry = 0xffffffffu;
constexpr uint32_t kSrcDense = 1u << 30, kSrcMain = 2u << 30, kIndexMask = (1u << 30) - 1u;

struct LatentSmem {
  static constexpr int D = 576;
  static constexpr int ROW = 2 * D;            // bytes per entry; the pad is a swizzle (lat_swz)
  static constexpr int TILE = kTile * ROW;
  static constexpr int PB = 3 * TILE;          // P^T: 2 x [4 head groups][64 lanes] x 16 bytes
  static constexpr int TAB = PB + 2 * 4096;    // entry codes; the loop fetches up to 3 tiles past the last
  static constexpr int TABN = kIdxCap + 3 * kTile;
  static constexpr int MASK = TAB + 4 * TABN;  // valid entries of each tile
  static constexpr int PMAX = MASK + 4 * (TABN / kTile + 5);  // [2 eh][64]; 16-byte aligned
  static constexpr int LSUM = PMAX + 512;      // [2 eh][64]
  static constexpr int RED = LSUM + 512;       // reduction scratch, redo, high
  static constexpr int LDS = RED + 64;
};

// 16-byte piece `piece` of row `e` sits at slot piece ^ (e & 7) of its row.  The LDS serves a
// 16-byte access in four phases of 16 lanes over its 64 banks; with 1152-byte rows this puts the
// 16 rows of a K operand's phase (8 rows of one piece, 8 others of its neighbour) on 16
// distinct bank quads, and so the stores of a tile (two rows, every piece or every second one)
// and the transposing reads of V^T.
__device__ __forceinline__ int lat_swz(int e) { return e & 7; }

constexpr float kRoomNear = kLazy, kRoomAbove = 100.0f;    // log2 units above the reference
constexpr float kMasked = -3.0e38f;                        // a masked entry's score: weight 0

// Rows of more scores than this are loaded in whole lines and passed on through LDS.  A thread's own 32
// scores are a line of their own, so loaded directly each instruction touches 64 lines: 8192 keys, one
// row x 64 heads 22.0 -> 21.7 us the launch and its merge, 64 rows 28.4 -> 27.9; at 4096 keys
// both take as long, at 512 LDS costs 0.15 us.
constexpr int kStageScores = 4096;

// A tile in flight: one thread's pieces of entry tid / 8.
template <int FMT>
struct LatRaw {
  static constexpr int NV = FMT == kFmtFp8 ? 5 : 9;
  u32x4 v[NV];
  u32x4 s;  // fp8: the entry's four block scales
};

template <int FMT, int NOPE, bool SEL>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1)))
sparse_mqa_latent_kernel(const AttnParams p) {
  using M = LatentSmem;
  constexpr int D = M::D, NT = 256, KS = D / 32, NI = D / 64;
  constexpr int EB = Layout<FMT, D, NOPE>::kEntryBytes;
  using RP = RowPlan<FMT, D, NOPE, NT>;
  extern __shared__ __align__(16) uint8_t smem[];
  uint32_t* const tab = reinterpret_cast<uint32_t*>(smem + M::TAB);
  uint32_t* const masks = reinterpret_cast<uint32_t*>(smem + M::MASK);
  float* const pmax = reinterpret_cast<float*>(smem + M::PMAX);
  float* const lsum = reinterpret_cast<float*>(smem + M::LSUM);
  int* const wred = reinterpret_cast<int*>(smem + M::RED);
  int* const redo = wred + 8;
  int* const high = wred + 9;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int eh = wave & 1, hh = wave >> 1;
  const int g = lane >> 4, e16 = lane & 15;
  RP rp;
  rp.template locate<true>(p, 64);

  // the index list (or scores), the position and the queries are requested together
  v4i pre[2];
  bool pre_ok = false;
  constexpr int SKPT = 32;
  float4 sc4[SEL ? SKPT / 4 : 1];
  if constexpr (SEL) {
    const float* srow = p.sel_scores + rp.row * p.sel_stride;
    const int G4 = static_cast<int>(p.G) - 4;
#pragma unroll
    for (int m = 0; m < SKPT / 4; ++m) {
      const int o = p.G > kStageScores ? 4 * (NT * m + tid) : SKPT * tid + 4 * m;
      sc4[m] = *reinterpret_cast<const float4*>(srow + (o <= G4 ? o : G4));
    }
  } else {
    pre_ok = rp.prefetch_list(p, tid, pre);
  }
  const int64_t row_pos = p.positions[rp.row];

  // q of the 64 heads is one contiguous run: requested whole lines at a time, and laid out as
  // the B operand of S^T through LDS once the entry table is built.  (Loaded straight into
  // the operand's layout, 64 bytes of a head at a time, it cost 11 K of a workgroup's cycles.)
  constexpr int QP = 18, QROW = D / 8;         // 16-byte pieces per thread, per head
  u32x4 qraw[QP];
  const int q_pieces = (p.H - rp.hgrp * 64 < 64 ? p.H - rp.hgrp * 64 : 64) * QROW;
  {
    const u32x4* qb = reinterpret_cast<const u32x4*>(p.q + (rp.row * p.H + rp.hgrp * 64) * D);
#pragma unroll
    for (int k = 0; k < QP; ++k) {
      const int at = tid + NT * k;
      qraw[k] = qb[at < q_pieces ? at : 0];
    }
  }
  // RoPE of q: the rope slice is the last two K-steps, 4 pairs per lane and step
  constexpr int RST = (D - NOPE) / 32;
  uint2 qrc[RST > 0 ? RST : 1], qrs[RST > 0 ? RST : 1];
  if constexpr (RST > 0) {
    const uint16_t* cb = p.rope_cos ? p.rope_cos : p.q;
    const uint16_t* sb = p.rope_cos ? p.rope_sin : p.q;
    const uint32_t roff = static_cast<uint32_t>(rp.row * ((D - NOPE) / 2)) + 4 * g;
#pragma unroll
    for (int r = 0; r < RST; ++r) {
      qrc[r] = *reinterpret_cast<const uint2*>(cb + roff + 16 * r);
      qrs[r] = *reinterpret_cast<const uint2*>(sb + roff + 16 * r);
    }
  }
  // in-launch merge: register the XCC this workgroup runs on with its (row, 64-head group)
  uint32_t* mrec = nullptr;
  if (p.merge_rec != nullptr) {
    const uint32_t nhg = static_cast<uint32_t>((p.H + 63) / 64);
    mrec = p.merge_rec + 4 * (static_cast<uint32_t>(rp.row) * nhg + static_cast<uint32_t>(rp.hgrp));
    if (tid == 0)
      __hip_atomic_fetch_add(reinterpret_cast<uint64_t*>(mrec), 1ull << (8 * xcc_id()), __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
  }
  if (tid == 0) *redo = *high = 0;

  // ---- the split's entry table -----------------------------------------------------------
  int32_t* const sidx = reinterpret_cast<int32_t*>(smem);  // the row's list, where tiles come later
  if constexpr (SEL) {
    rp.plan_row(p, row_pos);
    // the selection's LDS lies behind the list
    static_assert(SKPT * NT == 8192, "the selecting instance takes up to 8192 scores");
    int* const h1 = reinterpret_cast<int*>(smem + 4 * 8 * NT);
    int* const h2 = h1 + kHist1<NT>;
    int* const h3 = h2 + kBins;
    int* const sw = h3 + kBins / 2;
    static_assert(4 * 8 * NT + (kHist1<NT> + kBins + kBins / 2 + 16) * 4 <= M::PB, "selection LDS");
    const RowSelLds lds{h1, h2, h3, sw, sw + 8, sw + 12};
    const int G = static_cast<int>(p.G), k = p.topk;
    const bool search = G > k;
    // A long row's scores come in whole lines and reach their thread, 32 neighbours each, through
    // LDS: piece j of thread t's at slot j ^ (t / 2 & 7), so that both passes meet every bank once.
    const bool staged = p.G > kStageScores;  // uniform
    float4* const stage = reinterpret_cast<float4*>(smem + M::PB - 4 * 8192);
    static_assert(4 * 8 * NT + (kHist1<NT> + kBins + kBins / 2 + 16) * 4 <= M::PB - 4 * 8192, "behind the selection's LDS");
    if (staged) {
#pragma unroll
      for (int m = 0; m < SKPT / 4; ++m) {
        const int t = (NT / 8) * m + (tid >> 3);
        stage[8 * t + ((tid & 7) ^ ((t >> 1) & 7))] = sc4[m];
      }
    }
    if (search) row_sel_clear<NT>(lds, tid);
    if (search || staged) lds_barrier();
    if (staged) {
#pragma unroll
      for (int m = 0; m < SKPT / 4; ++m) sc4[m] = stage[8 * tid + (m ^ ((tid >> 1) & 7))];
    }
    const int i0 = SKPT * tid;
    uint32_t key[SKPT];
#pragma unroll
    for (int m = 0; m < SKPT / 4; ++m) {
      const float v[4] = {sc4[m].x, sc4[m].y, sc4[m].z, sc4[m].w};
#pragma unroll
      for (int c = 0; c < 4; ++c) key[4 * m + c] = order_key(v[c]) & key_mask(i0 + 4 * m + c, G);
    }
    uint32_t T;
    int need_eq;
    row_sel_threshold<SKPT, NT>(key, search, k, lds, T, need_eq);
    const RowTake tk = row_sel_take<SKPT, NT>(key, T, need_eq, sw);
    // The selection is bound by one wave's chain of instructions per SIMD (32 scores per thread,
    // some 10 K of a short step's 40 K cycles), so nothing in it is conditional per key: see
    // the spare words of topk_core.h.  The launch, against conditional counts and stores and
    // first-level counters side by side: one row over 8192 keys 21.0 -> 19.0 us, 8 rows 24.2 ->
    // 22.5, 32 rows 38.8 -> 36.8, one row over 512 keys 14.4 -> 13.6.
    // The list is in the top-k launch's form by construction: planned over its valid entries.
    // A thread's picks take list positions pos .. pos + popcount - 1, ascending with the
    // thread, so only the threads around this split's slice walk them -- and every thread of
    // the row's first workgroup, which writes the list
    rp.plan_split(p, tk.written);
    const bool lists = p.sel_out != nullptr && rp.split == 0 && rp.hgrp == 0;
    if (lists || (tk.pos < rp.v_end - rp.nwd && tk.pos + __builtin_popcount(tk.sel) > rp.sp_begin)) {
      int* const spare = row_sel_spare<NT>(lds, lane);
      int at = tk.pos;
#pragma unroll
      for (int j = 0; j < SKPT; ++j) {
        const int take = static_cast<int>((tk.sel >> j) & 1u);
        *(take ? sidx + at : spare) = i0 + j;
        at += take;
      }
    }
    if (lists) {
      lds_barrier();
      int32_t* const orow = p.sel_out + rp.row * p.sel_out_stride;
      for (int i = 4 * tid; i < k; i += 4 * NT) {
        v4i w = *reinterpret_cast<const v4i*>(sidx + i);
#pragma unroll
        for (int c = 0; c < 4; ++c) w[c] = i + c < tk.written ? w[c] : -1;
        *reinterpret_cast<v4i*>(orow + i) = w;
      }
    }
    pre_ok = true;
  } else {
    rp.plan(p, row_pos, pre_ok ? rp.valid_prefix_list(p, tid, pre, wred) : -1);
    if (pre_ok) rp.stage_list(sidx, tid, pre);
  }
  lds_barrier();
  const int n_ent = rp.v_end > rp.v_begin ? rp.v_end - rp.v_begin : 0;
  const int32_t* const idx_row = SEL || p.idx == nullptr ? nullptr : p.idx + rp.row * p.idx_row_stride;
  const int nt = rp.ntiles;
  const int n_tab = (nt + 3) * kTile;
  // An empty slot is fetched as another entry the row sees (its weight is 0 whatever it holds: K
  // is V, so what is not finite there is not finite in the entry's own product either): the
  // window's or the dense branch's first, or where the row has neither, the split's first.
  uint32_t any = rp.nw > 0 ? static_cast<uint32_t>(rp.win_first) : rp.nwd > 0 ? kSrcDense : kEmptyEntry;
  for (int e0 = 0; e0 < n_tab; e0 += NT) {
    const int e = e0 + tid;
    const int v = rp.v_begin + e;
    uint32_t code = kEmptyEntry;
    if (e < n_ent) {
      if (v < rp.nw) {
        int slot_w = rp.win_first + v;
        if (p.win_cap && slot_w >= p.win_cap) slot_w -= p.win_cap;
        code = static_cast<uint32_t>(slot_w);
      } else if (v < rp.nwd) {
        code = kSrcDense | static_cast<uint32_t>(v - rp.nw);
      } else {
        const int sp = v - rp.nwd;
        const int gi = pre_ok ? sidx[sp] : idx_row[sp];
        if (gi >= 0 && gi < rp.g_lim) code = kSrcMain | static_cast<uint32_t>(gi);
      }
    }
    const uint64_t bal = __ballot(code != kEmptyEntry);
    if (e < n_tab) {
      tab[e] = code != kEmptyEntry ? code : any;
      if ((lane & 31) == 0) masks[e / kTile] = static_cast<uint32_t>(lane ? bal >> 32 : bal);
    }
  }
  lds_barrier();
  int u0 = 0;  // leading tiles without an entry contribute nothing
  while (u0 < nt && masks[u0] == 0u) ++u0;
  if (any == kEmptyEntry && u0 < nt) {
    any = tab[u0 * kTile + __builtin_ctz(masks[u0])];
    for (int e = tid; e < n_tab; e += NT)
      if (tab[e] == kEmptyEntry) tab[e] = any;
    lds_barrier();
  }

  // ---- addresses -------------------------------------------------------------------------
  const int te = tid >> 3, tj = tid & 7;
  const int kx = g ^ lat_swz(e16);
  const uint32_t k_even = static_cast<uint32_t>((16 * eh + e16) * M::ROW + 16 * kx);
  const uint32_t k_odd = static_cast<uint32_t>((16 * eh + e16) * M::ROW + 16 * (kx ^ 4));
  const int vrow = 4 * g + (e16 >> 2);
  const uint32_t v_at = static_cast<uint32_t>(vrow * M::ROW + 16 * ((2 * wave + ((e16 >> 1) & 1)) ^ lat_swz(vrow)) +
                                              8 * (e16 & 1));
  const uint32_t st_at = static_cast<uint32_t>(
      FMT == kFmtFp8 ? te * M::ROW + 128 * (tj >> 2) + 16 * ((2 * (tj & 3)) ^ lat_swz(te))
                     : te * M::ROW + 16 * (tj ^ lat_swz(te)));
  const uint32_t rope_at = static_cast<uint32_t>(te * M::ROW + 1024 + 16 * (tj ^ lat_swz(te)));
  uint8_t* const pbuf = smem + M::PB;

  // the address of this thread's pieces of the entry with this code, and their loads
  // sums, not a choice among three: the compiler would keep the three in memory to index
  const uint64_t win_piece = reinterpret_cast<uint64_t>(rp.win_b) + 16u * tj;
  const uint64_t dense_piece = reinterpret_cast<uint64_t>(rp.dense_b) + 16u * tj;
  const uint64_t to_main = reinterpret_cast<uint64_t>(rp.main_b) - reinterpret_cast<uint64_t>(rp.dense_b);
  auto entry_at = [&](uint32_t code) __attribute__((always_inline)) -> gptr_t {
    uint64_t at = static_cast<uint64_t>(code & kIndexMask) * EB;
    at += code >= kSrcDense ? dense_piece : win_piece;
    at += code >= kSrcMain ? to_main : 0;
    return (gptr_t)at;
  };
  auto fetch_part = [&](gptr_t e, LatRaw<FMT>& r, int k) __attribute__((always_inline)) {
    if constexpr (FMT == kFmtFp8) {
      if (k < 4) r.v[k] = gload<u32x4>(e + 128 * k);
      if (k == 4) r.v[4] = gload<u32x4>(e + NOPE + 16);
      if (k == 5) r.s = gload<u32x4>(e - 16 * tj + NOPE);
    } else {
      if (k < 9) r.v[k] = gload<u32x4>(e + 128 * k);
    }
  };
  auto fetch_at = [&](gptr_t e, LatRaw<FMT>& r) __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < 9; ++k) fetch_part(e, r, k);
  };
  auto fetch = [&](int u, LatRaw<FMT>& r) __attribute__((always_inline)) { fetch_at(entry_at(tab[u * kTile + te]), r); };
  // part k (of 9) of a fetched tile into LDS: fp8 parts 2 q, 2 q + 1 are the halves of code
  // piece q (16 codes: two bf16 pieces), part 8 the rope slice
  auto store_part = [&](uint8_t* t, const LatRaw<FMT>& r, int k) __attribute__((always_inline)) {
    if constexpr (FMT == kFmtFp8) {
      if (k < 8) {
        const int q = k >> 1;
        const uint2 codes = k & 1 ? uint2{r.v[q].z, r.v[q].w} : uint2{r.v[q].x, r.v[q].y};
        *reinterpret_cast<uint4*>(t + ((k & 1 ? st_at ^ 16u : st_at) + 256 * q)) =
            dequant_fp8x8_bf16(codes, __uint_as_float(r.s[q]));
      } else {
        *reinterpret_cast<uint4*>(t + rope_at) = uint4{r.v[4].x, r.v[4].y, r.v[4].z, r.v[4].w};
      }
    } else {
      *reinterpret_cast<uint4*>(t + st_at + 128 * k) = uint4{r.v[k].x, r.v[k].y, r.v[k].z, r.v[k].w};
    }
  };
  auto store = [&](uint8_t* t, const LatRaw<FMT>& r) __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < 9; ++k) store_part(t, r, k);
  };
  auto k_frag = [&](const uint8_t* t, int st) __attribute__((always_inline)) -> v8bf {
    return __builtin_bit_cast(v8bf, *reinterpret_cast<const v4i*>(t + (st & 1 ? k_odd : k_even) + 128 * (st >> 1)));
  };

  float m4[4];          // the exponent's reference of this lane's head in each head group
  float m_own[2];       // ... of the two this wave's scores belong to
  float l_own[2];       // this lane's share of their row sums
  v4f acc[NI][4];
  v8bf qf[KS][2];       // the B operand of S^T: heads 32 hh + 16 b + e16, channels 32 st + 8 g .. + 7
  v4f s_acc[2];
  LatRaw<FMT> raw[2];   // two tiles of loads in flight

  // the lane's scaled, masked scores of tile u from s_acc
  auto scores = [&](int u, float (&v)[2][4]) __attribute__((always_inline)) {
    const uint32_t vmask = masks[u];
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) v[b][r] = s_acc[b][r] * p.scale_log2;
    // branch-free: a branch among the matrix instructions costs more than the selects
    const uint32_t bits = vmask >> (16 * eh + 4 * g);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const bool in = ((bits >> r) & 1u) != 0u;
      v[0][r] = in ? v[0][r] : -__builtin_huge_valf();
      v[1][r] = in ? v[1][r] : -__builtin_huge_valf();
    }
  };
  auto max4 = [](const float (&v)[4]) __attribute__((always_inline)) {
    return fmaxf(fmaxf(v[0], v[1]), fmaxf(v[2], v[3]));
  };
  // over the four lanes of a head
  auto head_max = [](float x) __attribute__((always_inline)) {
    x = fmaxf(x, __shfl_xor(x, 16, 64));
    return fmaxf(x, __shfl_xor(x, 32, 64));
  };
  // the heads' maxima over both entry halves into m4 / m_own (one barrier)
  auto agree_max = [&](float t0, float t1) __attribute__((always_inline)) {
    t0 = head_max(t0);
    t1 = head_max(t1);
    if (g == 0) {
      pmax[eh * 64 + 32 * hh + e16] = t0;
      pmax[eh * 64 + 32 * hh + 16 + e16] = t1;
    }
    lds_barrier();
#pragma unroll
    for (int hg = 0; hg < 4; ++hg) m4[hg] = fmaxf(pmax[16 * hg + e16], pmax[64 + 16 * hg + e16]);
    m_own[0] = fmaxf(pmax[32 * hh + e16], pmax[64 + 32 * hh + e16]);
    m_own[1] = fmaxf(pmax[32 * hh + 16 + e16], pmax[64 + 32 * hh + 16 + e16]);
  };
  // P^T of head group 2 hh + b: the weights, and their share of the row sum
  float m_seen[2];
  auto weights = [&](int b, const float (&v)[4]) __attribute__((always_inline)) -> uint2 {
    // v_exp_f32 directly: results below 2^-126 may flush to 0
    const float p0 = __builtin_amdgcn_exp2f(v[0] - m_own[b]);
    const float p1 = __builtin_amdgcn_exp2f(v[1] - m_own[b]);
    const float p2 = __builtin_amdgcn_exp2f(v[2] - m_own[b]);
    const float p3 = __builtin_amdgcn_exp2f(v[3] - m_own[b]);
    l_own[b] = l_own[b] + ((p0 + p1) + (p2 + p3));
    return uint2{pack_bf16x2(p0, p1), pack_bf16x2(p2, p3)};
  };
  // this lane's K-slots of tile u: the entries of eh = 0 first, then of eh = 1
  auto put_p = [&](int u, int b, uint2 w) __attribute__((always_inline)) {
    *reinterpret_cast<uint2*>(pbuf + (u & 1) * 4096 + 2048 * hh + 1024 * b + 16 * lane + 8 * eh) = w;
  };

  // ---- the pass ---------------------------------------------------------------------------
  // m4, l_own, acc hold the split after it, unless *redo is set: then again with m4 / m_own given
  auto pass = [&](bool given) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int hg = 0; hg < 4; ++hg) acc[i][hg] = v4f{};
    l_own[0] = l_own[1] = 0.0f;
    if (given) {
      fetch(u0, raw[0]);
      fetch(u0 + 1, raw[1]);
    }
    store(smem, raw[0]);
    // a split of one tile needs neither the second nor what follows it (the splits of a short list
    // over many workgroups: 640 entries of 2 rows in 32 splits 20.4 -> 19.9 us the launch and its merge)
    if (nt - u0 > 1) {  // uniform
      store(smem + M::TILE, raw[1]);
      const int odd = (nt - 1 - u0) & 1;  // set 1 is stored first then
      fetch(u0 + 2 + odd, raw[0]);
      fetch(u0 + 3 - odd, raw[1]);
    }
    lds_barrier();
    {
      const uint8_t* kt = smem;
      s_acc[0] = s_acc[1] = v4f{};
#pragma unroll
      for (int st = 0; st < KS; ++st) {
        const v8bf kf = k_frag(kt, st);
        s_acc[0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[st][0], s_acc[0], 0, 0, 0);
        s_acc[1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[st][1], s_acc[1], 0, 0, 0);
      }
      float v[2][4];
      scores(u0, v);
      if (!given) {
        agree_max(max4(v[0]), max4(v[1]));
        // a head without a finite score in its first tile (or with NaN): from the true maxima
#pragma unroll
        for (int hg = 0; hg < 4; ++hg)
          if (!(m4[hg] > -__builtin_huge_valf())) *redo = 1;
      }
      // the raw scores' maxima, for the check at the end (-inf where masked: the first tile's)
      m_seen[0] = m_seen[1] = -__builtin_huge_valf();
      put_p(u0, 0, weights(0, v[0]));
      put_p(u0, 1, weights(1, v[1]));
    }
    auto read_p = [&](int u, v8bf (&pf)[4]) __attribute__((always_inline)) {
#pragma unroll
      for (int hg = 0; hg < 4; ++hg)
        pf[hg] = __builtin_bit_cast(v8bf, *reinterpret_cast<const v4i*>(pbuf + (u & 1) * 4096 + 1024 * hg + 16 * lane));
    };
    auto read_v = [&](const uint8_t* vt, int i, v4s (&va)[2]) __attribute__((always_inline)) {
      const uint8_t* tp = vt + v_at + 128 * i;
      va[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(lds_v4s(tp));
      va[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(lds_v4s(tp + 16 * M::ROW));
    };
    // tiles u, u+1 and the one u+2 goes to, by turns
    uint32_t at_v = 0, at_k = M::TILE, at_w = 2 * M::TILE;
    // One wave per SIMD issues in order, so the iteration is laid out by hand: every LDS operand
    // is requested several matrix instructions before its use (K six steps, V^T four blocks),
    // the softmax, the stores and the loads are spread one slice after each matrix
    // instruction, whose 16 cycles they fill, and the last two blocks of PV(u-1), whose operands
    // are in registers by then, follow the barrier and cover the first reads of K.
    constexpr int AH = 6, VH = 4, LATE = 2;
    v4s va[VH + 1][2];
    v8bf pf[4];
    auto pv_block = [&](int i, auto&& fill) __attribute__((always_inline)) {
      const v4s a = va[i % (VH + 1)][0], b = va[i % (VH + 1)][1];
      const v8bf vf = __builtin_bit_cast(v8bf, v8s{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]});
#pragma unroll
      for (int hg = 0; hg < 4; ++hg) {
        acc[i][hg] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, pf[hg], acc[i][hg], 0, 0, 0);
        fill(hg);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
#pragma unroll
    for (int i = 0; i <= VH; ++i) va[i][0] = va[i][1] = v4s{0, 0, 0, 0};
#pragma unroll
    for (int hg = 0; hg < 4; ++hg) pf[hg] = __builtin_bit_cast(v8bf, v4i{0, 0, 0, 0});
    lds_barrier();  // P(u0) complete
    uint32_t vmask = masks[u0 + 1];  // of the tile whose scores come next
    auto step = [&](int u, LatRaw<FMT>& r) __attribute__((always_inline)) {
      // the barrier before: P(u) and tile u+1 complete; tile u-1 is read no more
      const uint8_t* vt = smem + at_v;
      const uint8_t* kt = smem + at_k;
      uint8_t* const wt = smem + at_w;
      v8bf kf[AH];
#pragma unroll
      for (int i = 0; i < AH; ++i) kf[i] = k_frag(kt, i);
      const uint32_t code = tab[(u + 4) * kTile + te];
      __builtin_amdgcn_sched_barrier(0);
      // masked entries start from kMasked instead of 0, so that no score needs a test
      const uint32_t bits = vmask >> (16 * eh + 4 * g);
      v4f init;
#pragma unroll
      for (int i = NI - LATE; i < NI; ++i)
        pv_block(i, [&](int hg) __attribute__((always_inline)) {
          const int k = 4 * (i - (NI - LATE)) + hg;
          if (k < 4) init[k] = ((bits >> k) & 1u) != 0u ? 0.0f : kMasked;
        });
      uint64_t next = 0;
#pragma unroll
      for (int st = 0; st < KS; ++st) {
        const v8bf cur = kf[st % AH];
        s_acc[0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(cur, qf[st][0], st == 0 ? init : s_acc[0], 0, 0, 0);
        if (st + AH < KS) kf[st % AH] = k_frag(kt, st + AH);
        __builtin_amdgcn_sched_barrier(0);
        s_acc[1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(cur, qf[st][1], st == 0 ? init : s_acc[1], 0, 0, 0);
        if (st == 1) vmask = masks[u + 2];
        if (st == 4) next = static_cast<uint64_t>(code & kIndexMask) * EB;
        if (st == 5) next += code >= kSrcDense ? dense_piece : win_piece;
        if (st == 6) next += code >= kSrcMain ? to_main : 0;
        if (st >= 8 && st < 12) {
          const int hg = st - 8;
          pf[hg] = __builtin_bit_cast(v8bf, *reinterpret_cast<const v4i*>(pbuf + (u & 1) * 4096 + 1024 * hg + 16 * lane));
        }
        if (st >= KS - VH - 2 && st < KS - 2) read_v(vt, st - (KS - VH - 2), va[st - (KS - VH - 2)]);
        if (st >= KS - 2) store_part(wt, r, 7 + st - (KS - 2));
        __builtin_amdgcn_sched_barrier(0);
      }
      const gptr_t from = (gptr_t)next;
      float v[2][4], pr[2][4];
      // slice k of what fills the matrix instructions of PV
      auto slice = [&](int k) __attribute__((always_inline)) {
        if (k >= 2 && k < 10) {
          const int b = (k - 2) >> 2, j = (k - 2) & 3;
          v[b][j] = s_acc[b][j];
          pr[b][j] = __builtin_fmaf(v[b][j], p.scale_log2, -m_own[b]);
        } else if (k >= 10 && k < 18) {  // v_exp_f32 directly: results below 2^-126 may flush to 0
          const int b = (k - 10) >> 2, j = (k - 10) & 3;
          pr[b][j] = __builtin_amdgcn_exp2f(pr[b][j]);
        } else if (k == 18 || k == 19) {
          const int b = k - 18;
          put_p(u + 1, b, uint2{pack_bf16x2(pr[b][0], pr[b][1]), pack_bf16x2(pr[b][2], pr[b][3])});
        } else if (k >= 20 && k < 22) {
          const int b = k - 20;
          l_own[b] = l_own[b] + ((pr[b][0] + pr[b][1]) + (pr[b][2] + pr[b][3]));
        } else if (k >= 22 && k < 24) {
          const int b = k - 22;
          m_seen[b] = fmaxf(fmaxf(m_seen[b], v[b][0]), fmaxf(v[b][1], fmaxf(v[b][2], v[b][3])));
        }
      };
#pragma unroll
      for (int i = 0; i < NI - LATE; ++i)
        pv_block(i, [&](int hg) __attribute__((always_inline)) {
          if (hg == 0 && i + VH < NI) read_v(vt, i + VH, va[(i + VH) % (VH + 1)]);
          slice(4 * i + hg);
          if (hg == 1) store_part(wt, r, i);
          // a piece is requested again, for tile u + 4, once all of it is stored
          if constexpr (FMT == kFmtFp8) {
            if (hg == 3 && (i & 1)) fetch_part(from, r, i >> 1);
            if (hg >= 2 && i == 6) fetch_part(from, r, hg == 2 ? 3 : 5);
            if (hg == 3 && i == 0) fetch_part(from, r, 4);
          } else {
            if (hg == 3) fetch_part(from, r, i);
            if (hg == 2 && i >= NI - 2 * LATE) fetch_part(from, r, i + LATE);
          }
        });
      lds_barrier();
      const uint32_t done = at_v;
      at_v = at_k;
      at_k = at_w;
      at_w = done;
    };
    // an odd number of steps takes one first: the loop is two steps long (two sets of loads in
    // flight) with a single exit, or every accumulator would be copied between its ends
    int u = u0;
    if ((nt - 1 - u0) & 1) {
      step(u++, raw[1]);
    }
#pragma unroll 1
    for (; u + 1 < nt; u += 2) {
      step(u, raw[0]);
      step(u + 1, raw[1]);
    }
    {  // the rest of the last but one, and the last tile
      const uint8_t* vt = smem + at_v;
#pragma unroll
      for (int i = NI - LATE; i < NI; ++i) pv_block(i, [](int) {});
      read_p(nt - 1, pf);
#pragma unroll
      for (int i = 0; i < VH; ++i) read_v(vt, i, va[i]);
#pragma unroll
      for (int i = 0; i < NI; ++i)
        pv_block(i, [&](int hg) __attribute__((always_inline)) {
          if (hg == 0 && i + VH < NI) read_v(vt, i + VH, va[(i + VH) % (VH + 1)]);
        });
    }
    if (!given) {
      const float rise = fmaxf(m_seen[0] * p.scale_log2 - m_own[0], m_seen[1] * p.scale_log2 - m_own[1]);
      if (rise > kRoomNear) *high = 1;
      if (rise > kRoomAbove) *redo = 1;
    }
  };

  // the true maxima of every head over the split (m4 / m_own): scores only
  auto max_pass = [&]() __attribute__((always_inline)) {
    float t0 = -__builtin_huge_valf(), t1 = t0;
#pragma unroll 1
    for (int u = u0; u < nt; ++u) {
      fetch(u, raw[0]);
      store(smem, raw[0]);
      lds_barrier();
      s_acc[0] = s_acc[1] = v4f{};
#pragma unroll
      for (int st = 0; st < KS; ++st) {
        const v8bf kf = k_frag(smem, st);
        s_acc[0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[st][0], s_acc[0], 0, 0, 0);
        s_acc[1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[st][1], s_acc[1], 0, 0, 0);
      }
      float v[2][4];
      scores(u, v);
      t0 = fmaxf(t0, max4(v[0]));
      t1 = fmaxf(t1, max4(v[1]));
      lds_barrier();
    }
    agree_max(t0, t1);
    // no finite score at all: the reference 0 makes every weight 0
#pragma unroll
    for (int hg = 0; hg < 4; ++hg) m4[hg] = m4[hg] == -__builtin_huge_valf() ? 0.0f : m4[hg];
#pragma unroll
    for (int b = 0; b < 2; ++b) m_own[b] = m_own[b] == -__builtin_huge_valf() ? 0.0f : m_own[b];
    lds_barrier();
  };

  float l4[4];  // row sums
  int e4[4];    // O^T is at 2^e4 times the scale of (m4, l4)
#pragma unroll
  for (int hg = 0; hg < 4; ++hg) {
    e4[hg] = 0;
    m4[hg] = -__builtin_huge_valf();
    l4[hg] = 0.0f;
#pragma unroll
    for (int i = 0; i < NI; ++i) acc[i][hg] = v4f{};
  }
  if (u0 < nt) {
    fetch(u0, raw[0]);
    fetch(u0 + 1, raw[1]);
    constexpr int QPITCH = 2 * D + 16;  // the pad spreads 16 heads' pieces over the banks
    static_assert(64 * QPITCH <= M::PB, "q in the tiles' place");
#pragma unroll
    for (int k = 0; k < QP; ++k) {
      const int at = tid + NT * k;
      const int h = at / QROW;
      *reinterpret_cast<u32x4*>(smem + h * QPITCH + 16 * (at - h * QROW)) = at < q_pieces ? qraw[k] : u32x4{0u, 0u, 0u, 0u};
    }
    lds_barrier();
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int st = 0; st < KS; ++st)
        qf[st][b] = __builtin_bit_cast(v8bf, *reinterpret_cast<const v4i*>(smem + (32 * hh + 16 * b + e16) * QPITCH + 64 * st + 16 * g));
    lds_barrier();
    if constexpr (RST > 0) {
      if (p.rope_cos != nullptr) {
#pragma unroll
        for (int r = 0; r < RST; ++r) {
          const uint32_t cw[2] = {qrc[r].x, qrc[r].y}, sw[2] = {qrs[r].x, qrs[r].y};
#pragma unroll
          for (int b = 0; b < 2; ++b) {
            v4i v = __builtin_bit_cast(v4i, qf[KS - RST + r][b]);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
              const uint32_t cp = cw[k >> 1], sp = sw[k >> 1];
              v[k] = static_cast<int>(rope_pair_bf16(static_cast<uint32_t>(v[k]),
                                                     bf16_to_f32(static_cast<uint16_t>((k & 1) ? cp >> 16 : cp & 0xffffu)),
                                                     bf16_to_f32(static_cast<uint16_t>((k & 1) ? sp >> 16 : sp & 0xffffu))));
            }
            qf[KS - RST + r][b] = __builtin_bit_cast(v8bf, v);
          }
        }
      }
    }
    // the first 24 query fragments live in accumulation registers beside O^T, which the matrix
    // instructions read directly; left to itself the compiler spills
#pragma unroll
    for (int st = 0; st < KS - 6; ++st)
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        v4i x = __builtin_bit_cast(v4i, qf[st][b]);
        asm volatile("" : "+a"(x));
        qf[st][b] = __builtin_bit_cast(v8bf, x);
      }
    for (bool given = false;; given = true) {
      pass(given);
      // each head's row sum: its four lanes, then the two entry halves
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        l_own[b] = l_own[b] + __shfl_xor(l_own[b], 16, 64);
        l_own[b] = l_own[b] + __shfl_xor(l_own[b], 32, 64);
        if (g == 0) lsum[eh * 64 + 32 * hh + 16 * b + e16] = l_own[b];
      }
      lds_barrier();
#pragma unroll
      for (int hg = 0; hg < 4; ++hg) l4[hg] = lsum[16 * hg + e16] + lsum[64 + 16 * hg + e16];
      if (__builtin_expect(!given && *high != 0, 0)) {  // uniform: set before the barrier above
        // O^T through the tiles' place, half of it at a time, each lane its own: a few stores
        // and a short loop.  Looked at in registers it took 3.6 KB of code, and a decode step
        // (whose kernel runs from a cold instruction cache) 1 us whether or not it was entered.
        float any_bad = 0.0f;  // NaN if an accumulator is not finite
        v4f* const slot = reinterpret_cast<v4f*>(smem) + tid;
        static_assert(2 * NI * NT * 16 <= M::PB, "half of O^T in the tiles' place");
#pragma unroll
        for (int half = 0; half < 2; ++half) {
#pragma unroll
          for (int k = 0; k < 2 * NI; ++k) slot[k * NT] = acc[k >> 1][2 * half + (k & 1)];
#pragma unroll 1
          for (int k = 0; k < 2 * NI; ++k) {
            const v4f x = slot[k * NT];
#pragma unroll
            for (int r = 0; r < 4; ++r) any_bad = __builtin_fmaf(x[r], 0.0f, any_bad);
          }
        }
        if (any_bad != 0.0f) *redo = 1;
        lds_barrier();
      }
      if (given || *redo == 0) break;  // uniform: set before the barrier above
      max_pass();
    }
    // (m, l) with l in [1, 2): the reference is not the maximum, so l may be far from 1
#pragma unroll
    for (int hg = 0; hg < 4; ++hg) {
      e4[hg] = l4[hg] > 0.0f && l4[hg] < __builtin_huge_valf() ? __builtin_amdgcn_frexp_expf(l4[hg]) - 1 : 0;
      l4[hg] = __builtin_amdgcn_ldexpf(l4[hg], -e4[hg]);
      m4[hg] = l4[hg] == 0.0f ? -__builtin_huge_valf() : m4[hg] + static_cast<float>(e4[hg]);
    }
  }

  // ---- the result -------------------------------------------------------------------------
  // acc[i][hg][r]: head 16 hg + e16, channel 16 (wave + 4 i) + 4 g + r
  const int h0 = rp.hgrp * 64;
  if (p.write_final) {
    // through LDS, so that the 64 heads' rows (one contiguous run) leave in whole lines
    constexpr int OPITCH = 2 * D + 16;
    const int64_t s_idx = rp.row % p.S;
#pragma unroll
    for (int hg = 0; hg < 4; ++hg) {
      const int head = h0 + 16 * hg + e16;
      if (head < p.H) {
        float m_fin = m4[hg], l_fin = l4[hg], o_scale;
        if (p.sinks) {
          const float sk = p.sinks[head] * kLog2e;
          const float mm = fmaxf(m_fin, sk);
          const float a = m_fin == -__builtin_huge_valf() ? 0.0f : exp2f(m_fin - mm);
          l_fin = l_fin * a + exp2f(sk - mm);
          m_fin = mm;
          o_scale = a / l_fin;
        } else {
          o_scale = 1.0f / l_fin;
        }
        o_scale = __builtin_amdgcn_ldexpf(o_scale, -e4[hg]);
        uint8_t* orow = smem + (16 * hg + e16) * OPITCH + 32 * wave + 8 * g;
#pragma unroll
        for (int i = 0; i < NI; ++i) {
          uint32_t w0 = pack_bf16x2(acc[i][hg][0] * o_scale, acc[i][hg][1] * o_scale);
          uint32_t w1 = pack_bf16x2(acc[i][hg][2] * o_scale, acc[i][hg][3] * o_scale);
          if constexpr (NOPE < D) {
            // the inverse rotation of the bf16 output (owlet1/attention.py:226): block 32 + wave
            if (i == NI - 1 && p.rope_cos) {
              const int64_t ci = rp.row * ((D - NOPE) / 2) + 8 * wave + 2 * g;
              const uint32_t cp = *reinterpret_cast<const uint32_t*>(p.rope_cos + ci);
              const uint32_t sp = *reinterpret_cast<const uint32_t*>(p.rope_sin + ci);
              w0 = rope_pair_bf16(w0, bf16_to_f32(static_cast<uint16_t>(cp & 0xffffu)),
                                  -bf16_to_f32(static_cast<uint16_t>(sp & 0xffffu)));
              w1 = rope_pair_bf16(w1, bf16_to_f32(static_cast<uint16_t>(cp >> 16)),
                                  -bf16_to_f32(static_cast<uint16_t>(sp >> 16)));
            }
          }
          *reinterpret_cast<uint2*>(orow + 128 * i) = uint2{w0, w1};
        }
        if (wave == hg && g == 0) p.lse[(rp.b * p.H + head) * p.S + s_idx] = (m_fin + __log2f(l_fin)) * kLn2;
      }
    }
    lds_barrier();
    u32x4* ob = reinterpret_cast<u32x4*>(p.out + (rp.row * p.H + h0) * D);
#pragma unroll
    for (int k = 0; k < QP; ++k) {
      const int at = tid + NT * k;
      const int h = at / QROW;
      if (at < q_pieces) ob[at] = *reinterpret_cast<const u32x4*>(smem + h * OPITCH + 16 * (at - h * QROW));
    }
  } else {
    // the split's own normalized output in bf16 (zeros for a split that saw no entry), in
    // 16-channel groups with the heads innermost: a store instruction covers 512 contiguous
    // bytes (through LDS, 2 KB a group, it took 2.4 K cycles longer)
    uint16_t* pbase = p.part_o + (rp.row * p.split_stride + rp.split) * p.H * static_cast<int64_t>(D);
    float* ml = p.part_ml + (rp.row * p.split_stride + rp.split) * p.H * 2;
#pragma unroll
    for (int hg = 0; hg < 4; ++hg) {
      const int head = h0 + 16 * hg + e16;
      if (head < p.H) {
        const float inv_l = l4[hg] > 0.0f ? __builtin_amdgcn_ldexpf(1.0f / l4[hg], -e4[hg]) : 0.0f;
#pragma unroll
        for (int i = 0; i < NI; ++i)
          *reinterpret_cast<uint2*>(pbase + static_cast<uint32_t>((wave + 4 * i) * p.H * 16 + head * 16 + 4 * g)) =
              uint2{pack_bf16x2(acc[i][hg][0] * inv_l, acc[i][hg][1] * inv_l),
                    pack_bf16x2(acc[i][hg][2] * inv_l, acc[i][hg][3] * inv_l)};
        if (wave == hg && g == 0) *reinterpret_cast<float2*>(ml + 2 * head) = float2{m4[hg], l4[hg]};
      }
    }
  }
  if (mrec != nullptr) merge_in_launch<D, NOPE, NT>(p, rp.row, h0, rp.split, mrec, tid);
}
