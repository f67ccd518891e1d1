// 32-row groups for problems of few query blocks, fp16 and bf16, head dim 64
// and 128.  Shared building blocks: fa2_common.h, fa2_d128.h.

#include "fa2_d128.h"

namespace fl {

namespace {

// ---------------------------------------------------------------------------
// One work-group of NW waves owns 32 query rows; wave w walks key tiles w,
// w + NW, ... through a K and a V slot of its own, so no barrier orders the
// walk: the waves only meet to publish Q and to merge.  K(i+1) is fetched by
// DMA as soon as the operands of K(i) are read, V(i+1) after those of V(i).
// Every wave issues the same 8 fetches per tile (past its range they land as
// zeros with no traffic), so "K(i) has landed" and "V(i) has landed" are both
// vmcnt <= 8.  The partial results merge through LDS at their largest
// stabiliser, each wave taking a share of the head dims of every row.
//
// What it is for: problems of few 32-row blocks, where the other schedules
// leave CUs idle or walk many tiles one after another.  A wave's walk is a
// chain of load latencies and of two dependent products per tile; four (or
// eight) independent chains per block shorten it to a quarter (or an eighth)
// of the tiles, where the 64-row split halves it.  NW = 4 keeps 64 KiB of
// tiles, two groups per CU; NW = 8, one group per CU, serves long walks.
// Against the configurations launched before it (fp16, us per call in a graph,
// new inputs each call): B1 H1 N128 4.66 -> 4.04, B2 H8 N256 6.8 -> 4.6, B2 H8
// N512 7.1 -> 5.9, B1 H8 N1024 9.2 -> 7.5 (bf16 9.4 -> 7.6), B1 H2 N4096 causal
// 22.9 -> 16.2, B1 H1 N8192 44.3 -> 31.9; head dim 128: B2 H8 N512 12.6 -> 7.45,
// B1 H2 N4096 54.3 -> 28.5.  Two tiles in flight per wave (128 KiB, one group
// per CU) measured 0-10% slower than one.
template <int D, class T, bool CAUSAL>
struct TileRows;

template <class T, bool CAUSAL>
struct TileRows<128, T, CAUSAL> : Rows128<CAUSAL, T> {
  using Base = Rows128<CAUSAL, T>;
  using V8 = typename Base::V8;
  static constexpr int kKeys = kBc2;
  struct Scores {
    float16_t s;
  };
  struct Probs {
    V8 p[2];
  };
  __device__ __forceinline__ void scores(const uint8_t* kt, Scores& s) const {
    this->gemm1(kt, s.s);
  }
  __device__ __forceinline__ void softmax(int t, int i, Scores& s, Probs& p) {
    this->mask(t, s.s);
    if (i == 0) this->first_tile(s.s);
    this->softmax_checked(s.s, p.p);
  }
  __device__ __forceinline__ void output(const uint8_t* vt, const Probs& p) {
    this->gemm2(vt, p.p);
  }
  __device__ __forceinline__ float stabiliser() const { return this->mc; }
};

template <class T, bool CAUSAL>
struct TileRows<64, T, CAUSAL> : Rows<CAUSAL, true, T> {
  using Base = Rows<CAUSAL, true, T>;
  using V8 = typename Base::V8;
  static constexpr int kKeys = kBc;
  struct Scores {
    float16_t s[2];
  };
  struct Probs {
    V8 p[2][2];
  };
  __device__ __forceinline__ void place(int lane, int qw, int seq, int kv_lim, int coff, float cr) {
    Base::place(lane, qw, seq, kv_lim, coff, cr);
    this->reset();
  }
  __device__ __forceinline__ void scores(const uint8_t* kt, Scores& s) const {
    V8 ka[2][4];
    this->read_k(kt, ka);
    this->gemm1(ka, s.s);
  }
  // The stabiliser is the exact row max over the first two tiles, so the
  // largest p of a walk of up to 512 keys is 1 and rounds to itself: a row's
  // error is mostly that of its few largest p (B2 H8 N512 against 64 bits
  // 2.78e-4 with the first tile's max, 2.66e-4 so; 0.3 us a call).
  __device__ __forceinline__ void softmax(int t, int i, Scores& s, Probs& p) {
    this->mask(t, s.s);
    if (i == 0)
      this->first_tile(s.s);
    else if (i == 1)
      this->raise_m(s.s);
    this->softmax_checked(s.s, p.p);
  }
  __device__ __forceinline__ void output(const uint8_t* vt, const Probs& p) {
    V8 va[2][4];
    this->read_v(vt, va);
    this->gemm2(va, p.p);
  }
  __device__ __forceinline__ float stabiliser() const { return this->m * this->cr; }
};

template <int D, int NW, bool CAUSAL, class T, bool KVSPLIT>
__global__ void __launch_bounds__(64 * NW, 2)
fa2_fwd_rows32_kernel(const T* Q, const T* __restrict__ K, const T* __restrict__ V, T* O,
                      const Geom geom, int nqb, float cq, float cr) {
  using RowsT = TileRows<D, T, CAUSAL>;
  using V8 = typename RowsT::V8;
  constexpr int kRowB = 2 * D;
  constexpr int kKeys = RowsT::kKeys;
  constexpr int kAcc = D / 2;  // O accumulators per lane
  static_assert(NW == 4 || NW == 8, "Q parts and merge shares");
  static_assert(kKeys * kRowB == kTileBytes, "tile size");
  static_assert(kAcc * 256 <= 2 * kTileBytes, "a wave's O fits its first slots");
  __shared__ __attribute__((aligned(16))) uint8_t buf[NW][2][kTileBytes];
  __shared__ __attribute__((aligned(16))) uint8_t qbuf[32 * kRowB];
  __shared__ float2 mlbuf[NW][64];

  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int bh, qb, chunk = 0;
  if constexpr (KVSPLIT)
    chunk_coords(nqb, geom.nsplit, geom.xcds, bh, chunk, qb);
  else
    wg_coords<false, 1>(nqb, geom.xcds, geom.cus_per_xcd, bh, qb);
  const HeadPtrs<T> hp = head_ptrs<T, kRowB>(geom, bh, Q, K, V, O);
  const int seq = geom.seq_q, q0 = 32 * qb;
  // The group's key tiles [tbeg, tiles), through its last row's diagonal and
  // its chunk's end; this wave takes tbeg + w + NW i, i < n (none in a chunk
  // past the diagonal).
  int tiles = max(1, (geom.seq_k + kKeys - 1) / kKeys), tbeg = 0;
  if constexpr (KVSPLIT) {
    const int per = (tiles + geom.nsplit - 1) / geom.nsplit;
    tbeg = chunk * per;
    tiles = min(tiles, tbeg + per);
  }
  if (CAUSAL) {
    const int last_key = min(q0 + 32, seq) - 1 + geom.coff;
    tiles = min(tiles, last_key < 0 ? 1 : last_key / kKeys + 1);
  }
  const int mine0 = tbeg + w;  // this wave's first tile
  const int n = tiles > mine0 ? (tiles - mine0 + NW - 1) / NW : 0;

  const FetchOff<8> fk = D == 64 ? fetch_offsets<8, false>(0, lane, 2 * geom.k_sr)
                                 : fetch_offsets128<8, false>(0, lane, 2 * geom.k_sr);
  const FetchOff<8> fv = D == 64 ? fetch_offsets<8, true>(0, lane, 2 * geom.v_sr)
                                 : fetch_offsets128<8, true>(0, lane, 2 * geom.v_sr);
  i32x4_t rk, rv;
  kv_rsrc_rows<T, kRowB>(geom, bh, K, V, tiles * kKeys, rk, rv);
  auto fetch_k = [&](int i) __attribute__((always_inline)) {
    fetch_tile_z<8>(rk, buf[w][0], mine0 + NW * i, tiles, 0, fk);
  };
  auto fetch_v = [&](int i) __attribute__((always_inline)) {
    fetch_tile_z<8>(rv, buf[w][1], mine0 + NW * i, tiles, 0, fv);
  };
  // A part of the block's Q first (its wait leaves the tiles in flight).
  if constexpr (D == 64)
    fetch_q_block<4>(hp.q, geom.q_sr, q0, seq, qbuf, lane, NW == 4 ? w : w & 3);
  else
    fetch_q_block128<NW>(hp.q, geom.q_sr, q0, seq, qbuf, lane, w);
  fetch_k(0);
  fetch_v(0);
  RowsT rows;
  rows.place(lane, q0, seq, min(geom.seq_k, tiles * kKeys), geom.coff, cr);
  sync_ring_ahead<16, 0>();  // Q
  rows.set_q_lds(qbuf, cq);
  for (int i = 0; i < n; ++i) {
    typename RowsT::Scores s;
    typename RowsT::Probs p;
    asm volatile("s_waitcnt vmcnt(8)" : : : "memory");  // K(i)
    rows.scores(buf[w][0], s);
    asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");  // its operands are in registers
    fetch_k(i + 1);
    rows.softmax(mine0 + NW * i, i, s, p);
    asm volatile("s_waitcnt vmcnt(8)" : : : "memory");  // V(i)
    rows.output(buf[w][1], p);
    asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
    fetch_v(i + 1);
  }
  // Nothing may still write this wave's slots: its O goes there.
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" : : : "memory");
  float4* const mine = reinterpret_cast<float4*>(buf[w][0]);
#pragma unroll
  for (int c = 0; c < kAcc / 4; ++c) {
    const float16_t& x = rows.o[c >> 2];
    const int r = 4 * (c & 3);
    mine[c * 64 + lane] = make_float4(x[r], x[r + 1], x[r + 2], x[r + 3]);
  }
  mlbuf[w][lane] = make_float2(rows.stabiliser(), rows.l);
  __syncthreads();
  // A range with no visible key (l = 0 across the lane pair) is skipped.
  float mm = ninf(), lt = 0.0f, a[NW];
  float2 ml[NW];
  bool has[NW];
#pragma unroll
  for (int j = 0; j < NW; ++j) {
    ml[j] = mlbuf[j][lane];
    has[j] = pair_sum(ml[j].y) > 0.0f;
    if (has[j]) mm = fmaxf(mm, ml[j].x);
  }
#pragma unroll
  for (int j = 0; j < NW; ++j) {
    a[j] = has[j] ? __builtin_amdgcn_exp2f(ml[j].x - mm) : 0.0f;
    lt += a[j] * ml[j].y;
  }
  const float l_tot = pair_sum(lt);
  const float inv = l_tot > 0.0f ? 1.0f / l_tot : 0.0f;
  const bool mine_row = rows.my_q < seq;
  constexpr int kPart = D == 64 ? kPartStride : kPartStride128;
  float* const prow = KVSPLIT ? geom.part + ((long long)(chunk * geom.batch_heads + bh) * seq +
                                             rows.my_q) * kPart
                              : nullptr;
  for (int c = w; c < D / 16; c += NW) {
    // 8-column piece c of the row: accumulators 8 (c & 1) .. + 7 of block c / 2
    float acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int j = 0; j < NW; ++j) {
      const float4* const pj = reinterpret_cast<const float4*>(buf[j][0]);
      const float4 x0 = pj[(2 * c) * 64 + lane], x1 = pj[(2 * c + 1) * 64 + lane];
      acc[0] += a[j] * x0.x;
      acc[1] += a[j] * x0.y;
      acc[2] += a[j] * x0.z;
      acc[3] += a[j] * x0.w;
      acc[4] += a[j] * x1.x;
      acc[5] += a[j] * x1.y;
      acc[6] += a[j] * x1.z;
      acc[7] += a[j] * x1.w;
    }
    const int col = 32 * (c >> 1) + 16 * (c & 1) + 8 * rows.g;
    if (!mine_row) continue;
    if constexpr (KVSPLIT) {
      *reinterpret_cast<float4*>(prow + col) = make_float4(acc[0], acc[1], acc[2], acc[3]);
      *reinterpret_cast<float4*>(prow + col + 4) = make_float4(acc[4], acc[5], acc[6], acc[7]);
    } else {
      V8 out;
#pragma unroll
      for (int e = 0; e < 8; ++e) out[e] = (T)(acc[e] * inv);
      *reinterpret_cast<V8*>(hp.o + (long long)rows.my_q * geom.o_sr + col) = out;
    }
  }
  if (w != 0 || rows.g != 0 || !mine_row) return;
  if constexpr (KVSPLIT) {
    prow[D] = l_tot > 0.0f ? mm : ninf();
    prow[D + 1] = l_tot;
  } else if (hp.lse != nullptr) {
    hp.lse[rows.my_q] =
        l_tot > 0.0f ? 0.693147180559945309f * (mm + __builtin_amdgcn_logf(l_tot)) : ninf();
  }
}

// Eight waves for blocks of at least 32 tiles at head dim 64, where they fit
// one round (B1 H1 N2048 9.2 against 9.7 us with four, N4096 13.5 against
// 15.1; N1024 equal, shorter ones up to 10% slower; at head dim 128 0-8%
// slower but for a tie at B1 H2 N2048).
template <int D, class T, bool KVSPLIT>
hipError_t launch_rows32_t(const FwdArgs& a, float* part, int nsplit, hipStream_t st) {
  const int nqb = (a.seq + 31) / 32;
  const Scales sc(a);
  Geom g = make_geom(a);
  g.part = part;
  g.nsplit = nsplit;
  const unsigned groups = (unsigned)(nqb * a.batch_heads * nsplit);
  const T *q = static_cast<const T*>(a.q), *k = static_cast<const T*>(a.k),
          *v = static_cast<const T*>(a.v);
  T* o = static_cast<T*>(a.o);
  auto go = [&](auto nw, auto causal) {
    constexpr int NW = decltype(nw)::value;
    hipLaunchKernelGGL((fa2_fwd_rows32_kernel<D, NW, decltype(causal)::value != 0, T, KVSPLIT>),
                       dim3(groups), dim3(64 * NW), 0, st, q, k, v, o, g, nqb, sc.cq, sc.cr);
  };
  if constexpr (D == 64 && !KVSPLIT) {
    if (a.seq_k >= 2048 && groups <= (unsigned)device_cus()) {
      a.causal ? go(Ic<8>{}, Ic<1>{}) : go(Ic<8>{}, Ic<0>{});
      return hipGetLastError();
    }
  }
  a.causal ? go(Ic<4>{}, Ic<1>{}) : go(Ic<4>{}, Ic<0>{});
  return hipGetLastError();
}

template <bool KVSPLIT>
hipError_t launch_rows32_any(const FwdArgs& a, float* part, int nsplit, hipStream_t st) {
  const bool bf = a.dtype == kDtypeBF16;
  if (a.head_dim == 128)
    return bf ? launch_rows32_t<128, __bf16, KVSPLIT>(a, part, nsplit, st)
              : launch_rows32_t<128, _Float16, KVSPLIT>(a, part, nsplit, st);
  return bf ? launch_rows32_t<64, __bf16, KVSPLIT>(a, part, nsplit, st)
            : launch_rows32_t<64, _Float16, KVSPLIT>(a, part, nsplit, st);
}

}  // namespace

hipError_t launch_rows32(const FwdArgs& a, hipStream_t st) {
  return launch_rows32_any<false>(a, nullptr, 1, st);
}

hipError_t launch_kvsplit_rows32(const FwdArgs& a, float* part, int nsplit, hipStream_t st) {
  const hipError_t e = launch_rows32_any<true>(a, part, nsplit, st);
  return e != hipSuccess ? e : launch_splitkv_combine(a, part, nsplit, st);
}

}  // namespace fl
