// Head dim 128: the slot schedule over 32-key tiles and its launchers, one
// source file per element type (fa2_d128.hip fp16, fa2_d128_bf16.hip bf16: the
// instantiations compile in parallel).
#pragma once

#include "fa2_d128.h"

namespace fl {

namespace {

// Slot-scheduled head-dim-128 pipeline: W waves of 32 query rows per key
// stream.  Iteration j: GEMM1 of tile j+1 (even slots), GEMM2 of tile j-1
// with P(j-1) (odd slots), the softmax of tile j (one exponential per slot),
// the LDS read of the operand of slot +kAhead.  S and P are double-buffered.
// The operands of the next iteration's first kAhead slots come from K(j+2)
// and V(j), so the barrier ending iteration j publishes K(j+3) and V(j+1); K
// is fetched FK tiles ahead and V FK-2 into rings of FK slots, FK-3 fetch
// groups in flight at a barrier.  Slot reuse: K(X) lands in the slot of
// K(X-FK), last read in iteration X-FK-1; V(X) in that of V(X-FK), last read
// in iteration X-FK+1 (fetched in iteration X-FK+2).  Iteration 0 has no
// GEMM2, and a wave's last tile drains the pipeline inside its iteration (as
// in fa2_fwd_slot_kernel: its P's first 16 keys are done by slot 7, so even
// slots 8-14 and four more MFMAs run its own GEMM2).  Masked tiles, per-wave
// tile counts, the range check and the checked recompute pass follow
// fa2_fwd_slot_kernel.
//
// SPLIT = 2: 2W waves hold the same 32W query rows; stream 0 walks the first
// half of the block's key tiles and stream 1 the rest, each through its own
// rings; at the end the two waves of a row block exchange halves of the head
// dim through one idle ring slot each, and each merges and stores its half.
// PAIR: such a group walks blocks p and nqb-1-p of a head (equal work under
// the causal mask), the second block's Q, K(0) and K(1) fetched during the
// first one's merge.
//
// What bounds it.  With every CU busy the loop runs at the chip's power
// limit: the 2 x 4-wave split takes 0.59 us per iteration on 64 CUs, 0.70 on
// 128 and 0.87 on 256, where 256 groups compute 1.23 PFLOP/s, what a large
// library GEMM reaches on the same box (1.25 fp16, 1.30 bf16).  Problems below
// that size are bound by their longest walk and its start and end, which is
// what SPLIT and PAIR shorten.  A DMA instruction waits at issue while the
// CU's memory pipeline is busy, so the iteration's fetches go out one every
// few slots instead of all at its start: B2 H8 N1024 15.6 -> 13.2 us and B1
// H2 N8192 causal 71.2 -> 65.5 on the 64-row split, 84.0 -> 76.3 on the
// 128-row one.  With one wave per SIMD (64-row groups) reading operands 8
// slots ahead instead of 4 takes those to 12.8 and 62.2; with two it is 0-4%
// slower.  The rings hold 4 tiles: 5 measured 0-5% slower.
template <int W, int FK, bool CAUSAL, class T, int SPLIT = 1, bool PAIR = false>
__global__ void __launch_bounds__(64 * W * SPLIT, 2)
fa2_fwd_d128_kernel(const T* Q, const T* __restrict__ K, const T* __restrict__ V, T* O,
                    const Geom geom, int nqb, float cq, float cr) {
  using RowsT = Rows128<CAUSAL, T>;
  using V8 = typename RowsT::V8;
  constexpr int FV = FK - 2;
  constexpr int kSlots = FK;
  constexpr int kUnroll = (kSlots % 2 == 0) ? kSlots : 2 * kSlots;
  constexpr int kBr = 32 * W;
  constexpr int kSegs = 8 / W;
  constexpr int kDmaPerIter = 2 * kSegs;
  constexpr int kDmaEvery = 16 / kDmaPerIter;  // slots per DMA instruction
  constexpr int kRingBytes = kSlots * kTileBytes;
  // Two work-groups share a CU when both rings fit its 160 KiB and the
  // waves fit two per SIMD (<= 4 waves each).
  constexpr int kWgPerCu = (W * SPLIT <= 4 && 2 * 2 * SPLIT * kRingBytes <= 160 * 1024) ? 2 : 1;
  // A stream's Q blocks pass through its V ring before the first V tile is
  // fetched, where they fit it and no other block's fetches overlap.
  constexpr bool kQInV = W <= kSlots && !PAIR;
  constexpr int kQBytes = W * kTileBytes;
  constexpr int kQParts = kQInV ? 1 : SPLIT;  // waves sharing a Q block's fetch
  // With one wave per SIMD the compiler's own order is left alone, and the
  // operands are read further ahead of their MFMA (slots).
  constexpr bool kFence = W * SPLIT * kWgPerCu > 4;
  constexpr int kAhead = kFence ? 4 : 8;
  constexpr int kTailReads = kAhead + kAhead / 2;  // K slots: 1 read, V slots: 2
  static_assert(kSegs * W == 8, "tile split");
  static_assert(FK >= 4 && FK <= 8, "fetch distance");
  static_assert(kAhead % 2 == 0 && kAhead >= 4 && kAhead < 16, "read-ahead");
  static_assert(kTileBytes == kBc2 * kRowBytes2, "tile size");
  static_assert(!PAIR || SPLIT == 2, "block pairs: key-range split groups");
  __shared__ __attribute__((aligned(16))) uint8_t
      lds[2 * SPLIT * kRingBytes + (kQInV ? 0 : kQBytes)];
  uint8_t* const kring = lds;
  uint8_t* const vring = lds + SPLIT * kRingBytes;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int stream = SPLIT == 1 ? 0 : wave / W;  // key-range half
  const int rw = wave - stream * W;              // 32-row block within the work-group
  int bh, qb, qb2 = 0, nblk = 1;
  if constexpr (PAIR) {
    int pr;
    pair_coords(nqb, geom.xcds, bh, pr);
    qb = nqb - 1 - pr;
    qb2 = pr;
    nblk = qb2 < qb ? 2 : 1;  // the middle block of an odd count walks alone
  } else {
    wg_coords<CAUSAL, kWgPerCu>(nqb, geom.xcds, geom.cus_per_xcd, bh, qb);
  }
  const HeadPtrs<T> hp = head_ptrs<T, kRowBytes2>(geom, bh, Q, K, V, O);
  const FetchOff<kSegs> fk = fetch_offsets128<kSegs, false>(rw, lane, 2 * geom.k_sr);
  const FetchOff<kSegs> fv = fetch_offsets128<kSegs, true>(rw, lane, 2 * geom.v_sr);
  const int seq = geom.seq_q;
  const StreamRings<kSlots> rings = {kring + stream * kRingBytes, vring + stream * kRingBytes};
  // The walk of block bi: its first query row, and this stream's key tiles
  // [tbeg, tend); iterations 0 .. t0 - 1 on tile tbeg + j (the shorter
  // stream's last tile lies past its range: masked, fetched as zeros).
  struct Walk {
    int q0, t0, tbeg, tend;
    i32x4_t rk, rv;
  };
  auto walk_of = [&](int bi) __attribute__((always_inline)) {
    Walk w;
    w.q0 = (bi == 0 ? qb : qb2) * kBr;
    int n = max(1, (geom.seq_k + kBc2 - 1) / kBc2);
    if (CAUSAL) n = min(n, causal_tiles32(min(w.q0 + kBr, seq), geom.coff));
    w.t0 = SPLIT == 2 ? (n + 1) / 2 : n;
    w.tbeg = stream == 0 ? 0 : w.t0;
    w.tend = stream == 0 ? w.t0 : n;
    kv_rsrc_rows<T, kRowBytes2>(geom, bh, K, V, w.tend * kBc2, w.rk, w.rv);
    return w;
  };
  uint8_t* const qblk =
      (kQInV ? rings.v : vring + SPLIT * kRingBytes) + rw * kTileBytes;
  bool prefetched = false;  // PAIR: Q, K(0), K(1) of the block are on their way
  auto run_block = [&](const int bi) __attribute__((always_inline)) {
  const Walk wk = walk_of(bi);
  const int q0 = wk.q0, t0 = wk.t0, tbeg = wk.tbeg, tend = wk.tend;
  const i32x4_t rk = wk.rk, rv = wk.rv;
  const int last = max(tend - 1, tbeg);  // fetch clamp of the checked pass
  const int tzero = tend;
  int nw = tend - tbeg;  // tiles this wave's rows need, at least one
  if (CAUSAL) nw = min(nw, causal_tiles32(min(q0 + 32 * rw + 32, seq), geom.coff) - tbeg);
  if (q0 + 32 * rw >= seq) nw = 1;
  nw = max(nw, 1);

  // Prologue: Q, K(0) and K(1) first, the remaining groups (-FK+2 .. -1)
  // after the first GEMM1.
  auto fetch_k = [&](auto i, int j) __attribute__((always_inline)) {
    fetch_tile_z<kSegs>(rk, rings.kslot(i), tbeg + j, tzero, rw, fk);
  };
  auto fetch_v = [&](auto i, int j) __attribute__((always_inline)) {
    fetch_tile_z<kSegs>(rv, rings.vslot(i), tbeg + j, tzero, rw, fv);
  };
  if (!PAIR || !prefetched) {
    fetch_q_block128<kQParts>(hp.q, geom.q_sr, q0 + 32 * rw, seq, qblk, lane,
                              kQInV ? 0 : stream);
    fetch_k(Ic<0>{}, 0);
    fetch_k(Ic<1>{}, 1);
  }
  RowsT rows;
  rows.place(lane, q0 + 32 * rw, seq, min(geom.seq_k, tend * kBc2), geom.coff, cr);
  // Iterations j < jm need no mask on tile tbeg + j + 1.
  int tm = rows.kv_lim / kBc2;
  if (CAUSAL) tm = min(tm, (rows.qd + 1) / kBc2);
  const int jm = max(0, tm - tbeg - 1);
  if constexpr (kQInV) {
    // The wave's own Q block: out of the V ring before any wave's V(0).
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" : : "n"(2 * kSegs) : "memory");
    rows.set_q_lds(qblk, cq);
  }
  sync_ring_ahead<kSegs, 0>();  // (Q,) K(0)
  if constexpr (!kQInV) rows.set_q_lds(qblk, cq);
  float16_t S0, S1;
  V8 P0[2], P1[2];
  rows.gemm1(rings.kslot(Ic<0>{}), S0);
  static_for(std::make_integer_sequence<int, FK - 2>{}, [&](auto i) __attribute__((always_inline)) {
    constexpr int N = decltype(i)::value;  // K(N + 2), V(N)
    fetch_k(Ic<N + 2>{}, N + 2);
    fetch_v(Ic<N>{}, N);
  });
  rows.mask(tbeg, S0);
  rows.first_tile(S0);
  // Iteration 0 refills K(0)'s slot: every wave's reads of it are done.
  sync_ring_ahead<(FK - 3) * kDmaPerIter, 0>();  // K(2), V(0)

  // Iteration kinds (bits): kFirst (j = 0) has no GEMM2; kLast (the wave's
  // last tile) has no GEMM1 and drains its own GEMM2.
  constexpr int kFull = 0, kFirst = 1, kLast = 2;
  constexpr int kLastTail = 4;
  constexpr auto runs = [](int kind, int L) {
    return (L & 1) ? (kind & kFirst) == 0 : ((kind & kLast) == 0 || L >= 8);
  };
  // kLast: even slot L >= 8 runs head-dim block fold_db(L) of its own key
  // step 0 (never the block of the odd slot beside it).
  constexpr auto fold_db = [](int L) { return (((L - 8) >> 1) + 2) & 3; };
  V8 ahead[kAhead];
  static_for(std::make_integer_sequence<int, kAhead / 2>{}, [&](auto i) __attribute__((always_inline)) {
    constexpr int a = 2 * decltype(i)::value;
    ahead[a] = rows.template read_slot<a>(rings.kslot(Ic<1>{}), rings.vslot(Ic<-1>{}));
  });

  uint64_t out_of_range = 0;
  auto iteration = [&](auto i, int j, float16_t& S, float16_t& Sn, V8 (&P)[2], const V8 (&Pp)[2],
                       auto masked, auto kind) __attribute__((always_inline)) {
    constexpr int I = decltype(i)::value;
    constexpr int Kd = decltype(kind)::value;
    constexpr bool kFold = (Kd & kLast) != 0;
    const int tbk = min(tbeg + j + FK, tzero) * fk.tile_bytes;
    const int tbv = min(tbeg + j + FV, tzero) * fv.tile_bytes;
    V8 op[16], top[kLastTail];
#pragma unroll
    for (int a = 0; a < kAhead; ++a)
      if (runs(Kd, a)) op[a] = ahead[a];
    float sum[4];
    static_for(std::make_integer_sequence<int, 16>{}, [&](auto sl) __attribute__((always_inline)) {
      constexpr int L = decltype(sl)::value;
      if constexpr (runs(Kd, L)) {
        if constexpr (kFold && L % 2 == 0)
          rows.o[fold_db(L)] = RowsT::E::mfma(op[L], P[0], rows.o[fold_db(L)]);
        else
          rows.template mfma_slot<L>(op[L], Sn, Pp);
      }
      if constexpr (kFence) __builtin_amdgcn_sched_barrier(0);
      // The iteration's fetches, one every kDmaEvery slots.
      if constexpr (L % kDmaEvery == 0) {
        constexpr int d = L / kDmaEvery;
        if constexpr (d < kSegs)
          fetch_seg<kSegs>(rk, rings.kslot(Ic<I + FK>{}), tbk, d, rw, fk);
        else
          fetch_seg<kSegs>(rv, rings.vslot(Ic<I + FV>{}), tbv, d - kSegs, rw, fv);
      }
      if constexpr (L + kAhead < 16) {
        constexpr int La = L + kAhead;
        if constexpr (runs(Kd, La)) {
          if constexpr (kFold && La % 2 == 0)
            op[La] = rows.read_v_op(rings.vslot(Ic<I>{}), fold_db(La), 0);
          else
            op[La] = rows.template read_slot<La>(rings.kslot(Ic<I + 1>{}), rings.vslot(Ic<I - 1>{}));
        }
      } else if constexpr (!kFold) {
        ahead[L + kAhead - 16] = rows.template read_slot<L + kAhead - 16>(
            rings.kslot(Ic<I + 2>{}), rings.vslot(Ic<I>{}));
      } else if constexpr (L + kAhead - 16 < kLastTail) {
        top[L + kAhead - 16] = rows.read_v_op(rings.vslot(Ic<I>{}), L + kAhead - 16, 1);
      }
      rows.template exp_slot<L>(S, P, sum);
      if constexpr (kFence) __builtin_amdgcn_sched_barrier(0);
    });
    if constexpr (kFold)
#pragma unroll
      for (int db = 0; db < kLastTail; ++db)
        rows.o[db] = RowsT::E::mfma(top[db], P[1], rows.o[db]);
    const float tot = (sum[0] + sum[1]) + (sum[2] + sum[3]);
    rows.l += tot;
    out_of_range |= __builtin_amdgcn_ballot_w64(!(tot <= kSumLimit));
    if constexpr (decltype(masked)::value && !kFold) rows.mask(tbeg + j + 1, Sn);
    sync_ring_ahead<(FK - 3) * kDmaPerIter, kFold ? 0 : kTailReads>();
  };
  auto group = [&](int j0, auto masked, auto first) __attribute__((always_inline)) {
    static_for(std::make_integer_sequence<int, kUnroll>{}, [&](auto i) __attribute__((always_inline)) {
      constexpr int I = decltype(i)::value;
      constexpr int Kd = decltype(first)::value && I == 0 ? kFirst : kFull;
      const int j = j0 + I;
      if (Kd == kFirst || !decltype(masked)::value || j < nw - 1) {
        if constexpr (I % 2 == 0)
          iteration(i, j, S0, S1, P0, P1, masked, Ic<Kd>{});
        else
          iteration(i, j, S1, S0, P1, P0, masked, Ic<Kd>{});
      }
    });
  };
  {
    if (nw >= 2) {
      int j0 = kUnroll;
      if (kUnroll <= jm) {
        group(0, Ic<false>{}, Ic<true>{});
        for (; j0 + kUnroll <= jm; j0 += kUnroll) group(j0, Ic<false>{}, Ic<false>{});
      } else {
        group(0, Ic<true>{}, Ic<true>{});
      }
      for (; j0 < nw - 1; j0 += kUnroll) group(j0, Ic<true>{}, Ic<false>{});
    }
    // the wave's last tile, at its unrolled position
    static_for(std::make_integer_sequence<int, kUnroll>{}, [&](auto i) __attribute__((always_inline)) {
      constexpr int I = decltype(i)::value;
      if ((nw - 1) % kUnroll == I) {
        if constexpr (I == 0) {
          if (nw == 1)
            iteration(i, 0, S0, S1, P0, P1, Ic<true>{}, Ic<kFirst | kLast>{});
          else
            iteration(i, nw - 1, S0, S1, P0, P1, Ic<true>{}, Ic<kLast>{});
        } else if constexpr (I % 2 == 0) {
          iteration(i, nw - 1, S0, S1, P0, P1, Ic<true>{}, Ic<kLast>{});
        } else {
          iteration(i, nw - 1, S1, S0, P1, P0, Ic<true>{}, Ic<kLast>{});
        }
      }
    });
    // Past its last tile a wave only fetches its share and meets the barriers.
    for (int j = nw; j < t0; ++j) {
      fetch_tile_z<kSegs>(rk, rings.k + kTileBytes * ((j + FK) % kSlots), tbeg + j + FK, tzero, rw,
                          fk);
      fetch_tile_z<kSegs>(rv, rings.v + kTileBytes * ((j + FV) % kSlots), tbeg + j + FV, tzero, rw,
                          fv);
      sync_ring_ahead<(FK - 3) * kDmaPerIter, 0>();
    }
  }

  // Checked pass (as in fa2_fwd_slot_kernel); the flag lives in the last 16
  // bytes of the V rings.
  __builtin_amdgcn_s_waitcnt(0);
  int* redo = reinterpret_cast<int*>(vring + SPLIT * kRingBytes - 16);
  __syncthreads();
  if (threadIdx.x == 0) *redo = 0;
  __syncthreads();
  if (out_of_range != 0 && lane == 0) *redo = 1;
  __syncthreads();
  if (*redo) {
    rows.launder();
    rows.reset();
    for (int t = 0; t < t0; ++t) {
      fetch_tile<kSegs>(rk, rings.kslot(Ic<0>{}), tbeg + t, last, rw, fk);
      fetch_tile<kSegs>(rv, rings.vslot(Ic<0>{}), tbeg + t, last, rw, fv);
      sync_ring_ahead<0, 0>();
      float16_t Sc;
      V8 Pc[2];
      rows.gemm1(rings.kslot(Ic<0>{}), Sc);
      rows.mask(tbeg + t, Sc);
      if (t == 0) rows.first_tile(Sc);
      rows.softmax_checked(Sc, Pc);
      rows.gemm2(rings.vslot(Ic<0>{}), Pc);
      sync_ring_ahead<0, 0>();
    }
  }
  if (PAIR && bi + 1 < nblk) {
    // Every wave is past its reads of the rings and of its Q block: the next
    // block's Q, K(0) and K(1) go out now, to land during the merge.
    const Walk nx = walk_of(bi + 1);
    fetch_q_block128<kQParts>(hp.q, geom.q_sr, nx.q0 + 32 * rw, seq, qblk, lane, stream);
    fetch_tile_z<kSegs>(nx.rk, rings.kslot(Ic<0>{}), nx.tbeg, nx.tend, rw, fk);
    fetch_tile_z<kSegs>(nx.rk, rings.kslot(Ic<1>{}), nx.tbeg + 1, nx.tend, rw, fk);
    prefetched = true;
  }
  rows.launder();
  if constexpr (SPLIT == 2) {
    // Exchange: wave (stream s, row block rw) leaves the half of its O that
    // the other stream's wave stores in slot 4 s + rw of {V slots 1-3 and K
    // slot 3 of stream 0, then of stream 1}, and its mc and l in K slot 2 of
    // stream 0; K slots 0 and 1 and the Q blocks take the next block's
    // fetches meanwhile.  (__syncthreads waits for LDS accesses only; the
    // DMA in flight writes none of these.)
    auto xslot = [&](int i) __attribute__((always_inline)) {
      const int r = i / 4, c = i % 4;
      return reinterpret_cast<float4*>(c < 3 ? vring + r * kRingBytes + (1 + c) * kTileBytes
                                             : kring + r * kRingBytes + 3 * kTileBytes);
    };
    float2* const ml = reinterpret_cast<float2*>(kring + 2 * kTileBytes);
    asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
    __syncthreads();
    if (stream == 0)
      rows.template save_half<1>(xslot(rw), lane);
    else
      rows.template save_half<0>(xslot(4 + rw), lane);
    ml[wave * 64 + lane] = make_float2(rows.mc, rows.l);
    __syncthreads();
    const float2 x = ml[(wave ^ W) * 64 + lane];
    if (stream == 0) {
      rows.template merge_half<0>(xslot(4 + rw), x.x, x.y, lane);
      rows.template store<0, 2>(hp.o, geom.o_sr, hp.lse);
    } else {
      rows.template merge_half<1>(xslot(rw), x.x, x.y, lane);
      rows.template store<2, 4>(hp.o, geom.o_sr, hp.lse);
    }
  } else {
    rows.template store<0, 4>(hp.o, geom.o_sr, hp.lse);
  }
  // every wave past its reads of the exchange before the next block's fetches
  if (PAIR && bi + 1 < nblk) __syncthreads();
  };  // run_block
  run_block(0);
  if constexpr (PAIR) {
    if (nblk > 1) run_block(1);
  }
}

template <int W, class T, int SPLIT = 1, bool PAIR = false>
hipError_t launch_d128_w(const FwdArgs& a, hipStream_t st) {
  constexpr int kFk = 4;
  const int nqb = (a.seq + 32 * W - 1) / (32 * W);
  const int groups = PAIR ? (nqb + 1) / 2 : nqb;
  const Scales sc(a);
  const Geom g = make_geom(a);
  const dim3 grid((unsigned)(groups * a.batch_heads));
  const dim3 block(64 * W * SPLIT);
  const T *q = static_cast<const T*>(a.q), *k = static_cast<const T*>(a.k),
          *v = static_cast<const T*>(a.v);
  T* o = static_cast<T*>(a.o);
  if (a.causal)
    hipLaunchKernelGGL((fa2_fwd_d128_kernel<W, kFk, true, T, SPLIT, PAIR>), grid, block, 0,
                       st, q, k, v, o, g, nqb, sc.cq, sc.cr);
  else
    hipLaunchKernelGGL((fa2_fwd_d128_kernel<W, kFk, false, T, SPLIT, PAIR>), grid, block,
                       0, st, q, k, v, o, g, nqb, sc.cq, sc.cr);
  return hipGetLastError();
}

template <class T>
hipError_t launch_d128_t(const FwdArgs& a, int cfg, hipStream_t stream) {
  switch (cfg) {
    case kSlotW8Config: return launch_d128_w<8, T>(a, stream);
    case kSlotW4Config: return launch_d128_w<4, T>(a, stream);
    case kCfgSplit2: return launch_d128_w<4, T, 2>(a, stream);
    case kCfgSplit2W2: return launch_d128_w<2, T, 2>(a, stream);
    case kCfgPair: return launch_d128_w<4, T, 2, true>(a, stream);
    case kCfgPairW2: return launch_d128_w<2, T, 2, true>(a, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace

}  // namespace fl
