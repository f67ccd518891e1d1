// Head dim 128 (fp16 and bf16): the row state and LDS layout of the slot
// schedule (fa2_d128_kernel.h).
#pragma once

#include "fa2_common.h"

namespace fl {

namespace {

// ---------------------------------------------------------------------------
// Head dim 128 (beyond the reference, whose kernels take D = 64 only,
// kernel_flash2.cu:756-757).  Key tiles of 32 rows x 256 bytes keep the
// 8 KiB tile of D = 64, so an iteration is again 16 MFMA slots: GEMM1 is one
// 32-key block over 8 head-dim steps (one chain), GEMM2 four head-dim
// blocks over 2 key steps.  With 16 scores per lane per tile there is one
// exponential per MFMA, so the softmax VALU work fits under the matrix
// core with room to spare and the row sums stay fp32.
constexpr int kBc2 = 32;
constexpr int kRowBytes2 = 2 * kD2;  // 256

// LDS swizzles of 256-byte rows.  A row is one whole sweep of the 64 banks,
// so unlike the 128-byte rows of D = 64 the row index does not move a read
// to other banks: the swizzles must use all 4 bits of the 16-byte chunk
// index.  K (ds_read_b128, 16 lanes = 16 rows per pass): chunk ^ (row % 16)
// puts the 16 rows of a pass on 16 different chunks.  V (ds_read_b64_tr_b16:
// 2 key-rows x 2 lane groups x 4 chunks x 2 halves per 32-lane pass): the
// D = 64 pattern (row bits 0-1 on chunk bits 1-2) plus row bit 0 on chunk
// bit 3.  Both are conflict-free for every lane pattern of read_k_op and
// read_v_op (the D = 64 swizzles left 2-way conflicts on both).
__device__ __forceinline__ int k_swz128(int row) { return row & 15; }
__device__ __forceinline__ int v_swz128(int row) { return ((row & 3) << 1) | ((row & 1) << 3); }

// DMA lane offsets for 256-byte rows: segment i of wave w is rows
// 4(w kSegs + i) .. +3; lane l lands at byte 16 l of it, i.e. row l/16,
// physical chunk l%16, which holds logical chunk (l%16) ^ swz(row).
template <int kSegs, bool IS_V>
__device__ __forceinline__ FetchOff<kSegs> fetch_offsets128(int wave, int lane, int row_bytes) {
  FetchOff<kSegs> f;
#pragma unroll
  for (int i = 0; i < kSegs; ++i) {
    const int seg = wave * kSegs + i;
    const int row = 4 * seg + (lane >> 4);
    const int phys = lane & 15;
    const int logical = phys ^ (IS_V ? v_swz128(row) : k_swz128(row));
    f.lane[i] = row * row_bytes + 16 * logical;
    asm volatile("" : "+v"(f.lane[i]));
  }
  f.tile_bytes = kBc2 * row_bytes;
  return f;
}

// The 32 query rows one wave owns at head dim 128 (same lane roles as Rows:
// one query per lane, 16 of a 32-key block's scores per lane).  Scores stay
// raw in the accumulators and the stabiliser is subtracted with the scale's
// multiply, p = 2^(s c - mc) in one fma: no accumulator-sized -m to keep (16
// registers) and the same instruction count.
template <bool CAUSAL, class T>
struct Rows128 {
  using E = Elem<T>;
  using V8 = typename E::v8;
  using V4 = typename E::v4;
  int g, col, qw, my_q, seq, qd, my_d, kv_lim, tr_row, tr_col;
  float cr;
  V8 qf[8];          // Q'^T B-operand, head-dim steps 0-7
  float16_t o[4];    // O^T accumulator, head-dim blocks 0-3
  float mc, l;       // stabiliser in base-2 logit units; this lane's share of the row sum

  // Lane placement (as Rows::place).
  __device__ __forceinline__ void place(int lane, int qw_, int seq_, int kv_lim_, int coff,
                                        float cr_) {
    g = lane >> 5;
    col = lane & 31;
    qw = qw_;
    my_q = qw + col;
    qd = qw + coff;
    my_d = my_q + coff;
    seq = seq_;
    kv_lim = kv_lim_;
    cr = cr_;
    const int trG = lane >> 4, trj = lane & 15;
    tr_row = 4 * (trG >> 1) + (trj >> 2);
    const int tr_x = trj & 3;
    tr_col = 16 * (trG & 1) + 4 * (((tr_x & 1) << 1) | (tr_x >> 1));
    reset();
  }
  // Q'^T from the wave's 32 rows staged in LDS like a K tile; the sign of
  // sm_scale is an exact flip of the sign bits.
  __device__ __forceinline__ void set_q_lds(const uint8_t* qblk, float cq) {
    const uint32_t s = cq < 0.0f ? 0x80008000u : 0u;
#pragma unroll
    for (int st = 0; st < 8; ++st)
      qf[st] = __builtin_bit_cast(
          V8, __builtin_bit_cast(u32x4_t, read_k_op(qblk, st)) ^ (u32x4_t){s, s, s, s});
  }
  __device__ __forceinline__ void launder() {
    asm volatile("" : "+v"(col), "+v"(g), "+v"(my_q), "+v"(tr_row), "+v"(tr_col));
  }
  __device__ __forceinline__ void reset() {
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
      for (int r = 0; r < 16; ++r) o[db][r] = 0.0f;
    mc = 0.0f;
    l = 0.0f;
  }
  __device__ __forceinline__ V8 read_k_op(const uint8_t* kt, int st) const {
    const int ch = 2 * st + g;
    return *reinterpret_cast<const V8*>(kt + col * kRowBytes2 + 16 * (ch ^ k_swz128(col)));
  }
  __device__ __forceinline__ V8 read_v_op(const uint8_t* vt, int db, int t) const {
    const int r1 = 16 * t + tr_row;
    const int r2 = r1 + 8;
    const int dcol = 32 * db + tr_col;
    const int ch = dcol >> 3, hb = ((dcol >> 2) & 1) * 8;
    const V4 lo = lds_read_tr<V4>(vt + r1 * kRowBytes2 + 16 * (ch ^ v_swz128(r1)) + hb);
    const V4 hi = lds_read_tr<V4>(vt + r2 * kRowBytes2 + 16 * (ch ^ v_swz128(r2)) + hb);
    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  }
  // GEMM1 of one tile: s = K . Q'^T.
  __device__ __forceinline__ void gemm1(const uint8_t* kt, float16_t& s) const {
    V8 ka[8];
#pragma unroll
    for (int st = 0; st < 8; ++st) ka[st] = read_k_op(kt, st);
#pragma unroll
    for (int st = 0; st < 8; ++st) s = E::mfma(ka[st], qf[st], st == 0 ? zero() : s);
  }
  // GEMM2 of one tile: O^T += V^T . P^T.
  __device__ __forceinline__ void gemm2(const uint8_t* vt, const V8 (&pp)[2]) {
    V8 va[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) va[u] = read_v_op(vt, u & 3, u >> 2);
#pragma unroll
    for (int u = 0; u < 8; ++u) o[u & 3] = E::mfma(va[u], pp[u >> 2], o[u & 3]);
  }
  __device__ __forceinline__ static float16_t zero() {
    return (float16_t){0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
  }
  // Slot map: L even, GEMM1 head-dim step L/2 of the next tile (one chain,
  // steps two slots apart); L odd, u = L/2: GEMM2 head-dim block u % 4 at
  // key step u / 4.
  template <int L>
  __device__ __forceinline__ V8 read_slot(const uint8_t* kt, const uint8_t* vt) const {
    constexpr int u = L >> 1;
    if constexpr ((L & 1) == 0)
      return read_k_op(kt, u);
    else
      return read_v_op(vt, u & 3, u >> 2);
  }
  template <int L>
  __device__ __forceinline__ void mfma_slot(const V8& a, float16_t& sn, const V8 (&pp)[2]) {
    constexpr int u = L >> 1;
    if constexpr ((L & 1) == 0)
      sn = E::mfma(a, qf[u], u == 0 ? zero() : sn);
    else
      o[u & 3] = E::mfma(a, pp[u >> 2], o[u & 3]);
  }
  __device__ __forceinline__ float logit(float s) const {
    return __builtin_fmaf(s, cr, -mc);
  }
  // Softmax share of slot L: score L -> one exponential, its element of
  // the P operand (P[t] holds keys 16t + 4g + {0..3, 8..11}) and the fp32
  // row sum in four chains.
  template <int L>
  __device__ __forceinline__ void exp_slot(const float16_t& s, V8 (&pn)[2], float (&sum)[4]) const {
    const float e = __builtin_amdgcn_exp2f(logit(s[L]));
    pn[L >> 3][L & 7] = (T)e;
    if constexpr (L < 4)
      sum[L] = e;
    else
      sum[L & 3] += e;
  }
  // Keys >= kv_lim and, causal, past the lane's diagonal, of tile t.
  __device__ __forceinline__ void mask(int t, float16_t& s) const {
    const int k0 = t * kBc2;
    if (k0 + kBc2 > kv_lim || (CAUSAL && k0 + kBc2 - 1 > qd)) {
      const int base = k0 + 4 * g;
      int lim = kv_lim - base;
      if (CAUSAL) lim = min(lim, my_d + 1 - base);
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int c = 8 * (r >> 2) + (r & 3);
        s[r] = c < lim ? s[r] : ninf();
      }
    }
  }
  // Row max of a tile in base-2 logit units (both halves of the row).
  __device__ __forceinline__ float tile_max(const float16_t& s) const {
    float mx = ninf();
#pragma unroll
    for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[r]);
    return pair_max(mx) * cr;
  }
  // The first tile's exact row max becomes the stabiliser (0 for a row with
  // no visible key there).
  __device__ __forceinline__ void first_tile(const float16_t& s) {
    const float m0 = tile_max(s);
    mc = m0 == ninf() ? 0.0f : m0;
  }
  __device__ __forceinline__ float exponentiate(const float16_t& s, V8 (&pn)[2]) const {
    float sum[2] = {0.0f, 0.0f};
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float e = __builtin_amdgcn_exp2f(logit(s[r]));
      pn[r >> 3][r & 7] = (T)e;
      sum[r & 1] += e;
    }
    return sum[0] + sum[1];
  }
  // As Rows::softmax_checked, for one 32-key tile.
  __device__ __forceinline__ void softmax_checked(const float16_t& s, V8 (&pn)[2]) {
    float sum = exponentiate(s, pn);
    if (__builtin_amdgcn_ballot_w64(!(sum <= kSumLimit)) != 0) {
      const float d = fmaxf(tile_max(s) - mc, 0.0f);
      const float alpha = __builtin_amdgcn_exp2f(-d);
      l *= alpha;
#pragma unroll
      for (int db = 0; db < 4; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[db][r] *= alpha;
      mc += d;
      sum = exponentiate(s, pn);
    }
    l += sum;
  }
  // Head-dim half H (blocks 2H, 2H+1) of this wave's O into one ring slot
  // (8 KiB), chunk-major in 16-byte pieces.
  template <int H>
  __device__ __forceinline__ void save_half(float4* slot, int lane) const {
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const int db = 2 * H + (c >> 2), r = 4 * (c & 3);
      slot[c * 64 + lane] = make_float4(o[db][r], o[db][r + 1], o[db][r + 2], o[db][r + 3]);
    }
  }
  // Folds the other key range's half H (and its mc and l share) into this
  // wave's; a row with no key in one range takes the other's values.
  template <int H>
  __device__ __forceinline__ void merge_half(const float4* slot, float m1, float l1, int lane) {
    const bool has0 = pair_sum(l) > 0.0f;
    const bool has1 = pair_sum(l1) > 0.0f;
    const float mm = has0 ? (has1 ? fmaxf(mc, m1) : mc) : m1;
    const float a0 = has0 ? __builtin_amdgcn_exp2f(mc - mm) : 0.0f;
    const float a1 = has1 ? __builtin_amdgcn_exp2f(m1 - mm) : 0.0f;
    l = a0 * l + a1 * l1;
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const int db = 2 * H + (c >> 2), r = 4 * (c & 3);
      const float4 x = slot[c * 64 + lane];
      o[db][r] = a0 * o[db][r] + a1 * x.x;
      o[db][r + 1] = a0 * o[db][r + 1] + a1 * x.y;
      o[db][r + 2] = a0 * o[db][r + 2] + a1 * x.z;
      o[db][r + 3] = a0 * o[db][r + 3] + a1 * x.w;
    }
    mc = mm;
  }
  // O = O^T / l of head-dim blocks [B0, B1), 16-byte stores of 8 contiguous
  // head dims; with block 0 the log-sum-exp as in Rows::store.
  template <int B0, int B1>
  __device__ __forceinline__ void store(T* Oh, int o_sr, float* lse) const {
    const float l_tot = pair_sum(l);
    const float inv = l_tot > 0.0f ? 1.0f / l_tot : 0.0f;
    if (B0 == 0 && lse != nullptr && g == 0 && my_q < seq) {
      const float lg = mc + __builtin_amdgcn_logf(l_tot);
      lse[my_q] = l_tot > 0.0f ? 0.693147180559945309f * lg : ninf();
    }
    if (my_q < seq) {
      T* orow = Oh + (long long)my_q * o_sr;
#pragma unroll
      for (int db = B0; db < B1; ++db)
#pragma unroll
        for (int hh = 0; hh < 2; ++hh) {
          V8 out;
#pragma unroll
          for (int e = 0; e < 8; ++e) out[e] = (T)(o[db][8 * hh + e] * inv);
          *reinterpret_cast<V8*>(orow + 32 * db + 16 * hh + 8 * g) = out;
        }
    }
  }
};

// Causal key tiles of 32 keys a block of query rows [q0, q_end) needs.
__device__ __forceinline__ int causal_tiles32(int q_end, int coff) {
  const int last_key = q_end - 1 + coff;
  return last_key < 0 ? 1 : last_key / kBc2 + 1;
}

// The 32 query rows [q, q + 32) of a head (rows >= N_q read as zeros) into
// `qblk`, laid out as a K tile: 8 fetches of 1 KiB by DMA, or with kParts
// waves sharing the block, the 8 / kParts of them of part `part`.  Rows
// further apart than 32-bit offsets reach go through registers.
template <int kParts, class T>
__device__ __forceinline__ void fetch_q_block128(const T* Qh, int q_sr, int q, int seq,
                                                 uint8_t* qblk, int lane, int part) {
  constexpr int kSegs = 8 / kParts;
  const int rows = min(32, seq - q);
  if (q_sr <= kDmaQRowStride) {
    const i32x4_t rq = buffer_rsrc(Qh + (long long)(rows > 0 ? q : 0) * q_sr,
                                   rows > 0 ? (rows - 1) * (2 * q_sr) + kRowBytes2 : 0);
    const FetchOff<kSegs> fq = fetch_offsets128<kSegs, false>(part, lane, 2 * q_sr);
    fetch_tile_z<kSegs>(rq, qblk, 0, 1, part, fq);
  } else {
#pragma unroll 1
    for (int i = 0; i < kSegs; ++i) {
      const int row = 4 * (part * kSegs + i) + (lane >> 4), chunk = lane & 15;
      u32x4_t x = {0, 0, 0, 0};
      if (row < rows)
        x = *reinterpret_cast<const u32x4_t*>(Qh + (long long)(q + row) * q_sr + 8 * chunk);
      *reinterpret_cast<u32x4_t*>(qblk + row * kRowBytes2 + 16 * (chunk ^ k_swz128(row))) = x;
    }
  }
}

}  // namespace

}  // namespace fl
