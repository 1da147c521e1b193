// Causal flash attention on the MFMA units for bf16 storage (registry ops 45, 47, 48; reference semantics:
// runtime/ref_gpt.py:279-364). Used when q, k, v, do, o, dq, dk, dv are bf16 storage with 16-byte aligned head
// slices, lse / delta are f32 and hd is 32, 64 or 128 (attn_form in ops_attn.h); other cases run the fp32 SIMT bodies
// there. T a multiple of 64 (and, backward, hd up to 64) takes the plain form, everything else the HP form.
//
// HP forms (T not a multiple of 64, and the backward at hd 128): the arithmetic of the SIMT bodies that these shapes took
// before. The probabilities and dS are f32 values and enter the second product whole, as three bf16 pieces (24 bits of
// significand are 8 + 8 + 8, and the other operand is bf16 storage, so every product is exact): three MFMAs instead of
// one. Exponentials are __expf of (score * scale - lse), not exp2 with log2(e) folded into the scale, whose rounding
// grows with the score and the lse instead of their difference. The SIMT bodies still take any task with a non-finite
// result: a masked key or query has weight 0, which a NaN or infinity in its row would turn into NaN here (0 * inf) where
// the SIMT loop skips the row. The HP form returns true then, with nothing stored. Rows past T are read as row T - 1
// (and masked).
//
// Scheme ("transposed space"): every product is computed with the reduction axis of the softmax on the MFMA's row
// axis, so that each lane owns one query (forward, dQ) or one key (dK/dV):
//   * S^T = K Q^T with v_mfma_f32_32x32x16_bf16 (A = 32 key rows, B = 32 query rows, k = head dim). The accumulator
//     holds D[key][query] with lane l owning query l % 32 and keys 8*(r/4) + 4*(l/32) + r%4 of its 32-key block:
//     the softmax statistics of a query live in lanes l and l ^ 32, combined with one lane exchange.
//   * O^T += V^T P^T: the bf16-rounded P^T accumulator registers are used directly as the B operand; the key order
//     inside each 16-key MFMA step is the one those registers already have (keys 0-3, 8-11 in lanes 0-31 and 4-7,
//     12-15 in lanes 32-63), and V^T is read in the same key order with LDS transpose reads. A dot product does not
//     depend on the order of its terms, so the permutation is free.
//   * O^T's accumulator has lane l owning query l % 32 again, so the online-softmax rescale is one multiply per
//     register and the output store is 4 consecutive head-dim elements per lane.
// Softmax exponentials are the hardware exp2 (v_exp_f32; __expf is the same after one product): every argument is <= 0 (a score minus the running max or the
// row's log-sum-exp), where it differs from the library exp2f only by flushing results below 2^-126 to zero.
// K/V (or Q/dO) blocks of 64 rows go from HBM straight into LDS (buffer_load ... lds), FA_NS stages deep. Each block
// is kept in one of two swizzled layouts: "kc" for MFMA operands read along the head dim (ds_read_b128), "tr" for
// operands read across rows (ds_read_b64_tr_b16); see ops_gemm.h for the transpose-read semantics.
#pragma once
#include "common.h"
#include "ops_gemm.h"

namespace kvm {

constexpr int FA_KB = 64;      // rows (keys or queries) per stage
constexpr int FA_NS = 3;       // stages (prefetch distance FA_NS - 1)

// KB: rows per staged block.
template <int HD, int KB = FA_KB> struct FaL {
  static constexpr int UPR = HD / 8;                       // 16-byte units per row
  static constexpr int NL = KB * HD * 2 / 1024 / KVM_WAVES;      // direct loads per thread per block
  static_assert(NL >= 1, "hd");
  // kc layout: 16 consecutive rows reading one unit hit every bank once
  __device__ static __forceinline__ int kswz(int row) { return (row / (16 / UPR)) % UPR; }
  // tr layout: 4 consecutive rows (row % 4 == 0) x 32 bytes per 16-lane group, 32 lanes per pass, conflict-free
  __device__ static __forceinline__ int tswz(int row) { return UPR >= 16 ? 4 * (row & 3) : UPR == 8 ? 4 * ((row >> 1) & 1) : 0; }
  __device__ static __forceinline__ int kc(int row, int unit) { return row * HD + 8 * (unit ^ kswz(row)); }
  __device__ static __forceinline__ int tr(int row, int col) { return row * HD + 8 * ((col >> 3) ^ tswz(row)) + (col & 7); }
  // Direct loads of rows [row0, row0 + KB), columns [c0, c0 + HD) of a bf16 matrix with `cols` columns (buffer
  // descriptor rs) into dst in the kc (TRL false) or tr (TRL true) layout. CL: rows past `last` read row `last`.
  template <bool TRL, bool CL = false> __device__ static __forceinline__ void issue(LDS uint16_t* dst, i32x4_t rs, int row0, int cols, int c0, int last = 0) {
#pragma unroll
    for (int q = 0; q < NL; ++q) {
      const int b = q * KVM_WAVES + wave(), u = 64 * b + lane(), row = u / UPR, ph = u % UPR;
      const int lu = ph ^ (TRL ? tswz(row) : kswz(row));
      dma16(rs, ((CL ? min(row0 + row, last) : row0 + row) * cols + c0 + 8 * lu) * 2, 0, dst + b * 512);
    }
  }
  // MFMA operand from the kc layout: 8 values of row rb + l % 32 at head-dim chunk kk*2 + l/32.
  __device__ static __forceinline__ bf16x8 frag_kc(const LDS uint16_t* s, int rb, int kk) {
    const int l = lane(), r = rb + (l & 31);
    return *(const LDS bf16x8*)(s + kc(r, kk * 2 + (l >> 5)));
  }
  // MFMA operand from the tr layout, rows = head dims db..db+31 (lane l: dim db + l % 32), k = 16 block rows starting
  // at `base` in the accumulator key order: lanes 0-31 rows base+0..3, base+8..11; lanes 32-63 rows base+4..7,
  // base+12..15.
  __device__ static __forceinline__ bf16x8 frag_tr(const LDS uint16_t* s, int db, int base) {
    const int l = lane(), G = l >> 4, i = l & 15;
    const int row = base + 4 * (G >> 1) + (i >> 2), col = db + 16 * (G & 1) + 4 * (i & 3);
    const LDS uint16_t* p0 = s + tr(row, col);
    const s16x4_t v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS s16x4_t*)p0);
    const s16x4_t v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS s16x4_t*)(p0 + 8 * HD));
    typedef short s16x8_t __attribute__((ext_vector_type(8)));
    return (bf16x8)__builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7);
  }
};

__device__ __forceinline__ bf16x8 pack_bf16(const float* p) {
  bf16x8 r;
#pragma unroll
  for (int i = 0; i < 8; ++i) r[i] = (__bf16)p[i];
  return r;
}

// f32 values as the second product's operand: their bf16 roundings and, for the HP forms, the bf16 roundings of what
// those leave, twice. Each remainder is exact in f32 and has 8 bits less, so that the three pieces sum to the value.
template <int NP> struct Pieces { bf16x8 p[NP]; };
template <int NP> __device__ __forceinline__ Pieces<NP> split_bf16(const float* x) {
  Pieces<NP> r;
  float y[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) y[i] = x[i];
#pragma unroll
  for (int k = 0; k < NP; ++k) {
    r.p[k] = pack_bf16(y);
#pragma unroll
    for (int i = 0; i < 8; ++i) y[i] -= (float)r.p[k][i];
  }
  return r;
}
// acc += a * (the sum of b's pieces), the smallest first
template <int NP> __device__ __forceinline__ f32x16 mfma_pieces(bf16x8 a, const Pieces<NP>& b, f32x16 acc) {
#pragma unroll
  for (int k = NP - 1; k >= 0; --k) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b.p[k], acc, 0, 0, 0);
  return acc;
}

// A block-wide vote on `bad` through the task's LDS, whose contents are no longer needed. All threads call it.
__device__ __forceinline__ bool fa_any(const Ctx& c, bool bad) {
  const bool w = __ballot(bad) != 0ull;
  LDS int* f = (LDS int*)c.smem;
  __syncthreads();
  if (lane() == 0) f[wave()] = w;
  __syncthreads();
  return (f[0] | f[1] | f[2] | f[3]) != 0;
}

// e^x as the SIMT bodies take it (HP), or 2^x
template <bool HP> __device__ __forceinline__ float fa_exp(float x) { return HP ? __expf(x) : __builtin_amdgcn_exp2f(x); }

__device__ __forceinline__ View uview(const Ctx& c, int k) { return uniform_view(c.buf(k)); }

// Whether a bf16 view's head slices can be read as 16-byte vectors through a buffer descriptor of T rows.
__device__ __forceinline__ bool fa_ok(const View& x, int T) {
  return x.ok() && x.dtype == 2 && (x.cols % 8) == 0 && (long long)T * x.cols * 2 < 0x7fffffffll;
}

// Forward for 128 queries of head h (op 45): lane l of wave w owns query q0 + 32w + l%32. Per 64-key block kb:
// S^T = K Q^T, P^T = exp2(S^T * scale * log2(e) - m), O^T += V^T P^T, with a running maximum m per query.
//   * Software pipeline over blocks: iteration kb computes the scores of block kb + 1 and then the softmax and P V of
//     block kb, so the MFMAs of the next scores and the VALU work of the current softmax are independent and the
//     scheduler interleaves them (one wave per SIMD: nothing else hides either). FA_FNS stages of K/V in LDS; the
//     buffer a new block loads into held block kb - 1, which every wave finished before the barrier of iteration kb.
//   * The causal mask is applied only in blocks that reach past the wave's first query.
//   * Lazy rescaling: m moves (and O, l are rescaled) only when a query's block maximum exceeds m by more than 8 (in
//     log2 units); P values are then at most 2^8, which fp32 sums and bf16 P hold with the same relative rounding. The
//     result O / l and the log-sum-exp m + log2(l) do not depend on which m was used.
constexpr int FA_FNS = 4;
template <int HD, bool HP = false> __device__ __noinline__ bool attn_fwd_mfma(const Ctx& c) {
  typedef FaL<HD> L;
  constexpr int NKK = HD / 16, NDB = HD / 32, NS = FA_FNS;
  const View q = uview(c, 0), k = uview(c, 1), v = uview(c, 2), o = uview(c, 3), lse = uview(c, 4);
  const int bb = rfl(c.i(5)), h = rfl(c.i(6)), q0 = rfl(c.i(7)), T = rfl(c.i(8)), H = rfl(c.i(9)), Hkv = rfl(c.i(10));
  const float sc = __int_as_float(rfl(__float_as_int(c.f(12))));
  const float sl2 = HP ? sc : sc * 1.4426950408889634f;   // the scores' unit: scale * log2(e), HP scale
  const float moved = HP ? 5.5f : 8.f;                     // a maximum moves by more than this (2^8, e^5.5)
  const int w = wave(), l = lane(), g = l >> 5, qi = l & 31;
  const int qrow = q0 + 32 * w + qi, kvh = h / (H / Hkv);
  const bool qok = qrow < T;
  bf16x8 qf[NKK];
#pragma unroll
  for (int kk = 0; kk < NKK; ++kk)
    qf[kk] = qok ? *(const GLOBAL bf16x8*)(q.h() + ((long long)bb * T + qrow) * q.cols + h * HD + kk * 16 + 8 * g) : bf16x8{};
  const int kend = min(T, q0 + 128), nkb = (kend + FA_KB - 1) / FA_KB;
  const int wfirst = rfl(q0 + 32 * w), wlast = rfl(min(T - 1, wfirst + 31));   // wave-uniform
  const i32x4_t rk = dma_rsrc((const void*)(k.h() + (long long)bb * T * k.cols), (long long)T * k.cols * 2);
  const i32x4_t rv = dma_rsrc((const void*)(v.h() + (long long)bb * T * v.cols), (long long)T * v.cols * 2);
  LDS uint16_t* lds = (LDS uint16_t*)c.smem;
  constexpr int ST = 2 * FA_KB * HD;                       // elements per stage: K then V
  static_assert(NS * ST * 2 <= KVM_LDS_BYTES, "LDS");
  auto issue = [&](int blk) {
    LDS uint16_t* d = lds + (blk % NS) * ST;
    L::template issue<false, HP>(d, rk, blk * FA_KB, k.cols, kvh * HD, T - 1);
    L::template issue<true, HP>(d + FA_KB * HD, rv, blk * FA_KB, v.cols, kvh * HD, T - 1);
  };
  auto scores = [&](int blk, f32x16 (&s)[2]) {
    const LDS uint16_t* Ks = lds + (blk % NS) * ST;
#pragma unroll
    for (int sb = 0; sb < 2; ++sb) {
      s[sb] = f32x16{};
#pragma unroll
      for (int kk = 0; kk < NKK; ++kk) s[sb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(L::frag_kc(Ks, sb * 32, kk), qf[kk], s[sb], 0, 0, 0);
    }
  };
  f32x16 oacc[NDB];
#pragma unroll
  for (int d = 0; d < NDB; ++d) oacc[d] = f32x16{};
  float m = -INFINITY, lsum = 0.f;                         // m in units of sl2 * score
  // One iteration: wait for block kb + 1, issue block kb + NS - 1, then (unless every key of block kb is after this
  // wave's queries) the mask of a diagonal block and the rescale, each behind a wave-uniform branch, and one
  // straight-line part: the fragment reads of block kb + 1's K and block kb's V, the softmax of kb, the scores of kb + 1
  // and P V of kb. The scores of kb + 1 are computed even where the wave does not use them (its last block), so that
  // the part has no branch and the scheduler can place the VALU softmax between the MFMAs. The barrier and the loads
  // are outside every per-wave condition.
  auto step = [&](int kb, f32x16 (&sa)[2], f32x16 (&sn)[2]) {
    if (kb + 1 < nkb) wait_vm(min(NS - 3, nkb - 2 - kb) * 2 * L::NL);
    __syncthreads();
    if (kb + NS - 1 < nkb) issue(kb + NS - 1);
    if (kb * FA_KB > wlast) return;                        // every key of the block is after this wave's queries
    if (kb * FA_KB + FA_KB - 1 > wfirst) {                 // a diagonal block: mask keys after each query
#pragma unroll
      for (int sb = 0; sb < 2; ++sb)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (kb * FA_KB + sb * 32 + 8 * (r >> 2) + 4 * g + (r & 3) > qrow) sa[sb][r] = -INFINITY;
    }
    float mx = sa[0][0];
#pragma unroll
    for (int sb = 0; sb < 2; ++sb)
#pragma unroll
      for (int r = 0; r < 16; ++r) mx = fmaxf(mx, sa[sb][r]);
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64)) * sl2;
    if (__ballot(mx > m + moved)) {                          // wave-uniform: some query's maximum moved far enough
      const float mn = fmaxf(m, mx), f = fa_exp<HP>(m - mn);
      lsum *= f;
#pragma unroll
      for (int d = 0; d < NDB; ++d) oacc[d] *= f;
      m = mn;
    }
    const LDS uint16_t* Kn = lds + ((kb + 1) % NS) * ST;
    const LDS uint16_t* Vs = lds + (kb % NS) * ST + FA_KB * HD;
    bf16x8 kfr[2][NKK], vfr[NDB][2][2];
#pragma unroll
    for (int sb = 0; sb < 2; ++sb)
#pragma unroll
      for (int kk = 0; kk < NKK; ++kk) kfr[sb][kk] = L::frag_kc(Kn, sb * 32, kk);
#pragma unroll
    for (int d = 0; d < NDB; ++d)
#pragma unroll
      for (int sb = 0; sb < 2; ++sb)
#pragma unroll
        for (int t = 0; t < 2; ++t) vfr[d][sb][t] = L::frag_tr(Vs, d * 32, sb * 32 + 16 * t);
    float ps = 0.f;
    Pieces<HP ? 3 : 1> pf[2][2];
#pragma unroll
    for (int sb = 0; sb < 2; ++sb)
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        float pv[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) { pv[i] = fa_exp<HP>(__builtin_fmaf(sa[sb][8 * t + i], sl2, -m)); ps += pv[i]; }
        pf[sb][t] = split_bf16<HP ? 3 : 1>(pv);
      }
#pragma unroll
    for (int sb = 0; sb < 2; ++sb) {
      sn[sb] = f32x16{};
#pragma unroll
      for (int kk = 0; kk < NKK; ++kk) sn[sb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kfr[sb][kk], qf[kk], sn[sb], 0, 0, 0);
    }
    lsum += ps + __shfl_xor(ps, 32, 64);
#pragma unroll
    for (int d = 0; d < NDB; ++d)
#pragma unroll
      for (int sb = 0; sb < 2; ++sb)
#pragma unroll
        for (int t = 0; t < 2; ++t) oacc[d] = mfma_pieces(vfr[d][sb][t], pf[sb][t], oacc[d]);
  };
  __syncthreads();                                         // the previous task may still read this LDS
#pragma unroll
  for (int p = 0; p < NS - 1; ++p)
    if (p < nkb) issue(p);
  wait_vm(min(NS - 2, nkb - 1) * 2 * L::NL);
  __syncthreads();
  f32x16 s0[2], s1[2];
  scores(0, s0);                                           // block 0 holds key 0 <= every query of the task
  int kb = 0;
  for (; kb + 1 < nkb; kb += 2) { step(kb, s0, s1); step(kb + 1, s1, s0); }
  if (kb < nkb) step(kb, s0, s1);
  const float inv = 1.f / lsum;
  if constexpr (HP) {
    float nf = 0.f;                                        // 0 unless some result of this query is not finite
#pragma unroll
    for (int d = 0; d < NDB; ++d)
#pragma unroll
      for (int r = 0; r < 16; ++r) nf += oacc[d][r] * inv * 0.f;
    if (fa_any(c, qok && !(nf == 0.f && fabsf(m) < INFINITY))) return true;
  }
  if (qok) {
    GLOBAL uint16_t* orow = o.h() + ((long long)bb * T + qrow) * o.cols + h * HD + 4 * g;
#pragma unroll
    for (int d = 0; d < NDB; ++d)
#pragma unroll
      for (int rq = 0; rq < 4; ++rq)
        stwt_bf4(orow + d * 32 + 8 * rq, oacc[d][4 * rq] * inv, oacc[d][4 * rq + 1] * inv, oacc[d][4 * rq + 2] * inv, oacc[d][4 * rq + 3] * inv);
    if (g == 0) stwt32(lse.f() + (((long long)bb * H + h) * T + qrow), HP ? m + logf(lsum) : (m + log2f(lsum)) * 0.6931471805599453f);
  }
  return false;
}


// dQ for 128 queries of head h (op 47): lane l of wave w owns query q0 + 32w + l%32.
//   S^T = K Q^T, dP^T = V dO^T (K, V from kc LDS copies; Q, dO in registers), P^T = exp(S^T*scale - lse),
//   dS^T = P^T (dP^T - delta), dQ^T += K^T dS^T (K^T from a tr LDS copy), dq = scale * dQ.
template <int HD, bool HP = false> __device__ __noinline__ bool attn_dq_mfma(const Ctx& c) {
  constexpr int KB = HD > 64 ? 32 : FA_KB;                 // rows per block (three operand copies and FA_NS stages in LDS)
  typedef FaL<HD, KB> L;
  constexpr int NKK = HD / 16, NDB = HD / 32, BK = KB * HD, ST = 3 * BK;
  static_assert(FA_NS * ST * 2 <= KVM_LDS_BYTES, "LDS");
  const View q = uview(c, 0), k = uview(c, 1), v = uview(c, 2), dO = uview(c, 3), lse = uview(c, 4), delta = uview(c, 5), dq = uview(c, 6);
  const int bb = rfl(c.i(7)), h = rfl(c.i(8)), q0 = rfl(c.i(9)), T = rfl(c.i(10)), H = rfl(c.i(11)), Hkv = rfl(c.i(12));
  const float sc = __int_as_float(rfl(__float_as_int(c.f(14)))), sl2 = HP ? sc : sc * 1.4426950408889634f;
  const int w = wave(), l = lane(), g = l >> 5, qi = l & 31;
  const int qrow = q0 + 32 * w + qi, kvh = h / (H / Hkv);
  const bool qok = qrow < T;
  const long long grow = (long long)bb * T + qrow;
  bf16x8 qf[NKK], df[NKK];
#pragma unroll
  for (int kk = 0; kk < NKK; ++kk) {
    qf[kk] = qok ? *(const GLOBAL bf16x8*)(q.h() + grow * q.cols + h * HD + kk * 16 + 8 * g) : bf16x8{};
    df[kk] = qok ? *(const GLOBAL bf16x8*)(dO.h() + grow * dO.cols + h * HD + kk * 16 + 8 * g) : bf16x8{};
  }
  const float l2 = qok ? lse.f()[((long long)bb * H + h) * T + qrow] * (HP ? 1.f : 1.4426950408889634f) : 0.f;
  const float di = qok ? delta.f()[((long long)bb * H + h) * T + qrow] : 0.f;
  const int kend = min(T, q0 + 128), nkb = (kend + KB - 1) / KB;
  const int wlast = min(T - 1, q0 + 32 * w + 31);
  const i32x4_t rk = dma_rsrc((const void*)(k.h() + (long long)bb * T * k.cols), (long long)T * k.cols * 2);
  const i32x4_t rv = dma_rsrc((const void*)(v.h() + (long long)bb * T * v.cols), (long long)T * v.cols * 2);
  LDS uint16_t* lds = (LDS uint16_t*)c.smem;
  auto issue = [&](int blk) {
    LDS uint16_t* d = lds + (blk % FA_NS) * ST;
    L::template issue<false, HP>(d, rk, blk * KB, k.cols, kvh * HD, T - 1);
    L::template issue<true, HP>(d + BK, rk, blk * KB, k.cols, kvh * HD, T - 1);
    L::template issue<false, HP>(d + 2 * BK, rv, blk * KB, v.cols, kvh * HD, T - 1);
  };
  f32x16 acc[NDB];
#pragma unroll
  for (int d = 0; d < NDB; ++d) acc[d] = f32x16{};
  __syncthreads();
#pragma unroll
  for (int p = 0; p < FA_NS - 1; ++p) if (p < nkb) issue(p);
  for (int kb = 0; kb < nkb; ++kb) {
    wait_vm(min(FA_NS - 2, nkb - 1 - kb) * 3 * L::NL);
    __syncthreads();
    if (kb + FA_NS - 1 < nkb) issue(kb + FA_NS - 1);
    if (kb * KB > wlast) continue;
    const LDS uint16_t* Kc = lds + (kb % FA_NS) * ST;
    const LDS uint16_t* Kt = Kc + BK;
    const LDS uint16_t* Vc = Kc + 2 * BK;
#pragma unroll
    for (int sb = 0; sb < KB / 32; ++sb) {
      f32x16 sv = f32x16{}, dp = f32x16{};
#pragma unroll
      for (int kk = 0; kk < NKK; ++kk) {
        sv = __builtin_amdgcn_mfma_f32_32x32x16_bf16(L::frag_kc(Kc, sb * 32, kk), qf[kk], sv, 0, 0, 0);
        dp = __builtin_amdgcn_mfma_f32_32x32x16_bf16(L::frag_kc(Vc, sb * 32, kk), df[kk], dp, 0, 0, 0);
      }
      Pieces<HP ? 3 : 1> dsf[2];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        float d8[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int r = 8 * t + i, key = kb * KB + sb * 32 + 8 * (r >> 2) + 4 * g + (r & 3);
          const float pr = key > qrow ? 0.f : fa_exp<HP>(sv[r] * sl2 - l2);
          d8[i] = pr * (dp[r] - di);
        }
        dsf[t] = split_bf16<HP ? 3 : 1>(d8);
      }
#pragma unroll
      for (int d = 0; d < NDB; ++d)
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const bf16x8 kt = L::frag_tr(Kt, d * 32, sb * 32 + 16 * t);
          acc[d] = mfma_pieces(kt, dsf[t], acc[d]);
        }
    }
  }
  if constexpr (HP) {
    float nf = 0.f;
#pragma unroll
    for (int d = 0; d < NDB; ++d)
#pragma unroll
      for (int r = 0; r < 16; ++r) nf += acc[d][r] * sc * 0.f;
    if (fa_any(c, qok && !(nf == 0.f))) return true;
  }
  if (qok) {
    GLOBAL uint16_t* orow = dq.h() + grow * dq.cols + h * HD + 4 * g;
#pragma unroll
    for (int d = 0; d < NDB; ++d)
#pragma unroll
      for (int rq = 0; rq < 4; ++rq)
        stwt_bf4(orow + d * 32 + 8 * rq, acc[d][4 * rq] * sc, acc[d][4 * rq + 1] * sc, acc[d][4 * rq + 2] * sc, acc[d][4 * rq + 3] * sc);
  }
  return false;
}

// dK / dV for 128 keys of kv head kvh (op 48), summed over the heads of its GQA group and every later query: lane l
// of wave w owns key k0 + 32w + l%32.
//   S = Q K^T, dP = dO V^T (Q, dO from kc LDS copies; K, V in registers), P = exp(S*scale - lse[q]),
//   dS = P (dP - delta[q]), dV^T += dO^T P, dK^T += Q^T dS (dO^T, Q^T from tr LDS copies), dk = scale * dK.
// lse / delta of the staged queries are loaded into LDS by one direct load per wave: 8 lanes of 16 bytes, in the HP form
// KB / 2 lanes of 4 bytes.
template <int HD, bool HP = false> __device__ __noinline__ bool attn_dkv_mfma(const Ctx& c) {
  constexpr int KB = HD > 64 ? 32 : FA_KB;
  typedef FaL<HD, KB> L;
  constexpr int NKK = HD / 16, NDB = HD / 32, BK = KB * HD, ST = 4 * BK + 2 * KB * 2;   // + lse, delta (f32)
  static_assert(FA_NS * ST * 2 <= KVM_LDS_BYTES, "LDS");
  const View q = uview(c, 0), k = uview(c, 1), v = uview(c, 2), dO = uview(c, 3), lse = uview(c, 4), delta = uview(c, 5);
  const View dk = uview(c, 6), dv = uview(c, 7);
  const int bb = rfl(c.i(8)), kvh = rfl(c.i(9)), k0 = rfl(c.i(10)), T = rfl(c.i(11)), H = rfl(c.i(12));
  const float sc = __int_as_float(rfl(__float_as_int(c.f(14)))), sl2 = HP ? sc : sc * 1.4426950408889634f;
  const int G = H / (k.cols / HD);
  const int w = wave(), l = lane(), g = l >> 5, ki = l & 31;
  const int krow = k0 + 32 * w + ki;
  const bool kok = krow < T;
  const long long grow = (long long)bb * T + krow;
  bf16x8 kf[NKK], vf[NKK];
#pragma unroll
  for (int kk = 0; kk < NKK; ++kk) {
    kf[kk] = kok ? *(const GLOBAL bf16x8*)(k.h() + grow * k.cols + kvh * HD + kk * 16 + 8 * g) : bf16x8{};
    vf[kk] = kok ? *(const GLOBAL bf16x8*)(v.h() + grow * v.cols + kvh * HD + kk * 16 + 8 * g) : bf16x8{};
  }
  const int qb0 = k0 / KB, nqb = (T + KB - 1) / KB - qb0, nit = G * nqb;
  const int wfirst = k0 + 32 * w;                          // this wave's first key: queries before it see none of its keys
  const i32x4_t rq = dma_rsrc((const void*)(q.h() + (long long)bb * T * q.cols), (long long)T * q.cols * 2);
  const i32x4_t rd = dma_rsrc((const void*)(dO.h() + (long long)bb * T * dO.cols), (long long)T * dO.cols * 2);
  LDS uint16_t* lds = (LDS uint16_t*)c.smem;
  auto issue = [&](int it) {
    const int hh = kvh * G + it / nqb, qb = qb0 + it % nqb;
    LDS uint16_t* d = lds + (it % FA_NS) * ST;
    L::template issue<false, HP>(d, rq, qb * KB, q.cols, hh * HD, T - 1);
    L::template issue<true, HP>(d + BK, rq, qb * KB, q.cols, hh * HD, T - 1);
    L::template issue<false, HP>(d + 2 * BK, rd, qb * KB, dO.cols, hh * HD, T - 1);
    L::template issue<true, HP>(d + 3 * BK, rd, qb * KB, dO.cols, hh * HD, T - 1);
    // lse / delta: wave 0, 1 -> the halves of lse; wave 2, 3 -> delta; 16 bytes per lane, or 4 where a row's length
    // leaves the sequence's values unaligned
    const View& src = w < 2 ? lse : delta;
    const i32x4_t rs = dma_rsrc((const void*)(src.f() + ((long long)bb * H + hh) * T), (long long)T * 4);
    if constexpr (HP) {
      if (l < KB / 2) dma4(rs, min(qb * KB + KB / 2 * (w & 1) + l, T - 1) * 4, 0, d + 4 * BK + (w >> 1) * (2 * KB) + (w & 1) * KB);
    } else if (l < 8)
      dma16(rs, (qb * KB + 32 * (w & 1) + 4 * l) * 4, 0, d + 4 * BK + (w >> 1) * 128 + (w & 1) * 64);
  };
  f32x16 adk[NDB], adv[NDB];
#pragma unroll
  for (int d = 0; d < NDB; ++d) { adk[d] = f32x16{}; adv[d] = f32x16{}; }
  constexpr int NLS = 4 * L::NL + 1;
  __syncthreads();
#pragma unroll
  for (int p = 0; p < FA_NS - 1; ++p) if (p < nit) issue(p);
  for (int it = 0; it < nit; ++it) {
    wait_vm(min(FA_NS - 2, nit - 1 - it) * NLS);
    __syncthreads();
    if (it + FA_NS - 1 < nit) issue(it + FA_NS - 1);
    const int qb = qb0 + it % nqb;
    if (qb * KB + KB - 1 < wfirst) continue;          // every query of the block is before this wave's keys
    const LDS uint16_t* Qc = lds + (it % FA_NS) * ST;
    const LDS uint16_t* Qt = Qc + BK;
    const LDS uint16_t* Dc = Qc + 2 * BK;
    const LDS uint16_t* Dt = Qc + 3 * BK;
    const LDS float* Ls = (const LDS float*)(Qc + 4 * BK);
    const LDS float* Es = Ls + KB;
#pragma unroll
    for (int sb = 0; sb < KB / 32; ++sb) {
      f32x16 sv = f32x16{}, dp = f32x16{};
#pragma unroll
      for (int kk = 0; kk < NKK; ++kk) {
        sv = __builtin_amdgcn_mfma_f32_32x32x16_bf16(L::frag_kc(Qc, sb * 32, kk), kf[kk], sv, 0, 0, 0);
        dp = __builtin_amdgcn_mfma_f32_32x32x16_bf16(L::frag_kc(Dc, sb * 32, kk), vf[kk], dp, 0, 0, 0);
      }
      Pieces<HP ? 3 : 1> pf[2], dsf[2];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        float p8[8], d8[8];
#pragma unroll
        for (int i4 = 0; i4 < 2; ++i4) {
          const int ql = sb * 32 + 8 * (2 * t + i4) + 4 * g;      // first of 4 consecutive queries in this register group
          const f32x4n lq = *(const LDS f32x4n*)(Ls + ql), eq = *(const LDS f32x4n*)(Es + ql);
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const int r = 8 * t + 4 * i4 + j, qq = qb * KB + ql + j;
            const float pr = qq < krow || (HP && qq >= T) ? 0.f : fa_exp<HP>(sv[r] * sl2 - lq[j] * (HP ? 1.f : 1.4426950408889634f));
            p8[4 * i4 + j] = pr;
            d8[4 * i4 + j] = pr * (dp[r] - eq[j]);
          }
        }
        pf[t] = split_bf16<HP ? 3 : 1>(p8);
        dsf[t] = split_bf16<HP ? 3 : 1>(d8);
      }
#pragma unroll
      for (int d = 0; d < NDB; ++d)
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const bf16x8 dt = L::frag_tr(Dt, d * 32, sb * 32 + 16 * t), qt = L::frag_tr(Qt, d * 32, sb * 32 + 16 * t);
          adv[d] = mfma_pieces(dt, pf[t], adv[d]);
          adk[d] = mfma_pieces(qt, dsf[t], adk[d]);
        }
    }
  }
  if constexpr (HP) {
    float nf = 0.f;
#pragma unroll
    for (int d = 0; d < NDB; ++d)
#pragma unroll
      for (int r = 0; r < 16; ++r) nf += (adk[d][r] * sc + adv[d][r]) * 0.f;
    if (fa_any(c, kok && !(nf == 0.f))) return true;
  }
  if (kok) {
    GLOBAL uint16_t* kr = dk.h() + grow * dk.cols + kvh * HD + 4 * g;
    GLOBAL uint16_t* vr = dv.h() + grow * dv.cols + kvh * HD + 4 * g;
#pragma unroll
    for (int d = 0; d < NDB; ++d)
#pragma unroll
      for (int rq = 0; rq < 4; ++rq) {
        stwt_bf4(kr + d * 32 + 8 * rq, adk[d][4 * rq] * sc, adk[d][4 * rq + 1] * sc, adk[d][4 * rq + 2] * sc, adk[d][4 * rq + 3] * sc);
        stwt_bf4(vr + d * 32 + 8 * rq, adv[d][4 * rq], adv[d][4 * rq + 1], adv[d][4 * rq + 2], adv[d][4 * rq + 3]);
      }
  }
  return false;
}

}  // namespace kvm
