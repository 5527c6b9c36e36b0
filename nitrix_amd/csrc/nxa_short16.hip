// 16-bit attention of short sequences (at most kShortMax queries and keys,
// head dims up to 64): windowed attention and small layers.
//
// Same math as the tuned kernels (nxa_fwd16.h, nxa_bwd16.h) and the
// reference's Pallas kernels (src/nitrix/_kernels/cuda/attention.py:85-156
// forward, :272-332 dK/dV, :335-387 dQ, :517-544 the sum of dbias over
// broadcast axes).
//
// The tuned kernels stream tiles past 128- or 256-row blocks, one barrier a
// tile; at a few hundred rows their prologue, the padding to whole blocks
// and the shared barriers cost more than the products.  Here one side of
// the problem (K and V, or Q and dO) fits the LDS whole: a block copies it
// once, passes one barrier, and its four waves then take 32-row strips of
// the other side independently, so waves of one SIMD overlap matrix and
// vector work without any schedule, and a (batch, head) pair is split over
// as many blocks as the chip needs.  Head dims up to 32 run at a padded width
// of 32 (half the products and LDS bytes of the 64 the tuned kernels pad to).
//
// A bias shared by many pairs (a window's relative position bias) is packed
// once per call into the accumulator layout of the score products, as fp32
// bias / scale, 4 KB per 32 x 32 block: a wave then reads its block with
// four coalesced 16-byte loads straight into the accumulators that K Q^T adds
// to, at any alignment, length or dtype of the caller's bias.
//
// dbias of such a bias is a sum over pairs.  Writing fp32 partials per pair
// costs 8 bytes of traffic per score; recomputing the scores costs two
// products and one exponential.  dbias_pairs_kernel therefore owns a block
// of the bias, walks its pairs recomputing dS, and keeps the sum in
// registers; the pairs are cut into a few ranges whose sums a last pass
// adds in a fixed order (deterministic).
//
// Measured (bf16, a bias [4, 343, 343] shared by 512 windows, head dim 32,
// forward + backward): 4.62 ms on the general kernels (dK/dV 3.0 in twelve
// launches with 284 us of reductions, the forward 0.78, dQ 0.55, both at
// one bias element per load), 0.42 here: packs 2 x 5 us, forward 104, dQ 115,
// dK/dV 128, dbias 112, its sum 7.  Without a bias (B 8, H 32, head dim 64,
// forward + backward on the GPU): 256 x 256 52 -> 42 us, 512 x 512 131 ->
// 118; a lone 512 x 512 call of 16 heads 43 -> 42.  The four kernels of the
// windowed call are bound by VALU issue (one exponential and about five
// operations per score): VALU instructions are in issue 54 to 60 % of the
// SIMDs' cycles at two or three waves a SIMD, the matrix cores 16 to 27 %.
#include "nxa_fwd16.h"
#include "nxa_launch.h"

#include <type_traits>

namespace nxa {

namespace {

// Resident bytes above which a block takes 8 waves instead of 4: with fewer
// than three 4-wave blocks sharing a CU's 160 KB its SIMDs would hold one or
// two waves (B 8, H 32, 512 x 512, head dim 64, forward: 47.9 us with 4
// waves, 31.7 with 8).  Below kShortFewBlocks blocks 4-wave ones spread over
// more CUs (16 heads, forward + backward: 49.9 us with 8, 41.6 with 4).
constexpr size_t kShortWideLds = 53 * 1024;
constexpr int kShortFewBlocks = 256;

// LDS word holding the 64-key keep bits of a tile (mask and key tail).
struct KeepBits {
  uint32_t lo, hi;
  __device__ __forceinline__ bool any() const { return (lo | hi) != 0; }
  __device__ __forceinline__ bool all() const { return (lo & hi) == 0xffffffffu; }
};

// Keep bits of keys k0 .. k0 + 63 of pair (b, h) under the key range and the
// query-broadcast mask (the only masks these kernels take).
__device__ __forceinline__ uint64_t keep_bits(const Params& p, int b, int h, int k0, int lane) {
  const int key = k0 + lane;
  bool keep = key < p.Lk;
  if (keep && p.has_mask) keep = p.mask[b * p.mask_str[0] + h * p.mask_str[1] + key] != 0;
  return __ballot(keep);
}

// Copies an [nrows, D] 16-bit matrix (row stride rs) into ntile swizzled
// [64 x DP] LDS tiles, the block's waves taking 1 KB copies in turn.  Rows
// past nrows and head-dim chunks past D are addressed outside the range and
// land as zeros.
template <int DP, int NW, typename T>
__device__ __forceinline__ void load_resident(const T* src, int64_t rs, int nrows, int ntile,
                                              int D, uint32_t lds, int wave, int lane) {
  constexpr int SPR = DP / 8;  // 16-byte slots per row
  const i32x4 r = make_rsrc(src, (uint32_t)(((int64_t)(nrows - 1) * rs + D) * 2));
  for (int m = wave; m < ntile * SPR; m += NW) {
    const int s = m * 64 + lane, row = s / SPR;
    const int ch = (s % SPR) ^ swz<DP>(row);
    const uint32_t off = row < nrows && ch * 8 < D ? 2u * (uint32_t)(row * (int)rs + ch * 8)
                                                   : 0xfffffff0u;
    dma16_buf(r, off, lds + m * 1024);
  }
}

// Row fragments of one 32-row strip of a [n, D] matrix in memory.
template <int NC, typename T>
__device__ __forceinline__ void strip_frags(typename Mma<T>::Frag (&f)[NC], const T* row, bool ok,
                                            int D, int g) {
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int d = c * 16 + g * 8;
    f[c] = ok && d < D ? ld16(row + d) : zero_frag<T>();
  }
}

// Packed bias block (32 x 32) as a score accumulator.
__device__ __forceinline__ f32x16 packed_block(const float* base, int64_t blk, int lane) {
  const f32x4* b = reinterpret_cast<const f32x4*>(base) + blk * 256 + lane;
  f32x16 r;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const f32x4 v = b[c * 64];
#pragma unroll
    for (int j = 0; j < 4; ++j) r[4 * c + j] = v[j];
  }
  return r;
}

__device__ __forceinline__ int bias_slot(const ShortParams& s, int b, int h) {
  return (s.OB > 1 ? b : 0) * s.OH + (s.OH > 1 ? h : 0);
}

// Keeps x where its key is kept (bit 8 (r / 4) + r % 4 of w: the lane
// half's keep bits) and, for CAUSAL, key <= query.
template <bool CAUSAL>
__device__ __forceinline__ void mask_block(f32x16& x, uint32_t w, int key0, int qrow) {
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int o = 8 * (r >> 2) + (r & 3);
    bool keep = (w >> o) & 1;
    if (CAUSAL) keep = keep && key0 + o <= qrow;
    x[r] = keep ? x[r] : -INFINITY;
  }
}

// Logits beyond this magnitude (log2 units) step by more than one unit in
// fp32: a product of which only one side is rounded (the exponent's FMA
// against a rounded reference) would be off by whole powers of two there, up
// to 2^64 at a bias of -1e9.  Both sides are then rounded alike.
constexpr float kBigLogit = 16777216.f;

// x cc + r with x cc rounded first (no contraction).
__device__ __forceinline__ float rounded_fma(float x, float cc, float r) {
#pragma clang fp contract(off)
  const float y = x * cc;
  return y + r;
}

// Exponents of a block's P from its scores x and -lse log2(e) of row r in
// nl(r).  BIG (some row's lse is beyond kBigLogit: masked throughout by a
// large finite bias): x cc is rounded as the reference was, and the exponent
// is held at 0, as no P is larger than 1 (a NaN stays one).
template <bool BIG, typename NL>
__device__ __forceinline__ void p_exponents(f32x16& x, float cc, NL&& nl) {
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    if constexpr (BIG) {
      const float e = rounded_fma(x[r], cc, nl(r));
      x[r] = e > 0.f ? 0.f : e;
    } else {
      x[r] = __builtin_fmaf(x[r], cc, nl(r));
    }
  }
}

// ---------------------------------------------------------------------------
// Packs bias / scale (fp32) into accumulator blocks.  One block of threads
// per 32 x 32 block; blockIdx.y 0 writes the S^T layout (lane = query, rows
// = keys; keys past Lk are -inf, which masks the tail), 1 the S layout
// (lane = key, rows = queries).  Finite biases whose quotient would overflow
// (or leave no room for the products) are mapped, in order and apart, onto
// [2^127, 2^128): a row masked throughout with the type's lowest value stays
// a row of equal finite logits, and a larger one in it still wins.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void bias_pack_kernel(const Params p, const ShortParams s) {
  const int lane = threadIdx.x & 63, c = threadIdx.x >> 6;
  const int g = lane >> 5, c32 = lane & 31;
  const int blk = blockIdx.x;
  const int kb = blk % s.nkb, qb = (blk / s.nkb) % s.nqb, slot = blk / (s.nkb * s.nqb);
  const int ob = slot / s.OH, oh = slot % s.OH;
  const bool rowmajor = blockIdx.y == 1;
  f32x4 v;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int o = 8 * c + 4 * g + j;
    const int q = qb * 32 + (rowmajor ? o : c32), key = kb * 32 + (rowmajor ? c32 : o);
    float x = key < p.Lk || rowmajor ? 0.f : -INFINITY;
    if (q < p.Lq && key < p.Lk) {
      const float bv = load_elem(p.bias_dtype, p.bias,
                                 ob * p.bias_str[0] + oh * p.bias_str[1] +
                                     (int64_t)q * p.bias_str[2] + key);
      x = bv * s.inv_scale;
      const float half = 1.70141183e38f;  // 2^127
      if (__builtin_isfinite(bv) && !(fabsf(x) <= half))
        x = __builtin_copysignf(__builtin_fmaf(0.499f, fabsf(bv), half), bv);
    }
    v[j] = x;
  }
  float* dst = rowmajor ? s.pack_s : s.pack_st;
  reinterpret_cast<f32x4*>(dst)[(int64_t)blk * 256 + c * 64 + lane] = v;
}

// ---------------------------------------------------------------------------
// Forward: K and V resident, waves take 32-query strips.
// ---------------------------------------------------------------------------
template <typename T, int DP, int NW, bool HAS_BIAS, bool CAUSAL>
__global__ __launch_bounds__(NW * 64, 2) void fwd_short_kernel(const Params p, const ShortParams sp) {
  using M = Mma<T>;
  using Frag = typename M::Frag;
  constexpr int NC = DP / 16, NDB = DP / 32, FPB = M::FRAGS_PER_BLOCK;
  constexpr int TILE_BYTES = 64 * DP * 2, HALF = 32 * DP * 2;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  __shared__ uint32_t kbits[2 * kShortMax / 64];

  const int vid = xcd_remap(blockIdx.x, p.B * p.H, sp.nsplit);
  const int bh = vid / sp.nsplit, part = vid % sp.nsplit;
  const int b = bh / p.H, h = bh % p.H;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 5, c32 = lane & 31;
  const int nkt = (p.Lk + 63) / 64, nst = (p.Lq + 31) / 32;
  const uint32_t k_lds = lds_offset(smem), v_lds = k_lds + nkt * TILE_BYTES;

  load_resident<DP, NW>((const T*)p.k + b * p.k_str[0] + h * p.k_str[1], p.k_str[2], p.Lk, nkt, p.D,
                    k_lds, wave, lane);
  load_resident<DP, NW>((const T*)p.v + b * p.v_str[0] + h * p.v_str[1], p.v_str[2], p.Lk, nkt, p.Dv,
                    v_lds, wave, lane);
  for (int t = wave; t < nkt; t += NW) {
    const uint64_t m = keep_bits(p, b, h, t * 64, lane);
    if (lane < 2) kbits[2 * t + lane] = (uint32_t)(m >> (32 * lane));
  }
  Resident<T, DP> rd;
  rd.init(lane);
  __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
  __syncthreads();

  const float cc = p.scale_log2;
  for (int st = part * NW + wave; st < nst; st += sp.nsplit * NW) {
    const int q0 = st * 32, qrow = q0 + c32;
    const bool qok = qrow < p.Lq;
    const int qc = qok ? qrow : p.Lq - 1;
    Frag qf[NC];
    strip_frags(qf, (const T*)p.q + b * p.q_str[0] + h * p.q_str[1] + (int64_t)qc * p.q_str[2], qok,
                p.D, g);
    f32x16 oacc[NDB];
#pragma unroll
    for (int db = 0; db < NDB; ++db) oacc[db] = splat16(0.f);
    float m_ref = -INFINITY, l_i = 0.f;
    bool big = false;  // a biased row's reference is beyond kBigLogit
    const int64_t blk0 = HAS_BIAS ? ((int64_t)bias_slot(sp, b, h) * sp.nqb + st) * sp.nkb : 0;
    const int nk = CAUSAL ? min(nkt, (q0 + 31) / 64 + 1) : nkt;
    for (int kt = 0; kt < nk; ++kt) {
      const KeepBits kb2 = {(uint32_t)__builtin_amdgcn_readfirstlane((int)kbits[2 * kt]),
                            (uint32_t)__builtin_amdgcn_readfirstlane((int)kbits[2 * kt + 1])};
      if (!kb2.any()) continue;
      const int k0 = kt * 64;
      f32x16 S[2];
      if constexpr (HAS_BIAS) {
        S[0] = packed_block(sp.pack_st, blk0 + 2 * kt, lane);
        S[1] = packed_block(sp.pack_st, blk0 + 2 * kt + 1, lane);
      }
      const uint32_t kat = k_lds + kt * TILE_BYTES;
#pragma unroll
      for (int m = 0; m < NC; ++m)
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
          const Frag a = rd.row(kat + kb * HALF, m);
          if (!HAS_BIAS && m == 0) S[kb] = M::first(a, qf[m]);
          else M::run(S[kb], a, qf[m]);
        }
      // The packed bias carries the key tail; a mask or a bias-free tail
      // takes the keep bits.
      const bool diag = CAUSAL && k0 + 63 > q0;
      if (diag || (!kb2.all() && (!HAS_BIAS || p.has_mask))) {
        mask_block<CAUSAL>(S[0], kb2.lo >> (4 * g), k0 + 4 * g, qrow);
        mask_block<CAUSAL>(S[1], kb2.hi >> (4 * g), k0 + 32 + 4 * g, qrow);
      }
      // Softmax as in nxa_fwd16.h: the tile is taken against the reference
      // in force and redone with a raised one only when a half-row sum
      // leaves the fp16 range of P (or the row has no reference yet).
      Frag pf[2][FPB];
      auto exp_tile = [&](auto big_tag) NXA_INLINE -> float {
        const float neg_m = m_ref == -INFINITY ? 0.f : -m_ref;
        float ts = 0.f;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
          f32x16 pt;
          float rs[4];
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            pt[r] = fast_exp2(decltype(big_tag)::value ? rounded_fma(S[kb][r], cc, neg_m)
                                                       : __builtin_fmaf(S[kb][r], cc, neg_m));
            rs[r & 3] = r < 4 ? pt[r] : rs[r & 3] + pt[r];
          }
          ts += (rs[0] + rs[1]) + (rs[2] + rs[3]);
#pragma unroll
          for (int f = 0; f < FPB; ++f) pf[kb][f] = M::pack(pt, f);
        }
        return ts;
      };
      float ts = 0.f;
      bool redo = big || __any(m_ref == -INFINITY);
      if (!redo) {
        ts = exp_tile(std::false_type{});
        redo = __any(!(ts <= kFwdSumLimit));
      }
      if (redo) {
        float mt = -INFINITY;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
          for (int r = 0; r < 16; ++r) mt = fmaxf(mt, S[kb][r]);
        mt = half_max(mt) * cc;
        const bool raise = mt > m_ref + kFwdRescaleSlack;
        const float alpha = raise ? fast_exp2(m_ref - mt) : 1.f;
        m_ref = raise ? mt : m_ref;
        l_i *= alpha;
        if (__any(raise)) {
#pragma unroll
          for (int db = 0; db < NDB; ++db)
#pragma unroll
            for (int r = 0; r < 16; ++r) oacc[db][r] *= alpha;
        }
        big = HAS_BIAS && __any(m_ref != -INFINITY && fabsf(m_ref) > kBigLogit);
        ts = big ? exp_tile(std::true_type{}) : exp_tile(std::false_type{});
      }
      l_i += ts;
      const uint32_t vat = v_lds + kt * TILE_BYTES;
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int f = 0; f < FPB; ++f)
#pragma unroll
          for (int db = 0; db < NDB; ++db)
            M::run(oacc[db], rd.tr(vat + kb * HALF, f, db), pf[kb][f]);
    }
    const float l = l_i + shfl_xor32(l_i);
    const float inv = 1.0f / l;
    if (qok) {
      T* op = (T*)p.o + b * p.o_str[0] + h * p.o_str[1] + (int64_t)qrow * p.o_str[2];
#pragma unroll
      for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const int d0 = db * 32 + 8 * c + 4 * g;
          if (d0 < p.Dv) store4(op + d0, oacc[db], 4 * c, inv);
        }
      if (g == 0 && p.lse)
        p.lse[((int64_t)b * p.H + h) * p.Lq + qrow] = (m_ref + __log2f(l)) * kLn2;
    }
  }
}

// ---------------------------------------------------------------------------
// dQ: K and V resident, waves take 32-query strips.  Also writes the rows'
// -delta and -lse log2(e), which dK/dV and dbias read.
// ---------------------------------------------------------------------------
template <typename T, int DP, int NW, bool HAS_BIAS, bool CAUSAL>
__global__ __launch_bounds__(NW * 64, 2) void dq_short_kernel(const Params p, const ShortParams sp) {
  using M = Mma<T>;
  using Frag = typename M::Frag;
  constexpr int NC = DP / 16, NDB = DP / 32, FPB = M::FRAGS_PER_BLOCK;
  constexpr int TILE_BYTES = 64 * DP * 2, HALF = 32 * DP * 2;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  __shared__ uint32_t kbits[2 * kShortMax / 64];

  const int vid = xcd_remap(blockIdx.x, p.B * p.H, sp.nsplit);
  const int bh = vid / sp.nsplit, part = vid % sp.nsplit;
  const int b = bh / p.H, h = bh % p.H;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 5, c32 = lane & 31;
  const int nkt = (p.Lk + 63) / 64, nst = (p.Lq + 31) / 32;
  const uint32_t k_lds = lds_offset(smem), v_lds = k_lds + nkt * TILE_BYTES;

  load_resident<DP, NW>((const T*)p.k + b * p.k_str[0] + h * p.k_str[1], p.k_str[2], p.Lk, nkt, p.D,
                    k_lds, wave, lane);
  load_resident<DP, NW>((const T*)p.v + b * p.v_str[0] + h * p.v_str[1], p.v_str[2], p.Lk, nkt, p.Dv,
                    v_lds, wave, lane);
  for (int t = wave; t < nkt; t += NW) {
    const uint64_t m = keep_bits(p, b, h, t * 64, lane);
    if (lane < 2) kbits[2 * t + lane] = (uint32_t)(m >> (32 * lane));
  }
  Resident<T, DP> rd;
  rd.init(lane);
  __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
  __syncthreads();

  for (int st = part * NW + wave; st < nst; st += sp.nsplit * NW) {
    const int q0 = st * 32, qrow = q0 + c32;
    const bool qok = qrow < p.Lq;
    const int qc = qok ? qrow : p.Lq - 1;
    Frag qf[NC], df[NC];
    strip_frags(qf, (const T*)p.q + b * p.q_str[0] + h * p.q_str[1] + (int64_t)qc * p.q_str[2], qok,
                p.D, g);
    const int64_t oo = b * p.o_str[0] + h * p.o_str[1] + (int64_t)qc * p.o_str[2];
    strip_frags(df, (const T*)p.dout + oo, qok, p.Dv, g);
    float dacc = 0.f;
    {
      Frag of[NC];
      strip_frags(of, (const T*)p.o + oo, qok, p.Dv, g);
#pragma unroll
      for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int e = 0; e < 8; ++e) dacc = __builtin_fmaf((float)of[c][e], (float)df[c][e], dacc);
    }
    const int64_t rowid = ((int64_t)b * p.H + h) * p.Lq + qc;
    const float ndlt = -(dacc + shfl_xor32(dacc));
    const float nlse2 = -p.lse[rowid] * kLog2e;
    const bool big = HAS_BIAS && __any(fabsf(nlse2) > kBigLogit);
    if (qok && g == 0) {
      p.ndelta[rowid] = ndlt;
      p.nlse2[rowid] = nlse2;
    }
    // The dP products start from -delta (exact in fp32, no extra work: the
    // first product of every block reads it as its accumulator input).
    const f32x16 nd16 = splat16(ndlt);
    f32x16 dq[NDB];
#pragma unroll
    for (int db = 0; db < NDB; ++db) dq[db] = splat16(0.f);
    const int64_t blk0 = HAS_BIAS ? ((int64_t)bias_slot(sp, b, h) * sp.nqb + st) * sp.nkb : 0;
    const int nk = CAUSAL ? min(nkt, (q0 + 31) / 64 + 1) : nkt;
    const auto tiles = [&](auto big_tag) NXA_INLINE {
      for (int kt = 0; kt < nk; ++kt) {
        const KeepBits kb2 = {(uint32_t)__builtin_amdgcn_readfirstlane((int)kbits[2 * kt]),
                              (uint32_t)__builtin_amdgcn_readfirstlane((int)kbits[2 * kt + 1])};
        if (!kb2.any()) continue;
        const int k0 = kt * 64;
        const bool diag = CAUSAL && k0 + 63 > q0;
        const bool masked = diag || (!kb2.all() && (!HAS_BIAS || p.has_mask));
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
          const uint32_t kat = k_lds + kt * TILE_BYTES + kb * HALF;
          const uint32_t vat = v_lds + kt * TILE_BYTES + kb * HALF;
          f32x16 s, dp = nd16;
          if constexpr (HAS_BIAS) s = packed_block(sp.pack_st, blk0 + 2 * kt + kb, lane);
#pragma unroll
          for (int m = 0; m < NC; ++m) {
            const Frag a = rd.row(kat, m);
            if (!HAS_BIAS && m == 0) s = M::first(a, qf[m]);
            else M::run(s, a, qf[m]);
            M::run(dp, rd.row(vat, m), df[m]);
          }
          const auto row_nl = [&](int) NXA_INLINE { return nlse2; };
          p_exponents<decltype(big_tag)::value>(s, p.scale_log2, row_nl);
          if (masked)
            mask_block<CAUSAL>(s, (kb ? kb2.hi : kb2.lo) >> (4 * g), k0 + 32 * kb + 4 * g, qrow);
#pragma unroll
          for (int r = 0; r < 16; ++r) dp[r] = fast_exp2(s[r]) * dp[r];
#pragma unroll
          for (int f = 0; f < FPB; ++f) {
            const Frag pd = M::pack(dp, f);
#pragma unroll
            for (int db = 0; db < NDB; ++db) M::run(dq[db], rd.tr(kat, f, db), pd);
          }
        }
      }
    };
    if (big) tiles(std::true_type{});
    else tiles(std::false_type{});
    if (qok) {
      T* dqp = (T*)p.dq + b * p.q_str[0] + h * p.q_str[1] + (int64_t)qrow * p.q_str[2];
#pragma unroll
      for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const int d0 = db * 32 + 8 * c + 4 * g;
          if (d0 < p.D) store4(dqp + d0, dq[db], 4 * c, p.scale);
        }
    }
  }
}

// ---------------------------------------------------------------------------
// dK / dV: Q and dO resident (with their rows' -lse2 and -delta), waves take
// 32-key strips.  Rows past Lq read as zeros with -lse2 = -inf, so P = 0.
// (Four waves a SIMD at head dim 32: both loops' registers but for a few that
// are written out once a strip.)
// ---------------------------------------------------------------------------
template <typename T, int DP, int NW, bool HAS_BIAS, bool CAUSAL>
__global__ __launch_bounds__(NW * 64, DP == 32 && !CAUSAL ? 4 : 2) void dkdv_short_kernel(
    const Params p, const ShortParams sp) {
  using M = Mma<T>;
  using Frag = typename M::Frag;
  constexpr int NC = DP / 16, NDB = DP / 32, FPB = M::FRAGS_PER_BLOCK;
  constexpr int TILE_BYTES = 64 * DP * 2, HALF = 32 * DP * 2;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  __shared__ __attribute__((aligned(16))) float nl_s[kShortMax], nd_s[kShortMax];

  const int vid = xcd_remap(blockIdx.x, p.B * p.H, sp.nsplit);
  const int bh = vid / sp.nsplit, part = vid % sp.nsplit;
  const int b = bh / p.H, h = bh % p.H;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 5, c32 = lane & 31;
  const int nqt = (p.Lq + 63) / 64, nst = (p.Lk + 31) / 32;
  const uint32_t q_lds = lds_offset(smem), d_lds = q_lds + nqt * TILE_BYTES;

  load_resident<DP, NW>((const T*)p.q + b * p.q_str[0] + h * p.q_str[1], p.q_str[2], p.Lq, nqt, p.D,
                    q_lds, wave, lane);
  load_resident<DP, NW>((const T*)p.dout + b * p.o_str[0] + h * p.o_str[1], p.o_str[2], p.Lq, nqt, p.Dv,
                    d_lds, wave, lane);
  const int64_t row0 = ((int64_t)b * p.H + h) * p.Lq;
  bool far = false;  // a row's lse beyond kBigLogit
  for (int i = tid; i < nqt * 64; i += NW * 64) {
    nl_s[i] = i < p.Lq ? p.nlse2[row0 + i] : -INFINITY;
    nd_s[i] = i < p.Lq ? p.ndelta[row0 + i] : 0.f;
    if (HAS_BIAS) far = far || (i < p.Lq && fabsf(nl_s[i]) > kBigLogit);
  }
  Resident<T, DP> rd;
  rd.init(lane);
  __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
  bool big = false;
  if constexpr (HAS_BIAS) big = __syncthreads_or(far);
  else __syncthreads();

  const int nqb = (p.Lq + 31) / 32;
  for (int st = part * NW + wave; st < nst; st += sp.nsplit * NW) {
    const int key0 = st * 32, key = key0 + c32;
    bool keep = key < p.Lk;
    const bool kok = keep;
    const int kc = kok ? key : p.Lk - 1;
    if (keep && p.has_mask) keep = p.mask[b * p.mask_str[0] + h * p.mask_str[1] + key] != 0;
    Frag kf[NC], vf[NC];
    strip_frags(kf, (const T*)p.k + b * p.k_str[0] + h * p.k_str[1] + (int64_t)kc * p.k_str[2], kok,
                p.D, g);
    strip_frags(vf, (const T*)p.v + b * p.v_str[0] + h * p.v_str[1] + (int64_t)kc * p.v_str[2], kok,
                p.Dv, g);
    f32x16 dk[NDB], dv[NDB];
#pragma unroll
    for (int db = 0; db < NDB; ++db) dk[db] = dv[db] = splat16(0.f);
    const int64_t slot0 = HAS_BIAS ? (int64_t)bias_slot(sp, b, h) * sp.nqb : 0;
    const bool some = __any(keep), every = __all(keep);
    const auto blocks = [&](auto big_tag) NXA_INLINE {
      for (int qb = CAUSAL ? st : 0; qb < (some ? nqb : 0); ++qb) {
        const uint32_t qat = q_lds + qb * HALF, dat = d_lds + qb * HALF;
        f32x16 x, d;
        float nl[16];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const f32x4 l4 = *reinterpret_cast<const f32x4*>(nl_s + qb * 32 + 8 * c + 4 * g);
          const f32x4 d4 = *reinterpret_cast<const f32x4*>(nd_s + qb * 32 + 8 * c + 4 * g);
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            nl[4 * c + j] = l4[j];
            d[4 * c + j] = d4[j];
          }
        }
        if constexpr (HAS_BIAS) x = packed_block(sp.pack_s, (slot0 + qb) * sp.nkb + st, lane);
#pragma unroll
        for (int m = 0; m < NC; ++m) {
          const Frag a = rd.row(qat, m);
          if (!HAS_BIAS && m == 0) x = M::first(a, kf[m]);
          else M::run(x, a, kf[m]);
          M::run(d, rd.row(dat, m), vf[m]);
        }
        // (read late in the rare variant: registers)
        const auto row_nl = [&](int r) NXA_INLINE {
          return decltype(big_tag)::value ? nl_s[qb * 32 + 8 * (r >> 2) + 4 * g + (r & 3)] : nl[r];
        };
        p_exponents<decltype(big_tag)::value>(x, p.scale_log2, row_nl);
        if (!every || (CAUSAL && qb == st)) {
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            bool kp = keep;
            if (CAUSAL) kp = kp && key <= qb * 32 + 8 * (r >> 2) + 4 * g + (r & 3);
            x[r] = kp ? x[r] : -INFINITY;
          }
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          x[r] = fast_exp2(x[r]);
          d[r] = x[r] * d[r];
        }
#pragma unroll
        for (int f = 0; f < FPB; ++f) {
          const Frag pp = M::pack(x, f), pd = M::pack(d, f);
#pragma unroll
          for (int db = 0; db < NDB; ++db) {
            M::run(dv[db], rd.tr(dat, f, db), pp);
            M::run(dk[db], rd.tr(qat, f, db), pd);
          }
        }
      }
    };
    if (big) blocks(std::true_type{});
    else blocks(std::false_type{});
    if (kok) {
      T* dkp = (T*)p.dk + b * p.k_str[0] + h * p.k_str[1] + (int64_t)key * p.k_str[2];
      T* dvp = (T*)p.dv + b * p.v_str[0] + h * p.v_str[1] + (int64_t)key * p.v_str[2];
#pragma unroll
      for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const int d0 = db * 32 + 8 * c + 4 * g;
          if (d0 < p.D) store4(dkp + d0, dk[db], 4 * c, p.scale);
          if (d0 < p.Dv) store4(dvp + d0, dv[db], 4 * c, 1.0f);
        }
    }
  }
}

// ---------------------------------------------------------------------------
// dbias of a shared bias.  A block owns a 128-query block of the bias by 64
// keys (4 waves; head dim 32, three blocks a CU) or 128 keys (8 waves; head
// dim 64, one), a wave 64 x 32 of it, walks the pairs of its range
// that share the bias and sums their dS in registers; the packed bias stays
// in registers too (nothing in the loop may wait on a load of its own: loads
// complete in order, behind the copies in flight).  A pair's rows (Q, dO, K,
// V of the block, -lse2 and -delta) come by direct copies, one pair ahead.  Range r of every block writes slab r [OB, OH, Lq,
// Lkp].  The blocks that read the same pairs sit on one XCD.
// ---------------------------------------------------------------------------
template <int DP>
constexpr int kDbiasWaves = DP == 32 ? 4 : 8;

template <typename T, int DP, bool CAUSAL>
__global__ __launch_bounds__(kDbiasWaves<DP> * 64, DP == 32 ? 3 : 2) void dbias_pairs_kernel(const Params p, const ShortParams sp) {
  using M = Mma<T>;
  constexpr int NC = DP / 16, SPR = DP / 8, NST = 2;
  constexpr int NW = kDbiasWaves<DP>, BK = NW * 16;
  constexpr int MAT = 128 * DP * 2, KMAT = BK * DP * 2, HALF = 32 * DP * 2;
  constexpr int ROWV = 2 * MAT + 2 * KMAT, STAGE = ROWV + 4 * 256;
  constexpr int ROWS = 64 / SPR, PER = ROWS < 16 ? 16 / ROWS : 1;
  __shared__ __attribute__((aligned(16))) char smem[NST * STAGE];

  const int nq = (p.Lq + 127) / 128, nk = (p.Lk + BK - 1) / BK, tiles = nq * nk;
  const int x = blockIdx.x % 8, rest = blockIdx.x / 8;
  const int group = (rest / tiles) * 8 + x, tile = rest % tiles;
  if (group >= sp.OB * sp.OH * sp.nrange) return;
  const int slot = group / sp.nrange, range = group % sp.nrange;
  const int bq = tile / nk, bk = tile % nk;
  const int ob = slot / sp.OH, oh = slot % sp.OH;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 5, c32 = lane & 31;
  const int q0 = bq * 128 + (wave & 1) * 64, k0 = bk * BK + (wave >> 1) * 32;
  const int nB = sp.OB > 1 ? 1 : p.B, nH = sp.OH > 1 ? 1 : p.H;
  const int pairs = nB * nH;
  const int j0 = (int)((int64_t)pairs * range / sp.nrange);
  const int j1 = (int)((int64_t)pairs * (range + 1) / sp.nrange);
  // Blocks above the causal diagonal only write zeros.
  const bool tile_dead = CAUSAL && bk * BK > bq * 128 + 127;
  const bool dead = q0 >= p.Lq || k0 >= p.Lk || (CAUSAL && k0 > q0 + 63);
  const bool diag = CAUSAL && k0 + 31 > q0;

  // This wave's matrix: rows r0 .. of `src`, D columns, rs apart (with 8
  // waves, w and w + 4 half of its copies each).
  const int mat = wave & 3, half = wave >> 2;
  const bool kv = mat >= 2;
  const T* src = (const T*)(mat == 0 ? p.q : mat == 1 ? p.dout : mat == 2 ? p.k : p.v);
  const int64_t* str = mat == 0 ? p.q_str : mat == 1 ? p.o_str : mat == 2 ? p.k_str : p.v_str;
  const int64_t sb = str[0], sh = str[1], rs = str[2];
  const int r0 = kv ? bk * BK : bq * 128, L = kv ? p.Lk : p.Lq;
  const int D = mat == 0 || mat == 2 ? p.D : p.Dv;
  const int rows = min(kv ? BK : 128, L - r0);
  const int ncpy = (kv ? BK : 128) / ROWS / (NW / 4);  // copies of this wave
  const uint32_t bytes = (uint32_t)(((int64_t)(rows - 1) * rs + D) * 2);
  // Copy m covers rows m * ROWS ..; the swizzle repeats every 16 rows.
  // Columns past D and (by the range) rows past L land as zeros.
  uint32_t off[PER];
#pragma unroll
  for (int m = 0; m < PER; ++m) {
    const int row = m * ROWS + lane / SPR, ch = (lane % SPR) ^ swz<DP>(row);
    off[m] = ch * 8 < D ? 2u * (uint32_t)(row * (int)rs + ch * 8) : 0xc0000000u;
  }
  const uint32_t step = 2u * (uint32_t)(16 * (int)rs);
  // Row values: wave 0 -lse2 of the first 64 rows, 1 of the others, 2 and 3 -delta
  // (4 to 7 copy nothing).
  const int v0 = bq * 128 + 64 * (wave & 1);
  const uint32_t vbytes = 4u * (uint32_t)max(0, min(64, p.Lq - v0));
  const float* vsrc = mat < 2 ? p.nlse2 : p.ndelta;
  const uint32_t lds0 = lds_offset(smem);
  auto pair_of = [&](int j, int& b, int& h) NXA_INLINE {
    b = sp.OB > 1 ? ob : j / nH;
    h = sp.OH > 1 ? oh : j % nH;
  };
  auto issue = [&](int j, int st) NXA_INLINE {
    int b, h;
    pair_of(j, b, h);
    const uint32_t at = lds0 + st * STAGE + (kv ? 2 * MAT + (mat - 2) * KMAT : mat * MAT);
    const i32x4 r = make_rsrc(src + b * sb + h * sh + (int64_t)r0 * rs, bytes);
#pragma unroll
    for (int i = 0; i < 128 / ROWS / (NW / 4); ++i)
      if (i < ncpy) {
        const int m = half * ncpy + i;
        dma16_buf(r, off[i % PER] + (m / PER) * step, at + m * 1024);
      }
    const i32x4 rv = make_rsrc(vsrc + ((int64_t)b * p.H + h) * p.Lq + v0, vbytes);
    if (half == 0) dma4_buf(rv, 4u * lane, lds0 + st * STAGE + ROWV + mat * 256);
  };

  Resident<T, DP> rd;
  rd.init(lane);
  f32x16 acc[2], bias[2];
#pragma unroll
  for (int qb = 0; qb < 2; ++qb) {
    acc[qb] = splat16(0.f);
    // (blocks past the packed extent belong to dead waves)
    if (!dead)
      bias[qb] = packed_block(sp.pack_st,
                              ((int64_t)slot * sp.nqb + q0 / 32 + qb) * sp.nkb + k0 / 32, lane);
  }
  // The packed blocks land here, so no wait in the loop covers them.
  __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
  const int je = tile_dead ? j0 : j1;
  if (j0 < je) issue(j0, 0);
  for (int j = j0; j < je; ++j) {
    const int st = (j - j0) & 1;
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
    barrier_nofence();  // pair j is resident; the other stage is free
    if (j + 1 < je) issue(j + 1, st ^ 1);
    if (dead) continue;
    uint32_t keep = 0xffffffffu;
    if (p.has_mask) {
      int b, h;
      pair_of(j, b, h);
      keep = (uint32_t)keep_bits(p, b, h, k0, lane);
      if (keep == 0) continue;
    }
    const uint32_t at = lds0 + st * STAGE;
    const uint32_t qat = at + (wave & 1) * 2 * HALF, kat = at + 2 * MAT + (wave >> 1) * HALF;
    typedef __attribute__((address_space(3))) float lds_f;
    const uint32_t vat = at + ROWV + (wave & 1) * 256 + 4 * c32;
#pragma unroll
    for (int qb = 0; qb < 2; ++qb) {
      // One 32 x 32 block at a time: left free, the scheduler keeps both in
      // flight and spills.
      __builtin_amdgcn_sched_barrier(0);
      const float nlse2 = *(const lds_f*)(uintptr_t)(vat + qb * 128);
      const float ndlt = *(const lds_f*)(uintptr_t)(vat + 512 + qb * 128);
      f32x16 s = bias[qb], dp = splat16(ndlt);
#pragma unroll
      for (int m = 0; m < NC; ++m) {
        M::run(s, rd.row(kat, m), rd.row(qat + qb * HALF, m));
        M::run(dp, rd.row(kat + KMAT, m), rd.row(qat + MAT + qb * HALF, m));
      }
      const auto row_nl = [&](int) NXA_INLINE { return nlse2; };
      if (__any(fabsf(nlse2) > kBigLogit)) p_exponents<true>(s, p.scale_log2, row_nl);
      else p_exponents<false>(s, p.scale_log2, row_nl);
      if (diag || keep != 0xffffffffu)
        mask_block<CAUSAL>(s, keep >> (4 * g), k0 + 4 * g, q0 + 32 * qb + c32);
#pragma unroll
      for (int r = 0; r < 16; ++r)
        acc[qb][r] = __builtin_fmaf(fast_exp2(s[r]), dp[r], acc[qb][r]);
    }
  }
  if (q0 >= p.Lq || k0 >= p.Lk) return;
#pragma unroll
  for (int qb = 0; qb < 2; ++qb) {
    const int q = q0 + 32 * qb + c32;
    if (q >= p.Lq) continue;
    float* out = sp.slabs + (((int64_t)range * sp.OB * sp.OH + slot) * p.Lq + q) * sp.Lkp;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int key = k0 + 8 * c + 4 * g;
      if (key < sp.Lkp) store4(out + key, acc[qb], 4 * c, 1.0f);
    }
  }
}

// Adds the ranges' slabs in order and writes dbias in its own dtype.
__global__ __launch_bounds__(256) void dbias_slabs_kernel(const Params p, const ShortParams sp,
                                                          void* out, int64_t s0, int64_t s1,
                                                          int64_t s2) {
  const int64_t n = (int64_t)sp.OB * sp.OH * p.Lq * p.Lk;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const int key = (int)(i % p.Lk);
  const int64_t row = i / p.Lk;  // (slot, q)
  const int64_t slab = (int64_t)sp.OB * sp.OH * p.Lq * sp.Lkp;
  float x = 0.f;
  for (int r = 0; r < sp.nrange; ++r) x += sp.slabs[r * slab + row * sp.Lkp + key];
  const int q = (int)(row % p.Lq), slot = (int)(row / p.Lq);
  store_elem(p.bias_dtype, out, (slot / sp.OH) * s0 + (slot % sp.OH) * s1 + q * s2 + key, x);
}

// Blocks per pair: one per NW strips (a strip per wave), fewer where the
// pairs alone give the chip more than enough waves.
int split_of(const Params& p, int rows, int nw) {
  const int groups = ((rows + 31) / 32 + nw - 1) / nw;
  const int64_t pairs = (int64_t)p.B * p.H;
  int64_t want = (1024 + pairs - 1) / pairs;
  return (int)(want < groups ? want : groups);
}

// Waves take strips of `strips` rows, against `resident` rows in LDS.
template <typename K4, typename K8>
void launch_strips(K4 k4, K8 k8, const Params& p, ShortParams sp, int strips, int resident, int dp,
                   hipStream_t stream) {
  const size_t lds = (size_t)2 * ((resident + 63) / 64) * 64 * dp * 2;
  // Few pairs: 4-wave blocks, which spread over twice as many CUs.
  const bool wide = lds > kShortWideLds &&
                    (int64_t)p.B * p.H * ((strips + 127) / 128) > kShortFewBlocks;
  sp.nsplit = split_of(p, strips, wide ? 8 : 4);
  const dim3 grid((unsigned)(p.B * p.H * sp.nsplit));
  if (wide)
    hipLaunchKernelGGL(k8, grid, dim3(512), lds, stream, p, sp);
  else
    hipLaunchKernelGGL(k4, grid, dim3(256), lds, stream, p, sp);
}

template <typename T, int DP, bool HB, bool CA>
void launch_part(const Params& p, const ShortParams& sp, ShortPart part, hipStream_t stream) {
  if (part == kShortFwd)
    launch_strips(fwd_short_kernel<T, DP, 4, HB, CA>, fwd_short_kernel<T, DP, 8, HB, CA>, p, sp,
                  p.Lq, p.Lk, DP, stream);
  else if (part == kShortDq)
    launch_strips(dq_short_kernel<T, DP, 4, HB, CA>, dq_short_kernel<T, DP, 8, HB, CA>, p, sp,
                  p.Lq, p.Lk, DP, stream);
  else if (part == kShortDkdv)
    launch_strips(dkdv_short_kernel<T, DP, 4, HB, CA>, dkdv_short_kernel<T, DP, 8, HB, CA>, p, sp,
                  p.Lk, p.Lq, DP, stream);
  else
    hipLaunchKernelGGL((dbias_pairs_kernel<T, DP, CA>),
                       dim3((unsigned)((sp.nrange * sp.OB * sp.OH + 7) / 8 * 8 *
                                       short_dbias_tiles(p.Lq, p.Lk, DP))),
                       dim3(kDbiasWaves<DP> * 64), 0, stream, p, sp);
}

template <typename T, int DP>
void launch_part_f(const Params& p, const ShortParams& sp, ShortPart part, hipStream_t stream) {
  if (p.has_bias) {
    if (p.causal) launch_part<T, DP, true, true>(p, sp, part, stream);
    else launch_part<T, DP, true, false>(p, sp, part, stream);
  } else {
    if (p.causal) launch_part<T, DP, false, true>(p, sp, part, stream);
    else launch_part<T, DP, false, false>(p, sp, part, stream);
  }
}

template <typename T>
void launch_part_d(const Params& p, const ShortParams& sp, ShortPart part, hipStream_t stream) {
  if (p.D <= 32 && p.Dv <= 32) launch_part_f<T, 32>(p, sp, part, stream);
  else launch_part_f<T, 64>(p, sp, part, stream);
}

}  // namespace

void launch_short(const Params& p, const ShortParams& sp, int io_dtype, ShortPart part,
                  hipStream_t stream) {
  if (io_dtype == kF16) launch_part_d<f16>(p, sp, part, stream);
  else launch_part_d<bf16>(p, sp, part, stream);
}

void launch_bias_pack(const Params& p, const ShortParams& sp, hipStream_t stream) {
  const int64_t blocks = (int64_t)sp.OB * sp.OH * sp.nqb * sp.nkb;
  hipLaunchKernelGGL(bias_pack_kernel, dim3((unsigned)blocks, sp.pack_s ? 2 : 1), dim3(256), 0,
                     stream, p, sp);
}

void launch_dbias_slabs(const Params& p, const ShortParams& sp, void* out, const int64_t* str,
                        hipStream_t stream) {
  const int64_t n = (int64_t)sp.OB * sp.OH * p.Lq * p.Lk;
  hipLaunchKernelGGL(dbias_slabs_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream,
                     p, sp, out, str[0], str[1], str[2]);
}

}  // namespace nxa
