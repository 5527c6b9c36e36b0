// 16-bit forward for few queries over many keys (prompt or latent tokens
// attending a long sequence, one decoding step): at most kSplitMaxQ queries,
// head dims up to 128, no bias, not causal, a mask (if any) that broadcasts
// over queries.
//
// Same math as nxa_fwd16.h (the reference's forward Pallas kernel,
// src/nitrix/_kernels/cuda/attention.py:85-156).  The call is bound by
// reading K and V once, but a grid of query blocks is one block per
// (batch, head): 32 blocks on 256 CUs, seven of whose eight waves hold no
// query (B 4, H 8, 28 queries, 8192 keys, head dim 64, fp16, key padding:
// 107 us for 42 MB).  Here the keys are split over blocks and, inside a
// block, over its four waves: every wave streams 32-key tiles of its own
// through a two-stage LDS ring of its own (no barrier in the loop), the
// block merges its waves' partial results in LDS, and a second kernel
// merges the blocks', O = sum 2^(m - M) O_i, l likewise, M = max m_i, in a
// fixed order.  Fully masked 32-key tiles are dropped from a wave's list
// before it copies anything, so no tile map is built.  That call: 18 us (14
// the splits, 4 the merge); one query over 32768 keys, 8 heads, head dim
// 128: 604 -> 31 us on the GPU.
#include "nxa_common.h"
#include "nxa_launch.h"

namespace nxa {

namespace {

constexpr int kSplitWaves = 4;
constexpr int kSplitTiles = 64;  // most tiles a wave lists

// Weights of N partial results with reference maxima m (all -inf: zeros).
template <int N>
__device__ __forceinline__ float merge_weights(const float (&m)[N], float (&sc)[N]) {
  float M = -INFINITY;
#pragma unroll
  for (int i = 0; i < N; ++i) M = fmaxf(M, m[i]);
#pragma unroll
  for (int i = 0; i < N; ++i) sc[i] = m[i] == -INFINITY ? 0.f : fast_exp2(m[i] - M);
  return M;
}

// Writes chunk ch = 4 db + c (four head-dim elements a lane) of a finished
// strip and, for ch 0, its log-sum-exp.
template <typename T>
__device__ __forceinline__ void store_chunk(const Params& p, int b, int h, int qrow, int g, int ch,
                                            const f32x4& o, float M, float l) {
  if (qrow >= p.Lq) return;
  const float inv = 1.0f / l;
  const int d0 = (ch >> 2) * 32 + 8 * (ch & 3) + 4 * g;
  if (d0 < p.Dv) {
    typedef T t4 __attribute__((ext_vector_type(4)));
    t4 v;
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = (T)(o[j] * inv);
    *reinterpret_cast<t4*>((T*)p.o + b * p.o_str[0] + h * p.o_str[1] + (int64_t)qrow * p.o_str[2] +
                           d0) = v;
  }
  if (ch == 0 && g == 0 && p.lse)
    p.lse[((int64_t)b * p.H + h) * p.Lq + qrow] = (M + __log2f(l)) * kLn2;
}

}  // namespace

// Partial results of a strip and split: NDB * 4 chunks of [64 lanes] float4,
// then m [64] and l [64] (both halves of a lane pair hold their row's).
template <int DP>
constexpr int kPartFloats = (DP / 32) * 4 * 256 + 128;

template <typename T, int DP>
__global__ __launch_bounds__(256, 2) void fwd_split_kernel(const Params p, const SplitParams sp) {
  using M = Mma<T>;
  using Frag = typename M::Frag;
  constexpr int NC = DP / 16, NDB = DP / 32, FPB = M::FRAGS_PER_BLOCK, NW = kSplitWaves;
  constexpr int SPR = DP / 8, ROWS = 64 / SPR, CPM = SPR / 2;  // copies per matrix per tile
  constexpr int TILE = 32 * DP * 2, STAGE = 2 * TILE, NST = 2;
  constexpr int MERGE = NW * (NDB * 16 + 2) * 64 * 4;
  constexpr int SMEM = NW * NST * STAGE > MERGE ? NW * NST * STAGE : MERGE;
  __shared__ __attribute__((aligned(16))) char smem[SMEM];
  __shared__ uint32_t bits_s[NW][kSplitTiles], tile_s[NW][kSplitTiles];

  int vid = blockIdx.x;
  const int strip = vid % sp.strips;
  vid /= sp.strips;
  const int split = vid % sp.splits, bh = vid / sp.splits;
  const int b = bh / p.H, h = bh % p.H;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 5, c32 = lane & 31;
  const int qrow = strip * 32 + c32;
  const bool qok = qrow < p.Lq;
  const int qc = qok ? qrow : p.Lq - 1;

  // This wave's tiles: t0 + wave, t0 + wave + NW, ... below t1.
  const int nt = (p.Lk + 31) / 32;
  const int t0 = (int)((int64_t)nt * split / sp.splits) + wave;
  const int t1 = (int)((int64_t)nt * (split + 1) / sp.splits);
  const int nw = t1 > t0 ? (t1 - t0 + NW - 1) / NW : 0;  // at most kSplitTiles
  const uint8_t* mrow = p.has_mask ? p.mask + b * p.mask_str[0] + h * p.mask_str[1] : nullptr;
  for (int i = 0; i < nw; i += 2) {
    const int key = (t0 + NW * (i + g)) * 32 + c32;
    bool keep = i + g < nw && key < p.Lk;
    if (keep && mrow) keep = mrow[key] != 0;
    const uint64_t m = __ballot(keep);
    if (c32 == 0 && i + g < nw) bits_s[wave][i + g] = (uint32_t)(g ? m >> 32 : m);
  }
  int n;
  {
    const uint32_t w = lane < nw ? bits_s[wave][lane] : 0u;
    const uint64_t act = __ballot(w != 0);
    const int pos = __popcll(act & ((1ull << lane) - 1));
    if (w != 0) {
      tile_s[wave][pos] = (uint32_t)(t0 + NW * lane);
      bits_s[wave][pos] = w;
    }
    n = __popcll(act);
  }

  Frag qf[NC];
  {
    const T* qp = (const T*)p.q + b * p.q_str[0] + h * p.q_str[1] + (int64_t)qc * p.q_str[2];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int d = c * 16 + g * 8;
      qf[c] = qok && d < p.D ? ld16(qp + d) : zero_frag<T>();
    }
  }

  // Copies: 1 KB covers ROWS rows; columns past D and rows past Lk land as
  // zeros (the swizzle repeats every 16 rows).
  const T* kp = (const T*)p.k + b * p.k_str[0] + h * p.k_str[1];
  const T* vp = (const T*)p.v + b * p.v_str[0] + h * p.v_str[1];
  const int64_t ks = p.k_str[2], vs = p.v_str[2];
  uint32_t koff[CPM], voff[CPM];
#pragma unroll
  for (int m = 0; m < CPM; ++m) {
    const int row = m * ROWS + lane / SPR, ch = (lane % SPR) ^ swz<DP>(row);
    koff[m] = ch * 8 < p.D ? 2u * (uint32_t)(row * ks + ch * 8) : 0xfffffff0u;
    voff[m] = ch * 8 < p.Dv ? 2u * (uint32_t)(row * vs + ch * 8) : 0xfffffff0u;
  }
  const uint32_t lds0 = lds_offset(smem) + wave * NST * STAGE;
  auto issue = [&](int i) NXA_INLINE {
    const int k0 = __builtin_amdgcn_readfirstlane((int)tile_s[wave][i]) * 32;
    const int rows = min(32, p.Lk - k0);
    const uint32_t at = lds0 + (i % NST) * STAGE;
    const i32x4 rk = make_rsrc(kp + (int64_t)k0 * ks, (uint32_t)(((int64_t)(rows - 1) * ks + p.D) * 2));
    const i32x4 rv = make_rsrc(vp + (int64_t)k0 * vs, (uint32_t)(((int64_t)(rows - 1) * vs + p.Dv) * 2));
    if (sp.strips == 1) {
      // Keys read once pass the caches by (B 16, H 32, 4096 keys, head dim
      // 128, 537 MB: 182 -> 165 us).
#pragma unroll
      for (int m = 0; m < CPM; ++m) {
        dma16_buf_nt(rk, koff[m], at + m * 1024);
        dma16_buf_nt(rv, voff[m], at + TILE + m * 1024);
      }
    } else {
#pragma unroll
      for (int m = 0; m < CPM; ++m) {
        dma16_buf(rk, koff[m], at + m * 1024);
        dma16_buf(rv, voff[m], at + TILE + m * 1024);
      }
    }
  };

  Resident<T, DP> rd;
  rd.init(lane);

  f32x16 oacc[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db) oacc[db] = splat16(0.f);
  float m_ref = -INFINITY, l_i = 0.f;
  // The Q loads complete here, so the waits below only count tile copies.
  __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
  if (n > 0) issue(0);
  if (n > 1) issue(1);
  for (int i = 0; i < n; ++i) {
    if (i + 1 < n) __builtin_amdgcn_s_waitcnt(vmcnt_imm(2 * CPM));
    else __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
    asm volatile("" ::: "memory");
    const uint32_t w = (uint32_t)__builtin_amdgcn_readfirstlane((int)bits_s[wave][i]);
    const uint32_t at = lds0 + (i % NST) * STAGE;
    f32x16 s;
#pragma unroll
    for (int m = 0; m < NC; ++m) {
      const Frag a = rd.row(at, m);
      if (m == 0) s = M::first(a, qf[m]);
      else M::run(s, a, qf[m]);
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] *= p.scale_log2;
    if (w != 0xffffffffu) {
      const uint32_t wg = w >> (4 * g);
#pragma unroll
      for (int r = 0; r < 16; ++r) s[r] = (wg >> (8 * (r >> 2) + (r & 3))) & 1 ? s[r] : -INFINITY;
    }
    float mt = s[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) mt = fmaxf(mt, s[r]);
    mt = fmaxf(mt, shfl_xor32(mt));
    const float mn = fmaxf(m_ref, mt);
    if (__any(mn > m_ref)) {
      // (a row whose kept scores are all -inf so far keeps -inf: no factor)
      const float alpha = mn > m_ref ? fast_exp2(m_ref - mn) : 1.f;
      l_i *= alpha;
#pragma unroll
      for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) oacc[db][r] *= alpha;
      m_ref = mn;
    }
    const float neg_m = m_ref == -INFINITY ? 0.f : -m_ref;
    float ts[4];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s[r] = fast_exp2(s[r] + neg_m);
      ts[r & 3] = r < 4 ? s[r] : ts[r & 3] + s[r];
    }
    l_i += (ts[0] + ts[1]) + (ts[2] + ts[3]);
#pragma unroll
    for (int f = 0; f < FPB; ++f) {
      const Frag pf = M::pack(s, f);
#pragma unroll
      for (int db = 0; db < NDB; ++db) M::run(oacc[db], rd.tr(at + TILE, f, db), pf);
    }
    // The next copies overwrite the stage that these reads used.
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(lgkmcnt_imm(0));
    if (i + NST < n) issue(i + NST);
  }

  // Merge the waves: [wave][field][lane], fields O (chunk-major), m, l.
  __syncthreads();
  float* ms = reinterpret_cast<float*>(smem);
  constexpr int F = NDB * 16 + 2;
#pragma unroll
  for (int db = 0; db < NDB; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) ms[(wave * F + db * 16 + r) * 64 + lane] = oacc[db][r];
  ms[(wave * F + F - 2) * 64 + lane] = m_ref;
  ms[(wave * F + F - 1) * 64 + lane] = l_i + shfl_xor32(l_i);
  __syncthreads();
  float mw[NW], sc[NW], l = 0.f;
#pragma unroll
  for (int w = 0; w < NW; ++w) mw[w] = ms[(w * F + F - 2) * 64 + lane];
  const float mx = merge_weights(mw, sc);
#pragma unroll
  for (int w = 0; w < NW; ++w) l = __builtin_fmaf(ms[(w * F + F - 1) * 64 + lane], sc[w], l);
  float* part = sp.splits > 1
                    ? sp.part + ((int64_t)(bh * sp.strips + strip) * sp.splits + split) * kPartFloats<DP>
                    : nullptr;
#pragma unroll
  for (int k = 0; k < NDB; ++k) {
    const int ch = wave * NDB + k;  // chunk: four fields
    f32x4 o;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float x = 0.f;
#pragma unroll
      for (int w = 0; w < NW; ++w) x = __builtin_fmaf(ms[(w * F + 4 * ch + j) * 64 + lane], sc[w], x);
      o[j] = x;
    }
    if (part)
      reinterpret_cast<f32x4*>(part)[ch * 64 + lane] = o;
    else
      store_chunk<T>(p, b, h, qrow, g, ch, o, mx, l);
  }
  if (part && wave == 0) {
    part[NDB * 4 * 256 + lane] = mx;
    part[NDB * 4 * 256 + 64 + lane] = l;
  }
}

// Merges the splits of a strip: one wave per chunk, the splits in order.
template <typename T, int DP>
__global__ __launch_bounds__(64) void split_merge_kernel(const Params p, const SplitParams sp) {
  constexpr int NCH = (DP / 32) * 4;
  const int lane = threadIdx.x, g = lane >> 5, c32 = lane & 31;
  const int ch = blockIdx.x % NCH, bs = blockIdx.x / NCH;
  const int strip = bs % sp.strips, bh = bs / sp.strips;
  const float* part = sp.part + (int64_t)bs * sp.splits * kPartFloats<DP>;
  float mx = -INFINITY;
#pragma unroll 8
  for (int s = 0; s < sp.splits; ++s) mx = fmaxf(mx, part[s * kPartFloats<DP> + NCH * 256 + lane]);
  f32x4 o = {0.f, 0.f, 0.f, 0.f};
  float l = 0.f;
#pragma unroll 8
  for (int s = 0; s < sp.splits; ++s) {
    const float* ps = part + s * kPartFloats<DP>;
    const float m = ps[NCH * 256 + lane];
    const float sc = m == -INFINITY ? 0.f : fast_exp2(m - mx);
    l = __builtin_fmaf(ps[NCH * 256 + 64 + lane], sc, l);
    const f32x4 v = reinterpret_cast<const f32x4*>(ps)[ch * 64 + lane];
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j] = __builtin_fmaf(v[j], sc, o[j]);
  }
  store_chunk<T>(p, bh / p.H, bh % p.H, strip * 32 + c32, g, ch, o, mx, l);
}

namespace {

template <typename T, int DP>
void launch_split_t(const Params& p, const SplitParams& sp, hipStream_t stream) {
  const unsigned bs = (unsigned)(p.B * p.H * sp.strips);
  hipLaunchKernelGGL((fwd_split_kernel<T, DP>), dim3(bs * sp.splits), dim3(256), 0, stream, p, sp);
  if (sp.splits > 1)
    hipLaunchKernelGGL((split_merge_kernel<T, DP>), dim3(bs * (DP / 32) * 4), dim3(64), 0, stream, p,
                       sp);
}

template <typename T>
void launch_split_d(const Params& p, const SplitParams& sp, int dp, hipStream_t stream) {
  if (dp == 32) launch_split_t<T, 32>(p, sp, stream);
  else if (dp == 64) launch_split_t<T, 64>(p, sp, stream);
  else launch_split_t<T, 128>(p, sp, stream);
}

}  // namespace

int split_count(int64_t strips, int Lk) {
  const int64_t tiles = ((int64_t)Lk + 31) / 32;
  // About one block per CU (more splits lengthen the merge: 8 heads of 32768
  // keys, head dim 128: 38.6 us in all with 256 blocks, 52 with 512, 79 with
  // 1024), at least two tiles a wave, at most kSplitTiles.
  int64_t n = (256 + strips - 1) / strips;
  const int64_t most = tiles / (2 * kSplitWaves), least = (tiles + kSplitWaves * kSplitTiles - 1) / (kSplitWaves * kSplitTiles);
  if (n > most) n = most;
  // Up to 2048 keys a second launch and its workspace cost the host more than
  // the split saves (4 heads, 1024 keys: 31 us a call split, 25 whole).
  if (tiles <= 64) n = 1;
  if (n < least) n = least;
  return (int)(n < 1 ? 1 : n);
}

size_t split_part_bytes(int dp) {
  return sizeof(float) * (dp == 32 ? kPartFloats<32> : dp == 64 ? kPartFloats<64> : kPartFloats<128>);
}

void launch_fwd_split(const Params& p, const SplitParams& sp, int io_dtype, int dp,
                      hipStream_t stream) {
  if (io_dtype == kF16) launch_split_d<f16>(p, sp, dp, stream);
  else launch_split_d<bf16>(p, sp, dp, stream);
}

}  // namespace nxa
