// Selective state-space scan of up to 16 states, forward and backward, over
// fp32, bf16 or fp16 x, delta, B and C (A, D and all arithmetic fp32).
//
// Same math as nxa_ssm.hip (the reference's recurrence,
// src/nitrix/nn/ssm/_reference.py:59-97, and its recompute adjoint,
// src/nitrix/_kernels/cuda/selective_scan.py:239-419), arranged so that each
// exponential is taken once per direction and no pass over chunks leaves the
// block.
//
// A block owns the channels of one wave (64 / LPC of them: LPC = NP / NPL
// lanes share a channel, NPL of its NP padded states each) of one batch and
// walks the whole sequence.  In one iteration its NW waves take NW
// consecutive chunks of T steps: every wave scans its chunk from a zero state
// keeping the decays in registers, publishes the chunk's end state and total
// decay in LDS, and after one barrier folds the chunks before its own into
// its entering state and walks the chunk again with the decays it kept (one
// multiply-add per state instead of another exponential).  The backward does
// the same from the last chunk on, with the states entering every 8 steps
// that the forward saved: states and decays of 8 steps stay in registers for
// the reverse walk.
//
// B and C rows are staged per wave (wave-private LDS, no barrier).  Loads go
// through buffer resources that end at the sequence's last row: steps past
// it read delta = x = dy = 0, i.e. decay 1 and no contribution, so no loop
// has a tail.  The next iteration's rows are loaded during this one.
//
// dB and dC sum over channels: per step a butterfly over the wave's channels
// (row and half swaps, DPP rotations), then one partial row per channel group
// that scan_reduce_kernel adds in a fixed order.  dA and dD accumulate in
// registers over the block's whole sequence.  Everything is deterministic.
//
// Measured: batch 8, L 2048, d 1536, n 16, fp32, forward + backward 792 us on
// the chunk-parallel kernels (nine launches, two exponentials a state step
// forward and three backward, 330 MB of chunk states and partial sums), 540
// here (forward 175 with its states, 150 without; backward 345; reduction
// 35, bound by reading 200 MB of partial rows).  Batch 1, L 5000, d 1000,
// n 16, bf16 forward: 121 -> 55 us (four upcasts, 44 us of serial carry).
// The walk is bound by VALU issue (VALU instructions are in issue 94 % of the
// SIMDs' cycles in the backward, 76 % in the forward); the saved states are written as whole
// lines (in [state][channel] order they cost 50 us more).
#include "nxa_common.h"
#include "nxa_launch.h"

#include <type_traits>

namespace nxa {

namespace {

typedef __amdgpu_buffer_rsrc_t Rsrc;

// Resource of `bytes` bytes from base (0: every load returns zero, every
// store is dropped).
__device__ __forceinline__ Rsrc buf(const void* base, int64_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)(uint32_t)bytes,
                                           0x00020000);
}

constexpr uint32_t kOob = 0xfffffff0u;

template <typename TX>
struct Io {  // 16-bit types
  typedef uint16_t raw;
  static __device__ __forceinline__ raw load(Rsrc r, uint32_t off) {
    return __builtin_amdgcn_raw_buffer_load_b16(r, off, 0, 0);
  }
  static __device__ __forceinline__ float cvt(raw v) { return (float)__builtin_bit_cast(TX, v); }
  static __device__ __forceinline__ void store(float x, Rsrc r, uint32_t off) {
    __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(uint16_t, (TX)x), r, off, 0, 0);
  }
};
template <>
struct Io<float> {
  typedef uint32_t raw;
  static __device__ __forceinline__ raw load(Rsrc r, uint32_t off) {
    return __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0);
  }
  static __device__ __forceinline__ float cvt(raw v) { return __builtin_bit_cast(float, v); }
  static __device__ __forceinline__ void store(float x, Rsrc r, uint32_t off) {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, x), r, off, 0, 0);
  }
};

template <int CTRL>
__device__ __forceinline__ float dpp(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xF, 0xF, true));
}

// x of lane K of each group of LPC lanes.
template <int LPC, int K>
__device__ __forceinline__ float bcast(float x) {
  if constexpr (LPC == 1) return x;
  else if constexpr (LPC == 2) return dpp<K | K << 2 | (K + 2) << 4 | (K + 2) << 6>(x);
  else if constexpr (LPC == 4) return dpp<K * 0x55>(x);
  else if constexpr (LPC == 8)
    return __int_as_float(__builtin_amdgcn_ds_swizzle(__float_as_int(x), 0x18 | K << 5));
  else return dpp<0x150 + K>(x);  // row_newbcast
}
// The value of step J of a chunk whose lane `sub` holds steps sub + LPC m in v[m].
template <int LPC, int J, int M>
__device__ __forceinline__ float step_of(const float (&v)[M]) {
  return bcast<LPC, J % LPC>(v[J / LPC]);
}
// f(integral_constant) for 0 .. T - 1 in order (or from the last on).
template <int T, bool REV = false, int I = 0, typename F>
__device__ __forceinline__ void for_steps(F&& f) {
  if constexpr (I < T) {
    f(std::integral_constant<int, REV ? T - 1 - I : I>{});
    for_steps<T, REV, I + 1>(f);
  }
}

// Sum over the LPC (1 .. 16) neighbouring lanes of a channel; every lane of
// the group gets it.  Quad permutes cover masks 1 and 2; with quads equal, the
// mirror of 8 (16) lanes brings the other quad (half row).
template <int LPC>
__device__ __forceinline__ float sum_lanes(float x) {
  if (LPC >= 2) x += dpp<0xB1>(x);
  if (LPC >= 4) x += dpp<0x4E>(x);
  if (LPC >= 8) x += dpp<0x141>(x);
  if (LPC >= 16) x += dpp<0x140>(x);
  return x;
}

__device__ __forceinline__ float swap32_sum(float lo, float hi) {
  const auto r =
      __builtin_amdgcn_permlane32_swap(__float_as_uint(lo), __float_as_uint(hi), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float swap16_sum(float lo, float hi) {
  const auto r =
      __builtin_amdgcn_permlane16_swap(__float_as_uint(lo), __float_as_uint(hi), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Sums each of v[0 .. NPL) over the wave's channels (lanes equal mod LPC).
// Swaps of half waves and of rows halve the values as they add: lane l ends
// with value index l / (64 / NPL); the rest are plain sums (row rotations by
// 8 and 4, quad permutes), so every lane of a row holds its row's result.
template <int NPL, int LPC>
__device__ __forceinline__ float sum_channels(const float (&v)[NPL]) {
  float s;
  if constexpr (NPL == 4) {
    // (after the half swap lanes < 32 hold indices 0, 1 and lanes >= 32 2, 3)
    const float a = swap32_sum(v[0], v[2]), b = swap32_sum(v[1], v[3]);
    s = swap16_sum(a, b);
  } else {
    static_assert(NPL == 2, "states per lane");
    s = swap32_sum(v[0], v[1]);
    s = swap16_sum(s, s);
  }
  if (LPC <= 8) s += dpp<0x128>(s);  // row_ror:8
  if (LPC <= 4) s += dpp<0x124>(s);  // row_ror:4
  if (LPC <= 2) s += dpp<0x4E>(s);
  if (LPC <= 1) s += dpp<0xB1>(s);
  return s;
}

// A log2(e).  A rate of -inf becomes the lowest finite one: the same decays
// (0 for every step above 1e-36), while the steps past the end of the
// sequence, whose delta is 0, keep the decay 1 and not 0 * -inf.
__device__ __forceinline__ float decay_rate(float a) {
  const float r = a * kLog2e;
  return r < -3.402823466e38f ? -3.402823466e38f : r;
}

// Block -> (batch, channel group): runs of neighbouring groups on one XCD,
// whose L2 then serves the 128-byte lines that neighbours share.
__device__ __forceinline__ bool scan_block(const ScanParams& p, int64_t& b, int& cg) {
  const int64_t n = p.nb * p.G, per = (n + 7) / 8;
  const int64_t i = (blockIdx.x % 8) * per + blockIdx.x / 8;
  if (blockIdx.x / 8 >= per || i >= n) return false;
  b = i / p.G;
  cg = (int)(i % p.G);
  return true;
}

// The chunk's B (or C) rows, element lane + 64 q of the padded [T][NP] block.
template <typename TX, int NQ>
__device__ __forceinline__ void load_rows_bc(typename Io<TX>::raw (&r)[NQ], const void* base,
                                             int64_t t0, int rows, int N, const uint32_t (&off)[NQ]) {
  const Rsrc rs = buf((const char*)base + t0 * N * (int64_t)sizeof(TX),
                      (int64_t)rows * N * (int64_t)sizeof(TX));
#pragma unroll
  for (int q = 0; q < NQ; ++q) r[q] = Io<TX>::load(rs, off[q]);
}

template <typename TX, int NP, int NQ>
__device__ __forceinline__ void bc_offsets(uint32_t (&off)[NQ], int N, int lane) {
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    const int e = q * 64 + lane, j = e / NP, n = e % NP;
    off[q] = n < N ? (uint32_t)((j * N + n) * (int)sizeof(TX)) : kOob;
  }
}

// Publishes a chunk's end value and total decay and folds the chunks of the
// iteration in wave order into carry; returns the value entering this wave's
// chunk in `in`.
template <int NPL, int NW>
__device__ __forceinline__ void fold_chunks(float (*agg)[2][64][NPL], int wave, int lane,
                                            const float (&end)[NPL], const float (&dec)[NPL],
                                            float (&carry)[NPL], float (&in)[NPL]) {
  typedef float vec __attribute__((ext_vector_type(NPL == 1 ? 2 : NPL)));
  vec ev, dv;
#pragma unroll
  for (int i = 0; i < NPL; ++i) {
    ev[i] = end[i];
    dv[i] = dec[i];
  }
  if constexpr (NPL == 1) {
    agg[wave][0][lane][0] = end[0];
    agg[wave][1][lane][0] = dec[0];
  } else {
    *reinterpret_cast<vec*>(agg[wave][0][lane]) = ev;
    *reinterpret_cast<vec*>(agg[wave][1][lane]) = dv;
  }
  // LDS only: the next iteration's rows stay in flight.
  __builtin_amdgcn_s_waitcnt(lgkmcnt_imm(0));
  barrier_nofence();
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    if constexpr (NPL == 1) {
      ev[0] = agg[w][0][lane][0];
      dv[0] = agg[w][1][lane][0];
    } else {
      ev = *reinterpret_cast<const vec*>(agg[w][0][lane]);
      dv = *reinterpret_cast<const vec*>(agg[w][1][lane]);
    }
#pragma unroll
    for (int i = 0; i < NPL; ++i) {
      if (w == wave) in[i] = carry[i];
      carry[i] = __builtin_fmaf(dv[i], carry[i], ev[i]);
    }
  }
}

// The lane's states, contiguous (channels' padded states one after another:
// a wave writes whole lines).
template <int NPL>
__device__ __forceinline__ void store_states(float* dst, const float (&h)[NPL]) {
  if constexpr (NPL == 4)
    *reinterpret_cast<f32x4*>(dst) = f32x4{h[0], h[1], h[2], h[3]};
  else
    dst[0] = h[0];
}

constexpr int kBwdT = 8;

template <typename TX, int NP, int NPL, int NW, int T>
__global__ __launch_bounds__(NW * 64, NPL == 4 ? 3 : 1) void scan_fwd_kernel(const ScanParams p) {
  constexpr int LPC = NP / NPL, CPW = 64 / LPC, NQ = T * NP / 64, MS = T / LPC;
  typedef typename Io<TX>::raw raw;
  __shared__ __attribute__((aligned(16))) float sB[NW][T][NP], sC[NW][T][NP];
  __shared__ __attribute__((aligned(16))) float agg[2][NW][2][64][NPL];
  int64_t b;
  int cg;
  if (!scan_block(p, b, cg)) return;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int sub = lane % LPC, n0 = sub * NPL;
  const int d = cg * CPW + lane / LPC;
  const bool ok = d < p.Dm;
  const int dc = ok ? d : p.Dm - 1;
  float al[NPL], carry[NPL];
#pragma unroll
  for (int i = 0; i < NPL; ++i) {
    al[i] = n0 + i < p.N ? decay_rate(p.A[(int64_t)dc * p.N + n0 + i]) : 0.f;
    carry[i] = 0.f;
  }
  const float Dd = p.D ? p.D[dc] : 0.f;
  const uint32_t xoff = (uint32_t)(dc * (int)sizeof(TX));
  uint32_t boff[NQ];
  bc_offsets<TX, NP>(boff, p.N, lane);
  const int64_t rb = b * p.L;
  const char* xb = (const char*)p.x + rb * p.Dm * (int64_t)sizeof(TX);
  const char* db = (const char*)p.delta + rb * p.Dm * (int64_t)sizeof(TX);
  const char* Bb = (const char*)p.B + rb * p.N * (int64_t)sizeof(TX);
  const char* Cb = (const char*)p.C + rb * p.N * (int64_t)sizeof(TX);
  raw xr[MS], dr[MS], br[NQ], cr[NQ];
  // Resources of the chunk's rows at step t (empty past the end).
  Rsrc rx, rd;
  auto rows_of = [&](int64_t t) NXA_INLINE -> int {
    return (int)min((int64_t)T, max((int64_t)0, p.L - t));
  };
  auto open = [&](int64_t t) NXA_INLINE {
    const int rows = rows_of(t);
    const int64_t o = t * p.Dm * (int64_t)sizeof(TX), n = (int64_t)rows * p.Dm * (int64_t)sizeof(TX);
    rd = buf(db + o, n);
    rx = buf(xb + o, n);
    load_rows_bc<TX, NQ>(br, Bb, t, rows, p.N, boff);
    load_rows_bc<TX, NQ>(cr, Cb, t, rows, p.N, boff);
  };
  // Lane `sub` of a channel loads (and stores) steps sub + LPC m: one load
  // brings LPC steps, which the group's lanes pass on by broadcasts.
  auto load_own = [&]() NXA_INLINE {
#pragma unroll
    for (int m = 0; m < MS; ++m) {
      const uint32_t o = xoff + (uint32_t)((sub + LPC * m) * p.Dm * (int)sizeof(TX));
      dr[m] = Io<TX>::load(rd, o);
      xr[m] = Io<TX>::load(rx, o);
    }
  };
  int64_t t0 = (int64_t)wave * T;
  open(t0);
  load_own();
  int par = 0;
  for (int64_t s0 = 0; s0 < p.L; s0 += NW * T, t0 += NW * T, par ^= 1) {
    float* Bw = &sB[wave][0][0];
    float* Cw = &sC[wave][0][0];
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      Bw[q * 64 + lane] = Io<TX>::cvt(br[q]);
      Cw[q * 64 + lane] = Io<TX>::cvt(cr[q]);
    }
    float dt[MS], xv[MS], dx[MS], sdt = 0.f;
#pragma unroll
    for (int m = 0; m < MS; ++m) {
      dt[m] = Io<TX>::cvt(dr[m]);
      xv[m] = Io<TX>::cvt(xr[m]);
      dx[m] = dt[m] * xv[m];
      sdt += dt[m];
    }
    sdt = sum_lanes<LPC>(sdt);
    open(t0 + NW * T);
    load_own();
    float a[T][NPL], h[NPL];
#pragma unroll
    for (int i = 0; i < NPL; ++i) h[i] = 0.f;
    for_steps<T>([&](auto jc) NXA_INLINE {
      constexpr int j = decltype(jc)::value;
      const float dtj = step_of<LPC, j>(dt), dxj = step_of<LPC, j>(dx);
#pragma unroll
      for (int i = 0; i < NPL; ++i) {
        a[j][i] = fast_exp2(dtj * al[i]);
        h[i] = __builtin_fmaf(a[j][i], h[i], dxj * sB[wave][j][n0 + i]);
      }
    });
    float dec[NPL], in[NPL];
#pragma unroll
    for (int i = 0; i < NPL; ++i) dec[i] = fast_exp2(al[i] * sdt);
    fold_chunks<NPL, NW>(agg[par], wave, lane, h, dec, carry, in);
#pragma unroll
    for (int i = 0; i < NPL; ++i) h[i] = in[i];
    const int rows = (int)min((int64_t)T, max((int64_t)0, p.L - t0));
    const Rsrc ry = buf(p.y + (rb + t0) * p.Dm, (int64_t)rows * p.Dm * 4);
    float yk = 0.f;
    for_steps<T>([&](auto jc) NXA_INLINE {
      constexpr int j = decltype(jc)::value;
      if (j % kSsmSub == 0 && p.hs && t0 + j < p.L && ok) {
        store_states<NPL>(p.hs + ((b * p.ns + (t0 + j) / kSsmSub) * p.Dm + d) * NP + n0, h);
      }
      const float dxj = step_of<LPC, j>(dx);
      float y = 0.f;
#pragma unroll
      for (int i = 0; i < NPL; ++i) {
        h[i] = __builtin_fmaf(a[j][i], h[i], dxj * sB[wave][j][n0 + i]);
        y = __builtin_fmaf(sC[wave][j][n0 + i], h[i], y);
      }
      y = sum_lanes<LPC>(y);
      yk = sub == j % LPC ? y : yk;
      if constexpr (j % LPC == LPC - 1)
        Io<float>::store(__builtin_fmaf(Dd, xv[j / LPC], yk), ry,
                         ok ? (uint32_t)(((j - (LPC - 1) + sub) * p.Dm + d) * 4) : kOob);
    });
  }
}

template <typename TX, int NP, int NPL, int NW>
__global__ __launch_bounds__(NW * 64, NPL == 4 && NP == 16 ? 3 : 2) void scan_bwd_kernel(const ScanParams p) {
  constexpr int T = kBwdT, LPC = NP / NPL, CPW = 64 / LPC, NQ = T * NP / 64, MS = T / LPC;
  static_assert(T % LPC == 0 && NQ * 64 == T * NP, "chunk shape");
  typedef typename Io<TX>::raw raw;
  __shared__ __attribute__((aligned(16))) float sB[NW][T][NP], sC[NW][T][NP];
  __shared__ __attribute__((aligned(16))) float red[NW][T][2 * NP];
  __shared__ __attribute__((aligned(16))) float agg[2][NW][2][64][NPL];
  int64_t b;
  int cg;
  if (!scan_block(p, b, cg)) return;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int sub = lane % LPC, n0 = sub * NPL;
  const int d = cg * CPW + lane / LPC;
  const bool ok = d < p.Dm;
  const int dc = ok ? d : p.Dm - 1;
  float al[NPL], carry[NPL], dA[NPL];
#pragma unroll
  for (int i = 0; i < NPL; ++i) {
    al[i] = n0 + i < p.N ? decay_rate(p.A[(int64_t)dc * p.N + n0 + i]) : 0.f;
    carry[i] = dA[i] = 0.f;
  }
  const float Dd = p.D ? p.D[dc] : 0.f;
  float dD = 0.f, dDe = 0.f;
  const uint32_t xoff = (uint32_t)(dc * (int)sizeof(TX));
  uint32_t boff[NQ];
  bc_offsets<TX, NP>(boff, p.N, lane);
  const int64_t rb = b * p.L;
  const char* xb = (const char*)p.x + rb * p.Dm * (int64_t)sizeof(TX);
  const char* db = (const char*)p.delta + rb * p.Dm * (int64_t)sizeof(TX);
  const char* Bb = (const char*)p.B + rb * p.N * (int64_t)sizeof(TX);
  const char* Cb = (const char*)p.C + rb * p.N * (int64_t)sizeof(TX);
  const float* yb = p.dy + rb * p.Dm;
  raw xr[MS], dr[MS], br[NQ], cr[NQ];
  uint32_t gr[MS], hr[NPL];
  // Lanes past the last channel read dy = 0: they add nothing to dB and dC
  // (their x, delta and states are those of the last channel).
  const uint32_t yoff = ok ? (uint32_t)(d * 4) : 0x80000000u;
  Rsrc rx, rd, rg;
  // Resources of chunk c's rows (empty before the first chunk).
  auto open = [&](int64_t c) NXA_INLINE {
    const int64_t t = max((int64_t)0, c) * T;
    const int rows = c < 0 ? 0 : (int)min((int64_t)T, p.L - t);
    const int64_t o = t * p.Dm, n = (int64_t)rows * p.Dm;
    rd = buf(db + o * (int64_t)sizeof(TX), n * (int64_t)sizeof(TX));
    rx = buf(xb + o * (int64_t)sizeof(TX), n * (int64_t)sizeof(TX));
    rg = buf(yb + o, n * 4);
    load_rows_bc<TX, NQ>(br, Bb, t, rows, p.N, boff);
    load_rows_bc<TX, NQ>(cr, Cb, t, rows, p.N, boff);
    const Rsrc rh = buf(p.hs + (b * p.ns + max((int64_t)0, c)) * NP * (int64_t)p.Dm,
                        c < 0 ? 0 : (int64_t)NP * p.Dm * 4);
    const uint32_t ho = (uint32_t)((dc * NP + n0) * 4);
    if constexpr (NPL == 4) {
      const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(rh, ho, 0, 0);
#pragma unroll
      for (int i = 0; i < NPL; ++i) hr[i] = v[i];
    } else {
      const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(rh, ho, 0, 0);
#pragma unroll
      for (int i = 0; i < NPL; ++i) hr[i] = v[i];
    }
  };
  // Lane `sub` of a channel loads and stores steps sub + LPC m.
  auto load_own = [&]() NXA_INLINE {
#pragma unroll
    for (int m = 0; m < MS; ++m) {
      const uint32_t o = (uint32_t)((sub + LPC * m) * p.Dm);
      dr[m] = Io<TX>::load(rd, xoff + o * (uint32_t)sizeof(TX));
      xr[m] = Io<TX>::load(rx, xoff + o * (uint32_t)sizeof(TX));
      gr[m] = Io<float>::load(rg, yoff + o * 4);
    }
  };
  // Chunks from the last on; wave w the w-th of an iteration.
  int64_t c = (int64_t)p.ns - 1 - wave;
  open(c);
  load_own();
  int par = 0;
  for (int64_t top = p.ns; top > 0; top -= NW, c -= NW, par ^= 1) {
    float* Bw = &sB[wave][0][0];
    float* Cw = &sC[wave][0][0];
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      Bw[q * 64 + lane] = Io<TX>::cvt(br[q]);
      Cw[q * 64 + lane] = Io<TX>::cvt(cr[q]);
    }
    float dt[MS], xv[MS], dyv[MS], dtx[MS], h[T + 1][NPL], sdt = 0.f, dDc = 0.f;
#pragma unroll
    for (int m = 0; m < MS; ++m) {
      dt[m] = Io<TX>::cvt(dr[m]);
      xv[m] = Io<TX>::cvt(xr[m]);
      dyv[m] = __uint_as_float(gr[m]);
      dtx[m] = dt[m] * xv[m];
      sdt += dt[m];
      dDc = __builtin_fmaf(dyv[m], xv[m], dDc);
    }
    {
      // Compensated: one value takes every chunk of a long sequence.
      const float v = dDc - dDe, t = dD + v;
      dDe = (t - dD) - v;
      dD = t;
    }
    sdt = sum_lanes<LPC>(sdt);
#pragma unroll
    for (int i = 0; i < NPL; ++i) h[0][i] = __uint_as_float(hr[i]);
    open(c - NW);
    load_own();
    float a[T][NPL];
    for_steps<T>([&](auto jc) NXA_INLINE {
      constexpr int j = decltype(jc)::value;
      const float dtj = step_of<LPC, j>(dt), dxj = step_of<LPC, j>(dtx);
#pragma unroll
      for (int i = 0; i < NPL; ++i) {
        a[j][i] = fast_exp2(dtj * al[i]);
        h[j + 1][i] = __builtin_fmaf(a[j][i], h[j][i], dxj * sB[wave][j][n0 + i]);
      }
    });
    float gh[NPL], dec[NPL], in[NPL];
#pragma unroll
    for (int i = 0; i < NPL; ++i) {
      gh[i] = 0.f;
      dec[i] = fast_exp2(al[i] * sdt);
    }
    for_steps<T, true>([&](auto jc) NXA_INLINE {
      constexpr int j = decltype(jc)::value;
      const float dyj = step_of<LPC, j>(dyv);
#pragma unroll
      for (int i = 0; i < NPL; ++i)
        gh[i] = a[j][i] * __builtin_fmaf(sC[wave][j][n0 + i], dyj, gh[i]);
    });
    fold_chunks<NPL, NW>(agg[par], wave, lane, gh, dec, carry, in);
#pragma unroll
    for (int i = 0; i < NPL; ++i) gh[i] = in[i];
    const int64_t t0 = max((int64_t)0, c) * T;
    const int rows = c < 0 ? 0 : (int)min((int64_t)T, p.L - t0);
    const int64_t gbytes = (int64_t)rows * p.Dm * (int64_t)sizeof(TX);
    const Rsrc ox = buf((char*)p.dx + (rb + t0) * p.Dm * (int64_t)sizeof(TX), gbytes);
    const Rsrc od = buf((char*)p.ddelta + (rb + t0) * p.Dm * (int64_t)sizeof(TX), gbytes);
    float kb = 0.f, ka = 0.f, dAc[NPL];
#pragma unroll
    for (int i = 0; i < NPL; ++i) dAc[i] = 0.f;
    for_steps<T, true>([&](auto jc) NXA_INLINE {
      constexpr int j = decltype(jc)::value;
      const float dtj = step_of<LPC, j>(dt), dyj = step_of<LPC, j>(dyv);
      const float dxj = step_of<LPC, j>(dtx);
      float sgb = 0.f, sga = 0.f, vb[NPL], vc[NPL];
#pragma unroll
      for (int i = 0; i < NPL; ++i) {
        const float g = __builtin_fmaf(sC[wave][j][n0 + i], dyj, gh[i]);
        const float u = g * (a[j][i] * h[j][i]);
        sgb = __builtin_fmaf(g, sB[wave][j][n0 + i], sgb);
        sga = __builtin_fmaf(u, al[i], sga);
        dAc[i] = __builtin_fmaf(u, dtj, dAc[i]);
        vb[i] = g * dxj;
        vc[i] = dyj * h[j + 1][i];
        gh[i] = a[j][i] * g;
      }
      sgb = sum_lanes<LPC>(sgb);
      sga = sum_lanes<LPC>(sga);
      // The lane whose step this is keeps the two sums: dx = D dy + delta
      // sum g B, ddelta = x sum g B + ln2 sum g al a h.
      kb = sub == j % LPC ? sgb : kb;
      ka = sub == j % LPC ? sga : ka;
      if constexpr (j % LPC == 0) {
        constexpr int m = j / LPC;
        const uint32_t o = ok ? (uint32_t)(((j + sub) * p.Dm + d) * (int)sizeof(TX)) : kOob;
        Io<TX>::store(__builtin_fmaf(dt[m], kb, Dd * dyv[m]), ox, o);
        Io<TX>::store(__builtin_fmaf(xv[m], kb, kLn2 * ka), od, o);
      }
      const float rB = sum_channels<NPL, LPC>(vb), rC = sum_channels<NPL, LPC>(vc);
      // One lane per value: the first channel of its row (or half).
      if ((lane % (64 / NPL)) < LPC) {
        const int q = n0 + lane / (64 / NPL);
        red[wave][j][q] = rB;
        red[wave][j][NP + q] = rC;
      }
    });
    // (a chunk's sum at a time: shorter chains of additions round less)
#pragma unroll
    for (int i = 0; i < NPL; ++i) dA[i] += dAc[i];
    // The chunk's partial rows [T][2 NP], contiguous.
    const Rsrc rp = buf(p.part + ((int64_t)cg * p.nb * p.L + rb + t0) * (2 * NP),
                        (int64_t)rows * (2 * NP) * 4);
    const float* rw = &red[wave][0][0];
#pragma unroll
    for (int e = 0; e < T * 2 * NP; e += 64)
      Io<float>::store(rw[e + lane], rp, (uint32_t)((e + lane) * 4));
  }
  // dA and dD of the block: the waves' sums in wave order.
  __syncthreads();
#pragma unroll
  for (int i = 0; i < NPL; ++i) agg[0][wave][0][lane][i] = dA[i];
  agg[1][wave][0][lane][0] = sum_lanes<LPC>(dD);  // (lanes hold their own steps')
  __syncthreads();
  if (wave != 0 || !ok) return;
#pragma unroll
  for (int i = 0; i < NPL; ++i) {
    float s = 0.f;
    for (int w = 0; w < NW; ++w) s += agg[0][w][0][lane][i];
    p.dApart[(b * NP + n0 + i) * p.Dm + d] = s;
  }
  if (sub == 0) {
    float s = 0.f;
    for (int w = 0; w < NW; ++w) s += agg[1][w][0][lane][0];
    p.dDpart[b * p.Dm + d] = s;
  }
}

// Sums of the partials in a fixed order: dB / dC over the channel groups
// (blocks below nbc, four values a thread), dA / dD over the batches.
template <typename TX, int NP>
__global__ __launch_bounds__(256) void scan_reduce_kernel(const ScanParams p, unsigned nbc) {
  if (blockIdx.x < nbc) {
    constexpr int V4 = 2 * NP / 4;
    const int64_t n = p.nb * p.L * V4;
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;  // (b, t, quad)
    if (i >= n) return;
    const f32x4* src = reinterpret_cast<const f32x4*>(p.part) + i;
    f32x4 s = {0.f, 0.f, 0.f, 0.f};
    // Eight groups at a time: all loads in flight, and chains of additions
    // that round less.
    for (int g0 = 0; g0 < p.G; g0 += 8) {
      f32x4 v[8];
#pragma unroll
      for (int g = 0; g < 8; ++g)
        v[g] = g0 + g < p.G ? src[(int64_t)(g0 + g) * n] : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < 4; ++k)
        s[k] += ((v[0][k] + v[1][k]) + (v[2][k] + v[3][k])) + ((v[4][k] + v[5][k]) + (v[6][k] + v[7][k]));
    }
    const int q = (int)(i % V4) * 4, n0 = q % NP;
    TX* out = (TX*)(q < NP ? p.dB : p.dC) + (i / V4) * p.N;
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (n0 + k < p.N) out[n0 + k] = (TX)s[k];
    return;
  }
  const int64_t i = (int64_t)(blockIdx.x - nbc) * 256 + threadIdx.x;
  const int64_t na = (int64_t)NP * p.Dm;
  if (i >= na + p.Dm) return;
  float s = 0.f;
  if (i < na) {
    for (int64_t b = 0; b < p.nb; ++b) s += p.dApart[b * na + i];
    const int n = (int)(i / p.Dm), d = (int)(i % p.Dm);
    if (n < p.N) p.dA[(int64_t)d * p.N + n] = s;
  } else if (p.dD) {
    for (int64_t b = 0; b < p.nb; ++b) s += p.dDpart[b * p.Dm + (i - na)];
    p.dD[i - na] = s;
  }
}

unsigned grid8(int64_t n) { return (unsigned)((n + 7) / 8 * 8); }

template <typename TX, int NP>
void launch_fwd_t(ScanParams p, hipStream_t stream) {
  // Four states a lane once that alone gives the chip two blocks of 8 waves
  // a CU; else one state a lane (four times the blocks), with 16 waves a
  // block while the blocks leave CUs idle.
  const int g4 = scan_groups(p.Dm, NP, 4), g1 = scan_groups(p.Dm, NP, 1);
  if (p.nb * g4 >= 512) {
    p.G = g4;
    hipLaunchKernelGGL((scan_fwd_kernel<TX, NP, 4, 4, 8>), dim3(grid8(p.nb * g4)), dim3(256), 0,
                       stream, p);
  } else {
    p.G = g1;
    if (p.nb * g1 > 512)
      hipLaunchKernelGGL((scan_fwd_kernel<TX, NP, 1, 8, 16>), dim3(grid8(p.nb * g1)), dim3(512), 0,
                         stream, p);
    else
      hipLaunchKernelGGL((scan_fwd_kernel<TX, NP, 1, 16, 16>), dim3(grid8(p.nb * g1)), dim3(1024), 0,
                         stream, p);
  }
}

template <typename TX, int NP>
void launch_bwd_t(ScanParams p, hipStream_t stream) {
  p.G = scan_groups(p.Dm, NP, scan_bwd_states(p.nb, p.Dm, NP));
  const dim3 grid(grid8(p.nb * p.G));
  if (scan_bwd_states(p.nb, p.Dm, NP) == 4)
    hipLaunchKernelGGL((scan_bwd_kernel<TX, NP, 4, 4>), grid, dim3(256), 0, stream, p);
  else if (p.nb * p.G > 256)
    hipLaunchKernelGGL((scan_bwd_kernel<TX, NP, 2, 8>), grid, dim3(512), 0, stream, p);
  else
    hipLaunchKernelGGL((scan_bwd_kernel<TX, NP, 2, 16>), grid, dim3(1024), 0, stream, p);
  const unsigned nbc = (unsigned)((p.nb * p.L * (2 * NP / 4) + 255) / 256);
  const unsigned na = (unsigned)(((int64_t)(NP + 1) * p.Dm + 255) / 256);
  hipLaunchKernelGGL((scan_reduce_kernel<TX, NP>), dim3(nbc + na), dim3(256), 0, stream, p, nbc);
}

template <typename TX>
void launch_scan_n(const ScanParams& p, bool bwd, hipStream_t stream) {
  const int NP = scan_padded_states(p.N);
  if (NP == 16) {
    if (bwd) launch_bwd_t<TX, 16>(p, stream);
    else launch_fwd_t<TX, 16>(p, stream);
  } else {
    // (states are padded to at least 8, so that a chunk's B rows fill a wave)
    if (bwd) launch_bwd_t<TX, 8>(p, stream);
    else launch_fwd_t<TX, 8>(p, stream);
  }
}

}  // namespace

int scan_padded_states(int N) { return N <= 8 ? 8 : 16; }

int scan_groups(int Dm, int NP, int npl) {
  const int cpw = 64 / (NP / npl);
  return (Dm + cpw - 1) / cpw;
}

int scan_bwd_states(int64_t nb, int Dm, int NP) {
  return nb * scan_groups(Dm, NP, 4) >= 512 ? 4 : 2;
}

void launch_scan(const ScanParams& p, int dtype, bool bwd, hipStream_t stream) {
  if (dtype == kF32) launch_scan_n<float>(p, bwd, stream);
  else if (dtype == kBF16) launch_scan_n<bf16>(p, bwd, stream);
  else launch_scan_n<f16>(p, bwd, stream);
}

}  // namespace nxa
