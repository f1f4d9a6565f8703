// plh_pack.hip -- the layout kernels of the forward: weight packing into per-lane MFMA fragments,
// x into B-fragment order, and small fills.
#include <algorithm>

#include "plh_device.h"

namespace plh {
namespace {

// ---------------------------------------------------------------------------------------------
// Weight packing: torch layout -> per-lane MFMA A fragments.
// For 16x16x32 f16, lane l of the A operand holds A[m = l % 16][k = 8 * (l / 16) + j], j < 8.
// Row m of tile (wave w, gate q) is gate column q*H + w*16 + m; K runs over [x | h] in chunks
// of 32: chunks [0, kci) index W_ih columns, [kci, kc) index W_hh columns; out-of-range -> 0.
template <int HP>
__global__ void pack_layer_kernel(const _Float16* __restrict__ w_ih, const _Float16* __restrict__ w_hh, int K,
                                  int H, _Float16* __restrict__ dst) {
  constexpr int kWaves = HP / 16, kKci = HP / 32, kKc = 2 * kKci;
  const size_t total = (size_t)kWaves * kKc * 4 * 64 * 8;
  const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= total) return;
  const int j = e & 7;
  const int lane = (e >> 3) & 63;
  const int q = (e >> 9) & 3;
  const int kc = (int)((e >> 11) % kKc);
  const int wv = (int)((e >> 11) / kKc);
  const int m = lane & 15, kgrp = lane >> 4;
  const int u = wv * 16 + m;
  const size_t col = (size_t)q * H + u;
  _Float16 v = (_Float16)0.0f;
  if (u < H) {
    if (kc < kKci) {
      const int k = kc * 32 + kgrp * 8 + j;
      if (k < K) v = w_ih[col * K + k];
    } else {
      const int k = (kc - kKci) * 32 + kgrp * 8 + j;
      if (k < H) v = w_hh[col * H + k];
    }
  }
  dst[e] = v;
}

// Sliced weights: [L][S][8 waves][2 KCH chunks][NJ tiles][64 lanes][8].  Wave w of slice s holds
// the gate rows of its 4 NJ units s HS + 4 NJ w + 0 .. 4 NJ - 1 over all of K: chunks 0 .. KCH - 1
// of W_ih (the layer input, zero past K), then KCH chunks of W_hh; row r of tile j is gate r % 4 of
// unit s HS + 4 NJ w + 4 j + r / 4, and lane l of chunk kc holds k = 32 kc + 8 (l / 16) + 0 .. 7.
template <int HP>
__global__ void pack_sliced_kernel(const _Float16* __restrict__ w_ih, const _Float16* __restrict__ w_hh, int K,
                                   int H, _Float16* __restrict__ dst) {
  using C = Sliced<HP>;
  constexpr int NJ = C::kNj, KCH = C::kKch;
  const size_t total = (size_t)C::kS * 8 * 2 * KCH * NJ * 64 * 8;
  const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= total) return;
  const int jj = e & 7;
  const int lane = (e >> 3) & 63;
  size_t rest = e >> 9;
  const int j = (int)(rest % NJ);
  rest /= NJ;
  const int kc = (int)(rest % (2 * KCH));
  rest /= 2 * KCH;
  const int wv = (int)(rest % 8);
  const int sl = (int)(rest / 8);
  const int r = lane & 15;
  const int u = sl * C::kHs + wv * 4 * NJ + 4 * j + (r >> 2);
  const size_t col = (size_t)(r & 3) * H + u;
  const int k = (kc % KCH) * 32 + (lane >> 4) * 8 + jj;
  _Float16 v = (_Float16)0.0f;
  if (u < H) {
    if (kc < KCH) {
      if (k < K) v = w_ih[col * K + k];
    } else {
      if (k < H) v = w_hh[col * H + k];
    }
  }
  dst[e] = v;
}

__global__ void pack_bias_kernel(const _Float16* __restrict__ b_ih, const _Float16* __restrict__ b_hh, int H, int HP,
                                 float* __restrict__ dst) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= 4 * HP) return;
  const int q = e / HP, u = e % HP;
  float v = 0.0f;
  if (u < H) {
    if (b_ih) v += (float)b_ih[q * H + u];
    if (b_hh) v += (float)b_hh[q * H + u];
  }
  dst[e] = v;
}

__global__ void pack_linear_kernel(const _Float16* __restrict__ w, const _Float16* __restrict__ b, int O, int H,
                                   int HP, float* __restrict__ wl, float* __restrict__ bl) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e < O * HP) {
    const int o = e / HP, k = e % HP;
    wl[e] = k < H ? (float)w[(size_t)o * H + k] : 0.0f;
  }
  if (e < O) bl[e] = b ? (float)b[e] : 0.0f;
}

// Forward prologue: x of rows [row0, row_end) into xp (B-fragment order: per tile and step, g0
// 8-wide K groups of `rows` f16x8, zero past I and past row_end), and the zeroing of the status and
// counters (u32) and of the ring (16-byte pieces), in one launch.
struct PrologueArgs {
  const _Float16* x;
  int T, I, row0, row_end, ntile, rows, g0;
  f16x8* xp;
  uint32_t *z0, *z1;
  f16x8* z2;
  size_t n0, n1, n2;
  uint32_t* uniform;  // DETECT: one word per block
};
// The 8 halfs of row b, step t from column k0 on, zero past I.
__device__ __forceinline__ f16x8 x_group(const PrologueArgs& p, int b, int t, int k0) {
  f16x8 v = {};
  const _Float16* src = p.x + ((size_t)b * p.T + t) * p.I;
#pragma unroll
  for (int j = 0; j < 8; ++j)
    if (k0 + j < p.I) v[j] = src[k0 + j];
  return v;
}
// (IDX: 32-bit element numbers where they fit, whose divisions cost a fraction of 64-bit ones: 13.3 -> 12.3 us
// for the headline batch with detection.)
// Element e; with `compare`, returns true if it belongs to a row that differs from row row0 there.
template <typename IDX>
__device__ __forceinline__ bool prologue_element(const PrologueArgs& p, IDX e, bool compare) {
  if (e < p.n0) p.z0[e] = 0u;
  if (e < p.n1) p.z1[e] = 0u;
  if (e < p.n2) p.z2[e] = f16x8{};
  const unsigned per = (unsigned)(p.g0 * p.rows);
  if (e >= (size_t)p.ntile * p.T * per) return false;
  const int f = (int)(e % per);
  const IDX tt = e / per;
  const int t = (int)(tt % (unsigned)p.T);
  const int tile = (int)(tt / (unsigned)p.T);
  const int b = p.row0 + tile * p.rows + f % p.rows;
  const int k0 = (f / p.rows) * 8;
  bool differs = false;
  f16x8 v = {};
  if (b < p.row_end) {
    v = x_group(p, b, t, k0);
    if (compare && b != p.row0) {
      typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
      const u32x4 d = __builtin_bit_cast(u32x4, v) ^ __builtin_bit_cast(u32x4, x_group(p, p.row0, t, k0));
      differs = (d[0] | d[1] | d[2] | d[3]) != 0u;
    }
  }
  p.xp[e] = v;
  return differs;
}
template <typename IDX>
__global__ void forward_prologue_kernel(PrologueArgs p) {
  (void)prologue_element<IDX>(p, (IDX)blockIdx.x * blockDim.x + threadIdx.x, false);
}
// The same with uniform-batch detection: at most as many blocks as there are words for their verdicts.  A
// thread that has seen a difference compares no further, so a batch of unequal rows reads little more than
// x once: the prologue of the headline batch (512 rows of 1000 steps) takes 12.3 us (9.2
// without the comparison), where the comparison as
// passes of its own (compare, reduce, copy, host synchronisation) took 25-35 us per forward.
template <typename IDX>
__global__ void __launch_bounds__(1024) forward_prologue_detect_kernel(PrologueArgs p, IDX n) {
  int differs = 0;
  for (IDX e = (IDX)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += gridDim.x * blockDim.x)
    differs |= prologue_element<IDX>(p, e, differs == 0) ? 1 : 0;
  differs = __syncthreads_or(differs);
  if (threadIdx.x == 0) p.uniform[blockIdx.x] = differs ? 1u : 0u;
}

__global__ void zero_u32_kernel(uint32_t* __restrict__ p, size_t n) {
  const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e < n) p[e] = 0u;
}

__global__ void repeat_first_row_kernel(const _Float16* __restrict__ in, _Float16* __restrict__ out, int rows, int cols) {
  const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e < (size_t)rows * cols) out[e] = in[e % cols];
}

inline unsigned blocks_for(size_t n, unsigned per) { return (unsigned)((n + per - 1) / per); }

}  // namespace

hipError_t launch_pack_layer(const Geometry& g, int layer, const _Float16* w_ih, const _Float16* w_hh, _Float16* wpack,
                             hipStream_t s) {
  const size_t per_layer = (size_t)(g.HP / 16) * g.kc * 4 * 64 * 8;
  _Float16* dst = wpack + per_layer * layer;
  const int K = layer == 0 ? g.I : g.H;
  const unsigned grid = blocks_for(per_layer, 256);
  switch (g.HP) {
    case 32: hipLaunchKernelGGL(pack_layer_kernel<32>, grid, 256, 0, s, w_ih, w_hh, K, g.H, dst); break;
    case 64: hipLaunchKernelGGL(pack_layer_kernel<64>, grid, 256, 0, s, w_ih, w_hh, K, g.H, dst); break;
    case 128: hipLaunchKernelGGL(pack_layer_kernel<128>, grid, 256, 0, s, w_ih, w_hh, K, g.H, dst); break;
    case 256: hipLaunchKernelGGL(pack_sliced_kernel<256>, grid, 256, 0, s, w_ih, w_hh, K, g.H, dst); break;
    case 512: hipLaunchKernelGGL(pack_sliced_kernel<512>, grid, 256, 0, s, w_ih, w_hh, K, g.H, dst); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_pack_bias(const Geometry& g, int layer, const _Float16* b_ih, const _Float16* b_hh, float* bias,
                            hipStream_t s) {
  hipLaunchKernelGGL(pack_bias_kernel, blocks_for(4 * g.HP, 256), 256, 0, s, b_ih, b_hh, g.H, g.HP,
                     bias + (size_t)layer * 4 * g.HP);
  return hipGetLastError();
}

hipError_t launch_pack_linear(const Geometry& g, const _Float16* w, const _Float16* b, float* wlin, float* blin,
                              hipStream_t s) {
  if (g.O == 0) return hipSuccess;
  hipLaunchKernelGGL(pack_linear_kernel, blocks_for((size_t)g.O * g.HP, 256), 256, 0, s, w, b, g.O, g.H, g.HP, wlin,
                     blin);
  return hipGetLastError();
}

hipError_t launch_forward_prologue(const Geometry& g, ForwardArgs& a, uint32_t* status, int g0,
                                   size_t ring_words, hipStream_t s) {
  const size_t npack = (size_t)a.ntile * a.T * g0 * a.tile_rows;
  const size_t nstat = status ? 1 : 0;
  // 16-byte pieces of the exchange ring (two u64 words each), or of the hand-off rings and their counters
  const bool wavefront = !g.rec && g.slices == 1;
  const size_t nctr = wavefront ? 0 : (size_t)g.L * a.ntile * counter_stride(g);
  size_t nring = ring_words / 2;
  if (wavefront) {
    nring = (size_t)(g.L - 1) * a.ntile * std::min(a.T, kHandoffSlots) * (g.HP / 8) * a.tile_rows;
    if (nring && a.T > kHandoffSlots) nring += (size_t)g.L * a.ntile * (kCounterStride / 4);
  }
  f16x8* const ring = wavefront ? a.hseq : reinterpret_cast<f16x8*>(a.xring);
  const size_t n = std::max(std::max(npack, nstat), std::max(nctr, nring));
  if (n == 0) return hipSuccess;
  const PrologueArgs p = {a.x,    a.T,        a.I,  a.row0, a.row_end, a.ntile, a.tile_rows, g0,
                          a.xp,   status,     a.counters, ring, nstat, nctr, nring, a.uniform};
  if (a.uniform) a.n_uniform = (int)std::min((size_t)a.n_uniform, (n + 1023) / 1024);
  const bool idx32 = n < ((size_t)1 << 31);
  if (a.uniform && idx32)
    hipLaunchKernelGGL(forward_prologue_detect_kernel<uint32_t>, a.n_uniform, 1024, 0, s, p, (uint32_t)n);
  else if (a.uniform)
    hipLaunchKernelGGL(forward_prologue_detect_kernel<uint64_t>, a.n_uniform, 1024, 0, s, p, (uint64_t)n);
  else if (idx32)
    hipLaunchKernelGGL(forward_prologue_kernel<uint32_t>, blocks_for(n, 256), 256, 0, s, p);
  else
    hipLaunchKernelGGL(forward_prologue_kernel<uint64_t>, blocks_for(n, 256), 256, 0, s, p);
  return hipGetLastError();
}

hipError_t launch_zero_u32(uint32_t* p, size_t n, hipStream_t s) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(zero_u32_kernel, blocks_for(n, 256), 256, 0, s, p, n);
  return hipGetLastError();
}

hipError_t launch_repeat_first_row(const _Float16* in, _Float16* out, int rows, int cols, hipStream_t s) {
  const size_t n = (size_t)rows * cols;
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(repeat_first_row_kernel, blocks_for(n, 256), 256, 0, s, in, out, rows, cols);
  return hipGetLastError();
}

}  // namespace plh
