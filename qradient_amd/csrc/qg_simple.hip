// Elementwise HIP kernels behind the device-resident State API and the
// generic (non-diagonal) observable path.  One thread per amplitude or pair;
// these are not the grad_run hot loop (qg_kernels.hip is), but they keep every
// State method of the reference on the GPU.
#include <hip/hip_runtime.h>
#include "qg_internal.h"
#include "qg_wave.hpp"

namespace qg {

template <class S>
struct V2;
template <>
struct V2<float> {
  typedef float2 T;
};
template <>
struct V2<double> {
  typedef double2 T;
};

// x0' = c x0 - i s (P x)_0 ; x1' = c x1 - i s (P x)_1 on global bit b
// (every 2x2 of the reference's rotations and their derivatives has this form).
template <class S>
__global__ void k_rot1(typename V2<S>::T* v, uint32_t npairs, int b, int type, double c, double s) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= npairs) return;
  const uint32_t lo = i & ((1u << b) - 1u);
  const uint32_t i0 = ((i >> b) << (b + 1)) | lo;
  const uint32_t i1 = i0 | (1u << b);
  const double ar = v[i0].x, ai = v[i0].y, br = v[i1].x, bi = v[i1].y;
  double r0, j0, r1, j1;
  if (type == G_X) {
    r0 = c * ar + s * bi; j0 = c * ai - s * br;
    r1 = c * br + s * ai; j1 = c * bi - s * ar;
  } else if (type == G_Y) {
    r0 = c * ar - s * br; j0 = c * ai - s * bi;
    r1 = c * br + s * ar; j1 = c * bi + s * ai;
  } else {
    r0 = c * ar + s * ai; j0 = c * ai - s * ar;
    r1 = c * br - s * bi; j1 = c * bi + s * br;
  }
  v[i0].x = (S)r0; v[i0].y = (S)j0;
  v[i1].x = (S)r1; v[i1].y = (S)j1;
}

// out[y] = in[map(y)] for a GF(2)-linear index map given by its columns.
template <class S>
__global__ void k_permute(const typename V2<S>::T* __restrict__ in, typename V2<S>::T* __restrict__ out,
                          uint32_t N, const uint32_t* __restrict__ map, int n) {
  const uint32_t y = blockIdx.x * blockDim.x + threadIdx.x;
  if (y >= N) return;
  uint32_t x = 0;
  for (int k = 0; k < n; ++k) x ^= map[k] & (0u - ((y >> k) & 1u));
  out[y] = in[x];
}

__device__ __forceinline__ double diag_at(const DTerm* __restrict__ t, int nt, uint32_t x) {
  double D = 0.0;
  for (int k = 0; k < nt; ++k) {
    double z = ((x >> t[k].a) & 1u) ? -1.0 : 1.0;
    if (t[k].b >= 0) z *= ((x >> t[k].b) & 1u) ? -1.0 : 1.0;
    D += t[k].w * z;
  }
  return D;
}

// v *= exp(-i * angle * D(x))   (and CZ-ladder sign when cz != 0 and nt == 0)
template <class S>
__global__ void k_diag_phase(typename V2<S>::T* v, uint32_t N, const DTerm* __restrict__ t, int nt, double angle,
                             int cz, int n) {
  const uint32_t x = blockIdx.x * blockDim.x + threadIdx.x;
  if (x >= N) return;
  double re = v[x].x, im = v[x].y;
  if (cz) {
    const uint32_t chain = (n >= 2) ? (uint32_t)((1ull << (n - 1)) - 1ull) : 0u;
    if (__popc(x & (x >> 1) & chain) & 1) { re = -re; im = -im; }
  } else {
    double sn, cs;
    sincos(angle * diag_at(t, nt, x), &sn, &cs);
    const double r = cs * re + sn * im, i = cs * im - sn * re;
    re = r; im = i;
  }
  v[x].x = (S)re;
  v[x].y = (S)im;
}

// O in, O = D(x) + sum_k w_k P_k (P in {X, Y} on global bit b_k): stored to
// out when given, and with part also part[block] = this block's share of
// Re<in|O in>, in a fixed order.  Bound by the reads of in (one per x / y
// term, mostly from the caches).  One pass instead of applying O, a dot product
// of both vectors and a sum of its parts; expectation values store nothing (a
// 19-qubit, 12-layer run, complex128: 174 -> 165 us on the device).
template <class S>
__global__ __launch_bounds__(256) void k_obs(const typename V2<S>::T* __restrict__ in, typename V2<S>::T* __restrict__ out,
                                             uint32_t N, const DTerm* __restrict__ dt, int ndt,
                                             const DTerm* __restrict__ xy, int nxy, double* __restrict__ part) {
  double acc = 0.0;
  const uint64_t step = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t at = blockIdx.x * blockDim.x + threadIdx.x; at < N; at += step) {
    const uint32_t x = (uint32_t)at;
    const double D = diag_at(dt, ndt, x);
    const double vr = in[x].x, vi = in[x].y;
    double re = D * vr, im = D * vi;
    for (int k = 0; k < nxy; ++k) {
      const int b = xy[k].a;
      const double w = xy[k].w;
      const uint32_t y = x ^ (1u << b);
      const double pr = in[y].x, pi = in[y].y;
      if (xy[k].b == 0) {  // X
        re += w * pr; im += w * pi;
      } else {             // Y: (Y v)_x = -i v_y if bit 0, +i v_y if bit 1
        const double sg = ((x >> b) & 1u) ? 1.0 : -1.0;
        re += w * (-sg * pi); im += w * (sg * pr);
      }
    }
    if (out) {
      out[x].x = (S)re;
      out[x].y = (S)im;
    }
    acc += vr * re + vi * im;
  }
  if (!part) return;
  __shared__ double red[4];
  const double w = wave_sum(acc, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = w;
  __syncthreads();
  if (threadIdx.x == 0) part[blockIdx.x] = ((red[0] + red[1]) + red[2]) + red[3];
}

// part[block] = sum over this block's elements of Re(conj(a) b) (mode 0),
// |a|^2 (mode 1), in FP64, fixed-order tree.
template <class S>
__global__ void k_dot(const typename V2<S>::T* __restrict__ a, const typename V2<S>::T* __restrict__ b, uint32_t N,
                      int mode, double* __restrict__ part) {
  __shared__ double red[256];
  double acc = 0.0;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < N; i += gridDim.x * blockDim.x) {
    const double ar = a[i].x, ai = a[i].y;
    if (mode == 0) acc += ar * (double)b[i].x + ai * (double)b[i].y;
    else acc += ar * ar + ai * ai;
  }
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int s = blockDim.x / 2; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

// part[(b * nt + k) * gridDim.x + block] = this block's share of <P_k> in state
// b = blockIdx.y (at v + b * N) for the terms t[0, nt), nt <= kTermsPerLaunch, in FP64:
//   Z / ZZ: |v_x|^2 z(x);  X: Re(conj(v_x) v_{x^m});  Y: Re(conj(v_x) (Y v)_x);
//   identity (kind 3): |v_x|^2
// with (Y v)_x = -i v_{x^m} on bit 0 and +i v_{x^m} on bit 1.  Fixed order:
// grid-stride sums, wave butterflies, then the block's waves in turn.
template <class S>
__global__ void __launch_bounds__(256) k_term_expec(const typename V2<S>::T* __restrict__ v, uint32_t N,
                                                    const PTerm* __restrict__ t, int nt, double* __restrict__ part) {
  __shared__ double red[4][kTermsPerLaunch];
  v += (size_t)blockIdx.y * N;
  part += (size_t)blockIdx.y * nt * gridDim.x;
  double acc[kTermsPerLaunch];
#pragma unroll
  for (int k = 0; k < kTermsPerLaunch; ++k) acc[k] = 0.0;
  for (uint32_t x = blockIdx.x * blockDim.x + threadIdx.x; x < N; x += gridDim.x * blockDim.x) {
    const double ar = v[x].x, ai = v[x].y;
    const double pr = ar * ar + ai * ai;
#pragma unroll
    for (int k = 0; k < kTermsPerLaunch; ++k) {
      if (k < nt) {
        const PTerm tk = t[k];
        if (tk.kind == 3) {
          acc[k] += pr;
        } else if (tk.kind == 0) {
          uint32_t par = (x >> tk.a) & 1u;
          if (tk.b >= 0) par ^= (x >> tk.b) & 1u;
          acc[k] += par ? -pr : pr;
        } else {
          const uint32_t bit = (x >> tk.a) & 1u;
          const uint32_t y = x ^ (1u << tk.a);
          const double cr = v[y].x, ci = v[y].y;
          if (tk.kind == 1) {
            acc[k] += ar * cr + ai * ci;
          } else {
            const double im = ar * ci - ai * cr;  // Im(conj(v_x) v_{x^m})
            acc[k] += bit ? -im : im;
          }
        }
      }
    }
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int k = 0; k < kTermsPerLaunch; ++k) {
    double s = acc[k];
    for (int m = 32; m > 0; m >>= 1) s += __shfl_xor(s, m, 64);
    if (lane == 0) red[wave][k] = s;
  }
  __syncthreads();
  if ((int)threadIdx.x < nt) {
    const int k = threadIdx.x;
    part[(size_t)k * gridDim.x + blockIdx.x] = ((red[0][k] + red[1][k]) + red[2][k]) + red[3][k];
  }
}

// The same sums for diagonal terms only (Z / ZZ, and the identity, kind 3):
// <P_k> sums |v_x|^2 (-1)^popc(x & m_k).  The grid stride is a power of two
// (2^sb amplitudes), so x = g + j 2^sb with g the thread's global index and j
// the iteration: the sign splits into (-1)^popc(g & m_k), fixed per thread,
// and (-1)^popc(j & (m_k >> sb)), the same for the whole grid at iteration j.
// A thread takes 16 iterations at a time: their Walsh-Hadamard transform (64
// additions) holds the sixteen probabilities summed with every sign pattern of
// the low four bits of j, so a term costs one read of the pattern it needs
// (from the thread's own LDS column, the pattern being uniform) and one
// addition per 16 amplitudes.
// A sign select and an FMA per term and amplitude, as before, was bound by
// those: 24 terms at 24 qubits, complex64, 75 us -> 53 us (one read of
// the state at the copy rate is 22 us).
template <class S>
__global__ void __launch_bounds__(256) k_term_expec_diag(const typename V2<S>::T* __restrict__ v, uint32_t N,
                                                         const PTerm* __restrict__ t, int nt, int sb,
                                                         double* __restrict__ part) {
  constexpr int NT = kDiagTermsPerLaunch;
  __shared__ double wht[16][256];
  __shared__ double red[4][NT];
  v += (size_t)blockIdx.y * N;
  part += (size_t)blockIdx.y * nt * gridDim.x;
  const uint32_t g = blockIdx.x * blockDim.x + threadIdx.x;
  auto mask_of = [&](int k) -> uint32_t {
    return (k < nt && t[k].kind == 0) ? (1u << t[k].a) | (t[k].b >= 0 ? (1u << t[k].b) : 0u) : 0u;
  };
  double acc[NT];
#pragma unroll
  for (int k = 0; k < NT; ++k) acc[k] = 0.0;
  const uint32_t iters = N >> sb;  // N and the stride are powers of two
  for (uint32_t jj = 0; jj * 16u < iters; ++jj) {
    double p[16];
#pragma unroll
    for (uint32_t r = 0; r < 16; ++r) {
      // fewer than 16 iterations in all: the missing ones hold nothing
      const uint32_t j = jj * 16u + r;
      p[r] = 0.0;
      if (j < iters) {
        const typename V2<S>::T a = v[g + (j << sb)];
        p[r] = (double)a.x * a.x + (double)a.y * a.y;
      }
    }
#pragma unroll
    for (int h = 1; h < 16; h <<= 1)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (!(r & h)) {
          const double x = p[r], y = p[r | h];
          p[r] = x + y;
          p[r | h] = x - y;
        }
#pragma unroll
    for (int r = 0; r < 16; ++r) wht[r][threadIdx.x] = p[r];
    // (the thread reads its own column only: no barrier)
#pragma unroll
    for (int k = 0; k < NT; ++k) {
      if (k < nt) {
        const uint32_t m = sb < 32 ? mask_of(k) >> sb : 0u;
        const double w = wht[m & 15u][threadIdx.x];
        acc[k] += (__popc(jj & (m >> 4)) & 1) ? -w : w;
      }
    }
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int k = 0; k < NT; ++k) {
    if (k < nt) {
      const double s = wave_sum((__popc(g & mask_of(k) & ((1u << sb) - 1u)) & 1) ? -acc[k] : acc[k], 64);
      if (lane == 0) red[wave][k] = s;
    }
  }
  __syncthreads();
  if ((int)threadIdx.x < nt) {
    const int k = threadIdx.x;
    part[(size_t)k * gridDim.x + blockIdx.x] = ((red[0][k] + red[1][k]) + red[2][k]) + red[3][k];
  }
}

// out[b * ldo + k] = sum of part[(b * nt + k) * np + 0 .. np), b = blockIdx.y: one
// 256-thread workgroup per term, coalesced strided partial sums, then a
// fixed-order tree.
__global__ void __launch_bounds__(256) k_sum_terms(const double* __restrict__ part, int np, int nt,
                                                   double* __restrict__ out, int ldo) {
  __shared__ double red[4];
  const int k = blockIdx.x;
  if (k >= nt) return;
  part += ((size_t)blockIdx.y * nt + k) * np;
  double s = 0.0;
  for (int i = threadIdx.x; i < np; i += 256) s += part[i];
  s = wave_sum(s, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) out[(size_t)blockIdx.y * ldo + k] = ((red[0] + red[1]) + red[2]) + red[3];
}

// Shifted copies of one state, copy b = blockIdx.y at out + b * N: op[b] applied to `in`.
template <class S>
__global__ void __launch_bounds__(256) k_shift_copies(const typename V2<S>::T* __restrict__ in,
                                                      typename V2<S>::T* __restrict__ out, uint32_t N,
                                                      const ShiftOp* __restrict__ op) {
  const uint32_t x = blockIdx.x * blockDim.x + threadIdx.x;
  if (x >= N) return;
  const ShiftOp o = op[blockIdx.y];
  const double re = in[x].x, im = in[x].y;
  double r, i;
  if (o.kind == 0) {
    const double s = (__popc(x & o.mask) & 1) ? -o.s : o.s;
    r = o.c * re + s * im;
    i = o.c * im - s * re;
  } else {
    const double pr = in[x ^ o.mask].x, pi = in[x ^ o.mask].y;
    r = o.c * re + o.s * pi;
    i = o.c * im - o.s * pr;
  }
  typename V2<S>::T w;
  w.x = (S)r;
  w.y = (S)i;
  out[(size_t)blockIdx.y * N + x] = w;
}

// *out = sum of part[0, np): one 256-thread workgroup, fixed-order tree.
__global__ void __launch_bounds__(256) k_sum(const double* __restrict__ part, int np, double* __restrict__ out) {
  __shared__ double red[256];
  if (blockIdx.x != 0) return;
  double s = 0.0;
  for (int i = threadIdx.x; i < np; i += 256) s += part[i];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h) red[threadIdx.x] += red[threadIdx.x + h];
    __syncthreads();
  }
  if (threadIdx.x == 0) *out = red[0];
}

// amp(x) = tab[popcount(x)]  (product initial states)
template <class S>
__global__ void k_init(typename V2<S>::T* v, uint32_t N, const double* __restrict__ tab) {
  const uint32_t x = blockIdx.x * blockDim.x + threadIdx.x;
  if (x >= N) return;
  v[x].x = (S)tab[__popc(x)];
  v[x].y = (S)0.0;
}

template <class S>
__global__ void k_convert_in(const double2* __restrict__ in, typename V2<S>::T* __restrict__ out, uint32_t N) {
  const uint32_t x = blockIdx.x * blockDim.x + threadIdx.x;
  if (x >= N) return;
  out[x].x = (S)in[x].x;
  out[x].y = (S)in[x].y;
}

template <class S>
__global__ void k_convert_out(const typename V2<S>::T* __restrict__ in, double2* __restrict__ out, uint32_t N) {
  const uint32_t x = blockIdx.x * blockDim.x + threadIdx.x;
  if (x >= N) return;
  out[x].x = (double)in[x].x;
  out[x].y = (double)in[x].y;
}

template <class S>
__global__ void k_scale(typename V2<S>::T* v, uint32_t N, double re, double im) {
  const uint32_t x = blockIdx.x * blockDim.x + threadIdx.x;
  if (x >= N) return;
  const double a = v[x].x, b = v[x].y;
  v[x].x = (S)(re * a - im * b);
  v[x].y = (S)(re * b + im * a);
}

// ---------------------------------------------------------------------------
// The elementwise kernels count amplitudes in 32 bits: states of up to 2^31.
constexpr int kSimpleMaxN = 31;

// ---------------------------------------------------------------------------
// Basis sampling: the inverse CDF of the distribution |v_x|^2 over positions
// k = 0 .. N-1, position k holding amplitude order[k] (or k without an
// order).  This is scipy's rv_discrete(values=(arange(N), dist)).rvs as the
// reference's dense sampled gradients call it (mc_clean.py:246-254,
// qaoa.py:196-198): a draw u maps to the first position whose cumulative
// probability reaches u, and to position 0 when none does
// (argmax(qvals >= u)).  Two levels: masses of 1024-position blocks and
// their prefix, then one wave per shot searches the prefix 64 entries at a
// time and scans its block 64 positions at a time.  blockIdx.y selects one of
// several states (state b at v + b * N, its masses, uniforms and positions
// behind each other).
//
// One thread per shot walking its block position by position waited for about
// 500 loads in a row: 170 us for 64 shots on 12 qubits, against 8.7 us with a
// wave per shot, whose sixteen loads are in flight together.
// ---------------------------------------------------------------------------
template <class S>
__device__ __forceinline__ double prob_at(const typename V2<S>::T* __restrict__ v, const int32_t* __restrict__ order,
                                          uint32_t k) {
  const uint32_t x = order ? (uint32_t)order[k] : k;
  const double re = v[x].x, im = v[x].y;
  return re * re + im * im;
}

template <class S>
__global__ void __launch_bounds__(256) k_block_mass(const typename V2<S>::T* __restrict__ v, uint32_t N,
                                                    const int32_t* __restrict__ order, double* __restrict__ mass) {
  __shared__ double red[4];
  v += (size_t)blockIdx.y * N;
  const uint32_t base = blockIdx.x * (uint32_t)kSampleBlock + threadIdx.x;
  double s = 0.0;
#pragma unroll
  for (uint32_t j = 0; j < 4; ++j)
    if (base + j * 256u < N) s += prob_at<S>(v, order, base + j * 256u);
  s = wave_sum(s, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) mass[(size_t)blockIdx.y * gridDim.x + blockIdx.x] = ((red[0] + red[1]) + red[2]) + red[3];
}

// Inclusive prefix sums of mass[0, nb) in place: one workgroup per state, 1024
// entries a round (a scan per wave, the waves' totals through LDS).
__global__ void __launch_bounds__(1024) k_mass_prefix(double* __restrict__ mass, int nb) {
  __shared__ double tot[16];
  mass += (size_t)blockIdx.x * nb;
  const int wave = threadIdx.x >> 6;
  double carry = 0.0;
  for (int b0 = 0; b0 < nb; b0 += 1024) {
    const int b = b0 + (int)threadIdx.x;
    double s = wave_scan(b < nb ? mass[b] : 0.0);
    if ((threadIdx.x & 63) == 63) tot[wave] = s;
    __syncthreads();
    double before = carry, all = carry;
    for (int w = 0; w < 16; ++w) {
      if (w == wave) before = all;
      all += tot[w];
    }
    if (b < nb) mass[b] = before + s;
    carry = all;
    __syncthreads();
  }
}

// Every wave takes shots in turn; states of one block (ONE) are read and summed
// once per wave.
template <class S, bool ONE>
__global__ void __launch_bounds__(256) k_basis_search(const typename V2<S>::T* __restrict__ v, uint32_t N,
                                                      const int32_t* __restrict__ order,
                                                      const double* __restrict__ pref, int nb,
                                                      const double* __restrict__ u, int shots,
                                                      int32_t* __restrict__ idx) {
  constexpr int J = kSampleBlock / 64;
  const uint32_t lane = threadIdx.x & 63;
  v += (size_t)blockIdx.y * N;
  pref += (size_t)blockIdx.y * nb;
  u += (size_t)blockIdx.y * shots;
  idx += (size_t)blockIdx.y * shots;
  const double all = pref[nb - 1];
  auto load = [&](uint32_t k0, uint32_t k1, double(&p)[J]) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const uint32_t k = k0 + (uint32_t)j * 64u + lane;
      p[j] = k < k1 ? prob_at<S>(v, order, k) : 0.0;
    }
  };
  double one[J];  // ONE: the cumulative probabilities
  if constexpr (ONE) {
    load(0, N, one);
    double acc = 0.0;
#pragma unroll
    for (int j = 0; j < J; ++j) {
      if (j && (uint32_t)j * 64u >= N) {
        one[j] = acc;  // past the state
      } else {
        const double c = wave_scan(one[j]);
        one[j] = acc + c;
        acc += wave_lane(c, 63);
      }
    }
  }
  for (int64_t s = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); s < shots; s += (int64_t)gridDim.x * 4) {
    const double us = u[s];
    if (!(all >= us)) {
      if (lane == 0) idx[s] = 0;
      continue;
    }
    // the first block whose prefix reaches us: [lo, hi] shrinks 64-fold a round
    int lo = 0, hi = ONE ? 0 : nb - 1;
    while (lo < hi) {
      const int step = (hi - lo + 64) / 64;
      const int e = min(lo + ((int)lane + 1) * step - 1, hi);
      const int f = __builtin_ctzll(__ballot(pref[e] >= us));  // the lane at hi always reaches
      hi = min(lo + (f + 1) * step - 1, hi);
      lo = lo + f * step;
    }
    double acc = lo ? pref[lo - 1] : 0.0;
    const uint32_t k0 = (uint32_t)lo * (uint32_t)kSampleBlock;
    const uint32_t k1 = min(N, k0 + (uint32_t)kSampleBlock);
    double p[J];
    if constexpr (!ONE) load(k0, k1, p);
    uint32_t found = k1 - 1;  // rounding between the two levels: the block's last position
    bool done = false;
#pragma unroll
    for (int j = 0; j < J; ++j) {
      if (!done) {
        const double c = ONE ? one[j] : wave_scan(p[j]);
        const unsigned long long m = __ballot((ONE ? c : acc + c) >= us);
        if (m) {
          found = min(k0 + (uint32_t)j * 64u + (uint32_t)__builtin_ctzll(m), k1 - 1);
          done = true;
        }
        if constexpr (!ONE) acc += wave_lane(c, 63);
      }
    }
    if (lane == 0) idx[s] = (int32_t)found;
  }
}

static inline dim3 grid_for(uint64_t n, int threads) { return dim3((unsigned)((n + threads - 1) / threads)); }

#define QG_DT_SWITCH(dtype, CALL) \
  do {                            \
    if ((dtype) == 1) {           \
      typedef float S;            \
      CALL;                       \
    } else {                      \
      typedef double S;           \
      CALL;                       \
    }                             \
  } while (0)

hipError_t simple_rot1(int dtype, void* v, int n, int b, int type, double c, double s, hipStream_t st) {
  if (n < 1 || n > kSimpleMaxN) return hipErrorInvalidValue;
  const uint32_t np = (uint32_t)(1ull << (n - 1));
  QG_DT_SWITCH(dtype, hipLaunchKernelGGL(k_rot1<S>, grid_for(np, 256), dim3(256), 0, st,
                                         (typename V2<S>::T*)v, np, b, type, c, s));
  return hipGetLastError();
}

hipError_t simple_permute(int dtype, const void* in, void* out, int n, const uint32_t* dmap, hipStream_t st) {
  if (n < 1 || n > kSimpleMaxN) return hipErrorInvalidValue;
  const uint32_t N = (uint32_t)(1ull << n);
  QG_DT_SWITCH(dtype, hipLaunchKernelGGL(k_permute<S>, grid_for(N, 256), dim3(256), 0, st,
                                         (const typename V2<S>::T*)in, (typename V2<S>::T*)out, N, dmap, n));
  return hipGetLastError();
}

hipError_t simple_diag_phase(int dtype, void* v, int n, const DTerm* dt, int nt, double angle, int cz,
                             hipStream_t st) {
  if (n < 1 || n > kSimpleMaxN) return hipErrorInvalidValue;
  const uint32_t N = (uint32_t)(1ull << n);
  QG_DT_SWITCH(dtype, hipLaunchKernelGGL(k_diag_phase<S>, grid_for(N, 256), dim3(256), 0, st,
                                         (typename V2<S>::T*)v, N, dt, nt, angle, cz, n));
  return hipGetLastError();
}

// out = O in (or nothing with out NULL).  With part, *blocks receives the
// number of partial sums of <in|O in> in part (at most kObsBlocks).
hipError_t simple_obs_apply(int dtype, const void* in, void* out, int n, const DTerm* dt, int ndt, const DTerm* xy,
                            int nxy, double* part, int* blocks, hipStream_t st) {
  if (n < 1 || n > kSimpleMaxN) return hipErrorInvalidValue;
  const uint32_t N = (uint32_t)(1ull << n);
  const dim3 grid = part ? dim3(std::min<uint32_t>((N + 255) / 256, kObsBlocks)) : grid_for(N, 256);
  if (blocks) *blocks = (int)grid.x;
  QG_DT_SWITCH(dtype, hipLaunchKernelGGL(k_obs<S>, grid, dim3(256), 0, st, (const typename V2<S>::T*)in,
                                         (typename V2<S>::T*)out, N, dt, ndt, xy, nxy, part));
  return hipGetLastError();
}

// out = sum: mode 0 Re<a|b>, mode 1 <a|a>; part needs `kDotBlocks` doubles.
constexpr int kDotBlocks = 512;
hipError_t simple_dot(int dtype, const void* a, const void* b, int n, int mode, double* part, double* out,
                      hipStream_t st) {
  if (n < 1 || n > kSimpleMaxN) return hipErrorInvalidValue;
  const uint32_t N = (uint32_t)(1ull << n);
  const int blocks = (int)((N + 255) / 256) < kDotBlocks ? (int)((N + 255) / 256) : kDotBlocks;
  QG_DT_SWITCH(dtype, hipLaunchKernelGGL(k_dot<S>, dim3(blocks), dim3(256), 0, st, (const typename V2<S>::T*)a,
                                         (const typename V2<S>::T*)b, N, mode, part));
  hipLaunchKernelGGL(k_sum, dim3(1), dim3(256), 0, st, (const double*)part, blocks, out);
  return hipGetLastError();
}

// Workgroups per state of a term launch over `batch` states, at most kTermBlocks
// in all.  The diagonal kernel takes 16 amplitudes per thread where the states
// fill the device that way (a thread's final cross-lane sums cost as much as
// some 30 amplitudes).  The general kernel's time is that of one thread's chain
// of amplitudes, so it takes one each: 480 x / y terms of 16 qubits, complex64, 422
// us against 2355 us with 16 per thread.
static int term_blocks(uint32_t N, int batch, bool diag) {
  const int most = kTermBlocks / batch;
  int b = 1;
  while (b * 2 <= most && (uint64_t)b * 2 * 256 * (diag ? 16 : 1) <= N) b *= 2;
  return b;
}

// Doubles of `part` that simple_term_expec needs.
size_t simple_term_part(int n, int batch) {
  return (size_t)term_blocks((uint32_t)(1ull << n), batch, false) * kTermPartRows * batch;
}

// out[b * nt + k] = <P_k> in state b for the nt terms t (device arrays) and
// the `batch` states behind each other at v; part: simple_term_part doubles.
// h_t: a host copy of t, or NULL; with it, a run of up to kDiagTermsPerLaunch
// diagonal terms takes one launch of the mask kernel, other terms go
// kTermsPerLaunch at a time to the general kernel.  Each term's sum does not
// depend on the other terms of its launch.
hipError_t simple_term_expec(int dtype, const void* v, int n, const PTerm* t, int nt, double* part, double* out,
                             hipStream_t st, const PTerm* h_t, int batch) {
  if (n < 1 || n > kSimpleMaxN || batch < 1 || batch > 65535) return hipErrorInvalidValue;
  const uint32_t N = (uint32_t)(1ull << n);
  auto is_diag = [&](int k) { return h_t[k].kind == 0 || h_t[k].kind == 3; };
  for (int k0 = 0, m = 0; k0 < nt; k0 += m) {
    // the diagonal kernel needs one thread per amplitude or fewer: N >= 256
    m = 0;
    if (h_t && N >= 256)
      while (m < kDiagTermsPerLaunch && k0 + m < nt && is_diag(k0 + m)) ++m;
    const bool diag = m > 0;
    if (!diag) m = nt - k0 < kTermsPerLaunch ? nt - k0 : kTermsPerLaunch;
    const int blocks = term_blocks(N, batch, diag);
    const dim3 grid(blocks, batch);
    if (diag) {
      int sb = 8;
      while ((1u << sb) < (uint32_t)blocks * 256u) ++sb;
      QG_DT_SWITCH(dtype, hipLaunchKernelGGL(k_term_expec_diag<S>, grid, dim3(256), 0, st,
                                             (const typename V2<S>::T*)v, N, t + k0, m, sb, part));
    } else {
      QG_DT_SWITCH(dtype, hipLaunchKernelGGL(k_term_expec<S>, grid, dim3(256), 0, st,
                                             (const typename V2<S>::T*)v, N, t + k0, m, part));
    }
    hipLaunchKernelGGL(k_sum_terms, dim3(m, batch), dim3(256), 0, st, (const double*)part, blocks, m, out + k0, nt);
  }
  return hipGetLastError();
}

// out state b = op[b] applied to in, b < batch (op: device array).
hipError_t simple_shift_copies(int dtype, const void* in, void* out, int n, const ShiftOp* op, int batch,
                               hipStream_t st) {
  if (n < 1 || n > kSimpleMaxN || batch < 1 || batch > 65535) return hipErrorInvalidValue;
  const uint32_t N = (uint32_t)(1ull << n);
  QG_DT_SWITCH(dtype, hipLaunchKernelGGL(k_shift_copies<S>, dim3((unsigned)((N + 255) / 256), batch), dim3(256), 0, st,
                                         (const typename V2<S>::T*)in, (typename V2<S>::T*)out, N, op));
  return hipGetLastError();
}

hipError_t simple_init(int dtype, void* v, int n, const double* tab, hipStream_t st) {
  if (n < 1 || n > kSimpleMaxN) return hipErrorInvalidValue;
  const uint32_t N = (uint32_t)(1ull << n);
  QG_DT_SWITCH(dtype, hipLaunchKernelGGL(k_init<S>, grid_for(N, 256), dim3(256), 0, st, (typename V2<S>::T*)v, N, tab));
  return hipGetLastError();
}

hipError_t simple_scale(int dtype, void* v, int n, double re, double im, hipStream_t st) {
  if (n < 1 || n > kSimpleMaxN) return hipErrorInvalidValue;
  const uint32_t N = (uint32_t)(1ull << n);
  QG_DT_SWITCH(dtype, hipLaunchKernelGGL(k_scale<S>, grid_for(N, 256), dim3(256), 0, st, (typename V2<S>::T*)v, N, re, im));
  return hipGetLastError();
}

hipError_t simple_convert_in(int dtype, const void* in_c128, void* out, int n, hipStream_t st) {
  if (n < 1 || n > kSimpleMaxN) return hipErrorInvalidValue;
  const uint32_t N = (uint32_t)(1ull << n);
  QG_DT_SWITCH(dtype, hipLaunchKernelGGL(k_convert_in<S>, grid_for(N, 256), dim3(256), 0, st, (const double2*)in_c128,
                                         (typename V2<S>::T*)out, N));
  return hipGetLastError();
}

hipError_t simple_convert_out(int dtype, const void* in, void* out_c128, int n, hipStream_t st) {
  if (n < 1 || n > kSimpleMaxN) return hipErrorInvalidValue;
  const uint32_t N = (uint32_t)(1ull << n);
  QG_DT_SWITCH(dtype, hipLaunchKernelGGL(k_convert_out<S>, grid_for(N, 256), dim3(256), 0, st,
                                         (const typename V2<S>::T*)in, (double2*)out_c128, N));
  return hipGetLastError();
}

constexpr int kSampleWgs = 8192;  // workgroups of a basis search

// Draws for `batch` states behind each other at v: u and idx hold shots
// entries per state, mass (2^n + kSampleBlock - 1) / kSampleBlock doubles of
// scratch per state.
hipError_t simple_sample_basis(int dtype, const void* v, int n, const int32_t* order, const double* u, int shots,
                               int32_t* idx, double* mass, int batch, hipStream_t st) {
  if (n < 1 || n > kSimpleMaxN || shots < 1 || batch < 1 || batch > 65535) return hipErrorInvalidValue;
  const uint32_t N = (uint32_t)(1ull << n);
  const int nb = (int)((N + kSampleBlock - 1) / kSampleBlock);
  QG_DT_SWITCH(dtype, hipLaunchKernelGGL(k_block_mass<S>, dim3(nb, batch), dim3(256), 0, st,
                                         (const typename V2<S>::T*)v, N, order, mass));
  hipLaunchKernelGGL(k_mass_prefix, dim3(batch), dim3(1024), 0, st, mass, nb);
  // as many workgroups as keep the device full; a state of one block is read
  // once per wave, so there a resident set.  A million shots, complex128, a wave
  // for each | now: 9 qubits 1430 | 1120 us, 11 qubits 1720 | 1710 us
  const dim3 grid((unsigned)std::min<int64_t>(((int64_t)shots + 3) / 4, std::max(1, (nb == 1 ? kSampleWgs / 4 : kSampleWgs) / batch)), batch);
  if (nb == 1)
    QG_DT_SWITCH(dtype, hipLaunchKernelGGL((k_basis_search<S, true>), grid, dim3(256), 0, st,
                                           (const typename V2<S>::T*)v, N, order, (const double*)mass, nb, u, shots, idx));
  else
    QG_DT_SWITCH(dtype, hipLaunchKernelGGL((k_basis_search<S, false>), grid, dim3(256), 0, st,
                                           (const typename V2<S>::T*)v, N, order, (const double*)mass, nb, u, shots, idx));
  return hipGetLastError();
}

}  // namespace qg
