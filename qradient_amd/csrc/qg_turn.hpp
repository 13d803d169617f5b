// Turning passes of the QAOA circuit.
//
// A layer is the cost phase (diagonal) and one X rotation per qubit, and a
// pass holds a window of the bits, so a layer takes P passes, one per window.
// The mixer's gates commute, so the windows of a layer may run in any order:
// the next layer starts with the window that this one ended on, and that
// pass runs this layer's gates, the phase between the layers and the next
// layer's gates on one read and write of the state.  L layers take
// (P - 1) L + 1 passes where one layer at a time takes P L.
//
// A pass is a list of rounds as in qg_sweep.hpp (four bits in registers, an
// LDS exchange between rounds), with one diagonal operation before round dq:
// the phase (evaluated in that round's layout, so a turn needs no exchange of
// its own) or, at the end of the forward circuit, E = sum D |psi|^2.
//
// The adjoint runs the rounds backwards on psi (the forward pass's output,
// from the history) and lambda: each round's reductions Im<lam|X_q|psi>,
// summed over the bits (they share one angle), then its inverse gates; at the
// diagonal operation d/dgamma = 2 sum D Im(conj(lam) psi) and the inverse
// phase.  The circuit's last pass forms lambda = D psi itself.  psi is never
// stored.
//
// A complex64 forward pass moves FP64 real parts through its 8-byte slots and
// then the imaginary parts (see qg_sweep.hpp), so psi is rounded where it is
// stored and nowhere else.  With FP32 exchanges E and the gradients of 15 qubits
// and 2 or 3 layers were less accurate than one layer at a time.  Error against
// complex128, 16 graphs, root mean square, one layer at a time | FP32 exchanges |
// now: E of 15 qubits, 2 layers, 6.4e-9 | 8.0e-9 | 4.1e-9, its gradient 1.14e-8 |
// 2.81e-8 | 1.38e-8; gradient of 20 qubits, 8 layers 9.1e-9 | 7.7e-9 | 6.7e-9, of
// 20 qubits, 30 layers 2.8e-7 | 1.9e-7 | 1.6e-7.  It costs 1 to 3% of a gradient
// run (256 circuits of 20 qubits, 8 layers 32.1 -> 32.5 ms).
//
// Bound: the vector ALU (gates, reductions, and the FP64 <-> FP32 conversions
// of the exchanges), then HBM: 84 GB of states would take 18 ms at the copy
// rate.  256 circuits of 20 qubits, 8 layers, complex64: 46.5 -> 32.5 ms (9 + 9
// passes instead of 16 + 16); one circuit of 17 qubits, 6 layers, complex128,
// real weights: 541 -> 251 us.
#pragma once
#include "qg_math.hpp"
#include "qg_sweep.hpp"

namespace qg {

// LDS bytes of a pass: the tile (the per-wave sums reuse it) and the phase table.
__host__ __device__ inline size_t turn_lds_bytes(int dtype, int K, int tab_bytes) {
  return (size_t)(1u << K) * (dtype == 1 ? 8 : 16) + (size_t)tab_bytes;
}

template <class S, bool TWO, int PH, bool BIG>
__device__ __forceinline__ void run_turn(const TurnDesc* __restrict__ d, void* lds, uint32_t tid_in, uint32_t blk,
                                         uint32_t nblk) {
  constexpr int R = 4, A = 16;
  typedef typename Store<S>::G G;   // HBM element type
  typedef typename Store<S>::L LT;  // LDS tile element type
  constexpr int GSH = sizeof(G) == 4 ? 3 : 4;
  constexpr int SH = sizeof(LT) == 4 ? 3 : 4;
  constexpr bool PF = !TWO;  // the next tile's loads in flight while this one is worked on
  constexpr bool HALVES = SH == 3 && !TWO;  // FP64 halves of an amplitude through its 8-byte slot (see above)
  warm_lines<(int)sizeof(TurnDesc)>(d);
  const int n = d->n, K = d->K, t = d->t, c = d->c, p = d->p;
  const uint32_t flags = d->flags;
  const uint32_t ntiles = 1u << (n - K);
  const uint32_t nthr = blockDim.x;
  const int nr = d->nr, dq = d->dq;
  double* tab = reinterpret_cast<double*>(reinterpret_cast<char*>(lds) + (sizeof(LT) * 2u << K));
  if (PH == TP_LUT && (flags & F_PHASE_PRE)) {
    const int nlut = 2 * (2 * d->lut_off + 1);
    for (int i = (int)tid_in; i < nlut; i += (int)nthr) tab[i] = d->lut[i];
    __syncthreads();
  }
  const bool init = !TWO && (flags & F_INIT_TAB);
  const bool obs = (flags & F_OBS_DIAG) != 0;
  const bool nt_a = (flags & F_NT_A) != 0;
  // tile order as in run_pass
  const bool xcd = (flags & F_XCD_ORDER) && (nblk >= 8) && (nblk % 8 == 0) && (ntiles % nblk == 0);
  const uint32_t per_x = ntiles / 8, slots = nblk / 8;
  const uint32_t rounds = xcd ? ntiles / nblk : (blk < ntiles ? (ntiles - 1 - blk) / nblk + 1 : 0u);
  auto tile_of = [&](uint32_t r) -> uint32_t {
    return xcd ? (blk % 8) * per_x + r * slots + blk / 8 : blk + r * nblk;
  };
  // global addresses of a thread's amplitudes in the natural layout
  auto addresses = [&](uint32_t tt, uint32_t(&adr)[A]) __attribute__((always_inline)) {
    constexpr int AS = BIG ? 0 : GSH;
    uint32_t tid = tid_in;
    asm volatile("" : "+v"(tid));
    uint32_t o[16], e[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) e[k] = (1u << gpos_of_local(t + k, c, p)) << AS;
    xor_table(o, e[0], e[1], e[2], e[3]);
    uint32_t base = (gl_tile(tt, c, p, K) | gl_local(tid, c, p)) << AS;
    asm volatile("" : "+v"(base));  // opaque (see lds_transpose)
#pragma unroll
    for (int a = 0; a < A; ++a) adr[a] = base ^ o[a];
  };
  Cx<G> ra[A];
  Cx<G> rb[TWO ? A : 1];
  auto fetch = [&](uint32_t tt) __attribute__((always_inline)) {
    if (init) return;
    uint32_t adr[A];
    addresses(tt, adr);
    if (nt_a) {
      asm volatile("");  // keeps the two load sequences apart (see run_pass)
#pragma unroll
      for (int a = 0; a < A; ++a)
        ra[a] = BIG ? Stor<G>::template ld_big<G>(d->a_in, adr[a]) : Stor<G>::template ld_o_nt<G>(d->a_in, adr[a]);
      asm volatile("");
    } else {
#pragma unroll
      for (int a = 0; a < A; ++a)
        ra[a] = BIG ? Stor<G>::template ld_big<G>(d->a_in, adr[a]) : Stor<G>::template ld_o<G>(d->a_in, adr[a]);
    }
    if constexpr (TWO) {
      if (!obs) {
#pragma unroll
        for (int a = 0; a < A; ++a)
          rb[a] = BIG ? Stor<G>::template ld_big<G>(d->b_in, adr[a]) : Stor<G>::template ld_o<G>(d->b_in, adr[a]);
      } else {
#pragma unroll
        for (int a = 0; a < A; ++a) rb[a] = {(G)0, (G)0};
      }
    }
  };
  if (init) {
#pragma unroll
    for (int a = 0; a < A; ++a) ra[a] = {(G)0, (G)0};
  }
  double acc0 = 0.0, acc1 = 0.0, accd = 0.0;
  if (PF && rounds > 0) fetch(tile_of(0));
#pragma unroll 1
  for (uint32_t r = 0; r < rounds; ++r) {
    const uint32_t tt = tile_of(r);
    if (!PF) {
      __builtin_amdgcn_s_setprio(2);
      fetch(tt);
      __builtin_amdgcn_s_setprio(0);
    }
    uint32_t tid = tid_in;
    asm volatile("" : "+v"(tid));
    Cd xa[A];
    Cd xb[TWO ? A : 1];
    if (init) {
      const double v = d->amp0;
#pragma unroll
      for (int a = 0; a < A; ++a) xa[a] = {v, 0.0};
    } else {
#pragma unroll
      for (int a = 0; a < A; ++a) xa[a] = {(double)ra[a].re, (double)ra[a].im};
    }
    if constexpr (TWO) {
#pragma unroll
      for (int a = 0; a < A; ++a) xb[a] = {(double)rb[a].re, (double)rb[a].im};
    }
    if (PF && r + 1 < rounds) {
      __builtin_amdgcn_s_setprio(2);
      fetch(tile_of(r + 1));
      __builtin_amdgcn_s_setprio(0);
    }
    int lo = t;
    // The exchange from the layout at hand into round rd's; each layout is
    // written to the slots it was read from, so only reads need a barrier
    // before them, and none inside a wave (see qg_sweep.hpp).
    auto exchange = [&](auto with_a, auto with_b, const TurnRound* __restrict__ rd) __attribute__((always_inline)) {
      const bool sync = ldc(&rd->sync, 0) != 0;
      auto barrier = [&]() __attribute__((always_inline)) {
        if (sync) {
          __syncthreads();
        } else {
          __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // the compiler keeps the order, no instruction
          __builtin_amdgcn_wave_barrier();
        }
      };
      uint32_t wo[16], ro[16];
      xor_table(wo, ldc(rd->we, 0), ldc(rd->we, 1), ldc(rd->we, 2), ldc(rd->we, 3));
      xor_table(ro, ldc(rd->re, 0), ldc(rd->re, 1), ldc(rd->re, 2), ldc(rd->re, 3));
      uint32_t bw = lds_addr(lds) + (swz<LT>(lidx<R>(tid, 0, lo)) << SH);
      uint32_t br = lds_addr(lds) + (swz<LT>(lidx<R>(tid, 0, ldc(&rd->lo, 0))) << SH);
      asm volatile("" : "+v"(bw), "+v"(br));  // opaque (see lds_transpose)
      if constexpr (HALVES) {
        // real parts, then imaginary parts, unrounded, through the same slots
        auto half = [&](double Cd::*part) __attribute__((always_inline)) {
#pragma unroll
          for (int a = 0; a < A; ++a) lds_st_d(bw ^ wo[a], xa[a].*part);
          barrier();
#pragma unroll
          for (int a = 0; a < A; ++a) xa[a].*part = lds_ld_d(br ^ ro[a]);
        };
        half(&Cd::re);
        barrier();
        asm volatile("" : "+v"(bw), "+v"(br));  // opaque again: shared addresses would all stay live
        half(&Cd::im);
      } else if constexpr (decltype(with_a)::value) {
#pragma unroll
        for (int a = 0; a < A; ++a) Stor<LT>::lds_st_a(bw ^ wo[a], xa[a]);
        barrier();
#pragma unroll
        for (int a = 0; a < A; ++a) xa[a] = Stor<LT>::template lds_ld_a<double>(br ^ ro[a]);
        if (TWO) barrier();
      }
      if constexpr (TWO && decltype(with_b)::value) {
        // opaque again: sharing lambda's addresses with psi's keeps them all live
        asm volatile("" : "+v"(bw), "+v"(br));
#pragma unroll
        for (int a = 0; a < A; ++a) Stor<LT>::lds_st_a(bw ^ wo[a], xb[a]);
        barrier();
#pragma unroll
        for (int a = 0; a < A; ++a) xb[a] = Stor<LT>::template lds_ld_a<double>(br ^ ro[a]);
      }
    };
    // the diagonal operation, in the layout at hand
    auto diagonal = [&]() __attribute__((always_inline)) {
      DiagParts<R> dp;
      uint32_t tl = tid_in;
      asm volatile("" : "+v"(tl));
      diag_prepare<R>(d, gl_tile(tt, c, p, K) | gl_local(lidx<R>(tl, 0, lo), c, p), dp);
      const bool phase = (flags & F_PHASE_PRE) != 0;
      const double gamma = ldc(&d->phase_gamma, 0);
      const int off = ldc(&d->lut_off, 0);
#pragma unroll
      for (int a = 0; a < A; ++a) {
        const double D = diag_value<R>(d, dp, a);
        if constexpr (TWO) {
          if (obs) xb[a] = {D * xa[a].re, D * xa[a].im};
          else accd += 2.0 * D * imcj(xb[a], xa[a]);
        } else {
          if (obs) accd += D * (xa[a].re * xa[a].re + xa[a].im * xa[a].im);
        }
        // taken here, from the unphased states (see run_pass)
        asm volatile("" : "+v"(accd));
        if (phase) {
          Cd ph;
          if constexpr (PH == TP_LUT) {
            const int idx = (int)rint(D) + off;
            ph = {tab[2 * idx], tab[2 * idx + 1]};
          } else {
            double sn, cs;
            if constexpr (PH == TP_SINCOS) sincos_reduced(gamma * D, &sn, &cs);
            else sincos(gamma * D, &sn, &cs);
            ph = {cs, -sn};
          }
          xa[a] = cmul(ph, xa[a]);
          if constexpr (TWO) xb[a] = cmul(ph, xb[a]);
        }
        // one amplitude at a time (register pressure)
        __builtin_amdgcn_sched_barrier(0);
      }
    };
#pragma unroll 1
    for (int q = 0; q < nr; ++q) {
      const TurnRound* __restrict__ rd = &d->r[q];
      const int lo_q = ldc(&rd->lo, 0);
      if (lo_q != lo) exchange(std::true_type{}, std::true_type{}, rd);
      lo = lo_q;
      if (q == dq) diagonal();
      const uint32_t mask = ldc(&rd->mask, 0);
      if constexpr (TWO) {
        double s = 0.0;
        static_for<R>([&](auto kc) __attribute__((always_inline)) {
          constexpr int kk = decltype(kc)::value;
          if ((mask >> kk) & 1u) s += red_bit<R, kk>(xb, xa, G_X);
          asm volatile("" : "+v"(s));  // taken here, before the gates
        });
        if (ldc(&rd->block, 0)) acc1 += s;
        else acc0 += s;
      }
      const double ga = ldc(&rd->a, 0), gb = ldc(&rd->b, 0);
      // psi is needed after the last round only by a diagonal operation there
      const bool rot_a = !TWO || q + 1 < nr || dq == nr;
      static_for<R>([&](auto kc) __attribute__((always_inline)) {
        constexpr int kk = decltype(kc)::value;
        const int ty = (mask >> kk) & 1u ? G_X : G_NONE;
        if (rot_a) gate_bit_s<R, kk>(xa, ty, ga, gb);
        if constexpr (TWO) gate_bit_s<R, kk>(xb, ty, ga, gb);
      });
    }
    if (!TWO && lo != t) {
      exchange(std::true_type{}, std::false_type{}, &d->r[nr]);
      lo = t;
    }
    if (dq == nr) diagonal();
    auto store = [&](void* out, const Cd(&x)[A]) __attribute__((always_inline)) {
      uint32_t adr[A];
      addresses(tt, adr);
#pragma unroll
      for (int a = 0; a < A; ++a) {
        if (BIG) Stor<G>::st_big(out, adr[a], x[a]);
        else Stor<G>::st_o(out, adr[a], x[a]);
      }
    };
    if constexpr (!TWO) {
      store(d->a_out, xa);
    } else if (flags & F_STORE_B) {
      if (lo != t) exchange(std::false_type{}, std::true_type{}, &d->r[nr]);
      store(d->b_out, xb);
    } else {
      __syncthreads();  // the slots of the last layout are still being read
    }
  }
  // fixed order: a thread's tiles in turn, the lanes of a wave, the waves in turn
  if (TWO || obs) {
    double* red = reinterpret_cast<double*>(lds);
    __syncthreads();
    const double v[3] = {wave_sum(TWO ? acc0 : accd, 64), wave_sum(acc1, 64), wave_sum(accd, 64)};
    if ((tid_in & 63u) == 0u)
      for (int i = 0; i < (TWO ? 3 : 1); ++i) red[(tid_in >> 6) * 3 + i] = v[i];
    __syncthreads();
    if (tid_in < (TWO ? 3u : 1u)) {
      double s = 0.0;
      for (uint32_t w = 0; w < nthr / 64; ++w) s += red[w * 3 + tid_in];
      d->part[(size_t)(d->row_base + (int)tid_in) * d->grid + blk] = s;
    }
  }
}

// blockIdx.y selects one of gridDim.y consecutive descriptors (batched circuits).
template <class S, bool TWO, int PH, bool BIG>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(kernel_dtype<S>() == 1 && PH == TP_LUT ? 3 : 2)))
void k_turn(const TurnDesc* __restrict__ d) {
  extern __shared__ __align__(16) char lds_dyn[];
  run_turn<S, TWO, PH, BIG>(d + blockIdx.y, lds_dyn, threadIdx.x, blockIdx.x, gridDim.x);
}

// With occ != NULL nothing is launched: *occ receives the workgroups per CU.
template <class S, bool TWO, int PH, bool BIG>
hipError_t launch_turn_t(const TurnDesc* d, int K, int grid, int batch, hipStream_t st, int* occ, int tab) {
  const int threads = 1 << (K - 4);
  const size_t lds = turn_lds_bytes(kernel_dtype<S>(), K, tab);
  if (occ) return hipOccupancyMaxActiveBlocksPerMultiprocessor(occ, k_turn<S, TWO, PH, BIG>, threads, lds);
  hipLaunchKernelGGL((k_turn<S, TWO, PH, BIG>), dim3(grid, batch), dim3(threads), lds, st, d);
  return hipGetLastError();
}

template <class S, bool TWO, int PH, bool BIG>
hipError_t set_turn_attr_t() {
  return hipFuncSetAttribute(reinterpret_cast<const void*>(&k_turn<S, TWO, PH, BIG>),
                             hipFuncAttributeMaxDynamicSharedMemorySize,
                             (int)turn_lds_bytes(kernel_dtype<S>(), kSweepMaxK, PH == TP_LUT ? 16 * kLutMax : 0));
}

}  // namespace qg
