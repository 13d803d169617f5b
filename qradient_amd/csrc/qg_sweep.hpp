// Multi-layer passes of the McClean circuit.
//
// A pass of qg_pass.hpp applies one layer's gates on the bits it holds, so a
// layer costs two or three reads and writes of the state and the passes run at
// the copy rate of the memory.  But a layer of the circuit (the CNOT or CZ
// ladder, one rotation per qubit) only couples neighbouring bits, so a tile
// that holds a window of consecutive bits can run several layers on it: at
// each layer every bond inside the window (or whose control is the tile bit
// just above it) and every rotation whose bonds are done.  The windows of
// successive passes overlap in a staircase, like the blocks of a stencil
// blocked in time; the planner (qg_sweep_plan.hpp) picks them.  At 24
// qubits and 20 layers this takes 18 passes where one layer at a time takes
// 60.
//
// A pass is a list of rounds.  A round holds four local bits in registers (16
// amplitudes per thread), reached by an LDS exchange, and rotates each once.
// The CNOTs before a round are a GF(2)-linear map of the local index (at most
// one bond of each of the ladder's two groups per bit, so the shift form of
// ladder_of holds), applied by the exchange's read addresses; the CNOTs before
// the first round are applied by the global load's addresses (forward) or the
// store's (adjoint).  Every target lies inside the window, so a tile only ever
// moves inside itself and passes may work in place.  A CZ ladder's signs are
// applied in registers.
//
// The adjoint pass runs the rounds backwards on psi (the forward pass's
// output) and lambda, taking each reduction Im<lam|P_q|psi> (the reference's
// gradient entries, mc_clean.py:68-76) where its bit is in registers.  psi is
// rotated back inside the tile and not stored (history mode), or stored
// (checkpoint mode).  The adjoint of the circuit's last pass forms lambda =
// D psi and E itself where the observable is diagonal (OBS).
//
// A complex64 forward pass (F32L64) keeps tiles of 8 bytes an amplitude: it moves
// the FP64 real parts through them and then the imaginary parts, so psi is
// rounded where it is stored and nowhere else; the adjoint rounds both states to
// FP32 at every exchange, as a pass of one layer does.  A pass of several layers
// has up to 14 exchanges, which in FP32 make a forward circuit less accurate than
// one layer at a time: geometric mean of the gradient's error over seeds, one
// layer at a time | FP32 forward exchanges | now: 18 qubits, 12 layers 1.78e-7 |
// 1.94e-7 | 1.20e-7; 24 qubits, 40 layers 6.14e-7 | 6.26e-7 | 3.87e-7; 25 qubits,
// 10 layers 1.83e-8 | 2.29e-8 | 1.15e-8.  It costs 1 to 3% of a gradient run (16
// qubits 553 -> 557 us, 24 qubits, 40 layers 10.65 -> 10.90 ms).  The adjoint's psi
// in halves too costs another 3 to 5% and leaves these errors as they are (24
// qubits, with FP32 forward exchanges: 6.26e-7 either way).
//
// Bound: the vector ALU.  A round costs 4 x 48 FMAs per thread and state and
// an exchange of about 130 instructions (in FP32 half of them conversions); the
// adjoint adds 4 x 32 FMAs of reductions.  The four sums of a round are reduced
// across the wave together: two lane swaps fold four values into one register,
// so they cost 21 instructions instead of 88.  Measured at 24 qubits, complex64,
// per layer: forward 145 -> 86 us (92 with FP64 exchanges), adjoint 288 -> 200 us.
#pragma once
#include "qg_pass.hpp"

namespace qg {

// The sixteen XOR combinations of four scalars, in scalar registers.
__device__ __forceinline__ void xor_table(uint32_t (&o)[16], uint32_t e0, uint32_t e1, uint32_t e2, uint32_t e3) {
  o[0] = 0;
  o[1] = e0;
  o[2] = e1;
  o[4] = e2;
  o[8] = e3;
  o[3] = e0 ^ e1;
  o[5] = e0 ^ e2;
  o[6] = e1 ^ e2;
  o[7] = o[3] ^ e2;
#pragma unroll
  for (int a = 1; a < 8; ++a) o[8 + a] = o[a] ^ e3;
#pragma unroll
  for (int a = 0; a < 16; ++a) o[a] = __builtin_amdgcn_readfirstlane(o[a]);
}

// Four values summed over the wave at once: lane 16 r holds the total of value
// {0, 2, 1, 3}[r].  v_permlane32_swap and v_permlane16_swap fold pairs of
// values into one register each, then four steps inside the rows of 16.
__device__ __forceinline__ double fold_half(double x, double y) {
  const unsigned long long u = __builtin_bit_cast(unsigned long long, x), v = __builtin_bit_cast(unsigned long long, y);
  const auto p = __builtin_amdgcn_permlane32_swap((unsigned)u, (unsigned)v, false, false);
  const auto q = __builtin_amdgcn_permlane32_swap((unsigned)(u >> 32), (unsigned)(v >> 32), false, false);
  return __builtin_bit_cast(double, (unsigned long long)p[0] | ((unsigned long long)q[0] << 32)) +
         __builtin_bit_cast(double, (unsigned long long)p[1] | ((unsigned long long)q[1] << 32));
}
__device__ __forceinline__ double fold_row(double x, double y) {
  const unsigned long long u = __builtin_bit_cast(unsigned long long, x), v = __builtin_bit_cast(unsigned long long, y);
  const auto p = __builtin_amdgcn_permlane16_swap((unsigned)u, (unsigned)v, false, false);
  const auto q = __builtin_amdgcn_permlane16_swap((unsigned)(u >> 32), (unsigned)(v >> 32), false, false);
  return __builtin_bit_cast(double, (unsigned long long)p[0] | ((unsigned long long)q[0] << 32)) +
         __builtin_bit_cast(double, (unsigned long long)p[1] | ((unsigned long long)q[1] << 32));
}
__device__ __forceinline__ double wave_sum4(double v0, double v1, double v2, double v3) {
  double v = fold_row(fold_half(v0, v1), fold_half(v2, v3));
  v += dpp_d<0xB1, 0xF>(v);
  v += dpp_d<0x4E, 0xF>(v);
  v += dpp_d<0x141, 0xF>(v);
  v += dpp_d<0x140, 0xF>(v);
  return v;
}
__device__ __forceinline__ int wave_sum4_slot(uint32_t tid) {  // the value whose total the lane's row holds
  const uint32_t r = (tid >> 4) & 3u;
  return (int)(((r & 1u) << 1) | (r >> 1));
}

// One FP64 value by absolute LDS address.
__device__ __forceinline__ void lds_st_d(uint32_t addr, double v) {
  *(__attribute__((address_space(3))) double*)(uintptr_t)addr = v;
}
__device__ __forceinline__ double lds_ld_d(uint32_t addr) {
  return *(const __attribute__((address_space(3))) double*)(uintptr_t)addr;
}

// LDS bytes of a pass: the tile, the per-wave sums and the initial-state table.
__host__ __device__ inline size_t sweep_lds_bytes(int dtype, int K, bool two, int tab_bytes) {
  return (size_t)(1u << K) * (dtype == 1 || sweep_halves(dtype, two) ? 8 : 16) +
         (two ? (size_t)(1u << (K - 4)) / 64 * kMaxRounds * 4 * 8 : 0) + (size_t)tab_bytes;
}

template <class S, bool TWO, bool BIG, bool OBS>
__device__ __forceinline__ void run_sweep(const SweepDesc* __restrict__ d, void* lds, uint32_t tid_in, uint32_t blk,
                                          uint32_t nblk) {
  constexpr int R = 4, A = 16;
  typedef typename Store<S>::G G;   // HBM element type
  typedef typename Store<S>::L LT;  // LDS tile element type
  constexpr int GSH = sizeof(G) == 4 ? 3 : 4;
  constexpr bool PF = !TWO;  // the next tile's loads in flight while this one is worked on
  // the exchange moves FP64 halves of an amplitude (see above)
  constexpr bool HALVES = sweep_halves(kernel_dtype<S>(), TWO);
  typedef typename std::conditional<HALVES, float, LT>::type SL;  // whose complex values fill an LDS slot
  constexpr int SH = sizeof(SL) == 4 ? 3 : 4;
  warm_lines<(int)sizeof(SweepDesc)>(d);
  const int n = d->n, K = d->K, t = d->t, c = d->c, p = d->p;
  const uint32_t flags = d->flags;
  const uint32_t ntiles = 1u << (n - K);
  const uint32_t nthr = blockDim.x;
  const int nr = d->nr;
  double* wacc = reinterpret_cast<double*>(reinterpret_cast<char*>(lds) + (1u << (K + SH)));
  double* itab = wacc + (TWO ? (nthr / 64) * kMaxRounds * 4 : 0);
  if constexpr (TWO) {
    for (uint32_t i = tid_in; i < (nthr / 64) * kMaxRounds * 4; i += nthr) wacc[i] = 0.0;
    __syncthreads();
  }
  const bool init = !TWO && (flags & F_INIT_TAB);
  if (init) {
    for (int i = (int)tid_in; i <= n; i += (int)nthr) itab[i] = d->init_tab[i];
    __syncthreads();
  }
  int rpos[R];
  uint32_t rbit[R];
#pragma unroll
  for (int k = 0; k < R; ++k) {
    rpos[k] = gpos_of_local(t + k, c, p);
    rbit[k] = 1u << rpos[k];
  }
  const bool nt_a = (flags & F_NT_A) != 0;
  // tile order as in run_pass
  const bool xcd = (flags & F_XCD_ORDER) && (nblk >= 8) && (nblk % 8 == 0) && (ntiles % nblk == 0);
  const uint32_t per_x = ntiles / 8, slots = nblk / 8;
  const uint32_t rounds = xcd ? ntiles / nblk : (blk < ntiles ? (ntiles - 1 - blk) / nblk + 1 : 0u);
  auto tile_of = [&](uint32_t r) -> uint32_t {
    return xcd ? (blk % 8) * per_x + r * slots + blk / 8 : blk + r * nblk;
  };
  // global addresses of a thread's amplitudes in the natural layout, through
  // the index map when `map`
  auto addresses = [&](bool map, uint32_t g, uint32_t(&adr)[A], auto shc) __attribute__((always_inline)) {
    constexpr int AS = decltype(shc)::value;
    uint32_t o[16];
    uint32_t e[4];
    const uint32_t m1 = map ? ldc(&d->g1, 0) : 0u, m2 = map ? ldc(&d->g2, 0) : 0u;
#pragma unroll
    for (int k = 0; k < 4; ++k) e[k] = ladder_of(rbit[k], m1, m2) << AS;
    xor_table(o, e[0], e[1], e[2], e[3]);
    uint32_t base = ladder_of(g, m1, m2) << AS;
    asm volatile("" : "+v"(base));  // opaque (see lds_transpose)
#pragma unroll
    for (int a = 0; a < A; ++a) adr[a] = base ^ o[a];
  };
  Cx<G> ra[A];
  Cx<G> rb[TWO ? A : 1];
  auto fetch = [&](uint32_t tt) __attribute__((always_inline)) {
    uint32_t tid = tid_in;
    asm volatile("" : "+v"(tid));
    uint32_t adr[A];
    addresses(!TWO && (flags & F_GATHER), gl_tile(tt, c, p, K) | gl_local(tid, c, p), adr, ic<BIG ? 0 : GSH>{});
    if (init) {
#pragma unroll
      for (int a = 0; a < A; ++a) ra[a] = {(G)0, (G)0};
    } else if (nt_a) {
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
#pragma unroll
      for (int a = 0; a < A; ++a)
        rb[a] = OBS   ? Cx<G>{(G)0, (G)0}
                : BIG ? Stor<G>::template ld_big<G>(d->b_in, adr[a])
                      : Stor<G>::template ld_o<G>(d->b_in, adr[a]);
    }
  };
  double energy = 0.0;  // OBS: this thread's share of E
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
    const uint32_t gthr = gl_tile(tt, c, p, K) | gl_local(tid, c, p);
    Cd xa[A];
    Cd xb[TWO ? A : 1];
    if (init) {
      uint32_t adr[A];
      addresses((flags & F_GATHER) != 0, gthr, adr, ic<0>{});
#pragma unroll
      for (int a = 0; a < A; ++a) xa[a] = {itab[__popc(adr[a])], 0.0};
    } else {
#pragma unroll
      for (int a = 0; a < A; ++a) xa[a] = {(double)ra[a].re, (double)ra[a].im};
    }
    if constexpr (OBS) {
      const DiagForm* __restrict__ form = d->obs;
      DiagParts<R> dp;
      diag_prepare<R>(form, gthr, dp);
#pragma unroll
      for (int a = 0; a < A; ++a) {
        const double D = diag_value<R>(form, dp, a);
        xb[a] = {D * xa[a].re, D * xa[a].im};
        energy += xa[a].re * xb[a].re + xa[a].im * xb[a].im;
        asm volatile("" : "+v"(energy));  // one amplitude at a time (register pressure)
        __builtin_amdgcn_sched_barrier(0);
      }
    } else if constexpr (TWO) {
#pragma unroll
      for (int a = 0; a < A; ++a) xb[a] = {(double)rb[a].re, (double)rb[a].im};
    }
    if (PF && r + 1 < rounds) {
      __builtin_amdgcn_s_setprio(2);
      fetch(tile_of(r + 1));
      __builtin_amdgcn_s_setprio(0);
    }
    // the tile bit above the window (bit K of the index maps)
    const uint32_t above = d->hi < 32 ? (gl_tile(tt, c, p, K) >> d->hi) & 1u : 0u;

    // The exchange into round rd, from register bits [lo_from, +4), through
    // the round's index map.  Each layout is written to the slots it was read
    // from, so only reads need a barrier before them, and mapped reads one
    // after them.  Where both layouts give the same bits to the wave index and
    // the map leaves those bits alone, a wave only meets its own slots, and
    // the LDS runs one wave's accesses in order: no barrier at all (adjoint passes of 24 qubits,
    // complex64: 222 -> 218 us).
    auto exchange = [&](auto with_a, auto with_b, const SweepRound* __restrict__ rd, int lo_from) __attribute__((always_inline)) {
      const uint32_t m1 = ldc(&rd->m1, 0), m2 = ldc(&rd->m2, 0);
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
      uint32_t bw = lds_addr(lds) + (swz<SL>(lidx<R>(tid, 0, lo_from)) << SH);
      uint32_t br = lds_addr(lds) +
                    ((swz<SL>(ladder_of(lidx<R>(tid, 0, ldc(&rd->lo, 0)), m1, m2)) << SH) ^ (above ? ldc(&rd->off, 0) : 0u));
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
      if (m1 | m2) barrier();
    };
    int lo = t;
#pragma unroll 1
    for (int q = 0; q < nr; ++q) {
      const SweepRound* __restrict__ rd = &d->r[q];
      const int lo_q = ldc(&rd->lo, 0);
      const uint32_t m1 = ldc(&rd->m1, 0), m2 = ldc(&rd->m2, 0);
      if (lo_q != lo || (m1 | m2)) exchange(std::true_type{}, std::true_type{}, rd, lo);
      lo = lo_q;
      const uint32_t cz = ldc(&rd->cz, 0);
      auto signs = [&]() __attribute__((always_inline)) {
        // sign of the bonds in cz, by the parity of x & (x >> 1)
        uint32_t l0 = lidx<R>(tid, 0, lo);
        const uint32_t gx = gl_tile(tt, c, p, K) | gl_local(l0, c, p);
#pragma unroll
        for (int a = 0; a < A; ++a) {
          const uint32_t x = gx | __builtin_amdgcn_readfirstlane(gl_local((uint32_t)a << lo, c, p));
          const uint64_t sb = (uint64_t)(__popc(x & (x >> 1) & cz) & 1) << 63;
          auto flip = [&](double v) { return __longlong_as_double(__double_as_longlong(v) ^ (long long)sb); };
          xa[a] = {flip(xa[a].re), flip(xa[a].im)};
          if constexpr (TWO) xb[a] = {flip(xb[a].re), flip(xb[a].im)};
        }
      };
      if (!TWO && cz) signs();
      if constexpr (TWO) {
        double v[4];
        static_for<R>([&](auto kc) __attribute__((always_inline)) {
          constexpr int kk = decltype(kc)::value;
          v[kk] = red_bit<R, kk>(xb, xa, ldc(rd->type, kk));
          asm volatile("" : "+v"(v[kk]));  // taken here, before the gates
        });
        const double s = wave_sum4(v[0], v[1], v[2], v[3]);
        if ((tid & 15u) == 0u) lds_add(&wacc[((tid >> 6) * kMaxRounds + q) * 4 + wave_sum4_slot(tid)], s);
      }
      // psi is needed after the last round's reductions only if it is stored
      const bool rot_a = !TWO || q + 1 < nr || (flags & F_STORE_A);
      static_for<R>([&](auto kc) __attribute__((always_inline)) {
        constexpr int kk = decltype(kc)::value;
        const int ty = ldc(rd->type, kk);
        const double ga = ldc(rd->a, kk), gb = ldc(rd->b, kk);
        if (rot_a) gate_bit_s<R, kk>(xa, ty, ga, gb);
        if constexpr (TWO) gate_bit_s<R, kk>(xb, ty, ga, gb);
      });
      if (TWO && cz) signs();
    }
    // back to the natural layout and out, psi before lambda: psi's registers
    // are free by then, and a join over whether it is stored costs a copy of it
    auto store = [&](void* out, const Cd(&x)[A]) __attribute__((always_inline)) {
      uint32_t gst = gthr;
      asm volatile("" : "+v"(gst));
      uint32_t adr[A];
      addresses(TWO && (flags & F_SCATTER), gst, adr, ic<BIG ? 0 : GSH>{});
#pragma unroll
      for (int a = 0; a < A; ++a) {
        if (BIG) Stor<G>::st_big(out, adr[a], x[a]);
        else Stor<G>::st_o(out, adr[a], x[a]);
      }
    };
    // a mapped pass without an exchange: every load of the tile before any store
    if (flags & F_SWEEP_SYNC) __syncthreads();
    if (!TWO || (flags & F_STORE_A)) {
      if (lo != t) exchange(std::true_type{}, std::false_type{}, &d->r[nr], lo);
      store(d->a_out, xa);
    }
    if constexpr (TWO) {
      if (flags & F_STORE_B) {
        if (lo != t) exchange(std::false_type{}, std::true_type{}, &d->r[nr], lo);
        store(d->b_out, xb);
      } else {
        __syncthreads();  // the slots of the last layout are still being read
      }
    }
  }
  if constexpr (TWO) {
    // fixed order: a wave's tiles in turn (above), then the waves in turn
    __syncthreads();
    for (uint32_t i = tid_in; i < (uint32_t)nr * 4u; i += nthr) {
      double v = 0.0;
      for (uint32_t w = 0; w < nthr / 64; ++w) v += wacc[w * kMaxRounds * 4 + i];
      d->part[(size_t)(d->row_base + (int)i) * d->grid + blk] = v;
    }
  }
  if constexpr (OBS) {
    double* red = reinterpret_cast<double*>(lds);  // the tile is done with
    const double w = wave_sum(energy, 64);
    if ((tid_in & 63u) == 0u) red[tid_in >> 6] = w;
    __syncthreads();
    if (tid_in == 0) {
      double v = 0.0;
      for (uint32_t i = 0; i < nthr / 64; ++i) v += red[i];
      d->part[(size_t)(d->row_base + nr * 4) * d->grid + blk] = v;
    }
  }
}

// blockIdx.y selects one of gridDim.y consecutive descriptors (batched
// circuits).  Three waves per SIMD where the LDS tiles allow it (8-byte slots):
// the complex64 adjoint at 24 qubits took 262 us per pass with 177 registers
// (two waves) and takes 222 us with at most 168.
template <class S, bool TWO, bool BIG, bool OBS>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(
    kernel_dtype<S>() == 1 || sweep_halves(kernel_dtype<S>(), TWO) ? 3 : 2)))
void k_sweep(const SweepDesc* __restrict__ d) {
  extern __shared__ __align__(16) char lds_dyn[];
  run_sweep<S, TWO, BIG, OBS>(d + blockIdx.y, lds_dyn, threadIdx.x, blockIdx.x, gridDim.x);
}

// With occ != NULL nothing is launched: *occ receives the workgroups per CU.
template <class S, bool TWO, bool BIG, bool OBS>
hipError_t launch_sweep_t(const SweepDesc* d, int K, int grid, int batch, hipStream_t st, int* occ, int tab) {
  const int threads = 1 << (K - 4);
  const size_t lds = sweep_lds_bytes(kernel_dtype<S>(), K, TWO, tab);
  if (occ) return hipOccupancyMaxActiveBlocksPerMultiprocessor(occ, k_sweep<S, TWO, BIG, OBS>, threads, lds);
  hipLaunchKernelGGL((k_sweep<S, TWO, BIG, OBS>), dim3(grid, batch), dim3(threads), lds, st, d);
  return hipGetLastError();
}

template <class S, bool TWO, bool BIG, bool OBS>
hipError_t set_sweep_attr_t() {
  return hipFuncSetAttribute(reinterpret_cast<const void*>(&k_sweep<S, TWO, BIG, OBS>),
                             hipFuncAttributeMaxDynamicSharedMemorySize,
                             (int)sweep_lds_bytes(kernel_dtype<S>(), kSweepMaxK, TWO, 8 * (kMaxQubits + 1)));
}

}  // namespace qg
