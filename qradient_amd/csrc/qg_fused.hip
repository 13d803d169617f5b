// Whole-circuit grad_run for states that fit one workgroup (n <= 13).
//
// One workgroup runs one circuit end to end: the 2^n amplitudes stay in
// registers (16 or 8 per thread) and LDS for every layer of the forward sweep,
// the observable and the adjoint sweep, so nothing but the parameters and the
// results crosses HBM.  psi is uncomputed alongside lambda in FP64 (no
// history: unitary FP64 uncompute drifts by ~1e-15 per layer), so complex64
// and complex128 requests give the same FP64-quality result here.  A batch of
// circuits is one launch with one workgroup per circuit.
//
// McClean (reference qradient/circuit_logic/mc_clean.py:47-78): RY(pi/4)
// initial layer (table by popcount), per layer the CNOT ladder as an LDS
// permutation (or the CZ sign) then one rotation per qubit.  QAOA
// (qaoa.py:40-70): |+>, per layer exp(-i gamma C) then RX(beta) on all qubits.
//
// The kernel is bound by latency and by LDS traffic: one workgroup on one CU,
// every layer waiting for the one before.  So the qubit number is a template
// parameter and every layout below is known at compile time:
//
//   layout 0 (natural)  registers hold the top 4 index bits, threads the rest
//   layout 1 (n >= 10)  index bits 4, 5 swapped into registers from the lane
//                       bits with v_permlane16/32_swap: no LDS, no wait
//   layout 2 (n >= 10)  index bits 0-3 in registers: an LDS exchange inside
//                       each wave, so no barrier
//   layout 3 (n >= 12)  the wave bits in registers: an LDS exchange across
//                       waves
//
// and the ladder's permutation (or the plain way back) is the exchange into
// layout 0 of the next layer: three LDS round trips a layer where a stage of
// four bits at a time needs five.  10 and 11 qubits would have one and two
// waves that way and wait alone for every instruction; they hold 8 amplitudes
// per thread (registers: the top 3 bits; bits 0-2, then 3-5, exchanged inside
// the waves; the wave bits) in two and four waves: 97 -> 76 us and 124 -> 94
// us for 10 layers.  At 12 qubits the same form took 126 us against 174 for
// one circuit but 119 against 110 for a batch of 512, which fills the CUs
// either way, so 12 qubits keep 16 per thread.
//
// A layout is written to the slots it was read from, so only reads across
// waves need a barrier.  Up to 11 qubits psi and lambda have a buffer each and
// share their barriers; above, they take turns in one buffer, which leaves
// room for a second workgroup on the CU at 12 qubits.  Rotations are the
// in-place shears of the pass kernels, which need no second copy of the state:
// the earlier form (direct 2x2 products, all gate types joined by branches)
// spilled 259 registers.
//
// Measured (kernel time, MI355X; before -> now): 10 qubits x 10 layers
// 209 -> 76 us, 13 x 20 959 -> 435 us, 64 QAOA circuits of 12 qubits x 4
// layers 476 -> 70 us.  At 13 qubits the two waves of a SIMD issue vector
// instructions in 55% of its cycles; the rest waits on LDS and barriers.
#include "qg_math.hpp"
#include "qg_pass.hpp"

namespace qg {

struct FusedDesc {
  int32_t n, L;
  int32_t ent;            // McClean: 0 CNOT ladder, 1 CZ ladder
  const int32_t* gtype;   // McClean: [L][n] gate type per layer and qubit
  const double* gab;      // tan(phi / 2), sin(phi) of the rotations (see PassDesc::ga):
                          // [L][n][2] (McClean) or [L][2] (QAOA, every qubit's mixer)
  const double* gamma;    // QAOA: [L]
  const DTerm* dterms;    // diagonal observable / classical Hamiltonian
  int32_t ndterms;
  const DTerm* xy;        // x / y terms: a = bit, b = 0 (X) or 1 (Y)
  int32_t nxy;
  int32_t lut_w;          // FM_QAOA_LUT: |C(x)| <= lut_w
  uint32_t lad1, lad2;    // CNOT ladder gather map in shift form (ladder_of)
  uint32_t inv1, inv2;    // and its inverse
  const double* init_tab; // n + 1 entries
  double* out;            // [1 + L*n] (McClean) or [1 + 2L] (QAOA)
  int32_t grad;           // 0: forward and E only
  int32_t psi_c64;        // psi_out element type: 0 complex128, 1 complex64
  void* psi_out;          // final forward state (natural order) or NULL
};

// ---------------------------------------------------------------------------
// layouts
// ---------------------------------------------------------------------------
struct Layout {
  int reg[4];   // index bit held by register bit k
  int thr[16];  // index bit held by thread bit j
};

template <int N>
struct Shape {
  static constexpr int R = N < kRegBits ? N : N == 10 || N == 11 ? 3 : kRegBits;
  static constexpr int T = N - R;              // thread bits
  static constexpr int NT = 1 << T;            // threads
  static constexpr int W = T > 6 ? T - 6 : 0;  // wave bits
  // stages per layer, each with its layout
  static constexpr int NS = N >= 10 ? 4 : T == 0 ? 1 : T <= 4 ? 2 : 3;
  static constexpr bool TWO_BUF = N <= 11;     // psi and lambda have an LDS buffer each
};

template <int N>
constexpr Layout layout(int s) {
  constexpr int R = Shape<N>::R, T = Shape<N>::T, W = Shape<N>::W;
  Layout o{};
  if (N < 10 || s == 0) {
    // registers at [lo, lo + R), threads the rest in order
    int lo = T - R * s;
    if (lo < 0) lo = 0;
    for (int k = 0; k < R; ++k) o.reg[k] = lo + k;
    for (int j = 0; j < T; ++j) o.thr[j] = j < lo ? j : j + R;
    return o;
  }
  for (int k = 0; k < R; ++k) o.reg[k] = T + k;
  for (int j = 0; j < T; ++j) o.thr[j] = j;
  // lanes are ordered so that the first four cover the four low slot bits
  // under the swizzle (no bank conflicts)
  if constexpr (R == 3) {
    if (s < 3) {
      for (int k = 0; k < 3; ++k) o.reg[k] = 3 * (s - 1) + k;
      const int lanes[2][2][6] = {{{3, 4, 5, 9, 7, 8}, {3, 4, 5, 9, 8, 10}}, {{0, 1, 2, 7, 8, 9}, {0, 1, 2, 10, 8, 9}}};
      for (int j = 0; j < 6; ++j) o.thr[j] = lanes[s - 1][N - 10][j];
    } else {
      // the wave bits into registers, filled up with bits 5 and 4
      for (int k = 0; k < 3; ++k) o.reg[k] = k < W ? 6 + k : 5 - (k - W);
      const int lanes[2][6] = {{0, 1, 2, 3, 7, 8}, {0, 1, 2, 3, 4, 8}};
      for (int j = 0; j < 6; ++j) o.thr[j] = lanes[N - 10][j];
      for (int k = 0; k < W; ++k) o.thr[6 + k] = 9 + k;
    }
  } else if (s == 1) {
    o.reg[0] = 4;
    o.reg[1] = 5;
    o.thr[4] = T;
    o.thr[5] = T + 1;
  } else if (s == 2) {
    // lanes: the six bits 4, 5, T .. T + 3
    for (int k = 0; k < 4; ++k) o.reg[k] = k;
    const int lanes[2][6] = {{4, 5, 10, 11, 8, 9}, {4, 5, 10, 11, 9, 12}};
    for (int j = 0; j < 6; ++j) o.thr[j] = lanes[N - 12][j];
  } else {
    // wave bits into registers, register bits into the waves
    for (int k = 0; k < W; ++k) {
      o.reg[k] = 6 + k;
      o.thr[6 + k] = T + k;
    }
  }
  return o;
}

// Register bit k of stage s holds an index bit that no earlier stage held in
// a register: its gate is applied in this stage.
template <int N>
constexpr bool gates_here(int s, int k) {
  const int b = layout<N>(s).reg[k];
  for (int e = 0; e < s; ++e)
    for (int j = 0; j < Shape<N>::R; ++j)
      if (layout<N>(e).reg[j] == b) return false;
  return true;
}

// LDS slot of index j: the bits from 4 up are folded into the low four, so
// that 16 consecutive lanes of every layout above fall on 16 different slots
// modulo 16 (16-byte slots, 64 banks).
template <int N>
__host__ __device__ constexpr uint32_t fslot(uint32_t j) {
  if constexpr (Shape<N>::R == 3) return j ^ (((j >> 4) ^ (j >> 7) ^ (j >> 10)) & 15u);
  else return j ^ (((j >> 4) ^ (j >> 8) ^ (j >> 12)) & 15u);
}

template <int N, int S>
__device__ __forceinline__ uint32_t thread_index(uint32_t tid) {
  uint32_t x = 0;
  static_for<Shape<N>::T>([&](auto jc) __attribute__((always_inline)) {
    constexpr int j = decltype(jc)::value;
    constexpr int b = layout<N>(S).thr[j];
    x |= ((tid >> j) & 1u) << b;
  });
  return x;
}
template <int N, int S>
constexpr uint32_t reg_index(int a) {
  uint32_t x = 0;
  for (int k = 0; k < Shape<N>::R; ++k)
    if ((a >> k) & 1) x |= 1u << layout<N>(S).reg[k];
  return x;
}

// A point past which every thread of the wave (ACROSS: of the workgroup) sees
// the LDS writes before it.  One wave's LDS accesses complete in order, so
// inside a wave only the compiler has to keep the order.
template <bool ACROSS>
__device__ __forceinline__ void lds_point() {
  if constexpr (ACROSS) {
    __syncthreads();
  } else {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
}

template <int N, int S>
__device__ __forceinline__ void put(const Cd (&x)[1 << Shape<N>::R], uint32_t base) {
  // opaque: otherwise the sixteen addresses of every layout are hoisted out of
  // the layer loop, which costs more registers than the XORs cost time
  asm volatile("" : "+v"(base));
  static_for<(1 << Shape<N>::R)>([&](auto ac) __attribute__((always_inline)) {
    constexpr int a = decltype(ac)::value;
    constexpr uint32_t c = fslot<N>(reg_index<N, S>(a)) << 4;
    Stor<double>::lds_st_a(base ^ c, x[a]);
  });
}
template <int N, int S>
__device__ __forceinline__ void get(Cd (&x)[1 << Shape<N>::R], uint32_t base) {
  asm volatile("" : "+v"(base));  // opaque (see put)
  static_for<(1 << Shape<N>::R)>([&](auto ac) __attribute__((always_inline)) {
    constexpr int a = decltype(ac)::value;
    constexpr uint32_t c = fslot<N>(reg_index<N, S>(a)) << 4;
    x[a] = Stor<double>::template lds_ld_a<double>(base ^ c);
  });
}
// reads into layout 0 through the ladder map (m1, m2) of the index
template <int N>
__device__ __forceinline__ void get_map(Cd (&x)[1 << Shape<N>::R], uint32_t base, uint32_t m1, uint32_t m2) {
  asm volatile("" : "+v"(base));  // opaque (see put)
  static_for<(1 << Shape<N>::R)>([&](auto ac) __attribute__((always_inline)) {
    constexpr int a = decltype(ac)::value;
    const uint32_t c = __builtin_amdgcn_readfirstlane(fslot<N>(ladder_of(reg_index<N, 0>(a), m1, m2)) << 4);
    x[a] = Stor<double>::template lds_ld_a<double>(base ^ c);
  });
}

// Swaps register bit k with lane bit 4 (k = 0) and 5 (k = 1) of one FP64
// value pair: the 32-bit halves move with v_permlane16_swap / 32_swap.
template <bool HALF>
__device__ __forceinline__ void swap_lanes(double& lo, double& hi) {
  unsigned long long u = __builtin_bit_cast(unsigned long long, lo), v = __builtin_bit_cast(unsigned long long, hi);
  unsigned r0, r1, q0, q1;
  if constexpr (HALF) {
    auto p = __builtin_amdgcn_permlane32_swap((unsigned)u, (unsigned)v, false, false);
    auto q = __builtin_amdgcn_permlane32_swap((unsigned)(u >> 32), (unsigned)(v >> 32), false, false);
    r0 = p[0], r1 = p[1], q0 = q[0], q1 = q[1];
  } else {
    auto p = __builtin_amdgcn_permlane16_swap((unsigned)u, (unsigned)v, false, false);
    auto q = __builtin_amdgcn_permlane16_swap((unsigned)(u >> 32), (unsigned)(v >> 32), false, false);
    r0 = p[0], r1 = p[1], q0 = q[0], q1 = q[1];
  }
  lo = __builtin_bit_cast(double, (unsigned long long)r0 | ((unsigned long long)q0 << 32));
  hi = __builtin_bit_cast(double, (unsigned long long)r1 | ((unsigned long long)q1 << 32));
}
__device__ __forceinline__ void layout_0_to_1(Cd (&x)[16]) {
#pragma unroll
  for (int a = 0; a < 16; ++a)
    if (!(a & 1)) {
      swap_lanes<false>(x[a].re, x[a | 1].re);
      swap_lanes<false>(x[a].im, x[a | 1].im);
    }
#pragma unroll
  for (int a = 0; a < 16; ++a)
    if (!(a & 2)) {
      swap_lanes<true>(x[a].re, x[a | 2].re);
      swap_lanes<true>(x[a].im, x[a | 2].im);
    }
}

// ---------------------------------------------------------------------------
// one circuit
// ---------------------------------------------------------------------------
// What a kernel runs: the diagonal phase of a QAOA layer from a table
// (integer-valued C), by the reduced sincos, or, for angles past its range,
// by the library's.  Kernels of their own: the code of one in another cost the
// others registers.
enum FusedMode : int32_t {
  FM_MCCLEAN = 0,
  FM_QAOA_LUT = 1,
  FM_QAOA_SINCOS = 2,
  FM_QAOA_LARGE = 3,     // angles past sincos_reduced
  FM_QAOA_LUT_LARGE = 4  // the same, from a table
};

template <int N, int MODE>
struct Fused {
  static constexpr bool QAOA = MODE != FM_MCCLEAN, TABLE = MODE == FM_QAOA_LUT || MODE == FM_QAOA_LUT_LARGE;
  static constexpr int R = Shape<N>::R, A = 1 << R, T = Shape<N>::T, NT = Shape<N>::NT, NS = Shape<N>::NS;
  static constexpr int NW = (NT + 63) / 64;
  static constexpr int WIDTH = NT < 64 ? NT : 64;
  static constexpr bool MANY = NW > 1, TWO_BUF = Shape<N>::TWO_BUF;
  static constexpr uint32_t BUF = 16u << N;
  // LDS: the state buffer(s) at address 0, then [2][N][NW] sums, then the phase table
  static constexpr uint32_t RED = BUF * (TWO_BUF ? 2 : 1);
  static constexpr uint32_t LUT = RED + 2 * 16 * 8 * sizeof(double);

  const FusedDesc& d;
  const uint32_t tid;
  uint32_t b0, b1, b2, b3;  // byte addresses of the thread's amplitude 0 in each layout

  __device__ __forceinline__ Fused(const FusedDesc& d_, uint32_t t) : d(d_), tid(t) {
    b0 = fslot<N>(thread_index<N, 0>(t)) << 4;
    b1 = NS > 1 ? fslot<N>(thread_index<N, (NS > 1 ? 1 : 0)>(t)) << 4 : 0u;
    b2 = NS > 2 ? fslot<N>(thread_index<N, (NS > 2 ? 2 : 0)>(t)) << 4 : 0u;
    b3 = NS > 3 ? fslot<N>(thread_index<N, (NS > 3 ? 3 : 0)>(t)) << 4 : 0u;
  }
  template <int S>
  __device__ __forceinline__ uint32_t base(int buf) const {
    const uint32_t b = S == 0 ? b0 : S == 1 ? b1 : S == 2 ? b2 : b3;
    return b + (TWO_BUF ? buf * BUF : 0u);
  }
  __device__ __forceinline__ double* lds_d(void* lds, uint32_t off) const {
    return reinterpret_cast<double*>(reinterpret_cast<char*>(lds) + off);
  }

  // layout S -> S + 1, of psi and (TWO) lambda
  template <int S, bool TWO>
  __device__ __forceinline__ void next(Cd (&psi)[A], Cd (&lam)[A]) const {
    if constexpr (N >= 10 && R == 4 && S == 0) {
      layout_0_to_1(psi);
      if constexpr (TWO) layout_0_to_1(lam);
    } else {
      constexpr bool across = N >= 10 && S == 2;
      put<N, S>(psi, base<S>(0));
      if constexpr (TWO && TWO_BUF) put<N, S>(lam, base<S>(1));
      lds_point<across>();
      get<N, S + 1>(psi, base<S + 1>(0));
      if constexpr (TWO && TWO_BUF) get<N, S + 1>(lam, base<S + 1>(1));
      if constexpr (TWO && !TWO_BUF) {
        lds_point<across>();
        put<N, S>(lam, base<S>(0));
        lds_point<across>();
        get<N, S + 1>(lam, base<S + 1>(0));
      }
      // a layout is written to the slots it was read from: what comes next
      // needs no point here
      if constexpr (!across) lds_point<false>();
    }
  }

  // the last layout -> layout 0, through the ladder map (MAP) or straight
  template <bool MAP, bool TWO>
  __device__ __forceinline__ void back(Cd (&psi)[A], Cd (&lam)[A], uint32_t m1, uint32_t m2) const {
    const uint32_t mb = MAP ? fslot<N>(ladder_of(thread_index<N, 0>(tid), m1, m2)) << 4 : b0;
    auto rd = [&](Cd (&x)[A], int buf) __attribute__((always_inline)) {
      if constexpr (MAP) get_map<N>(x, mb + (TWO_BUF ? buf * BUF : 0u), m1, m2);
      else get<N, 0>(x, base<0>(buf));
    };
    // in one buffer lambda goes first: it was the last to be read from it, so
    // its slots of this layout are this thread's
    if constexpr (TWO && !TWO_BUF) {
      put<N, NS - 1>(lam, base<NS - 1>(0));
      lds_point<MANY>();
      rd(lam, 0);
      lds_point<MANY>();
    }
    put<N, NS - 1>(psi, base<NS - 1>(0));
    if constexpr (TWO && TWO_BUF) put<N, NS - 1>(lam, base<NS - 1>(1));
    lds_point<MANY>();
    rd(psi, 0);
    if constexpr (TWO && TWO_BUF) rd(lam, 1);
    lds_point<MANY>();
  }

  // The workgroup's sum of v, in every thread.
  __device__ __forceinline__ double block_sum(double v, void* lds) const {
    v = wave_sum(v, WIDTH);
    if constexpr (!MANY) return v;
    double* red = lds_d(lds, RED);
    __syncthreads();
    if ((tid & 63) == 0) red[tid >> 6] = v;
    __syncthreads();
    double s = 0.0;
#pragma unroll
    for (int w = 0; w < NW; ++w) s += red[w];
    __syncthreads();
    return s;
  }

  // The single-qubit layer i: forward (TWO false), or its reductions
  // Im<lam|P_q|psi> and its inverse on both states.  The gates of a layer
  // commute, so each stage reduces and undoes the bits it holds.  Leaves the
  // states in the last layout.  bsum: QAOA, this thread's sum over all qubits.
  template <bool TWO>
  __device__ __forceinline__ void layer_rot(Cd (&psi)[A], Cd (&lam)[A], int i, void* lds, double& bsum) const {
    static_for<NS>([&](auto sc) __attribute__((always_inline)) {
      constexpr int s = decltype(sc)::value;
      if constexpr (s > 0) next<s - 1, TWO>(psi, lam);
      static_for<R>([&](auto kc) __attribute__((always_inline)) {
        constexpr int kk = decltype(kc)::value;
        if constexpr (gates_here<N>(s, kk)) {
          constexpr int q = N - 1 - layout<N>(s).reg[kk];
          const int ty = QAOA ? (int)G_X : ldc(d.gtype, i * N + q);
          double ga = ldc(d.gab, QAOA ? 2 * i : 2 * (i * N + q));
          double gb = ldc(d.gab, QAOA ? 2 * i + 1 : 2 * (i * N + q) + 1);
          if constexpr (TWO) {
            const double v = red_bit<R, kk>(lam, psi, ty);
            if constexpr (QAOA) {
              bsum += v;
              asm volatile("" : "+v"(bsum));  // taken here: sunk past the gates it would keep both states' old values live
            } else {
              const double w = wave_sum(v, WIDTH);
              if constexpr (MANY) {
                if ((tid & 63) == 0) lds_d(lds, RED)[((i & 1) * 16 + q) * 8 + (tid >> 6)] = w;
              } else {
                if (tid == 0) d.out[1 + i * N + q] = w;
              }
            }
            ga = -ga;
            gb = -gb;
          }
          gate_bit_s<R, kk>(psi, ty, ga, gb);
          if constexpr (TWO) gate_bit_s<R, kk>(lam, ty, ga, gb);
        }
      });
    });
  }

  // D(x) of the thread's amplitudes in layout 0.
  __device__ __forceinline__ void diagonal(double (&D)[A]) const {
    const uint32_t x = thread_index<N, 0>(tid);
#pragma unroll
    for (int a = 0; a < A; ++a) D[a] = 0.0;
    const int nt = d.ndterms;
#pragma unroll 1
    for (int k = 0; k < nt; ++k) {
      const DTerm t = ldc(d.dterms, k);
      const uint32_t m = (1u << t.a) | (t.b >= 0 ? 1u << t.b : 0u);
      const double w = flipw(t.w, x & m);
      const uint32_t r = m >> T;  // the register bits of the term
#pragma unroll
      for (int a = 0; a < A; ++a) D[a] += flipw(w, (uint32_t)a & r);
    }
  }

  // This layer's phase table exp(-i g k), k = -W .. W, in LDS (integer D).
  __device__ __forceinline__ void fill_lut(double g, void* lds) const {
    double* lut = lds_d(lds, LUT);
    const int w = d.lut_w;
    lds_point<MANY>();  // the previous layer's reads are done
    for (int k = (int)tid; k <= w; k += NT) {
      double sn, cs;
      if constexpr (MODE == FM_QAOA_LUT) sincos_reduced(g * (double)k, &sn, &cs);
      else sincos_phase(g * (double)k, &sn, &cs);
      lut[2 * (w + k)] = cs;
      lut[2 * (w + k) + 1] = -sn;
      lut[2 * (w - k)] = cs;
      lut[2 * (w - k) + 1] = sn;
    }
    lds_point<MANY>();
  }
  // psi (and with TWO lambda) *= exp(-i g D); with TWO, returns this thread's
  // share of 2 sum D Im(conj(lam) psi), taken first.  One amplitude at a time:
  // the scheduler would otherwise evaluate all sixteen phases ahead of their
  // products and spill.
  template <bool TWO>
  __device__ __forceinline__ double apply_phase(Cd (&psi)[A], Cd (&lam)[A], const double (&D)[A], double g,
                                                void* lds) const {
    double cr = 0.0;
    auto mul = [&](int a, Cd ph) __attribute__((always_inline)) {
      if constexpr (TWO) {
        cr += 2.0 * D[a] * imcj(lam[a], psi[a]);
        asm volatile("" : "+v"(cr));
        lam[a] = cmul(ph, lam[a]);
      }
      psi[a] = cmul(ph, psi[a]);
    };
    if constexpr (TABLE) {
      fill_lut(g, lds);
      const double* lut = lds_d(lds, LUT) + 2 * d.lut_w;
#pragma unroll
      for (int a = 0; a < A; ++a) {
        double Da = D[a];
        asm volatile("" : "+v"(Da));  // opaque: the table addresses are not kept across layers
        const double* e = lut + 2 * (int)Da;
        mul(a, {e[0], e[1]});
        __builtin_amdgcn_sched_barrier(0);
      }
    } else if constexpr (MODE == FM_QAOA_SINCOS) {
#pragma unroll
      for (int a = 0; a < A; ++a) {
        double sn, cs;
        sincos_reduced(g * D[a], &sn, &cs);
        mul(a, {cs, -sn});
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
      // angles past the reduced sincos: one instance of the library's in a
      // rolled loop, its arguments and results in the thread's own LDS slots
      uint32_t bx = b0;
      asm volatile("" : "+v"(bx));
#pragma unroll
      for (int a = 0; a < A; ++a) Stor<double>::lds_st_a(bx ^ (fslot<N>(reg_index<N, 0>(a)) << 4), Cd{g * D[a], 0.0});
      lds_point<false>();
#pragma unroll 1
      for (uint32_t a = 0; a < (uint32_t)A; ++a) {
        const uint32_t at = bx ^ (fslot<N>(a << T) << 4);
        double sn, cs;
        sincos(Stor<double>::template lds_ld_a<double>(at).re, &sn, &cs);
        Stor<double>::lds_st_a(at, Cd{cs, -sn});
      }
      lds_point<false>();
#pragma unroll
      for (int a = 0; a < A; ++a) {
        mul(a, Stor<double>::template lds_ld_a<double>(bx ^ (fslot<N>(reg_index<N, 0>(a)) << 4)));
        __builtin_amdgcn_sched_barrier(0);
      }
      lds_point<false>();
    }
    return cr;
  }

  __device__ __forceinline__ void run(void* lds) const {
    const int L = d.L;
    Cd psi[A], lam[A];
    double none = 0.0;
    const uint32_t x0 = thread_index<N, 0>(tid);
    double D[A];
    if constexpr (QAOA) diagonal(D);
    // ---- initial state; the first layer's ladder is a map of the index ----
#pragma unroll
    for (int a = 0; a < A; ++a) {
      uint32_t x = x0 | ((uint32_t)a << T);
      if (!QAOA && d.ent == 0) x = ladder_of(x, d.lad1, d.lad2);
      psi[a] = {d.init_tab[__popc(x)], 0.0};
    }
    auto cz = [&](Cd (&v)[A]) __attribute__((always_inline)) {
      uint32_t xb = x0;
      asm volatile("" : "+v"(xb));  // opaque: the sixteen signs are not kept across layers
#pragma unroll
      for (int a = 0; a < A; ++a) {
        const double sg = cz_sign(xb | ((uint32_t)a << T), N);
        v[a] = {sg * v[a].re, sg * v[a].im};
      }
    };
    // ---- forward sweep ----
#pragma unroll 1
    for (int i = 0; i < L; ++i) {
      if (i > 0) {
        if (!QAOA && d.ent == 0) back<true, false>(psi, lam, d.lad1, d.lad2);
        else back<false, false>(psi, lam, 0, 0);
      }
      if constexpr (QAOA) {
        apply_phase<false>(psi, lam, D, ldc(d.gamma, i), lds);
      } else if (d.ent != 0) {
        cz(psi);
      }
      layer_rot<false>(psi, lam, i, lds, none);
    }
    back<false, false>(psi, lam, 0, 0);
    // ---- lambda = O psi, E = <psi|O|psi> ----
    if constexpr (!QAOA) diagonal(D);
#pragma unroll
    for (int a = 0; a < A; ++a) lam[a] = {D[a] * psi[a].re, D[a] * psi[a].im};
    if (d.nxy > 0) {
      put<N, 0>(psi, b0);
      lds_point<MANY>();
#pragma unroll 1
      for (int k = 0; k < d.nxy; ++k) {
        const DTerm t = ldc(d.xy, k);
        const uint32_t px = b0 ^ (fslot<N>(1u << t.a) << 4);
        static_for<A>([&](auto ac) __attribute__((always_inline)) {
          constexpr int a = decltype(ac)::value;
          constexpr uint32_t c = fslot<N>(reg_index<N, 0>(a)) << 4;
          const Cd p = Stor<double>::template lds_ld_a<double>(px ^ c);
          if (t.b == 0) {
            lam[a].re += t.w * p.re;
            lam[a].im += t.w * p.im;
          } else {
            const double sg = (((x0 | ((uint32_t)a << T)) >> t.a) & 1u) ? 1.0 : -1.0;
            lam[a].re += t.w * (-sg * p.im);
            lam[a].im += t.w * (sg * p.re);
          }
        });
      }
      lds_point<MANY>();
    }
    double e = 0.0;
#pragma unroll
    for (int a = 0; a < A; ++a) e += psi[a].re * lam[a].re + psi[a].im * lam[a].im;
    e = block_sum(e, lds);
    if (tid == 0) d.out[0] = e;
    if (d.psi_out) {
#pragma unroll
      for (int a = 0; a < A; ++a) {
        const uint32_t x = x0 | ((uint32_t)a << T);
        if (d.psi_c64) Stor<float>::st(d.psi_out, x, psi[a]);
        else Stor<double>::st(d.psi_out, x, psi[a]);
      }
    }
    if (!d.grad) return;
    // ---- adjoint sweep ----
#pragma unroll 1
    for (int i = L - 1; i >= 0; --i) {
      double bsum = 0.0;
      layer_rot<true>(psi, lam, i, lds, bsum);
      if constexpr (QAOA) {
        back<false, true>(psi, lam, 0, 0);
        const double cr = apply_phase<true>(psi, lam, D, -ldc(d.gamma, i), lds);
        const double sb = block_sum(bsum, lds), sc = block_sum(cr, lds);
        if (tid == 0) {
          d.out[1 + 2 * i] = sb;
          d.out[2 + 2 * i] = sc;
        }
      } else {
        if (i > 0 || MANY) {
          // L^-1: the inverse gather of the forward ladder's
          if (d.ent == 0) {
            back<true, true>(psi, lam, d.inv1, d.inv2);
          } else {
            back<false, true>(psi, lam, 0, 0);
            cz(psi);
            cz(lam);
          }
        }
        if constexpr (MANY) {
          // every wave's sums are in LDS (the exchange's barriers are past);
          // the next layer writes the other half
          if (tid < (uint32_t)N) {
            const double* r = lds_d(lds, RED) + ((i & 1) * 16 + tid) * 8;
            double s = 0.0;
#pragma unroll
            for (int w = 0; w < NW; ++w) s += r[w];
            d.out[1 + i * N + (int)tid] = s;
          }
        }
      }
    }
  }
};

template <int N, int MODE>
__global__ __launch_bounds__(Shape<N>::NT < 64 ? 64 : Shape<N>::NT) __attribute__((amdgpu_waves_per_eu(2, 2)))
void k_fused(const FusedDesc* __restrict__ descs) {
  extern __shared__ __align__(16) char lds[];
  const FusedDesc d = descs[blockIdx.x];
  Fused<N, MODE>(d, threadIdx.x).run(lds);
}

// With st_attr the kernel's LDS limit is set instead of a launch (every
// kernel whose LDS may pass the 64 KiB a launch gets without asking).
template <int N, int MODE>
static hipError_t launch_n(const FusedDesc* d, int batch, int lut_w, hipStream_t st, bool st_attr) {
  const int w = st_attr ? kLutMax / 2 : lut_w;
  const size_t lds = (size_t)Fused<N, MODE>::LUT + (Fused<N, MODE>::TABLE ? 16 * (size_t)(2 * w + 1) : 0);
  if (st_attr)
    return lds <= 65536 ? hipSuccess
                        : hipFuncSetAttribute(reinterpret_cast<const void*>(&k_fused<N, MODE>),
                                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  hipLaunchKernelGGL((k_fused<N, MODE>), dim3(batch), dim3(Shape<N>::NT), lds, st, d);
  return hipGetLastError();
}

template <int N>
static hipError_t launch_mode(const FusedDesc* d, int batch, int mode, int lut_w, hipStream_t st, bool st_attr) {
  switch (mode) {
    case FM_MCCLEAN: return launch_n<N, FM_MCCLEAN>(d, batch, lut_w, st, st_attr);
    case FM_QAOA_LUT: return launch_n<N, FM_QAOA_LUT>(d, batch, lut_w, st, st_attr);
    case FM_QAOA_SINCOS: return launch_n<N, FM_QAOA_SINCOS>(d, batch, lut_w, st, st_attr);
    case FM_QAOA_LARGE: return launch_n<N, FM_QAOA_LARGE>(d, batch, lut_w, st, st_attr);
    case FM_QAOA_LUT_LARGE: return launch_n<N, FM_QAOA_LUT_LARGE>(d, batch, lut_w, st, st_attr);
  }
  return hipErrorInvalidValue;
}

static hipError_t launch_any(const FusedDesc* d, int batch, int n, int mode, int lut_w, hipStream_t st, bool st_attr) {
  switch (n) {
#define QG_N(N) case N: return launch_mode<N>(d, batch, mode, lut_w, st, st_attr);
    QG_N(1) QG_N(2) QG_N(3) QG_N(4) QG_N(5) QG_N(6) QG_N(7) QG_N(8) QG_N(9) QG_N(10) QG_N(11) QG_N(12) QG_N(13)
#undef QG_N
  }
  return hipErrorInvalidValue;
}

// lut_w: the largest lut_w of the batch (FM_QAOA_LUT).
hipError_t launch_fused(const void* descs, int batch, int n, int mode, int lut_w, hipStream_t st) {
  if ((mode == FM_QAOA_LUT || mode == FM_QAOA_LUT_LARGE) && (lut_w < 0 || 2 * lut_w + 1 > kLutMax)) return hipErrorInvalidValue;
  return launch_any((const FusedDesc*)descs, batch, n, mode, lut_w, st, false);
}

hipError_t set_fused_attributes() {
  hipError_t e = hipSuccess;
  for (int n = 1; n <= kFusedMaxN && e == hipSuccess; ++n)
    for (int mode = FM_MCCLEAN; mode <= FM_QAOA_LUT_LARGE && e == hipSuccess; ++mode)
      e = launch_any(nullptr, 0, n, mode, 0, nullptr, true);
  return e;
}

size_t fused_desc_size() { return sizeof(FusedDesc); }

}  // namespace qg
