// Register-resident Stockham transforms of a fixed length.
//
// The stages of a length (radix 4, then one radix 2, then radix 3; the engine
// in les_common.h) are taken in phases of consecutive stages.  A phase with
// total radix G that starts at span p splits into n/G closed groups: group i0
// (k = i0 mod p) maps the inputs i0 + t n/G (t < G) to the outputs
// (i0 - k) G + k + c p (c < G).  So one thread holds a group's G values in
// registers for the whole phase, and LDS is touched once between two phases
// instead of once per stage.  Inside a phase stage s (radix R, span P) sees
// G' = G / (radices before it) positions of every sub-problem sp (the outputs
// chosen so far): its butterflies combine positions j + r G'/R with twiddles
// of index k + sp p, and output r goes to sub-problem sp + r (radices before).
// The butterflies, their twiddles and their operands are those of the staged
// engine, so the results are the same bit for bit.
//
// The first stage's twiddles (span 1) are all one and are not multiplied in:
// fma(a, 1, -(b 0)) is a for every finite a and b.
#pragma once
#include "les_common.h"

#define LES_MAX_PHASES 3
// lambdas over register arrays: a call left out of line would move them to scratch
#define LES_INLINE __attribute__((always_inline))

struct PhasePlan {
  int np;                        // phases
  int s[LES_MAX_PHASES + 1];     // first stage of each phase (s[np] = number of stages)
  int g[LES_MAX_PHASES];         // total radix
};

constexpr int ph_prod(int n, int s0, int s1) { int g = 1; for (int s = s0; s < s1; ++s) g *= cp_R(n, s); return g; }

// Two phases with the smallest larger radix, or three when that exceeds maxg
// (the values a thread can hold).
constexpr PhasePlan ph_plan(int n, int maxg) {
  const int nst = cp_nst(n);
  PhasePlan b{1, {0, nst, 0, 0}, {n, 1, 1}};
  if (nst == 1) return b;
  int best = 1 << 30;
  for (int s = 1; s < nst; ++s) {
    const int g0 = ph_prod(n, 0, s), g1 = ph_prod(n, s, nst), m = g0 > g1 ? g0 : g1;
    if (m <= best) { best = m; b = PhasePlan{2, {0, s, nst, 0}, {g0, g1, 1}}; }
  }
  if (best <= maxg || nst == 2) return b;
  best = 1 << 30;
  for (int s = 1; s < nst - 1; ++s)
    for (int t = s + 1; t < nst; ++t) {
      const int g0 = ph_prod(n, 0, s), g1 = ph_prod(n, s, t), g2 = ph_prod(n, t, nst);
      int m = g0 > g1 ? g0 : g1;
      m = (m > g2 ? m : g2) * 4096 + g0 + g1 + g2;
      if (m < best) { best = m; b = PhasePlan{3, {0, s, t, nst}, {g0, g1, g2}}; }
    }
  return b;
}

// groups of phase q per thread when a line has t threads
constexpr int ph_ng(const PhasePlan& p, int n, int q, int t) { return (n / p.g[q] + t - 1) / t; }
// values a thread holds
constexpr int ph_vals(const PhasePlan& p, int n, int t) {
  int e = 0;
  for (int q = 0; q < p.np; ++q) { const int v = ph_ng(p, n, q, t) * p.g[q]; e = v > e ? v : e; }
  return e;
}
// thread time of a line: threads times the values each works on, all phases
constexpr int ph_cost(const PhasePlan& p, int n, int t) {
  int c = 0;
  for (int q = 0; q < p.np; ++q) c += ph_ng(p, n, q, t) * p.g[q];
  return c * t;
}
constexpr int ph_maxg(const PhasePlan& p) {
  int m = 0;
  for (int q = 0; q < p.np; ++q) m = p.g[q] > m ? p.g[q] : m;
  return m;
}
// Threads per line: the least thread time with at most max(G, 18) values per
// thread, the larger count on a tie.  n2 != 0: the same for a pair of lengths
// transformed by the same threads.
constexpr int ph_threads(int n, int n2, int maxg) {
  const PhasePlan a = ph_plan(n, maxg), b = n2 ? ph_plan(n2, maxg) : a;
  int cap = ph_maxg(a) > ph_maxg(b) ? ph_maxg(a) : ph_maxg(b);
  if (cap < 18) cap = 18;
  int best = 1 << 30, bt = 1;
  for (int t = 1; t <= (n > n2 ? n : n2); ++t) {
    if (ph_vals(a, n, t) > cap || (n2 && ph_vals(b, n2, t) > cap)) continue;
    const int c = ph_cost(a, n, t) + (n2 ? ph_cost(b, n2, t) : 0);
    if (c <= best) { best = c; bt = t; }
  }
  return bt;
}

// One phase of one group in registers: X[t] = z[i0 + t N/G] in, X[c] =
// z'[(i0 - k) G + k + c p] out.  tw: the forward table of the plan of length
// N; the inverse takes the conjugates (equal to the inverse table bit for bit).
template <typename T, int N, int S, int SEND, int P0, int G, int DONE, bool INVERSE>
__device__ __forceinline__ void ph_stages(Cplx<T>* X, const Cplx<T>* __restrict__ tw, int k) {
  if constexpr (S < SEND) {
    constexpr int R = cp_R(N, S), P = cp_P(N, S), OFF = cp_OFF(N, S), GREM = G / DONE, M = GREM / R;
    static_assert(P == P0 * DONE, "span of a stage inside its phase");
    Cplx<T> Y[G];
#pragma unroll
    for (int sp = 0; sp < DONE; ++sp) {
      Cplx<T> w[R];
      if constexpr (P > 1) {
#pragma unroll
        for (int r = 1; r < R; ++r) {
          w[r] = tw[OFF + (r - 1) * P + sp * P0 + k];
          if (INVERSE) w[r].y = -w[r].y;
        }
      }
#pragma unroll
      for (int j = 0; j < M; ++j) {
        Cplx<T> x[4];
#pragma unroll
        for (int r = 0; r < R; ++r) {
          x[r] = X[sp * GREM + j + r * M];
          if constexpr (P > 1) {
            if (r > 0) x[r] = c_mul(x[r], w[r]);
          }
        }
        bfly(x, R, INVERSE ? 1 : -1);
#pragma unroll
        for (int r = 0; r < R; ++r) Y[(sp + r * DONE) * M + j] = x[r];
      }
    }
#pragma unroll
    for (int t = 0; t < G; ++t) X[t] = Y[t];
    ph_stages<T, N, S + 1, SEND, P0, G, DONE * R, INVERSE>(X, tw, k);
  }
}

// A line of N values shared by NT threads (this one is number a), through an
// LDS line of its own.  MAXG: the most values per group (the phase split).
// PADX: between two phases the line has one unused slot after every G0 values
// (G0 the first phase's radix, when even), so that neighbouring threads, which
// write at stride G0, meet different banks; the line then holds XLEN values.
template <typename T, int N, int NT, int MAXG, bool PADX = false>
struct RegLine {
  static constexpr PhasePlan plan = ph_plan(N, MAXG);
  static constexpr int PG = PADX && plan.np > 1 && plan.g[0] % 2 == 0 ? plan.g[0] : 0;
  static constexpr int XLEN = N + (PG ? N / PG : 0);
  static constexpr int xstep(int d) { return PG && d % (PG ? PG : 1) == 0 ? d + d / (PG ? PG : 1) : d; }
  static __device__ __forceinline__ int xpos(int e) { return PG ? e + e / (PG ? PG : 1) : e; }
  static constexpr int NP = plan.np, LAST = plan.np - 1;
  static constexpr int VALS = ph_vals(plan, N, NT);
  template <int Q>
  static constexpr int ng() { return ph_ng(plan, N, Q, NT); }
  template <int Q>
  static constexpr int groups() { return N / plan.g[Q]; }
  // the layout a transform ends in is the one it starts from
  static constexpr bool SAME = NP == 2 && plan.g[0] == plan.g[1] && ph_ng(plan, N, 0, NT) == 1;

  // fn(v, r) for every value v this thread holds in the starting (Q = 0) or
  // ending (Q = LAST) layout: its row is a + r, r the same in every thread.
  template <int Q, int GI = 0, typename FN>
  static __device__ __forceinline__ void rows(int a, FN&& fn) {
    if constexpr (GI < ng<Q>()) {
      constexpr int G = plan.g[Q], NGR = N / G;
      if (NGR % NT == 0 || a + NT * GI < NGR) {
#pragma unroll
        for (int t = 0; t < G; ++t) fn(GI * G + t, NT * GI + t * NGR);
      }
      rows<Q, GI + 1>(a, fn);
    }
  }

  // Per group g of a thread, by recursion: with the group's offset in X a
  // constant the arrays stay in registers.
  template <int Q, bool INVERSE, int GI = 0>
  static __device__ __forceinline__ void phase(Cplx<T>* X, const Cplx<T>* __restrict__ tw, int a) {
    if constexpr (GI < ng<Q>()) {
      constexpr int G = plan.g[Q], NGR = N / G, P0 = cp_P(N, plan.s[Q]);
      const int i0 = a + NT * GI;
      if (NGR % NT == 0 || i0 < NGR) {
        const int k = Q == 0 ? 0 : (Q == LAST ? i0 : i0 % P0);
        ph_stages<T, N, plan.s[Q], plan.s[Q + 1], P0, G, 1, INVERSE>(X, tw, k);
      }
      phase<Q, INVERSE, GI + 1>(X + G, tw, a);
    }
  }
  // outputs of phase Q to the line, inputs of phase Q + 1 from it (padded
  // places between two phases; the ending and starting layouts in place)
  template <int Q, int GI = 0>
  static __device__ __forceinline__ void put(const Cplx<T>* X, Cplx<T>* line, int a) {
    if constexpr (GI < ng<Q>()) {
      constexpr int G = plan.g[Q], NGR = N / G, P0 = cp_P(N, plan.s[Q]);
      const int i0 = a + NT * GI;
      if (NGR % NT == 0 || i0 < NGR) {
        const int k = Q == 0 ? 0 : (Q == LAST ? i0 : i0 % P0);
        Cplx<T>* __restrict__ o = line + (Q == LAST ? (i0 - k) * G + k : Q == 0 ? i0 * xstep(G) : xpos((i0 - k) * G + k));
#pragma unroll
        for (int c = 0; c < G; ++c) lds_st(o + c * (Q == LAST ? P0 : xstep(P0)), X[c]);
      }
      put<Q, GI + 1>(X + G, line, a);
    }
  }
  template <int Q, int GI = 0>
  static __device__ __forceinline__ void get(Cplx<T>* X, const Cplx<T>* line, int a) {
    if constexpr (GI < ng<Q>()) {
      constexpr int G = plan.g[Q], NGR = N / G;
      const int i0 = a + NT * GI;
      if (NGR % NT == 0 || i0 < NGR) {
#pragma unroll
        for (int t = 0; t < G; ++t) X[t] = lds_ld(line + (Q == 0 ? i0 + t * NGR : xpos(i0) + t * xstep(NGR)));
      }
      get<Q, GI + 1>(X + G, line, a);
    }
  }
  // The whole transform, X from the starting to the ending layout.  The
  // caller's earlier reads of the lines are behind a sync; after it, so are
  // this transform's (a sync follows every get).
  template <bool INVERSE, typename SYNC>
  static __device__ __forceinline__ void fft(Cplx<T>* X, Cplx<T>* line, const Cplx<T>* __restrict__ tw, int a, SYNC&& sync) {
    phase<0, INVERSE>(X, tw, a);
    if constexpr (NP > 1) {
      put<0>(X, line, a);
      sync();
      get<1>(X, line, a);
      sync();
      phase<1, INVERSE>(X, tw, a);
    }
    if constexpr (NP > 2) {
      put<1>(X, line, a);
      sync();
      get<2>(X, line, a);
      sync();
      phase<2, INVERSE>(X, tw, a);
    }
  }
  // ending layout -> starting layout (between a forward and an inverse transform)
  template <typename SYNC>
  static __device__ __forceinline__ void relay(Cplx<T>* X, Cplx<T>* line, int a, SYNC&& sync) {
    if constexpr (!SAME) {
      put<LAST>(X, line, a);
      sync();
      get<0>(X, line, a);
      sync();
    }
  }
};

// most values per group in the column kernels: FP32 32 (64 VGPRs), FP64 24 (96 VGPRs)
template <typename T>
constexpr int col_maxg() { return sizeof(T) == 4 ? 32 : 24; }

// Addresses: a tile's first plane is the same for the whole block, so every
// access is a uniform base (field, plane, row offset) plus one 32-bit byte
// offset per thread (its column, its plane past the first, its row a).
template <typename T>
__device__ __forceinline__ T at_bytes(const T* base, unsigned off) {
  return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + off);
}
template <typename T>
__device__ __forceinline__ void put_bytes(T* base, unsigned off, T v) {
  *reinterpret_cast<T*>(reinterpret_cast<char*>(base) + off) = v;
}

// Lengths a plan accepts (2^a 3^b, a multiple of 4, 3/2 of it at most
// LES_MAX_N), in parts compiled side by side.
#define LES_LENGTHS_0(X) X(8) X(12) X(16) X(24) X(32) X(36) X(48)
#define LES_LENGTHS_1(X) X(64) X(72) X(96) X(108) X(128) X(144)
#define LES_LENGTHS_2(X) X(192) X(216) X(256) X(288) X(324)
#define LES_LENGTHS_3(X) X(384) X(432) X(512) X(576) X(648)
