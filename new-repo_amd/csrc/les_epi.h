// What the inverse x transforms store besides a plain field: the right-hand
// side update of the stress divergence and the projection of the pressure step.
#pragma once
#include "fft_kernels.h"
#include "fft_reg.h"

// rhs(k) += d/dx tx + d/dy ty + d/dz tz for k = 1..nz, plus the forcing of
// compute_RHS_adv; optionally the pressure BC layers
// (src/compute_derivatives.f90:545-574; src/LES_engine.f90:547-562).
template <typename T>
struct DivEpiArgs {
  double* rhs;
  const T* tz;
  int stag, save_wk;
  double *bottom_wk, *top_wk;
  double cz;
  long np;
  int nz;
  int forcing;  // 1: x forcing, 2: y forcing
  double pf, coriol, geo;
  const double* vel;  // v for x, u for y (Coriolis)
  int coriolis;
};

// Chunks of LES_EPI_CHUNK values of a thread: the loads of a chunk are issued
// together, then its stores.  (One value at a time, the compiler has to keep
// each load behind the store before it, which may alias: the wait for a load
// then waits for that store too.)
#define LES_EPI_CHUNK 4

// rhs(k) += (horizontal divergence) + dz(tz) + forcing, applied as the store
// of the inverse x transform of the divergence spectrum, so the divergence
// never goes through HBM; levels 1..nz+1 (nz+1 only for top_wk).  The thread's
// values: X[v].x at q + r of plane k, X[v].y one row (N) further, (v, r) from
// rows.
template <typename T, int N, int VX, int LO = 0, typename ROWS>
__device__ __forceinline__ void div_epi_rows(const DivEpiArgs<T>& a, int k, long q, ROWS&& rows, const Cplx<T>* X) {
  const long c = (long)k * a.np + q;
  if (k > a.nz) {
    if (a.save_wk)
      rows([&](int v, int r) LES_INLINE {
        a.top_wk[q + r] = (double)X[v].x;
        a.top_wk[q + r + N] = (double)X[v].y;
      });
    return;
  }
  if constexpr (LO < VX) {
    double R[2 * LES_EPI_CHUNK], V[2 * LES_EPI_CHUNK];
    T U[2 * LES_EPI_CHUNK], D[2 * LES_EPI_CHUNK];
    double* __restrict__ rhs = a.rhs + c;
    const T* __restrict__ up = a.stag ? a.tz + c + a.np : a.tz + c;
    const T* __restrict__ dn = a.stag ? a.tz + c : a.tz + c - a.np;
    const double* __restrict__ vel = a.vel + c;
    const bool cor = a.forcing && a.coriolis;
    rows([&](int v, int r) LES_INLINE {
      if (v >= LO && v < LO + LES_EPI_CHUNK) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int i = 2 * (v - LO) + h, o = r + h * N;
          R[i] = rhs[o];
          U[i] = up[o];
          D[i] = dn[o];
          V[i] = cor ? vel[o] : 0.0;
        }
      }
    });
    rows([&](int v, int r) LES_INLINE {
      if (v >= LO && v < LO + LES_EPI_CHUNK) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int i = 2 * (v - LO) + h, o = r + h * N;
          const double dh = h == 0 ? (double)X[v].x : (double)X[v].y;
          double x = R[i] + dh + a.cz * ((double)U[i] - (double)D[i]);
          if (a.forcing) x = x + a.pf;
          if (cor) {
            if (a.forcing == 1) x = x + a.coriol * V[i] - a.coriol * a.geo;
            else x = x - a.coriol * V[i] + a.coriol * a.geo;
          }
          rhs[o] = x;
        }
      }
    });
    if (a.save_wk && k == 1)
      rows([&](int v, int r) LES_INLINE {
        if (v >= LO && v < LO + LES_EPI_CHUNK) {
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const int o = r + h * N;
            const double dh = h == 0 ? (double)X[v].x : (double)X[v].y;
            a.bottom_wk[q + o] = dh + a.cz * ((double)a.tz[c + o] - (double)a.tz[q + o]);
          }
        }
      });
    div_epi_rows<T, N, VX, LO + LES_EPI_CHUNK>(a, k, q, rows, X);
  }
}

template <typename T>
struct DivEpi3 {
  DivEpiArgs<T> c[3];  // per component (blockIdx.y)
};

// ---- the step's projection, fused with the pressure-gradient transforms.
// The x and y components are projected as the store of the inverse x
// transform of i kx phat and i ky phat (blockIdx.y 0 and 1); blockIdx.y 2
// stores p.  The gradient then never goes through HBM: dpdx, dpdy and dpdz
// are formed again from phat and p only when the host asks for them
// (refresh_gradp).  The arithmetic per value is k_proj's.
struct ProjEpiArgs {
  double *vel, *r;          // u or v, rhsx or rhsy (null for the p component)
  const double *rf, *lbc;   // rhs_f, lbc_u or lbc_v
  double* p;                // p (component 2)
  int neu;                  // top BC Neumann
  double ubc;
};
struct ProjEpi3 {
  ProjEpiArgs c[3];
  double dt, t1, t2, dtt, dz;
  long np;
  int nz;
};

// the thread's values as in div_epi_rows
template <int N, int VX, int LO = 0, typename ROWS>
__device__ __forceinline__ void proj_epi_rows(const ProjEpi3& e, const ProjEpiArgs& a, int k, long q, ROWS&& rows,
                                              const Cplx<double>* X) {
  const long c = (long)k * e.np + q;
  if (a.p) {
    double* __restrict__ p = a.p + c;
    rows([&](int v, int r) LES_INLINE {
      p[r] = X[v].x;
      p[r + N] = X[v].y;
    });
    return;
  }
  if (k < 1 || k > e.nz) return;
  if constexpr (LO < VX) {
    double R[2 * LES_EPI_CHUNK], U[2 * LES_EPI_CHUNK], P[2 * LES_EPI_CHUNK];
    double* __restrict__ vel = a.vel + c;
    double* __restrict__ rhs = a.r + c;
    const double* __restrict__ rf = a.rf + c;
    rows([&](int v, int r) LES_INLINE {
      if (v >= LO && v < LO + LES_EPI_CHUNK) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int i = 2 * (v - LO) + h, o = r + h * N;
          R[i] = rhs[o];
          U[i] = vel[o];
          P[i] = rf[o];
        }
      }
    });
    rows([&](int v, int r) LES_INLINE {
      if (v >= LO && v < LO + LES_EPI_CHUNK) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int i = 2 * (v - LO) + h, o = r + h * N;
          const double g = h == 0 ? X[v].x : X[v].y;
          double us = U[i];
          us = us + e.dt * (e.t1 * R[i] + e.t2 * P[i]);
          const double un = us - e.dtt * g;
          rhs[o] = R[i] - g;
          vel[o] = un;
          // the ghost plane's values (planes 0 and nz + 1 have no other writer)
          if (k == 1) a.vel[q + o] = un - a.lbc[q + o] * e.dz;
          if (k == e.nz) vel[o + e.np] = a.neu ? un + a.ubc * e.dz : 2.0 * a.ubc - un;
        }
      }
    });
    proj_epi_rows<N, VX, LO + LES_EPI_CHUNK>(e, a, k, q, rows, X);
  }
}

// The same for items in another order: item u has z.x at in-plane point q of
// plane k, z.y one row (N) further.
template <int N>
__device__ __forceinline__ void proj_epi_chunk(const ProjEpi3& e, const ProjEpiArgs& a, const int* k, const int* q,
                                               const bool* ok, const Cplx<double>* z) {
  if (a.p) {
#pragma unroll
    for (int u = 0; u < LES_EPI_CHUNK; ++u)
      if (ok[u]) {
        const long c = (long)k[u] * e.np + q[u];
        a.p[c] = z[u].x;
        a.p[c + N] = z[u].y;
      }
    return;
  }
  double R[2 * LES_EPI_CHUNK], U[2 * LES_EPI_CHUNK], P[2 * LES_EPI_CHUNK];
#pragma unroll
  for (int u = 0; u < LES_EPI_CHUNK; ++u)
    if (ok[u] && k[u] >= 1 && k[u] <= e.nz) {
      const long c = (long)k[u] * e.np + q[u];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        R[2 * u + h] = a.r[c + h * N];
        U[2 * u + h] = a.vel[c + h * N];
        P[2 * u + h] = a.rf[c + h * N];
      }
    }
#pragma unroll
  for (int u = 0; u < LES_EPI_CHUNK; ++u)
    if (ok[u] && k[u] >= 1 && k[u] <= e.nz) {
      const long c = (long)k[u] * e.np + q[u];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const long o = c + h * N;
        const double g = h == 0 ? z[u].x : z[u].y;
        double us = U[2 * u + h];
        us = us + e.dt * (e.t1 * R[2 * u + h] + e.t2 * P[2 * u + h]);
        const double un = us - e.dtt * g;
        a.r[o] = R[2 * u + h] - g;
        a.vel[o] = un;
        // the ghost planes' values (planes 0 and nz + 1 have no other writer)
        if (k[u] == 1) a.vel[q[u] + h * N] = un - a.lbc[q[u] + h * N] * e.dz;
        if (k[u] == e.nz) a.vel[o + e.np] = a.neu ? un + a.ubc * e.dz : 2.0 * a.ubc - un;
      }
    }
}
