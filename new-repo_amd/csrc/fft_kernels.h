// Arguments and point-wise parts of the batched horizontal transform kernels
// (rows_reg.h, cols_reg.h, colres_reg.h).
//
// Replaces the reference's FFTW/2DECOMP path (src/decomp_2d_fft_2d.f90:397-577
// r2c_1d_x / c2c_1d_y / c2r_1d_x, src/compute_convective_padd.f90:274-388
// transpose_to_big / dealias): the pencil transposes become strided column
// passes over a single device allocation.
//
// Layout: a real field is (nx, ny, planes) with x fastest; a spectral field is
// (lhx, ny, planes) complex, lhx = nx/2 + 1.  Row kernels take row pairs
// (j, j+1) of a plane as one complex line z = a + i b; column kernels take a
// block of adjacent kx columns, counted through the planes.
#pragma once
#include "les_common.h"

#define LES_BLOCK 256
// fields a launch takes (the dynamic models filter up to 21 at once, two results each)
#define LES_MAX_FIELDS 6
#define LES_R2C_FIELDS 21
#define LES_C2R_FIELDS 42
#define LES_COL_JOBS 21

// ------------------------------------------------------------------ row r2c
// Load modes of the real input.
// LOAD_AB2_SCALE_DIV: the AB2 predictor u + dt (t1 r + t2 r_f) of each
// value (the arithmetic of k_ab2, src/LES_engine.f90:253-283), then
// LOAD_SCALE_DIV: the pressure right-hand side straight from u, rhs, rhs_f.
// LOAD_PCLEAN: the TKE budget's cleaned pressure
// p - (u u + v v + W W) / 2, W = (w(k) + w(k+1)) / 2, from p (src) and u, v, w
// (ab_r), 0 on the planes 0 and nz+1.
enum { LOAD_SCALE = 0, LOAD_SCALE_DIV = 1, LOAD_AB2_SCALE_DIV = 2, LOAD_PCLEAN = 3 };
// the load modes compiled for transforms of precision T
template <typename T>
constexpr bool r2c_has(int mode) { return sizeof(T) == 8 ? mode >= LOAD_SCALE && mode <= LOAD_PCLEAN : mode == LOAD_SCALE; }

template <typename TI, typename T>
struct RowR2CArgs {
  const TI* src[LES_R2C_FIELDS];
  Cplx<T>* dst[LES_R2C_FIELDS];
  int nx, ny, lhx;
  int k0, nplanes;  // planes [k0, k0+nplanes)
  T scale, div;
  const TI* ab_r[3];  // LOAD_AB2_SCALE_DIV: rhs and rhs_f of field f
  const TI* ab_f[3];
  T ab_dt, ab_t1, ab_t2;
  int pc_nz;          // LOAD_PCLEAN: nz (planes 0 and nz+1 are ghosts)
  // k_rows_r2c_nyq: the FP64 Nyquist sums of the raw input (row sums A,
  // column partials P of each band of 8 rows), and the strides between fields
  double *nyq_a, *nyq_p;
  long nyq_as, nyq_ps;
};

// ------------------------------------------------------------------ row c2r
template <typename T, typename TO>
struct RowC2RArgs {
  const Cplx<T>* src[LES_C2R_FIELDS];
  TO* dst[LES_C2R_FIELDS];
  int nx, ny, lhx;
  int k0, nplanes;
};

// ------------------------------------------------------------------ columns
// Spectral-space operations applied between the forward and inverse y passes.
enum { COP_GRAD = 0, COP_DIV = 1, COP_FILT2 = 2, COP_FILT1 = 3, COP_COPY = 4, COP_PGRAD = 5 };

// The instances (op, outputs, forward and inverse transform) a step uses: FP32
// has no pressure operations, FP64 no two-output gradient.
#define LES_COL_INSTANCES(X)                                                                                     \
  X(COP_DIV, 1, true, true) X(COP_FILT1, 1, true, true) X(COP_FILT2, 2, true, true) X(COP_COPY, 1, true, false)   \
  X(COP_COPY, 1, false, true)
#define LES_COL_INSTANCES_F32(X) X(COP_GRAD, 2, true, true)
#define LES_COL_INSTANCES_F64(X) X(COP_GRAD, 3, true, true) X(COP_DIV, 1, true, false) X(COP_PGRAD, 3, false, true)
template <typename T>
constexpr bool cols_has(int op, int nout, bool fwd, bool inv) {
#define X(OP, NOUT, FWD, INV) || (op == OP && nout == NOUT && fwd == FWD && inv == INV)
  return (false LES_COL_INSTANCES(X)) || (sizeof(T) == 4 && (false LES_COL_INSTANCES_F32(X))) ||
         (sizeof(T) == 8 && (false LES_COL_INSTANCES_F64(X)));
#undef X
}

template <typename T>
struct ColArgs {  // k_cols_reg, cols_reg.h
  // per job (blockIdx.y):
  // the same op on up to LES_COL_JOBS independent input/output sets
  const Cplx<T>* in[LES_COL_JOBS][2];
  Cplx<T>* out[LES_COL_JOBS][3];
  const T* kkx;
  const T* kky;
  const T* g0;
  const T* g1;
  int lhx;
  int k0, nplanes;
};

// ------------------------------------------------------------------ 3/2 resampling
// Padding keeps modes |k| < n/2 (Nyquist dropped) of a length-n1 line in a
// length-n2 spectrum; truncation is the mirror image
// (src/compute_convective_padd.f90:288-319, 352-382).
// Convection source planes padded in x: which = 0..5 -> -c u, -c v, -c w,
// c (dw/dy - dv/dz), c (du/dz - dw/dx), c (dv/dx - du/dy), with the wall-law
// first level of the vorticities (src/compute_convective_padd.f90:133-169).
template <typename TI>
struct ConvSrc {
  const double *u, *v, *w;
  const TI *dudy, *dudz, *dvdx, *dvdz, *dwdx, *dwdy;
};

template <typename T, typename TI>
__device__ __forceinline__ T conv_src(const ConvSrc<TI>& s, int which, int k, long q, long np, T c) {
  const long a = (long)k * np + q;
  switch (which) {
    case 0: return (T)(-((double)c * s.u[a]));
    case 1: return (T)(-((double)c * s.v[a]));
    case 2: return (T)(-((double)c * s.w[a]));
    case 3:
      if (k == 1) return c * ((T)0.5 * ((T)s.dwdy[a] + (T)s.dwdy[a + np]) - (T)s.dvdz[a]);
      return c * ((T)s.dwdy[a] - (T)s.dvdz[a]);
    case 4:
      if (k == 1) return c * ((T)s.dudz[a] - (T)0.5 * ((T)s.dwdx[a] + (T)s.dwdx[a + np]));
      return c * ((T)s.dudz[a] - (T)s.dwdx[a]);
    default: return c * ((T)s.dvdx[a] - (T)s.dudy[a]);
  }
}

// Row resampling (k_rows_resample_reg, rows_reg.h): padding computes the
// convection sources (field = blockIdx.y) from ConvSrc, truncation reads src.
template <typename T, typename TI, typename TO>
struct RowResArgs {
  const T* src[LES_MAX_FIELDS];
  TO* dst[LES_MAX_FIELDS];
  ConvSrc<TI> cs;
  T cconv;
  int ny;
  int k0, nplanes;
  // truncation: the planes k0 - 1 and k0 + nplanes are filled with `ghost`
  double ghost;
};

// Column resampling: column pairs (i, i+1) of a real (W, h1) plane -> (W, h2)
// as complex lines (k_colres_reg, colres_reg.h).
template <typename T>
struct ColResArgs {
  const T* src[LES_MAX_FIELDS];
  T* dst[LES_MAX_FIELDS];
  int W;  // real columns
  int k0, nplanes;
  long src_plane, dst_plane;  // plane strides (elements)
};
