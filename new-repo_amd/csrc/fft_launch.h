// Launchers of the kernels that have one instance per transform length,
// compiled in parts (fft_cols.hip, once per precision and part).
#pragma once
#include "fft_kernels.h"

#define LES_LENGTH_PARTS 4

// Column op on njobs sets, forward and / or inverse y transforms of length
// ny; tw: the forward twiddle table of ny.  attr: only raise the kernels' LDS
// limits.  False: the length is not one of this part.
template <typename T, int PART>
bool cols_reg_part(bool attr, int ny, int op, int nout, bool fwd, bool inv, const ColArgs<T>& a, int njobs,
                   const Cplx<T>* tw, hipStream_t s);
// Column resampling n <-> 3 n / 2 of nf fields; twn, twb: the forward tables
// of n and 3 n / 2.
template <typename T, int PART>
bool colres_reg_part(bool attr, int n, bool pad, const ColResArgs<T>& a, int nf, const Cplx<T>* twn, const Cplx<T>* twb,
                     hipStream_t s);

template <typename T, int PART = 0>
static bool cols_reg(bool attr, int ny, int op, int nout, bool fwd, bool inv, const ColArgs<T>& a, int njobs,
                     const Cplx<T>* tw, hipStream_t s) {
  if (cols_reg_part<T, PART>(attr, ny, op, nout, fwd, inv, a, njobs, tw, s)) return true;
  if constexpr (PART + 1 < LES_LENGTH_PARTS) return cols_reg<T, PART + 1>(attr, ny, op, nout, fwd, inv, a, njobs, tw, s);
  return false;
}
template <typename T, int PART = 0>
static bool colres_reg(bool attr, int n, bool pad, const ColResArgs<T>& a, int nf, const Cplx<T>* twn, const Cplx<T>* twb,
                       hipStream_t s) {
  if (colres_reg_part<T, PART>(attr, n, pad, a, nf, twn, twb, s)) return true;
  if constexpr (PART + 1 < LES_LENGTH_PARTS) return colres_reg<T, PART + 1>(attr, n, pad, a, nf, twn, twb, s);
  return false;
}
