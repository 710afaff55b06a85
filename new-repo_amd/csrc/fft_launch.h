// Launchers of the kernels that have one instance per transform length,
// compiled in parts (fft_cols.hip and fft_rows.hip, once per precision and part).
#pragma once
#include "fft_kernels.h"
#include "les_epi.h"

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
// Row transforms of length n (nf fields; tw: the forward table of n), the
// resampling n <-> 3 n / 2 (twn, twb).  attr and the result as above.
template <typename TI, typename T, int PART>
bool rows_r2c_part(bool attr, int n, int mode, const RowR2CArgs<TI, T>& a, int nf, const Cplx<T>* tw, hipStream_t s);
template <typename T, int PART>
bool rows_nyq_part(bool attr, int n, const RowR2CArgs<double, T>& a, int nf, const Cplx<T>* tw, hipStream_t s);
template <typename T, typename TO, int PART>
bool rows_c2r_part(bool attr, int n, const RowC2RArgs<T, TO>& a, int nf, const Cplx<T>* tw, hipStream_t s);
template <typename T, int PART>
bool rows_div_part(bool attr, int n, const RowC2RArgs<T, T>& a, const DivEpi3<T>& ep, int nf, const Cplx<T>* tw, hipStream_t s);
template <typename T, int PART>
bool rows_proj_part(bool attr, int n, const RowC2RArgs<T, T>& a, const ProjEpi3& ep, int nf, const Cplx<T>* tw, hipStream_t s);
template <typename T, int PART>
bool rows_pad_part(bool attr, int n, const RowResArgs<T, T, T>& a, int nf, const Cplx<T>* twn, const Cplx<T>* twb, hipStream_t s);
template <typename T, int PART>
bool rows_trunc_part(bool attr, int n, const RowResArgs<T, T, double>& a, int nf, const Cplx<T>* twn, const Cplx<T>* twb,
                     hipStream_t s);

// The part that has length n, over all parts.  Operation and load mode are
// template arguments: a kernel that is not compiled is an error of the build
// and not a call that launches nothing.  That the lengths have kernels is
// checked once, by les_init (attr).
#define LES_EACH_PART(CALL) CALL(0) || CALL(1) || CALL(2) || CALL(3)
static_assert(LES_LENGTH_PARTS == 4, "LES_EACH_PART lists the parts");
template <typename T, int OP, int NOUT, bool FWD, bool INV>
static bool cols_reg(bool attr, int ny, const ColArgs<T>& a, int njobs, const Cplx<T>* tw, hipStream_t s) {
  static_assert(cols_has<T>(OP, NOUT, FWD, INV), "no column kernel of this operation and precision (LES_COL_INSTANCES)");
#define C(P) (cols_reg_part<T, P>(attr, ny, OP, NOUT, FWD, INV, a, njobs, tw, s))
  return LES_EACH_PART(C);
#undef C
}
template <typename T>
static bool colres_reg(bool attr, int n, bool pad, const ColResArgs<T>& a, int nf, const Cplx<T>* twn, const Cplx<T>* twb,
                       hipStream_t s) {
#define C(P) (colres_reg_part<T, P>(attr, n, pad, a, nf, twn, twb, s))
  return LES_EACH_PART(C);
#undef C
}
template <typename TI, typename T, int MODE>
static bool rows_r2c_reg(bool attr, int n, const RowR2CArgs<TI, T>& a, int nf, const Cplx<T>* tw, hipStream_t s) {
  static_assert(r2c_has<T>(MODE), "no forward row kernel of this load mode and precision");
#define C(P) (rows_r2c_part<TI, T, P>(attr, n, MODE, a, nf, tw, s))
  return LES_EACH_PART(C);
#undef C
}
template <typename T>
static bool rows_nyq_reg(bool attr, int n, const RowR2CArgs<double, T>& a, int nf, const Cplx<T>* tw, hipStream_t s) {
#define C(P) (rows_nyq_part<T, P>(attr, n, a, nf, tw, s))
  return LES_EACH_PART(C);
#undef C
}
template <typename T, typename TO>
static bool rows_c2r_reg(bool attr, int n, const RowC2RArgs<T, TO>& a, int nf, const Cplx<T>* tw, hipStream_t s) {
#define C(P) (rows_c2r_part<T, TO, P>(attr, n, a, nf, tw, s))
  return LES_EACH_PART(C);
#undef C
}
template <typename T>
static bool rows_div_reg(bool attr, int n, const RowC2RArgs<T, T>& a, const DivEpi3<T>& ep, int nf, const Cplx<T>* tw,
                         hipStream_t s) {
#define C(P) (rows_div_part<T, P>(attr, n, a, ep, nf, tw, s))
  return LES_EACH_PART(C);
#undef C
}
template <typename T>
static bool rows_proj_reg(bool attr, int n, const RowC2RArgs<T, T>& a, const ProjEpi3& ep, int nf, const Cplx<T>* tw,
                          hipStream_t s) {
#define C(P) (rows_proj_part<T, P>(attr, n, a, ep, nf, tw, s))
  return LES_EACH_PART(C);
#undef C
}
template <typename T>
static bool rows_pad_reg(bool attr, int n, const RowResArgs<T, T, T>& a, int nf, const Cplx<T>* twn, const Cplx<T>* twb,
                         hipStream_t s) {
#define C(P) (rows_pad_part<T, P>(attr, n, a, nf, twn, twb, s))
  return LES_EACH_PART(C);
#undef C
}
template <typename T>
static bool rows_trunc_reg(bool attr, int n, const RowResArgs<T, T, double>& a, int nf, const Cplx<T>* twn, const Cplx<T>* twb,
                           hipStream_t s) {
#define C(P) (rows_trunc_part<T, P>(attr, n, a, nf, twn, twb, s))
  return LES_EACH_PART(C);
#undef C
}
