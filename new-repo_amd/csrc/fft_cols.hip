// Column kernels of one precision (LES_T) for the lengths of one part
// (LES_PART); the build compiles this file once per pair.
#include "cols_reg.h"
#include "colres_reg.h"
#include "fft_launch.h"

#define LES_CAT_(a, b) a##b
#define LES_CAT(a, b) LES_CAT_(a, b)
#define LES_MY_LENGTHS LES_CAT(LES_LENGTHS_, LES_PART)

template <>
bool cols_reg_part<LES_T, LES_PART>(bool attr, int ny, int op, int nout, bool fwd, bool inv, const ColArgs<LES_T>& a,
                                    int njobs, const Cplx<LES_T>* tw, hipStream_t s) {
  switch (ny) {
#define X(N) case N: return cols_reg_n<LES_T, N>(attr, op, nout, fwd, inv, a, njobs, tw, s);
    LES_MY_LENGTHS(X)
#undef X
  }
  return false;
}

template <>
bool colres_reg_part<LES_T, LES_PART>(bool attr, int n, bool pad, const ColResArgs<LES_T>& a, int nf,
                                      const Cplx<LES_T>* twn, const Cplx<LES_T>* twb, hipStream_t s) {
  switch (n) {
#define X(N) case N: return colres_reg_n<LES_T, N>(attr, pad, a, nf, twn, twb, s);
    LES_MY_LENGTHS(X)
#undef X
  }
  return false;
}
