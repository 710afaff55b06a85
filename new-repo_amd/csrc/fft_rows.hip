// Row kernels of one precision (LES_T) for the lengths of one part (LES_PART);
// the build compiles this file once per pair.
#include "rows_reg.h"
#include "fft_launch.h"

#define LES_CAT_(a, b) a##b
#define LES_CAT(a, b) LES_CAT_(a, b)
#define LES_MY_LENGTHS LES_CAT(LES_LENGTHS_, LES_PART)

// one launch of kernel K over the row pairs of nplanes planes and EXTRA blocks
// past them, or (attr) only its LDS limit
#define LES_ROW_LAUNCH(SHAPE, K, ...) LES_ROW_LAUNCH_X(SHAPE, 0, K, __VA_ARGS__)
#define LES_ROW_LAUNCH_X(SHAPE, EXTRA, K, ...)                                                                    \
  do {                                                                                                            \
    using S_ = SHAPE;                                                                                             \
    if (attr) {                                                                                                   \
      hipFuncSetAttribute((const void*)K, hipFuncAttributeMaxDynamicSharedMemorySize, (int)S_::LDS);              \
    } else {                                                                                                      \
      const long jobs_ = (long)a.nplanes * (a.ny / 2);                                                            \
      hipLaunchKernelGGL((K), dim3((unsigned)((jobs_ + S_::LB - 1) / S_::LB + (EXTRA)), (unsigned)nf),            \
                         dim3(S_::THREADS), S_::LDS, s, a, __VA_ARGS__);                                          \
    }                                                                                                             \
  } while (0)

template <typename TI, typename T, int N>
static void r2c_n(bool attr, int mode, const RowR2CArgs<TI, T>& a, int nf, const Cplx<T>* tw, hipStream_t s) {
  using SH = RowShape<T, N>;
  if constexpr (sizeof(T) == 8) {
    if (attr || mode == LOAD_SCALE_DIV) LES_ROW_LAUNCH(SH, (k_rows_r2c_reg<TI, T, N, LOAD_SCALE_DIV, false>), tw);
    if (attr || mode == LOAD_AB2_SCALE_DIV) LES_ROW_LAUNCH(SH, (k_rows_r2c_reg<TI, T, N, LOAD_AB2_SCALE_DIV, r2c_stream(N)>), tw);
    if (attr || mode == LOAD_PCLEAN) LES_ROW_LAUNCH(SH, (k_rows_r2c_reg<TI, T, N, LOAD_PCLEAN, r2c_stream(N)>), tw);
  }
  if (attr || mode == LOAD_SCALE) LES_ROW_LAUNCH(SH, (k_rows_r2c_reg<TI, T, N, LOAD_SCALE, false>), tw);
}

#define LES_ROW_SWITCH(n, CALL)   \
  switch (n) {                    \
    LES_MY_LENGTHS(CALL)          \
  }                               \
  return false

template <>
bool rows_r2c_part<double, LES_T, LES_PART>(bool attr, int n, int mode, const RowR2CArgs<double, LES_T>& a, int nf,
                                            const Cplx<LES_T>* tw, hipStream_t s) {
#define X(N) case N: r2c_n<double, LES_T, N>(attr, mode, a, nf, tw, s); return true;
  LES_ROW_SWITCH(n, X);
#undef X
}

template <>
bool rows_c2r_part<LES_T, double, LES_PART>(bool attr, int n, const RowC2RArgs<LES_T, double>& a, int nf,
                                            const Cplx<LES_T>* tw, hipStream_t s) {
#define X(N) case N: { using SH = RowShape<LES_T, N>; LES_ROW_LAUNCH(SH, (k_rows_c2r_reg<LES_T, double, N>), tw); return true; }
  LES_ROW_SWITCH(n, X);
#undef X
}

template <>
bool rows_div_part<LES_T, LES_PART>(bool attr, int n, const RowC2RArgs<LES_T, LES_T>& a, const DivEpi3<LES_T>& ep, int nf,
                                    const Cplx<LES_T>* tw, hipStream_t s) {
#define X(N) case N: { using SH = RowShape<LES_T, N>; LES_ROW_LAUNCH(SH, (k_rows_c2r_div_reg<LES_T, N>), ep, tw); return true; }
  LES_ROW_SWITCH(n, X);
#undef X
}

template <>
bool rows_pad_part<LES_T, LES_PART>(bool attr, int n, const RowResArgs<LES_T, LES_T, LES_T>& a, int nf, const Cplx<LES_T>* twn,
                                    const Cplx<LES_T>* twb, hipStream_t s) {
#define X(N)                                                                          \
  case N: {                                                                           \
    using SH = RowShape<LES_T, N, 3 * N / 2>;                                         \
    LES_ROW_LAUNCH(SH, (k_rows_resample_reg<LES_T, LES_T, N, true>), twn, twb);       \
    return true;                                                                      \
  }
  LES_ROW_SWITCH(n, X);
#undef X
}

template <>
bool rows_trunc_part<LES_T, LES_PART>(bool attr, int n, const RowResArgs<LES_T, LES_T, double>& a, int nf,
                                      const Cplx<LES_T>* twn, const Cplx<LES_T>* twb, hipStream_t s) {
#define X(N)                                                                          \
  case N: {                                                                           \
    using SH = RowShape<LES_T, N, 3 * N / 2>;                                         \
    const long fill = ((long)N * a.ny + 8 * SH::THREADS - 1) / (8 * SH::THREADS);     \
    LES_ROW_LAUNCH_X(SH, fill, (k_rows_resample_reg<LES_T, double, N, false>), twn, twb); \
    return true;                                                                      \
  }
  LES_ROW_SWITCH(n, X);
#undef X
}

#if LES_FP32
template <>
bool rows_nyq_part<float, LES_PART>(bool attr, int n, const RowR2CArgs<double, float>& a, int nf, const Cplx<float>* tw,
                                    hipStream_t s) {
#define X(N) case N: { using SH = NyqShape<float, N>; LES_ROW_LAUNCH(SH, (k_rows_r2c_nyq<float, N>), tw); return true; }
  LES_ROW_SWITCH(n, X);
#undef X
}
template <>
bool rows_r2c_part<float, float, LES_PART>(bool attr, int n, int mode, const RowR2CArgs<float, float>& a, int nf, const Cplx<float>* tw,
                                           hipStream_t s) {
#define X(N) case N: r2c_n<float, float, N>(attr, mode, a, nf, tw, s); return true;
  LES_ROW_SWITCH(n, X);
#undef X
}
template <>
bool rows_c2r_part<float, float, LES_PART>(bool attr, int n, const RowC2RArgs<float, float>& a, int nf, const Cplx<float>* tw,
                                           hipStream_t s) {
#define X(N) case N: { using SH = RowShape<float, N>; LES_ROW_LAUNCH(SH, (k_rows_c2r_reg<float, float, N>), tw); return true; }
  LES_ROW_SWITCH(n, X);
#undef X
}
#else
template <>
bool rows_proj_part<double, LES_PART>(bool attr, int n, const RowC2RArgs<double, double>& a, const ProjEpi3& ep, int nf,
                              const Cplx<double>* tw, hipStream_t s) {
#define X(N) case N: { using SH = RowShape<double, N>; LES_ROW_LAUNCH(SH, (k_rows_c2r_proj_reg<N>), ep, tw); return true; }
  LES_ROW_SWITCH(n, X);
#undef X
}
#endif
