// Column (y) transforms of the spectral planes, register resident, one
// instance per length (fft_cols.hip).
//
// A block owns a tile of CB adjacent columns, counted through the planes (the
// columns of plane k + 1 follow those of plane k, so only the last tile of
// the launch is partly filled whatever lhx is), with NT threads per column.
// Thread (c, a) loads its rows of column c straight into registers: the CB
// lanes of one row read one 128-byte segment.  Transform, spectral operation
// and inverse transform then run as register phases (fft_reg.h) with one LDS
// exchange between two phases, and the result is stored from registers.
//
// LDS: CB lines of an odd number of values, so that the lanes that share a
// row (one 128-byte LDS cycle) fall into different banks whatever row it is.
//
// Bound by memory from about 128 columns and levels on, below that by the
// latency of a block's load, exchanges and store.  Against lines that are
// exchanged in LDS at every stage the column kernels of five steps took 3.01
// -> 1.08 ms at 192x144x65 in FP64, of five mixed steps at 128^3 1.75 -> 1.46.
#pragma once
#include "fft_kernels.h"
#include "fft_reg.h"

template <typename T, int N>
struct ColShape {
  static constexpr int NT = ph_threads(N, 0, col_maxg<T>());  // threads per column
  // 128-byte row segments; FP64 256-byte ones for the lengths 192..288, where
  // two such blocks fit the LDS of a CU (256: test filters 174 -> 150 us,
  // gradients 221 -> 200; no difference at 144 and 64)
  static constexpr int CB0 = sizeof(T) == 8 && (N < 192 || N > 288) ? 8 : 16;
  // at least one wavefront per block
  static constexpr int CB = NT * CB0 >= 64 ? CB0 : NT * CB0 * 2 >= 64 ? 2 * CB0 : NT * CB0 * 4 >= 64 ? 4 * CB0 : 8 * CB0;
  static constexpr int LS = N | 1;                            // odd line stride
  static constexpr int THREADS = NT * CB;
  static constexpr size_t LDS = (size_t)CB * LS * sizeof(Cplx<T>);
};

// by value: choosing between two lvalues would put the register array in memory
template <typename T>
__device__ __forceinline__ Cplx<T> cut_if(bool cut, Cplx<T> x) {
  return {cut ? (T)0 : x.x, cut ? (T)0 : x.y};
}

// OP on NOUT outputs; FWD / INV: forward transform before it, inverse after.
// The tables kkx, kky are zero on the Nyquist row and column; elsewhere kkx
// depends on the column only and kky on the row only, so row 0 and column 0
// of the tables serve.
template <typename T, int N, int OP, int NOUT, bool FWD, bool INV>
__global__ void __launch_bounds__((ColShape<T, N>::THREADS)) __attribute__((amdgpu_waves_per_eu(2)))
k_cols_reg(ColArgs<T> a, const Cplx<T>* __restrict__ tw) {
  using S = ColShape<T, N>;
  using L = RegLine<T, N, S::NT, col_maxg<T>()>;
  constexpr int CB = S::CB, VX = L::VALS;
  constexpr int QOP = FWD ? L::LAST : 0;    // layout the operation runs in
  constexpr int QST = INV ? L::LAST : QOP;  // layout of the result
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int c = threadIdx.x % CB, ar = threadIdx.x / CB;
  Cplx<T>* line = reinterpret_cast<Cplx<T>*>(smem_raw) + c * S::LS;
  const int job = blockIdx.y, lhx = a.lhx;
  const int total = a.nplanes * lhx, g0 = xcd_tile(blockIdx.x, gridDim.x) * CB;
  const bool valid = g0 + c < total;
  const int g = valid ? g0 + c : total - 1;
  const int pl0 = g0 / lhx, pl = g / lhx, kx = g - pl * lhx;
  const long plane0 = (long)(a.k0 + pl0) * N * lhx;
  const unsigned off = ((unsigned)((pl - pl0) * N + ar) * lhx + kx) * (unsigned)sizeof(Cplx<T>);
  const unsigned toff = (unsigned)(ar * lhx + kx) * (unsigned)sizeof(T), yoff = (unsigned)(ar * lhx) * (unsigned)sizeof(T);
  const bool nyqx = kx == lhx - 1;
  auto sync = []() LES_INLINE { block_sync_lds(); };

  Cplx<T> X[VX];
  {
    const Cplx<T>* __restrict__ src = a.in[job][0] + plane0;
    L::template rows<0>(ar, [&](int v, int r) LES_INLINE { X[v] = at_bytes(src + (long)r * lhx, off); });
  }
  if constexpr (FWD) L::template fft<false>(X, line, tw, ar, sync);
  // from the operation's layout through the inverse transform to memory
  auto finish = [&](Cplx<T>* Y, int o) LES_INLINE {
    if constexpr (INV) {
      if constexpr (FWD) L::relay(Y, line, ar, sync);
      L::template fft<true>(Y, line, tw, ar, sync);
    }
    Cplx<T>* __restrict__ dst = a.out[job][o] + plane0;
    if (valid) L::template rows<QST>(ar, [&](int v, int r) LES_INLINE { put_bytes(dst + (long)r * lhx, off, Y[v]); });
  };
  if constexpr (OP == COP_DIV) {
    // i kx X0 is formed before the second input is loaded (the transforms'
    // barriers keep its loads after), so one input line and the partial sum
    // are live at a time
    static_assert(FWD && NOUT == 1, "the divergence transforms its inputs");
    const T kxv = nyqx ? (T)0 : a.kkx[kx];
    L::template rows<QOP>(ar, [&](int v, int r) LES_INLINE {
      const bool nyq = nyqx || ar + r == N / 2;
      X[v] = c_ik(nyq ? (T)0 : kxv, cut_if(nyq, X[v]));
    });
    Cplx<T> X1[VX];
    const Cplx<T>* __restrict__ src = a.in[job][1] + plane0;
    L::template rows<0>(ar, [&](int v, int r) LES_INLINE { X1[v] = at_bytes(src + (long)r * lhx, off); });
    L::template fft<false>(X1, line, tw, ar, sync);
    L::template rows<QOP>(ar, [&](int v, int r) LES_INLINE {
      const bool nyq = nyqx || ar + r == N / 2;
      const T ky = at_bytes(a.kky + (long)r * lhx, yoff);
      X[v] = c_add(X[v], c_ik(nyq ? (T)0 : ky, cut_if(nyq, X1[v])));
    });
    finish(X, 0);
  } else if constexpr (OP == COP_COPY) {
    finish(X, 0);
  } else if constexpr (OP == COP_FILT1 || OP == COP_FILT2) {
    auto filter = [&](int o, const T* __restrict__ gt) LES_INLINE {
      Cplx<T> Y[VX];
      L::template rows<QOP>(ar, [&](int v, int r) LES_INLINE { Y[v] = c_scale(X[v], at_bytes(gt + (long)r * lhx, toff)); });
      finish(Y, o);
    };
    filter(0, a.g0);
    if constexpr (NOUT > 1) filter(1, a.g1);
  } else {
    // COP_GRAD (Nyquist modes removed) and COP_PGRAD: i kx, i ky, the field
    const T kxv = nyqx ? (T)0 : a.kkx[kx];
    auto cut = [&](int v, int r) LES_INLINE {
      return OP == COP_GRAD ? cut_if(nyqx || ar + r == N / 2, X[v]) : X[v];
    };
    {
      Cplx<T> Y[VX];
      L::template rows<QOP>(ar, [&](int v, int r) LES_INLINE { Y[v] = c_ik(ar + r == N / 2 ? (T)0 : kxv, cut(v, r)); });
      finish(Y, 0);
    }
    {
      Cplx<T> Y[VX];
      L::template rows<QOP>(ar, [&](int v, int r) LES_INLINE {
        const T ky = at_bytes(a.kky + (long)r * lhx, yoff);
        Y[v] = c_ik(nyqx || ar + r == N / 2 ? (T)0 : ky, cut(v, r));
      });
      finish(Y, 1);
    }
    if constexpr (NOUT > 2) {
      Cplx<T> Y[VX];
      L::template rows<QOP>(ar, [&](int v, int r) LES_INLINE { Y[v] = cut(v, r); });
      finish(Y, 2);
    }
  }
}

// Launches the instance of op (nout outputs, fwd, inv) of length N; with attr
// set only raises every instance's LDS limit.
template <typename T, int N>
static bool cols_reg_n(bool attr, int op, int nout, bool fwd, bool inv, const ColArgs<T>& a, int njobs, const Cplx<T>* tw,
                       hipStream_t s) {
  using S = ColShape<T, N>;
  const dim3 g((unsigned)(((long)a.nplanes * a.lhx + S::CB - 1) / S::CB), (unsigned)njobs);
#define X(OP, NOUT, FWD, INV)                                                                             \
  if (attr) {                                                                                             \
    hipFuncSetAttribute((const void*)k_cols_reg<T, N, OP, NOUT, FWD, INV>,                                \
                        hipFuncAttributeMaxDynamicSharedMemorySize, (int)S::LDS);                         \
  } else if (op == OP && nout == NOUT && fwd == FWD && inv == INV) {                                      \
    hipLaunchKernelGGL((k_cols_reg<T, N, OP, NOUT, FWD, INV>), g, dim3(S::THREADS), S::LDS, s, a, tw);    \
    return true;                                                                                          \
  }
  LES_COL_INSTANCES(X)
  if constexpr (sizeof(T) == 4) {
    LES_COL_INSTANCES_F32(X)
  } else {
    LES_COL_INSTANCES_F64(X)
  }
#undef X
  return attr;
}
