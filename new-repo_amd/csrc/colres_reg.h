// Column (y) resampling of the padded convection, register resident, one
// instance per length.
//
// A block takes CB adjacent complex lines (pairs of real columns, 128-byte row
// segments), counted through the planes as in cols_reg.h, with NT threads per
// line: forward transform of length N1, padding or truncation while the
// spectrum is re-laid through LDS, inverse transform of length N2.  Padding
// keeps the modes |k| < N/2 (N the shorter length; its Nyquist mode is
// dropped, the rest is zero), truncation is the mirror image
// (src/compute_convective_padd.f90:288-319, 352-382).
#pragma once
#include "fft_kernels.h"
#include "fft_reg.h"

// N: the shorter length; 3 N / 2 the longer
template <typename T, int N>
struct ColResShape {
  static constexpr int NB = 3 * N / 2;
  static constexpr int NT = ph_threads(N, NB, col_maxg<T>());
  // 128-byte segments; FP32 from 384 on 64-byte ones, where two blocks or one
  // of 16 lines would fill the LDS of a CU (512 <-> 768, 256 levels: padding
  // 2055 -> 1740 us, truncation 958 -> 825; 384 <-> 576 padding 448 -> 423)
  static constexpr int CB0 = sizeof(T) == 8 || N >= 384 ? 8 : 16;
  static constexpr int CB = NT * CB0 >= 64 ? CB0 : NT * CB0 * 2 >= 64 ? 2 * CB0 : NT * CB0 * 4 >= 64 ? 4 * CB0 : 8 * CB0;
  static constexpr int LS = NB | 1;
  static constexpr int THREADS = NT * CB;
  static constexpr size_t LDS = (size_t)CB * LS * sizeof(Cplx<T>);
};

template <typename T, int N, bool PAD>
__global__ void __launch_bounds__((ColResShape<T, N>::THREADS)) __attribute__((amdgpu_waves_per_eu(2)))
k_colres_reg(ColResArgs<T> a, const Cplx<T>* __restrict__ twn, const Cplx<T>* __restrict__ twb) {
  using S = ColResShape<T, N>;
  constexpr int N1 = PAD ? N : S::NB, N2 = PAD ? S::NB : N, NT = S::NT, CB = S::CB, H = N / 2;
  using L1 = RegLine<T, N1, NT, col_maxg<T>()>;
  using L2 = RegLine<T, N2, NT, col_maxg<T>()>;
  constexpr int VX = L1::VALS > L2::VALS ? L1::VALS : L2::VALS;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int c = threadIdx.x % CB, ar = threadIdx.x / CB;
  Cplx<T>* line = reinterpret_cast<Cplx<T>*>(smem_raw) + c * S::LS;
  const int f = blockIdx.y, nl = a.W / 2;
  const int total = a.nplanes * nl, g0 = xcd_tile(blockIdx.x, gridDim.x) * CB;
  const bool valid = g0 + c < total;
  const int g = valid ? g0 + c : total - 1;
  const int pl0 = g0 / nl, pl = g / nl, l = g - pl * nl;
  const Cplx<T>* __restrict__ src = reinterpret_cast<const Cplx<T>*>(a.src[f] + (long)(a.k0 + pl0) * a.src_plane);
  Cplx<T>* __restrict__ dst = reinterpret_cast<Cplx<T>*>(a.dst[f] + (long)(a.k0 + pl0) * a.dst_plane);
  const unsigned soff = ((unsigned)(pl - pl0) * (unsigned)(a.src_plane / 2) + ar * nl + l) * (unsigned)sizeof(Cplx<T>);
  const unsigned doff = ((unsigned)(pl - pl0) * (unsigned)(a.dst_plane / 2) + ar * nl + l) * (unsigned)sizeof(Cplx<T>);
  auto sync = []() LES_INLINE { block_sync_lds(); };
  const Cplx<T>* __restrict__ tw1 = PAD ? twn : twb;
  const Cplx<T>* __restrict__ tw2 = PAD ? twb : twn;
  Cplx<T> X[VX];
  L1::template rows<0>(ar, [&](int v, int r) LES_INLINE { X[v] = at_bytes(src + (long)r * nl, soff); });
  L1::template fft<false>(X, line, tw1, ar, sync);
  // spectrum row m of N1 -> row of N2; the rows left without a mode are zero
  L1::template rows<L1::LAST>(ar, [&](int v, int r) LES_INLINE {
    const int m = ar + r;
    if (PAD) {
      if (m != H) lds_st(line + (m < H ? m : m + H), X[v]);
    } else {
      if (m < H) lds_st(line + m, X[v]);
      else if (m > N) lds_st(line + m - H, X[v]);
    }
  });
  const Cplx<T> zero = {(T)0, (T)0};
  if (PAD) {
#pragma unroll
    for (int e = H; e <= N; e += NT)
      if (e + ar <= N) lds_st(line + e + ar, zero);
  } else {
    if (ar == 0) lds_st(line + H, zero);
  }
  sync();
  L2::template get<0>(X, line, ar);
  sync();
  L2::template fft<true>(X, line, tw2, ar, sync);
  if (valid) L2::template rows<L2::LAST>(ar, [&](int v, int r) LES_INLINE { put_bytes(dst + (long)r * nl, doff, X[v]); });
}

// with attr set only raises the instances' LDS limits
template <typename T, int N>
static bool colres_reg_n(bool attr, bool pad, const ColResArgs<T>& a, int nf, const Cplx<T>* twn, const Cplx<T>* twb,
                         hipStream_t s) {
  using S = ColResShape<T, N>;
  if (attr) {
    hipFuncSetAttribute((const void*)k_colres_reg<T, N, true>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)S::LDS);
    hipFuncSetAttribute((const void*)k_colres_reg<T, N, false>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)S::LDS);
    return true;
  }
  const dim3 g((unsigned)(((long)a.nplanes * (a.W / 2) + S::CB - 1) / S::CB), (unsigned)nf);
  if (pad) hipLaunchKernelGGL((k_colres_reg<T, N, true>), g, dim3(S::THREADS), S::LDS, s, a, twn, twb);
  else hipLaunchKernelGGL((k_colres_reg<T, N, false>), g, dim3(S::THREADS), S::LDS, s, a, twn, twb);
  return true;
}
