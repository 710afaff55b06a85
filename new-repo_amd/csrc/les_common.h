// Shared device-side building blocks of the LES library: complex arithmetic,
// the butterflies and stage plans of every horizontal transform (fft_reg.h).
//
// FFT algorithm (fixed so results are reproducible across devices and against
// the CPU restatement used in testing): complex length-n transforms with
// n = 2^a 3^b as a Stockham autosort sweep of radix-4 stages, one radix-2
// stage when a is odd, then radix-3 stages.  Stage s (radix R, span p = the
// product of earlier radices): for i < n/R with k = i mod p the inputs
// x_r = in[i + r n/R] (r >= 1) are multiplied by exp(sign 2 pi i r k/(pR))
// (fused multiply-adds: (fma(a.x, w.x, -(a.y w.y)), fma(a.x, w.y, a.y w.x))),
// combined by a size-R DFT and written to out[(i - k) R + k + r p].  The
// transforms are unnormalised like FFTW's (src/decomp_2d_fft_2d.f90:397-577).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#define LES_MAX_STAGES 10

template <typename T>
struct Cplx {
  T x, y;
};

template <typename T>
__device__ __forceinline__ Cplx<T> c_add(Cplx<T> a, Cplx<T> b) { return {a.x + b.x, a.y + b.y}; }
template <typename T>
__device__ __forceinline__ Cplx<T> c_sub(Cplx<T> a, Cplx<T> b) { return {a.x - b.x, a.y - b.y}; }
// Twiddle product with fused multiply-adds (one rounding each), four
// instructions instead of six.
template <typename T>
__device__ __forceinline__ Cplx<T> c_mul(Cplx<T> a, Cplx<T> w) {
  return {fma(a.x, w.x, -(a.y * w.y)), fma(a.x, w.y, a.y * w.x)};
}
template <typename T>
__device__ __forceinline__ Cplx<T> c_scale(Cplx<T> a, T s) { return {a.x * s, a.y * s}; }
// i*k*a with k real, as the reference's eye*kkx*f_hat
template <typename T>
__device__ __forceinline__ Cplx<T> c_ik(T k, Cplx<T> a) { return {-(k * a.y), k * a.x}; }

// Plan of one transform length (host-built, passed by value to kernels).
struct FftPlan {
  int n, nst;
  int R[LES_MAX_STAGES], P[LES_MAX_STAGES], off[LES_MAX_STAGES];
  int twf;  // offset of the forward twiddle table in the twiddle pool (inverse transforms use the conjugates)
};

template <typename T>
__device__ __forceinline__ void bfly(Cplx<T>* x, int R, int sgn) {
  if (R == 4) {
    Cplx<T> t0 = c_add(x[0], x[2]), t1 = c_sub(x[0], x[2]);
    Cplx<T> t2 = c_add(x[1], x[3]), t3 = c_sub(x[1], x[3]);
    Cplx<T> t3r = (sgn < 0) ? Cplx<T>{t3.y, -t3.x} : Cplx<T>{-t3.y, t3.x};
    x[0] = c_add(t0, t2);
    x[2] = c_sub(t0, t2);
    x[1] = c_add(t1, t3r);
    x[3] = c_sub(t1, t3r);
  } else if (R == 2) {
    Cplx<T> y0 = c_add(x[0], x[1]), y1 = c_sub(x[0], x[1]);
    x[0] = y0;
    x[1] = y1;
  } else {
    const T h = (T)0.86602540378443864676372317075294;
    Cplx<T> t1 = c_add(x[1], x[2]);
    Cplx<T> t2 = {x[0].x - (T)0.5 * t1.x, x[0].y - (T)0.5 * t1.y};
    Cplx<T> t3 = c_sub(x[1], x[2]);
    Cplx<T> t3r = (sgn < 0) ? Cplx<T>{h * t3.y, -(h * t3.x)} : Cplx<T>{-(h * t3.y), h * t3.x};
    x[0] = c_add(x[0], t1);
    x[1] = c_add(t2, t3r);
    x[2] = c_sub(t2, t3r);
  }
}

#define LES_WAVE 64
#define LES_MAX_N 1024

// One 8- or 16-byte LDS access per complex value (ds_read_b64 / _b128)
// instead of two 4- or 8-byte ones.
template <typename T>
struct Vec2T;
template <>
struct Vec2T<float> { using type = float2; };
template <>
struct Vec2T<double> { using type = double2; };
template <typename T>
__device__ __forceinline__ Cplx<T> lds_ld(const Cplx<T>* p) {
  const typename Vec2T<T>::type v = *reinterpret_cast<const typename Vec2T<T>::type*>(p);
  return {v.x, v.y};
}
template <typename T>
__device__ __forceinline__ void lds_st(Cplx<T>* p, Cplx<T> a) {
  typename Vec2T<T>::type v;
  v.x = a.x;
  v.y = a.y;
  *reinterpret_cast<typename Vec2T<T>::type*>(p) = v;
}

__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The stages of a length at compile time, by the host's rule (radix-4 stages, one
// radix-2 stage when the power of two is odd, then radix-3 stages).
constexpr int cp_a(int n) { int a = 0; while (n % 2 == 0) { n /= 2; ++a; } return a; }
constexpr int cp_b(int n) { while (n % 2 == 0) n /= 2; int b = 0; while (n % 3 == 0) { n /= 3; ++b; } return b; }
constexpr int cp_nst(int n) { return cp_a(n) / 2 + (cp_a(n) & 1) + cp_b(n); }
constexpr int cp_R(int n, int s) {
  return s < cp_a(n) / 2 ? 4 : ((cp_a(n) & 1) && s == cp_a(n) / 2 ? 2 : 3);
}
constexpr int cp_P(int n, int s) { int p = 1; for (int t = 0; t < s; ++t) p *= cp_R(n, t); return p; }
constexpr int cp_OFF(int n, int s) { int o = 0; for (int t = 0; t < s; ++t) o += (cp_R(n, t) - 1) * cp_P(n, t); return o; }

// Block barrier for LDS exchange only: waits for the wavefront's LDS
// operations, not for its outstanding global loads (a prefetch stays in
// flight across it, unlike __syncthreads, whose workgroup fence can wait for
// them).  The memory clobber keeps the compiler from moving memory accesses
// across it.
__device__ __forceinline__ void block_sync_lds() { __asm__ volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// XCD-aware tile order.  Workgroups are dispatched round-robin over the 8
// XCDs (block b on XCD b % 8), each with its own L2.  Tiles that share
// 128-byte lines (adjacent column tiles of narrower rows) must run on one XCD
// at nearly the same time, so physical block b = 8 m + x runs logical tile
// s_x + m, where XCD x owns the contiguous range [s_x, s_x + size_x) of the
// n tiles (sizes q + 1 for x < n % 8, q = n / 8 otherwise).  A bijection on
// [0, n).
#define LES_NXCD 8
__device__ __forceinline__ int xcd_tile(int b, int n) {
  const int q = n / LES_NXCD, r = n % LES_NXCD;
  const int x = b % LES_NXCD, m = b / LES_NXCD;
  return x * q + (x < r ? x : r) + m;
}

#define LES_CHECK(x)                                                                     \
  do {                                                                                   \
    hipError_t e_ = (x);                                                                 \
    if (e_ != hipSuccess) {                                                              \
      les_set_error("%s failed: %s (%s:%d)", #x, hipGetErrorString(e_), __FILE__, __LINE__); \
      return 5;                                                                          \
    }                                                                                    \
  } while (0)

void les_set_error(const char* fmt, ...);
