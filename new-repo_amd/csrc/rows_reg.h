// Row (x) transforms, register resident, one instance per length.
//
// Pairs of real rows (2 jp, 2 jp + 1) of a plane are one complex line a + i b.
// A line has NT threads; thread a of a line reads its elements of both rows
// straight into registers (the NT threads of a line take consecutive
// elements), runs the phases of fft_reg.h with one LDS exchange between two of
// them, and the forward transform goes through LDS once more because the
// unpacking needs Z(k) and Z(n - k) together; the inverse transform packs into
// LDS and stores its real rows from registers.  Against a kernel that keeps the
// line in LDS that is two or three round trips instead of one per stage and two.
// Bound by memory (FP64, and FP32 from 256 points: 4-5 TB/s).  Measured
// (MI355X) per launch: FP64 192x144x65 r2c 27 -> 16 us, c2r 33 -> 21, padding
// and truncation 91 -> 69 and 29, divergence store 61 -> 41; FP32 256^3 c2r of
// two fields 95 -> 80, padding 392 -> 309, divergence store 300 -> 224.  The FP64
// stores with the projection are faster below 64 points and at 648 (48x64x512 68 ->
// 45 us, 648x64x48 66 -> 51), within 10% either way from 128 to 512, and slower at
// 64, 96 and 256 on some grids: 64x64x488 66 -> 84, 96x64x325 63 -> 87, 256^3 402 ->
// 420, 256x64x122 41 -> 55.
//
// Where NT divides a wavefront the threads of a line are in one wavefront and
// no block barrier is needed.  Consecutive row pairs are consecutive in memory,
// planes included, so addresses are a uniform base per block plus one 32-bit
// offset per thread.
#pragma once
#include "fft_kernels.h"
#include "fft_reg.h"
#include "les_epi.h"

// Lines of one or two lengths (n2 = 0: one) in a block.
template <typename T, int N, int N2 = 0>
struct RowShape {
  static constexpr int NT = ph_threads(N, N2, col_maxg<T>());  // threads per line
  static constexpr bool WAVE = 64 % NT == 0;
  // about 256 threads (64 for short lines, where a wavefront holds many); the
  // line count with the fewest idle lanes where a block's threads straddle wavefronts
  static constexpr int lines() {
    if (WAVE) return (N >= 128 ? 256 : 64) / NT;
    int best = 1, idle = 1 << 30;
    for (int l = 1; l * NT <= 256 || l == 1; ++l) {
      const int t = l * NT, w = (t + 63) / 64 * 64, i = (w - t) * 256 / w;
      if (t >= 128 || (l + 1) * NT > 256) {
        if (i <= idle) { idle = i; best = l; }
      }
    }
    return best;
  }
  static constexpr int LB = lines();
  static constexpr int THREADS = LB * NT;
  using L1 = RegLine<T, N, NT, col_maxg<T>(), true>;
  using L2 = RegLine<T, N2 ? N2 : N, NT, col_maxg<T>(), true>;
  static constexpr int need() { return L1::XLEN > L2::XLEN ? L1::XLEN : L2::XLEN; }
  // line stride: lines that share an LDS cycle follow one another in the banks
  static constexpr int stride() {
    constexpr int S = 128 / (int)sizeof(Cplx<T>);
    int s = need();
    while (s % S != (NT < S ? NT % S : 1)) ++s;
    return s;
  }
  static constexpr int LS = stride();
  static constexpr size_t LDS = (size_t)LB * LS * sizeof(Cplx<T>);
  static constexpr int VX = L1::VALS > L2::VALS ? L1::VALS : L2::VALS;
};

template <bool WAVE>
__device__ __forceinline__ void row_sync() {
  if constexpr (WAVE) wave_sync();
  else block_sync_lds();
}

// This thread's line: number l of the block, thread a of it, row pair job.
template <typename S>
struct RowAt {
  int a;
  long job0;    // first row pair of the block
  int dj;       // row pairs past it (clamped to the last one)
  bool valid;
  __device__ __forceinline__ RowAt(long njobs) {
    const int l = threadIdx.x / S::NT;
    a = threadIdx.x - l * S::NT;
    job0 = (long)blockIdx.x * S::LB;
    valid = job0 + l < njobs;
    dj = valid ? l : (int)(njobs - 1 - job0);
  }
  __device__ __forceinline__ int line() const { return threadIdx.x / S::NT; }
};

// The other order of a block's elements: consecutive lanes take consecutive
// elements of a row (512 bytes of FP64 per access instead of NT values), a
// wavefront over its own lines where they are in one wavefront, else the block
// over all.  item(i): line number and element of this thread's i-th item.
template <typename S, int N>
struct RowStream {
  static constexpr int W = S::WAVE ? 64 : S::THREADS, LINES = S::WAVE ? 64 / S::NT : S::LB;
  static constexpr int IT = (LINES * N + W - 1) / W;
  static constexpr bool FULL = LINES * N % W == 0;
  int t, l0;  // place in the group, its first line
  __device__ __forceinline__ RowStream() : t(S::WAVE ? threadIdx.x & 63 : threadIdx.x), l0(S::WAVE ? threadIdx.x / 64 * LINES : 0) {}
  __device__ __forceinline__ bool item(int i, int& l, int& n) const {
    const int idx = t + i * W;
    if (W % N == 0 || N % W == 0) {  // one line at a time, or whole lines
      l = l0 + (N % W == 0 ? i / (N % W == 0 ? N / W : 1) : idx / N);
      n = N % W == 0 ? t + i % (N % W == 0 ? N / W : 1) * W : idx % N;
    } else {
      l = l0 + idx / N;
      n = idx % N;
    }
    return FULL || idx < LINES * N;
  }
};

// The transformed line of a row pair in natural order -> the half spectra of
// both rows; dst: the block's first row.
template <typename S, typename T, int N, typename AT>
__device__ __forceinline__ void row_unpack(const Cplx<T>* line, Cplx<T>* __restrict__ dst, const AT& at) {
  constexpr int LHX = N / 2 + 1, NT = S::NT;
  const unsigned doff = (unsigned)(2 * at.dj * LHX + at.a) * (unsigned)sizeof(Cplx<T>);
#pragma unroll
  for (int q = 0; q < LHX; q += NT) {
    const int kk = q + at.a;
    if (q + NT <= LHX || kk < LHX) {
      const Cplx<T> zk = lds_ld(line + kk), zm = lds_ld(line + (q == 0 && at.a == 0 ? 0 : N - kk));
      const Cplx<T> A = {(T)0.5 * (zk.x + zm.x), (T)0.5 * (zk.y - zm.y)};
      const Cplx<T> B = {(T)0.5 * (zk.y + zm.y), (T)0.5 * (zm.x - zk.x)};
      put_bytes(dst + q, doff, A);
      put_bytes(dst + q + LHX, doff, B);
    }
  }
}

// ------------------------------------------------------------------ r2c
// STREAM: the input is read in RowStream order into LDS, else by each thread
// into its registers (one field: 64 points 10 -> 6 us, 192 19 -> 16).  The AB2
// predictor and the cleaned pressure, which read three and four FP64 fields per
// value, are streamed from 108 points on.  Registers against streamed, AB2: 48^3
// 8.2 us against 11.7, 64^3 14.2 and 14.6, 96x48x37 11.9 and 15.7, then 108x108x64
// 23.6 and 19.5, 128x64x64 23.8 and 16.0, 192x144x65 57.3 and 36.5, 512x512x256
// 1487 and 1204; cleaned pressure: 48^3 10.2 and 13.1, 64^3 11.7 and 15.1, 96x48x37
// 14.7 and 17.8, 192x144x65 23.0 and 19.7.
// At 256 and 512 points lines of one wavefront each, transformed in LDS stage by
// stage, read both faster (AB2 256^3 272 us against 317, 512x512x32 175 and 195;
// cleaned pressure 256^3 123 and 136): a block's 70 KB leave two wavefronts per
// SIMD, each with four rounds of loads waited for one after the other.
constexpr bool r2c_stream(int n) { return n >= 108; }
template <typename TI, typename T, int N, int MODE, bool STREAM>
__global__ void __launch_bounds__((RowShape<T, N>::THREADS)) k_rows_r2c_reg(RowR2CArgs<TI, T> a, const Cplx<T>* __restrict__ tw) {
  using S = RowShape<T, N>;
  using L = typename S::L1;
  constexpr int LHX = N / 2 + 1;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const RowAt<S> at((long)a.nplanes * (a.ny / 2));
  Cplx<T>* line = reinterpret_cast<Cplx<T>*>(smem_raw) + at.line() * S::LS;
  const int f = blockIdx.y;
  const long row0 = (long)a.k0 * a.ny + 2 * at.job0;
  auto sync = []() LES_INLINE { row_sync<S::WAVE>(); };
  const long e0 = row0 * N;
  const TI* __restrict__ src = a.src[f] + e0;
  // the line's value from both rows' inputs at element e of the block (row one, row two at e + N)
  auto value = [&](int r, unsigned off, long job) LES_INLINE {
    T v0 = (T)at_bytes(src + r, off), v1 = (T)at_bytes(src + N + r, off);
    if constexpr (MODE == LOAD_AB2_SCALE_DIV) {
      const TI* __restrict__ ar = a.ab_r[f] + e0 + r;
      const TI* __restrict__ af = a.ab_f[f] + e0 + r;
      v0 = v0 + a.ab_dt * (a.ab_t1 * (T)at_bytes(ar, off) + a.ab_t2 * (T)at_bytes(af, off));
      v1 = v1 + a.ab_dt * (a.ab_t1 * (T)at_bytes(ar + N, off) + a.ab_t2 * (T)at_bytes(af + N, off));
    }
    if constexpr (MODE == LOAD_PCLEAN) {
      const int k = a.k0 + (int)(job / (a.ny / 2));
      if (k == 0 || k == a.pc_nz + 1) {
        v0 = (T)0;
        v1 = (T)0;
      } else {
        const long pl = (long)a.ny * N;
        const TI* __restrict__ u = a.ab_r[0] + e0 + r;
        const TI* __restrict__ vv = a.ab_r[1] + e0 + r;
        const TI* __restrict__ w = a.ab_r[2] + e0 + r;
        const T u0 = (T)at_bytes(u, off), u1 = (T)at_bytes(u + N, off);
        const T w0 = (T)at_bytes(vv, off), w1 = (T)at_bytes(vv + N, off);
        const T h0 = (T)0.5 * ((T)at_bytes(w, off) + (T)at_bytes(w + pl, off));
        const T h1 = (T)0.5 * ((T)at_bytes(w + N, off) + (T)at_bytes(w + N + pl, off));
        v0 = v0 - (T)0.5 * ((u0 * u0 + w0 * w0) + h0 * h0);
        v1 = v1 - (T)0.5 * ((u1 * u1 + w1 * w1) + h1 * h1);
      }
    }
    if constexpr (MODE == LOAD_SCALE_DIV || MODE == LOAD_AB2_SCALE_DIV)
      return Cplx<T>{a.scale * (v0 / a.div), a.scale * (v1 / a.div)};
    else
      return Cplx<T>{a.scale * v0, a.scale * v1};
  };
  Cplx<T> X[S::VX];
  if constexpr (STREAM) {
    const RowStream<S, N> st;
    Cplx<T>* lines = reinterpret_cast<Cplx<T>*>(smem_raw);
    const long njobs = (long)a.nplanes * (a.ny / 2);
#pragma unroll
    for (int i = 0; i < RowStream<S, N>::IT; ++i) {
      int l, n;
      if (st.item(i, l, n) && at.job0 + l < njobs)
        lds_st(lines + l * S::LS + n, value(0, (unsigned)(2 * l * N + n) * (unsigned)sizeof(TI), at.job0 + l));
    }
    sync();
    L::template get<0>(X, line, at.a);
    sync();
  } else {
    const unsigned off = (unsigned)(2 * at.dj * N + at.a) * (unsigned)sizeof(TI);
    L::template rows<0>(at.a, [&](int v, int r) LES_INLINE { X[v] = value(r, off, at.job0 + at.dj); });
  }
  L::template fft<false>(X, line, tw, at.a, sync);
  L::template put<L::LAST>(X, line, at.a);
  sync();
  if (at.valid) row_unpack<S, T, N>(line, a.dst[f] + row0 * LHX, at);
}

// k_rows_r2c_reg of FP64 fields with the first pass of the mixed mode's FP64
// Nyquist removal folded into the load (the sums k_nyq_reduce forms, from the
// values this kernel reads anyway): A_j = sum_i (-1)^i f_ij / nx of both rows
// (the same lane-strided sums and butterfly as k_nyq_reduce), and per band of
// 4 row pairs the column partial sum_j (-1)^j f_ij.  A wavefront reads a whole
// band, 64 consecutive values at a time, and keeps the column partials in
// registers, the 4 pairs added in order; the lines go to LDS and from there
// into the transform's layout.  Lengths that divide a wavefront read their own
// lines and need no block barrier.
// Needs ny % 8 == 0: a band lies in one plane and is whole.
// Bound by memory: u, v, w at 128^3 34.5 -> 20.1 us against lines transformed
// in LDS by one wavefront each, 192x192x64 31.0 -> 18.0, 384x384x64 138 -> 101,
// 512x256x64 139 -> 102, 256x256x128 89 -> 85 (3.6 TB/s).  Where a block has
// fewer bands than wavefronts some only wait while the others load (576 points:
// 52 -> 55 us at 256x64, equal at 512x128).
template <typename T, int N>
struct NyqShape {
  using R = RowShape<T, N>;
  static constexpr int NT = R::NT, LS = R::LS;
  static constexpr bool WAVE = R::WAVE;
  // whole bands; short lines in one wavefront (96x48x37: 17 -> 12 us), long ones
  // in four (288x288x64: 53 -> 50).  A wavefront sums its bands in turn: at most
  // four of them, also where lines of one or two threads would fill it with 8 or
  // 16 (grad_velocity_filt at ny 16, 8 levels: 12 points 35.0 -> 16.6 us, 24 23.7 ->
  // 17.3, 8 20.1 -> 15.2; at ny 64, 512 levels 12 points 40.3 -> 24.3).
  static constexpr int TH = N < 256 ? 64 : 256;
  static constexpr int LB = !WAVE ? (TH / NT >= 4 ? TH / NT / 4 * 4 : 4) : R::THREADS == 64 && R::LB > 16 ? 16 : R::LB;
  static constexpr int THREADS = (LB * NT + 63) / 64 * 64, LINES = (THREADS + NT - 1) / NT;  // whole wavefronts
  static constexpr int NW = THREADS / 64, BW = (LB / 4 + NW - 1) / NW;  // wavefronts, bands of one
  static constexpr size_t LDS = (size_t)LINES * LS * sizeof(Cplx<T>);
  static constexpr int VX = R::VX;
  static_assert(LB % 4 == 0 && (!WAVE || 64 / NT % 4 == 0), "wavefronts hold whole bands");
};

template <typename T, int N>
__global__ void __launch_bounds__((NyqShape<T, N>::THREADS)) k_rows_r2c_nyq(RowR2CArgs<double, T> a, const Cplx<T>* __restrict__ tw) {
  using S = NyqShape<T, N>;
  using L = typename S::R::L1;
  // bands of a wavefront: its own lines', else every NW-th
  constexpr int J = (N + 63) / 64, NW = S::NW, BW = S::BW;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const long njobs = (long)a.nplanes * (a.ny / 2);
  RowAt<S> at(njobs);
  at.valid = at.valid && at.line() < S::LB;  // the last lanes may have no line to store
  Cplx<T>* lines = reinterpret_cast<Cplx<T>*>(smem_raw);
  Cplx<T>* line = lines + at.line() * S::LS;
  const int f = blockIdx.y, lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  auto sync = []() LES_INLINE { row_sync<S::WAVE>(); };
  for (int i = 0; i < BW; ++i) {
    const int b = S::WAVE ? wave * BW + i : wave + i * NW;
    const long job = at.job0 + 4 * b;
    if (b >= S::LB / 4 || job >= njobs) break;
    const long row0 = (long)a.k0 * a.ny + 2 * job;
    const double* __restrict__ src = a.src[f] + row0 * N;
    double acc[J], s[8];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      double s0 = 0.0, s1 = 0.0;
      Cplx<T>* z = lines + (4 * b + t) * S::LS;
#pragma unroll
      for (int j = 0; j < J; ++j) {
        const int n = lane + 64 * j;
        if (N % 64 == 0 || n < N) {
          const double r0 = src[2 * t * N + n], r1 = src[(2 * t + 1) * N + n];
          s0 += (lane & 1) ? -r0 : r0;
          s1 += (lane & 1) ? -r1 : r1;
          acc[j] = t == 0 ? r0 - r1 : acc[j] + (r0 - r1);
          lds_st(z + n, Cplx<T>{a.scale * (T)r0, a.scale * (T)r1});
        }
      }
      s[2 * t] = s0;
      s[2 * t + 1] = s1;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1)
#pragma unroll
      for (int r = 0; r < 8; ++r) s[r] += __shfl_xor(s[r], o, 64);
    double* __restrict__ A = a.nyq_a + f * a.nyq_as + row0;
    if (lane == 0) {
#pragma unroll
      for (int r = 0; r < 8; ++r) A[r] = s[r] / (double)N;
    }
    double* __restrict__ P = a.nyq_p + f * a.nyq_ps + job / 4 * N;
#pragma unroll
    for (int j = 0; j < J; ++j)
      if (N % 64 == 0 || lane + 64 * j < N) P[lane + 64 * j] = acc[j];
  }
  sync();
  Cplx<T> X[S::VX];
  L::template get<0>(X, line, at.a);
  sync();
  L::template fft<false>(X, line, tw, at.a, sync);
  L::template put<L::LAST>(X, line, at.a);
  sync();
  if (at.valid) row_unpack<S, T, N>(line, a.dst[f] + ((long)a.k0 * a.ny + 2 * at.job0) * (N / 2 + 1), at);
}

// ------------------------------------------------------------------ c2r
// The half spectra of a row pair as one line, inverse transform: X ends with
// row 2 jp in .x and row 2 jp + 1 in .y.
template <typename S, typename T, int N, typename AT, typename SYNC>
__device__ __forceinline__ void row_c2r_line(Cplx<T>* X, Cplx<T>* line, const Cplx<T>* __restrict__ src, const AT& at,
                                             const Cplx<T>* __restrict__ tw, SYNC&& sync) {
  using L = typename S::L1;
  constexpr int LHX = N / 2 + 1, H = N / 2, NT = S::NT;
  const unsigned off = (unsigned)(2 * at.dj * LHX + at.a) * (unsigned)sizeof(Cplx<T>);
  constexpr int M = (LHX + NT - 1) / NT, CH = M > 5 ? (M + 1) / 2 : M;
  // two batches of loads at most, so that they are in flight together
#pragma unroll
  for (int b = 0; b < M; b += CH) {
    Cplx<T> A[CH], B[CH];
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      const int q = (b + i) * NT;
      if (b + i < M && (q + NT <= LHX || q + at.a < LHX)) {
        A[i] = at_bytes(src + q, off);
        B[i] = at_bytes(src + q + LHX, off);
      }
    }
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      const int q = (b + i) * NT, kk = q + at.a;
      if (b + i < M && (q + NT <= LHX || kk < LHX)) {
        const bool edge = kk == 0 || kk == H;
        if (edge) {
          A[i].y = (T)0;
          B[i].y = (T)0;
        }
        lds_st(line + kk, Cplx<T>{A[i].x - B[i].y, A[i].y + B[i].x});
        if (!edge) lds_st(line + N - kk, Cplx<T>{A[i].x + B[i].y, B[i].x - A[i].y});
      }
    }
  }
  sync();
  L::template get<0>(X, line, at.a);
  sync();
  L::template fft<true>(X, line, tw, at.a, sync);
}

template <typename T, typename TO, int N>
__global__ void __launch_bounds__((RowShape<T, N>::THREADS)) k_rows_c2r_reg(RowC2RArgs<T, TO> a, const Cplx<T>* __restrict__ tw) {
  using S = RowShape<T, N>;
  using L = typename S::L1;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const RowAt<S> at((long)a.nplanes * (a.ny / 2));
  Cplx<T>* line = reinterpret_cast<Cplx<T>*>(smem_raw) + at.line() * S::LS;
  const long row0 = (long)a.k0 * a.ny + 2 * at.job0;
  auto sync = []() LES_INLINE { row_sync<S::WAVE>(); };
  Cplx<T> X[S::VX];
  row_c2r_line<S, T, N>(X, line, a.src[blockIdx.y] + row0 * (N / 2 + 1), at, tw, sync);
  if (at.valid) {
    TO* __restrict__ dst = a.dst[blockIdx.y] + row0 * N;
    const unsigned off = (unsigned)(2 * at.dj * N + at.a) * (unsigned)sizeof(TO);
    L::template rows<L::LAST>(at.a, [&](int v, int r) LES_INLINE {
      put_bytes(dst + r, off, (TO)X[v].x);
      put_bytes(dst + r + N, off, (TO)X[v].y);
    });
  }
}

// c2r with an epilogue as the store, in RowStream order through LDS: epi(k, q,
// n, ok, z) gets chunks of LES_EPI_CHUNK items (plane, in-plane start of row 2 jp,
// element, value) so that it can issue a chunk's loads together.
template <typename S, typename T, int N, typename EPI>
__device__ __forceinline__ void row_epilogue(Cplx<T>* X, Cplx<T>* lines, const RowAt<S>& at, int k0, int ny, long njobs, EPI&& epi) {
  using L = typename S::L1;
  using ST = RowStream<S, N>;
  L::template put<L::LAST>(X, lines + at.line() * S::LS, at.a);
  row_sync<S::WAVE>();
  const ST st;
  const int npairs = ny / 2;
#pragma unroll
  for (int b = 0; b < ST::IT; b += LES_EPI_CHUNK) {
    int k[LES_EPI_CHUNK], q[LES_EPI_CHUNK];
    bool ok[LES_EPI_CHUNK];
    Cplx<T> z[LES_EPI_CHUNK];
#pragma unroll
    for (int u = 0; u < LES_EPI_CHUNK; ++u) {
      int l = 0, n = 0;
      ok[u] = b + u < ST::IT && st.item(b + u, l, n) && at.job0 + l < njobs;
      const int job = ok[u] ? (int)at.job0 + l : 0, pl = job / npairs;
      k[u] = k0 + pl;
      q[u] = (job - pl * npairs) * 2 * N + n;
      if (ok[u]) z[u] = lds_ld(lines + l * S::LS + n);
    }
    epi(k, q, ok, z);
  }
}

// c2r with the stress divergence's rhs update as the store (per component).
template <typename T, int N>
__global__ void __launch_bounds__((RowShape<T, N>::THREADS)) k_rows_c2r_div_reg(RowC2RArgs<T, T> a, DivEpi3<T> ep,
                                                                                const Cplx<T>* __restrict__ tw) {
  using S = RowShape<T, N>;
  using L = typename S::L1;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const RowAt<S> at((long)a.nplanes * (a.ny / 2));
  Cplx<T>* line = reinterpret_cast<Cplx<T>*>(smem_raw) + at.line() * S::LS;
  const long row0 = (long)a.k0 * a.ny + 2 * at.job0;
  auto sync = []() LES_INLINE { row_sync<S::WAVE>(); };
  Cplx<T> X[S::VX];
  row_c2r_line<S, T, N>(X, line, a.src[blockIdx.y] + row0 * (N / 2 + 1), at, tw, sync);
  if (at.valid) {
    const DivEpiArgs<T>& e = ep.c[blockIdx.y];
    const int job = (int)(at.job0 + at.dj), npairs = a.ny / 2, pl = job / npairs;
    const long q = (long)(job - pl * npairs) * 2 * N + at.a;
    div_epi_rows<T, N, S::VX>(e, a.k0 + pl, q, [&](auto&& fn) LES_INLINE { L::template rows<L::LAST>(at.a, fn); }, X);
  }
}

// c2r of the pressure-gradient spectra with the projection as the store: from
// registers, or (STREAM) in RowStream order through LDS.  The projection reads
// three FP64 fields per value and writes two; the wider accesses win from 128
// points (128: 63 -> 54 us, 256 435 -> 416 us at 256 levels), lose below (64:
// 15 -> 23 us) and make no difference beyond 384.
constexpr bool proj_stream(int n) { return n >= 128 && n <= 384; }
template <int N>
__global__ void __launch_bounds__((RowShape<double, N>::THREADS)) k_rows_c2r_proj_reg(RowC2RArgs<double, double> a, ProjEpi3 ep,
                                                                                      const Cplx<double>* __restrict__ tw) {
  using S = RowShape<double, N>;
  using L = typename S::L1;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const long njobs = (long)a.nplanes * (a.ny / 2);
  const RowAt<S> at(njobs);
  Cplx<double>* lines = reinterpret_cast<Cplx<double>*>(smem_raw);
  const long row0 = (long)a.k0 * a.ny + 2 * at.job0;
  auto sync = []() LES_INLINE { row_sync<S::WAVE>(); };
  Cplx<double> X[S::VX];
  row_c2r_line<S, double, N>(X, lines + at.line() * S::LS, a.src[blockIdx.y] + row0 * (N / 2 + 1), at, tw, sync);
  const ProjEpiArgs& e = ep.c[blockIdx.y];
  if constexpr (proj_stream(N)) {
    row_epilogue<S, double, N>(X, lines, at, a.k0, a.ny, njobs,
                               [&](const int* k, const int* q, const bool* ok, const Cplx<double>* z) LES_INLINE {
                                 proj_epi_chunk<N>(ep, e, k, q, ok, z);
                               });
  } else if (at.valid) {
    const int job = (int)(at.job0 + at.dj), npairs = a.ny / 2, pl = job / npairs;
    const long q = (long)(job - pl * npairs) * 2 * N + at.a;
    proj_epi_rows<N, S::VX>(ep, e, a.k0 + pl, q, [&](auto&& fn) LES_INLINE { L::template rows<L::LAST>(at.a, fn); }, X);
  }
}

// ------------------------------------------------------------------ 3/2 resampling
// Source `which` of the convection (conv_src) for a thread's elements: body(fn)
// with fn(r) the value at element e0 + off + r, k the thread's plane.
template <typename T, typename BODY>
__device__ __forceinline__ void conv_src_rows(const ConvSrc<T>& s, int which, int k, long e0, unsigned off, long np, T c,
                                              BODY&& body) {
  const unsigned o8 = off * 8u, ot = off * (unsigned)sizeof(T);
  const bool wall = k == 1;
  if (which < 3) {
    const double* __restrict__ f = (which == 0 ? s.u : which == 1 ? s.v : s.w) + e0;
    body([&](int r) LES_INLINE { return (T)(-((double)c * at_bytes(f + r, o8))); });
  } else if (which == 3) {
    const T* __restrict__ wy = s.dwdy + e0;
    const T* __restrict__ vz = s.dvdz + e0;
    body([&](int r) LES_INLINE {
      T w = at_bytes(wy + r, ot);
      if (wall) w = (T)0.5 * (w + at_bytes(wy + r + np, ot));
      return c * (w - at_bytes(vz + r, ot));
    });
  } else if (which == 4) {
    const T* __restrict__ uz = s.dudz + e0;
    const T* __restrict__ wx = s.dwdx + e0;
    body([&](int r) LES_INLINE {
      T w = at_bytes(wx + r, ot);
      if (wall) w = (T)0.5 * (w + at_bytes(wx + r + np, ot));
      return c * (at_bytes(uz + r, ot) - w);
    });
  } else {
    const T* __restrict__ vx = s.dvdx + e0;
    const T* __restrict__ uy = s.dudy + e0;
    body([&](int r) LES_INLINE { return c * (at_bytes(vx + r, ot) - at_bytes(uy + r, ot)); });
  }
}

// N: the shorter length.  PAD: the convection sources (conv_src, one per
// blockIdx.y) N -> 3 N / 2; else rows of src 3 N / 2 -> N.
template <typename T, typename TO, int N, bool PAD>
__global__ void __launch_bounds__((RowShape<T, N, 3 * N / 2>::THREADS)) k_rows_resample_reg(
    RowResArgs<T, T, TO> a, const Cplx<T>* __restrict__ twn, const Cplx<T>* __restrict__ twb) {
  using S = RowShape<T, N, 3 * N / 2>;
  constexpr int NB = 3 * N / 2, N1 = PAD ? N : NB, N2 = PAD ? NB : N, H = N / 2, NT = S::NT;
  using L1 = RegLine<T, N1, NT, col_maxg<T>(), true>;
  using L2 = RegLine<T, N2, NT, col_maxg<T>(), true>;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  if constexpr (!PAD) {
    // the blocks past the row pairs fill the ghost planes below and above
    const long np = (long)N * a.ny, nb = ((long)a.nplanes * (a.ny / 2) + S::LB - 1) / S::LB;
    if ((long)blockIdx.x >= nb) {
      TO* __restrict__ lo = a.dst[blockIdx.y] + (a.k0 - 1) * np;
      TO* __restrict__ hi = a.dst[blockIdx.y] + (a.k0 + a.nplanes) * np;
      for (long q = (blockIdx.x - nb) * S::THREADS + threadIdx.x; q < np; q += (gridDim.x - nb) * S::THREADS) {
        lo[q] = (TO)a.ghost;
        hi[q] = (TO)a.ghost;
      }
      return;
    }
  }
  const RowAt<S> at((long)a.nplanes * (a.ny / 2));
  Cplx<T>* line = reinterpret_cast<Cplx<T>*>(smem_raw) + at.line() * S::LS;
  const int f = blockIdx.y;
  const long row0 = (long)a.k0 * a.ny + 2 * at.job0;
  auto sync = []() LES_INLINE { row_sync<S::WAVE>(); };
  Cplx<T> X[S::VX];
  if constexpr (PAD) {
    const int k = a.k0 + (int)((at.job0 + at.dj) / (a.ny / 2));
    const long e0 = row0 * N;
    const unsigned off = (unsigned)(2 * at.dj * N + at.a);
    conv_src_rows<T>(a.cs, f, k, e0, off, (long)N * a.ny, a.cconv, [&](auto&& fn) LES_INLINE {
      L1::template rows<0>(at.a, [&](int v, int r) LES_INLINE { X[v] = Cplx<T>{fn(r), fn(r + N)}; });
    });
  } else {
    const T* __restrict__ src = a.src[f] + row0 * NB;
    const unsigned off = (unsigned)(2 * at.dj * NB + at.a) * (unsigned)sizeof(T);
    L1::template rows<0>(at.a, [&](int v, int r) LES_INLINE {
      X[v] = Cplx<T>{at_bytes(src + r, off), at_bytes(src + r + NB, off)};
    });
  }
  L1::template fft<false>(X, line, PAD ? twn : twb, at.a, sync);
  L1::template rows<L1::LAST>(at.a, [&](int v, int r) LES_INLINE {
    const int m = at.a + r;
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
      if (e + at.a <= N) lds_st(line + e + at.a, zero);
  } else {
    if (at.a == 0) lds_st(line + H, zero);
  }
  sync();
  L2::template get<0>(X, line, at.a);
  sync();
  L2::template fft<true>(X, line, PAD ? twb : twn, at.a, sync);
  if (at.valid) {
    TO* __restrict__ dst = a.dst[f] + row0 * N2;
    const unsigned off = (unsigned)(2 * at.dj * N2 + at.a) * (unsigned)sizeof(TO);
    L2::template rows<L2::LAST>(at.a, [&](int v, int r) LES_INLINE {
      put_bytes(dst + r, off, (TO)X[v].x);
      put_bytes(dst + r + N2, off, (TO)X[v].y);
    });
  }
}
