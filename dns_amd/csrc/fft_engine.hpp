// Device-side Stockham FFT engine for gfx950 (CDNA4).
//
// A length-N pencil is owned by TPP = N/E threads; thread t holds the E
// elements at positions t + TPP*c (c = 0..E-1) in registers.  Each stage of
// radix r performs E/r butterflies per thread:
//   butterfly j = t + q*TPP reads x[j + m*N/r] (= register q + m*E/r),
//   multiplies by w^(m*(j mod Ns)) with w = exp(-+2 pi i/(Ns r)), applies a
//   radix-r DFT and writes y[(j/Ns)*Ns*r + j%Ns + m*Ns].
// Between stages the values go through LDS; after the last stage
// (Ns = N/r) the outputs land back on the load positions t + TPP*c, so a
// pencil is read from and written to HBM with the same, coalesced pattern.
//
// Twiddles come from a per-N table (generated on the host in long double,
// rounded once to the working precision); stage 0 needs none.
#pragma once
#include <hip/hip_runtime.h>
#include <type_traits>
#include <utility>

// All arithmetic from here on is rounded as written: sums of products use fm()
// where a fused multiply-add is wanted.  Left to the compiler, which product
// of a sum is fused depends on the code around it, and launch shapes of one
// kernel (which have to give bitwise identical results) came out different.
#pragma clang fp contract(off)

namespace dnsk {

// a * b + c, rounded once
__device__ __forceinline__ double fm(double a, double b, double c) { return __builtin_fma(a, b, c); }
__device__ __forceinline__ float fm(float a, float b, float c) { return __builtin_fmaf(a, b, c); }

template <typename R> struct cx_of;
template <> struct cx_of<double> { using type = double2; };
template <> struct cx_of<float> { using type = float2; };
template <typename R> using cx = typename cx_of<R>::type;

template <typename R> __device__ __forceinline__ cx<R> mk(R a, R b) {
  cx<R> z;
  z.x = a;
  z.y = b;
  return z;
}
template <typename R> __device__ __forceinline__ cx<R> cadd(cx<R> a, cx<R> b) { return mk<R>(a.x + b.x, a.y + b.y); }
template <typename R> __device__ __forceinline__ cx<R> csub(cx<R> a, cx<R> b) { return mk<R>(a.x - b.x, a.y - b.y); }
template <typename R> __device__ __forceinline__ cx<R> cmul(cx<R> a, cx<R> b) {
  return mk<R>(fm(a.x, b.x, -(a.y * b.y)), fm(a.x, b.y, a.y * b.x));
}
template <typename R> __device__ __forceinline__ cx<R> cmulc(cx<R> a, cx<R> b) {  // a * conj(b)
  return mk<R>(fm(a.x, b.x, a.y * b.y), fm(a.y, b.x, -(a.x * b.y)));
}
// multiply by -i (forward) or +i (inverse)
template <typename R, bool INV> __device__ __forceinline__ cx<R> rot(cx<R> a) {
  return INV ? mk<R>(-a.y, a.x) : mk<R>(a.y, -a.x);
}

// Streaming stores: every pass writes each element exactly once and the next
// pass reads it from HBM, so stores use the non-temporal path.
#ifndef DNS_NT_STORES
#define DNS_NT_STORES 1
#endif
template <typename R> __device__ __forceinline__ void st(cx<R> *p, cx<R> v) {
#if DNS_NT_STORES
  typedef R v2 __attribute__((ext_vector_type(2)));
  v2 t = {v.x, v.y};
  __builtin_nontemporal_store(t, (v2 *)p);
#else
  *p = v;
#endif
}
// Non-temporal load of a complex element that its pass reads once: the x
// pass with these loads runs 3.7% (FP64) and 5% (float) faster at n=512,
// the inverse y pass 4%, the z pass 3-5% (its Hermitian loads fetch each
// element once and pass the mirrored half between lanes; loading both
// halves non-temporally instead costs 7%).
template <typename T> __device__ __forceinline__ T ldnt(const T *p) {
  typedef decltype(p->x) E;
  typedef E v2 __attribute__((ext_vector_type(2)));
  v2 t = __builtin_nontemporal_load((const v2 *)p);
  T r;
  r.x = t.x;
  r.y = t.y;
  return r;
}
// Load of one element of a tile row of COLS consecutive elements: non-
// temporal when the row covers whole 128-byte lines.  Narrower rows share
// their lines with the neighbouring tile's block, which finds the other
// half in L2 only with ordinary loads (n=1024, 64-byte rows: non-temporal
// loads cost 13%).
template <int COLS, typename T> __device__ __forceinline__ T ld_row(const T *p) {
  if constexpr (COLS * sizeof(T) >= 128) return ldnt(p);
  else return *p;
}
// Load of one element of a state-layout tile row (two x rows share each
// line; see srow): non-temporal when the tile's two rows cover whole lines.
template <int COLS, typename T> __device__ __forceinline__ T ld_state(const T *p) {
  if constexpr (2 * COLS * sizeof(T) >= 128) return ldnt(p);
  else return *p;
}
template <typename R> __device__ __forceinline__ void st_real(R *p, R v) {
#if DNS_NT_STORES
  __builtin_nontemporal_store(v, p);
#else
  *p = v;
#endif
}

// ---------------------------------------------------------------------------
// Radix schedules.  E = elements per thread, so a pencil takes N/E threads.
// The first and last radix divide E; a middle one need not (fft_pencil).  E
// and the number of stages were chosen by hand from builds of one size,
// the radix order of the power-of-two grids from 128 on by
// dns_amd/tune_radix.py, which times the other orders of a size against the row
// below (a candidate build replaces it with -DDNS_SCHED_N=n -DDNS_SCHED_E=e
// -DDNS_SCHED_R=r0,r1,...).
//
// Each stage costs an exchange through LDS and two barriers, and 12
// elements per thread are what held most grids with a factor 3 back: the
// FP64 z pass then takes all 512 registers (one wave per SIMD) and the x pass
// spills.  Microseconds a step of the former 12- and 6-element schedules of
// radices 4, 3, 2 -> these (one box): FP64 n=96 390 -> 290, n=216 3970 -> 2800,
// n=432 35600 -> 21600, n=486 58300 -> 29900; mixed n=162 903 -> 752, n=384
// 9560 -> 8050, n=648 119200 -> 46500, n=972 376700 -> 174000.  Measured
// and not taken: n=486 and n=648 with 6 elements (28.1 and 63.6 ms mixed:
// tiles of 4 columns), n=576 8-9-8 (61.7 ms FP64 against 56.1, mixed
// 33.6 against 28.6), n=128 and n=256 with radix 16 (683 against 573 us, 3.99
// against 3.74 ms FP64).
template <int N> struct SchedTable;
#define DNS_SCHED(N_, E_, ...)                                \
  template <> struct SchedTable<N_> {                         \
    static constexpr int E = E_;                              \
    static constexpr int r[] = {__VA_ARGS__};                 \
    static constexpr int NS = sizeof(r) / sizeof(r[0]);       \
  };
DNS_SCHED(8, 4, 4, 2)
DNS_SCHED(12, 6, 6, 2)
DNS_SCHED(16, 4, 4, 4)
DNS_SCHED(18, 6, 6, 3)
DNS_SCHED(24, 4, 4, 3, 2)
DNS_SCHED(32, 4, 4, 2, 4)
DNS_SCHED(36, 6, 6, 6)
DNS_SCHED(48, 4, 4, 3, 4)
DNS_SCHED(54, 6, 6, 3, 3)
DNS_SCHED(64, 4, 4, 4, 4)
DNS_SCHED(72, 6, 6, 2, 6)
DNS_SCHED(96, 4, 4, 6, 4)
DNS_SCHED(108, 6, 6, 3, 6)
DNS_SCHED(128, 8, 8, 8, 2)
DNS_SCHED(144, 6, 6, 4, 6)
DNS_SCHED(162, 6, 6, 9, 3)
DNS_SCHED(192, 8, 8, 3, 8)
DNS_SCHED(216, 6, 6, 6, 6)
DNS_SCHED(256, 8, 8, 4, 8)
DNS_SCHED(288, 6, 6, 8, 6)
DNS_SCHED(324, 6, 6, 9, 6)
DNS_SCHED(384, 8, 8, 6, 8)
DNS_SCHED(432, 9, 9, 16, 3)
DNS_SCHED(486, 9, 9, 6, 9)
DNS_SCHED(512, 8, 8, 8, 8)
DNS_SCHED(576, 12, 12, 4, 12)
DNS_SCHED(648, 12, 12, 9, 6)
DNS_SCHED(768, 12, 12, 16, 4)
DNS_SCHED(864, 12, 12, 6, 12)
DNS_SCHED(972, 9, 9, 12, 9)
DNS_SCHED(1024, 8, 8, 8, 4, 4)
#undef DNS_SCHED
// Float kernels of a size whose float schedule is another one.  n=64: one
// twiddle stage instead of two leaves four mixed steps an error of 1.66e-7 of
// what they change instead of 1.80e-7, and the plane pass two stages instead of
// three (mixed 125 -> 118 us a step, six members 321 -> 300); in FP64 it takes 4%
// longer (165 us instead of 159 as a batch of one).
template <int N> struct SchedFloat : SchedTable<N> {};
#define DNS_SCHED_FLOAT(N_, E_, ...)                          \
  template <> struct SchedFloat<N_> {                         \
    static constexpr int E = E_;                              \
    static constexpr int r[] = {__VA_ARGS__};                 \
    static constexpr int NS = sizeof(r) / sizeof(r[0]);       \
  };
DNS_SCHED_FLOAT(64, 8, 8, 8)
#undef DNS_SCHED_FLOAT
template <int N, typename R> struct Sched : std::conditional_t<sizeof(R) == 4, SchedFloat<N>, SchedTable<N>> {};
#ifdef DNS_SCHED_N
template <typename R> struct Sched<DNS_SCHED_N, R> {
  static constexpr int E = DNS_SCHED_E;
  static constexpr int r[] = {DNS_SCHED_R};
  static constexpr int NS = sizeof(r) / sizeof(r[0]);
};
#endif

template <int N, typename R> constexpr int stage_Ns(int s) {
  int ns = 1;
  for (int q = 0; q < s; q++) ns *= Sched<N, R>::r[q];
  return ns;
}
template <int N, typename R> constexpr int stage_twoff(int s) {
  int off = 0, ns = 1;
  for (int q = 0; q < s; q++) {
    off += ns * (Sched<N, R>::r[q] - 1);
    ns *= Sched<N, R>::r[q];
  }
  return off;
}
template <int N, typename R> constexpr int tw_size() { return stage_twoff<N, R>(Sched<N, R>::NS); }

template <int I, int END, class F> __device__ __forceinline__ void static_for(F &&f) {
  if constexpr (I < END) {
    f(std::integral_constant<int, I>{});
    static_for<I + 1, END>(f);
  }
}

// ---------------------------------------------------------------------------
// Radix-r DFTs in registers (unnormalised; INV selects exp(+i)).
template <typename R, bool INV> __device__ __forceinline__ void dft2(cx<R> *a) {
  cx<R> t = a[0];
  a[0] = cadd<R>(t, a[1]);
  a[1] = csub<R>(t, a[1]);
}
template <typename R, bool INV> __device__ __forceinline__ void dft4(cx<R> *a) {
  cx<R> s0 = cadd<R>(a[0], a[2]), d0 = csub<R>(a[0], a[2]);
  cx<R> s1 = cadd<R>(a[1], a[3]), d1 = rot<R, INV>(csub<R>(a[1], a[3]));
  a[0] = cadd<R>(s0, s1);
  a[2] = csub<R>(s0, s1);
  a[1] = cadd<R>(d0, d1);
  a[3] = csub<R>(d0, d1);
}
template <typename R, bool INV> __device__ __forceinline__ void dft3(cx<R> *a) {
  const R s3 = (R)0.86602540378443864676372317075294;  // sin(2 pi / 3)
  cx<R> t1 = cadd<R>(a[1], a[2]);
  const cx<R> t2 = mk<R>(fm((R)-0.5, t1.x, a[0].x), fm((R)-0.5, t1.y, a[0].y));
  const cx<R> d = rot<R, INV>(csub<R>(a[1], a[2]));
  a[0] = cadd<R>(a[0], t1);
  a[1] = mk<R>(fm(s3, d.x, t2.x), fm(s3, d.y, t2.y));
  a[2] = mk<R>(fm(-s3, d.x, t2.x), fm(-s3, d.y, t2.y));
}
template <typename R, bool INV> __device__ __forceinline__ void dft8(cx<R> *a) {
  const R h = (R)0.70710678118654752440084436210485;  // 1/sqrt(2)
  cx<R> s[4], d[4];
#pragma unroll
  for (int m = 0; m < 4; m++) {
    s[m] = cadd<R>(a[m], a[m + 4]);
    d[m] = csub<R>(a[m], a[m + 4]);
  }
  // d[m] *= w8^m, w8 = exp(-+ i pi/4); the factor h of d[1] and d[3] is left
  // to the fused sums below
  d[2] = rot<R, INV>(d[2]);
  if (INV) {
    d[1] = mk<R>(d[1].x - d[1].y, d[1].x + d[1].y);
    d[3] = mk<R>(-(d[3].x + d[3].y), d[3].x - d[3].y);
  } else {
    d[1] = mk<R>(d[1].x + d[1].y, d[1].y - d[1].x);
    d[3] = mk<R>(d[3].y - d[3].x, -(d[3].x + d[3].y));
  }
  dft4<R, INV>(s);
  const cx<R> s0 = cadd<R>(d[0], d[2]), d0 = csub<R>(d[0], d[2]);
  const cx<R> s1 = cadd<R>(d[1], d[3]), d1 = rot<R, INV>(csub<R>(d[1], d[3]));
  a[1] = mk<R>(fm(h, s1.x, s0.x), fm(h, s1.y, s0.y));
  a[3] = mk<R>(fm(h, d1.x, d0.x), fm(h, d1.y, d0.y));
  a[5] = mk<R>(fm(-h, s1.x, s0.x), fm(-h, s1.y, s0.y));
  a[7] = mk<R>(fm(-h, d1.x, d0.x), fm(-h, d1.y, d0.y));
#pragma unroll
  for (int p = 0; p < 4; p++) a[2 * p] = s[p];
}
// a *= c -+ i s, c = cos x, s = sin x (exp(-i x), INV exp(+i x))
template <typename R, bool INV> __device__ __forceinline__ cx<R> turn(cx<R> a, R c, R s) {
  return INV ? mk<R>(fm(c, a.x, -(s * a.y)), fm(c, a.y, s * a.x)) : mk<R>(fm(c, a.x, s * a.y), fm(c, a.y, -(s * a.x)));
}
template <typename R, bool INV> __device__ __forceinline__ void dft9(cx<R> *a) {
  // 3 x 3: columns a[m], a[m+3], a[m+6], twiddles w9^(m q), rows
  const R c1 = (R)0.7660444431189780352023926505554, s1 = (R)0.6427876096865393263226434099073;   // 2 pi / 9
  const R c2 = (R)0.1736481776669303488517166267693, s2 = (R)0.9848077530122080593667430245895;   // 4 pi / 9
  const R c4 = (R)-0.9396926207859083840541092773247, s4 = (R)0.3420201433256687330440996146823;  // 8 pi / 9
  cx<R> b[3][3];
#pragma unroll
  for (int m = 0; m < 3; m++) {
    b[m][0] = a[m];
    b[m][1] = a[m + 3];
    b[m][2] = a[m + 6];
    dft3<R, INV>(b[m]);
  }
  b[1][1] = turn<R, INV>(b[1][1], c1, s1);
  b[1][2] = turn<R, INV>(b[1][2], c2, s2);
  b[2][1] = turn<R, INV>(b[2][1], c2, s2);
  b[2][2] = turn<R, INV>(b[2][2], c4, s4);
#pragma unroll
  for (int q = 0; q < 3; q++) {
    cx<R> r[3] = {b[0][q], b[1][q], b[2][q]};
    dft3<R, INV>(r);
    a[q] = r[0];
    a[q + 3] = r[1];
    a[q + 6] = r[2];
  }
}
template <typename R, bool INV> __device__ __forceinline__ void dft16(cx<R> *a) {
  // 4 x 4: columns a[m], a[m+4], .., twiddles w16^(m q), rows
  const R h = (R)0.70710678118654752440084436210485;
  const R c = (R)0.9238795325112867561281831893968, s = (R)0.3826834323650897717284599840304;  // pi / 8
  cx<R> b[4][4];
#pragma unroll
  for (int m = 0; m < 4; m++) {
#pragma unroll
    for (int q = 0; q < 4; q++) b[m][q] = a[m + 4 * q];
    dft4<R, INV>(b[m]);
  }
  b[1][1] = turn<R, INV>(b[1][1], c, s);
  b[1][2] = turn<R, INV>(b[1][2], h, h);
  b[1][3] = turn<R, INV>(b[1][3], s, c);
  b[2][1] = turn<R, INV>(b[2][1], h, h);
  b[2][2] = rot<R, INV>(b[2][2]);
  b[2][3] = turn<R, INV>(b[2][3], -h, h);
  b[3][1] = turn<R, INV>(b[3][1], s, c);
  b[3][2] = turn<R, INV>(b[3][2], -h, h);
  b[3][3] = turn<R, INV>(b[3][3], -c, -s);
#pragma unroll
  for (int q = 0; q < 4; q++) {
    cx<R> r[4] = {b[0][q], b[1][q], b[2][q], b[3][q]};
    dft4<R, INV>(r);
#pragma unroll
    for (int m = 0; m < 4; m++) a[q + 4 * m] = r[m];
  }
}
// Radix PA * PB of coprime factors (Good's mapping, no twiddles): input
// PB n1 + PA n2 and output IB PB k1 + IA PA k2 modulo PA PB, IB = PB^-1 mod
// PA, IA = PA^-1 mod PB.
template <typename R, int RAD, bool INV> __device__ __forceinline__ void dft(cx<R> *a);
template <typename R, int PA, int PB, int IB, int IA, bool INV> __device__ __forceinline__ void dft_coprime(cx<R> *a) {
  constexpr int M = PA * PB;
  cx<R> b[PB][PA];
#pragma unroll
  for (int n2 = 0; n2 < PB; n2++) {
#pragma unroll
    for (int n1 = 0; n1 < PA; n1++) b[n2][n1] = a[(PB * n1 + PA * n2) % M];
    dft<R, PA, INV>(b[n2]);
  }
#pragma unroll
  for (int k1 = 0; k1 < PA; k1++) {
    cx<R> r[PB];
#pragma unroll
    for (int n2 = 0; n2 < PB; n2++) r[n2] = b[n2][k1];
    dft<R, PB, INV>(r);
#pragma unroll
    for (int k2 = 0; k2 < PB; k2++) a[(IB * PB * k1 + IA * PA * k2) % M] = r[k2];
  }
}
template <typename R, int RAD, bool INV> __device__ __forceinline__ void dft(cx<R> *a) {
  if constexpr (RAD == 2) dft2<R, INV>(a);
  else if constexpr (RAD == 3) dft3<R, INV>(a);
  else if constexpr (RAD == 4) dft4<R, INV>(a);
  else if constexpr (RAD == 6) dft_coprime<R, 2, 3, 1, 2, INV>(a);
  else if constexpr (RAD == 8) dft8<R, INV>(a);
  else if constexpr (RAD == 9) dft9<R, INV>(a);
  else if constexpr (RAD == 12) dft_coprime<R, 4, 3, 3, 1, INV>(a);
  else {
    static_assert(RAD == 16, "radix");
    dft16<R, INV>(a);
  }
}

// Twiddle table staged in LDS by the whole block.  LDS reads are waited for
// separately from global memory operations, so a transform that follows a
// batch of global stores does not stall until those stores complete (a
// global twiddle load would: loads and stores share one counter).
template <int N, typename R>
__device__ __forceinline__ const cx<R> *stage_twiddles(cx<R> *twl, const cx<R> *__restrict__ tw) {
  for (int i = threadIdx.x; i < tw_size<N, R>(); i += blockDim.x) twl[i] = tw[i];
  __syncthreads();
  return twl;
}

// ---------------------------------------------------------------------------
// LDS slot maps.  One dummy row every 8 positions breaks the power-of-two
// strides of the first stages' scattered writes.
template <int N> __device__ __forceinline__ int padpos(int pos) { return pos + (pos >> 3); }
template <int N> constexpr int padlen() { return N + N / 8; }

// Tile of T pencils, pencil index fastest (strided-axis passes).
template <int N, int T> struct TileSlot {
  int p;
  __device__ __forceinline__ int operator()(int pos) const { return padpos<N>(pos) * T + p; }
};
// Pencil-major (contiguous-axis passes).
template <int N> struct PencilSlot {
  int base;
  __device__ __forceinline__ int operator()(int pos) const { return base + padpos<N>(pos); }
};

// In-register FFT of one pencil.  v[c] holds position t + TPP*c on entry
// and the transform's coefficient at the same position on exit.
// All threads of the block must call it together (it uses __syncthreads).
// E (elements per thread) defaults to the schedule's; any multiple of the
// first and last radix works (fewer threads per pencil, more registers).  A
// middle stage may have a radix that does not divide E: its N/r butterflies
// then leave the last round of threads partly idle.
template <int N, typename R, bool INV, class Slot, int E>
__device__ __forceinline__ void fft_pencil(cx<R> (&v)[E], int t, cx<R> *lds, Slot slot,
                                           const cx<R> *__restrict__ tw) {
  constexpr int NS = Sched<N, R>::NS, TPP = N / E;
  static_assert(stage_Ns<N, R>(NS) == N && N % E == 0 && E % Sched<N, R>::r[0] == 0 && E % Sched<N, R>::r[NS - 1] == 0,
                "the radices multiply to N, E divides N, the first and last radix divide E");
  static_for<0, NS>([&](auto S) {
    constexpr int s = decltype(S)::value;
    constexpr int r = Sched<N, R>::r[s];
    constexpr int Ns = stage_Ns<N, R>(s);
    constexpr int toff = stage_twoff<N, R>(s);
    constexpr int B = N / r;                  // butterflies of the stage
    constexpr int Q = (B + TPP - 1) / TPP;    // per thread
    constexpr bool FULL = E % r == 0;         // every thread has all of its Q
    cx<R> x[FULL ? 1 : Q][r];                 // a partly filled stage reads its own inputs
    if constexpr (!FULL) {
#pragma unroll
      for (int q = 0; q < Q; q++) {
        const int j = t + q * TPP;
        if (j < B) {
#pragma unroll
          for (int m = 0; m < r; m++) x[q][m] = lds[slot(j + m * B)];
        }
      }
      __syncthreads();
    }
#pragma unroll
    for (int q = 0; q < Q; q++) {
      const int j = t + q * TPP;
      if (!FULL && j >= B) continue;
      cx<R> a[r];
#pragma unroll
      for (int m = 0; m < r; m++) {
        if constexpr (FULL) a[m] = v[q + m * Q];
        else a[m] = x[q][m];
      }
      if constexpr (s > 0) {
        const int k = j % Ns;
        const cx<R> *w = tw + toff + k * (r - 1);
#pragma unroll
        for (int m = 1; m < r; m++) a[m] = INV ? cmulc<R>(a[m], w[m - 1]) : cmul<R>(a[m], w[m - 1]);
      }
      dft<R, r, INV>(a);
      if constexpr (s == NS - 1) {
#pragma unroll
        for (int m = 0; m < r; m++) v[q + m * Q] = a[m];
      } else {
        const int base = (j / Ns) * Ns * r + (j % Ns);
#pragma unroll
        for (int m = 0; m < r; m++) lds[slot(base + m * Ns)] = a[m];
      }
    }
    if constexpr (s < NS - 1) {
      __syncthreads();
      if constexpr (E % Sched<N, R>::r[s + 1] == 0) {
#pragma unroll
        for (int c = 0; c < E; c++) v[c] = lds[slot(t + TPP * c)];
        __syncthreads();
      }
    }
  });
}

}  // namespace dnsk
