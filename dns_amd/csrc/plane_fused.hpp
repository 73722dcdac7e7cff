// Passes B, C and D of one RK stage in one launch, for small grids: a block
// holds one x-plane and runs the inverse y transforms, the fused z pass and
// the forward y transforms of the nonlinear term on it (kernels.hpp), with
// the plane in LDS between them.
//
// Small grids are bound by latency: a pass is a chain of transforms that one
// wave per SIMD at most works on, and each launch adds its start and drain.
// One launch takes the place of three here, and the chain is 9 transforms
// where the passes B, C and D take 6 + 5 + 3: the y transforms of two fields
// run side by side, and so do the forward ones of all three.  n=16 FP64: a
// step takes 80 us with three launches a stage, 55 with one.  The other side of it
// is that a plane has one CU to itself and the rest idle; where the line lies
// is measured at Engine::PLANE.
//
// Fields are taken in pairs (the two halves of one complex z transform): the
// pair's N/2+1 columns each lie side by side in the rows of one LDS plane,
// row j = [X_0 .. X_H | Y_0 .. Y_H], N + 2 <= RS slots, which is also room for
// the row's own z transform.  Threads take column q of the plane (consecutive
// lanes = consecutive kz, as in global memory) for y and row q for z; there
// are C >= N column slots, so the last C - N "rows" have no data: their
// threads transform what lies in spare LDS rows and store nothing.
#pragma once
#include "kernels.hpp"

namespace dnsk {

// #{m >= 0 : m < kmax}, kmax = 2/3 (n/2+1) (main.c:231-238), as dns_api.hip
// counts it.
constexpr int box_count(int n) {
  int m = 0;
  while (m <= n / 2 && (double)m < 2. / 3. * (n / 2 + 1)) m++;
  return m;
}

template <int N, int E> struct Plane {
  static constexpr int TPP = N / E, NF = N / 2 + 1, NK = box_count(N);
  static constexpr int C = 2 * NF > 3 * NK ? 2 * NF : 3 * NK;  // columns (threads: C * TPP)
  static constexpr int RS = C > padlen<N>() ? C : padlen<N>();  // slots per row
  static constexpr int THREADS = C * TPP, SLOTS = C * RS;
};

struct ColumnSlot {
  int q, rs;
  __device__ __forceinline__ int operator()(int pos) const { return pos * rs + q; }
};

// MODE, REC as k_zfused.  Grid (N, 1, members), Plane::THREADS threads.
template <int N, typename R, int MODE, typename UR, int E, bool REC = false>
__global__ __launch_bounds__((Plane<N, E>::THREADS)) void k_plane(cx<R> *__restrict__ W, UR *__restrict__ us, Geo g,
                                                                  R invn3, const cx<R> *__restrict__ tw,
                                                                  double *__restrict__ rec = nullptr) {
  using P = Plane<N, E>;
  constexpr int TPP = P::TPP, NF = P::NF, H = N / 2, NK = P::NK, C = P::C, RS = P::RS;
  __shared__ cx<R> lds[P::SLOTS];
  __shared__ cx<R> twl[tw_size<N, R>()];
  tw = stage_twiddles<N, R>(twl, tw);
  cx<R> *w = W + blockIdx.z * g.mW + blockIdx.x * g.wps;
  // column q of the plane, y positions ty + TPP*c
  const int q = threadIdx.x % C, ty = threadIdx.x / C;
  const bool second = q >= NF, col = q < 2 * NF;
  const int k = second ? q - NF : q;
  const ColumnSlot ycol{q, RS};
  // row `row` of the plane, z positions tz + TPP*c
  const int row = threadIdx.x / TPP, tz = threadIdx.x % TPP;
  const bool live = row < N;
  const PencilSlot<N> zrow{row * RS};
  const long at = ((long)blockIdx.x * N + row) * N + tz;  // physical fields
  us += blockIdx.z * g.mR;

  // column elements of the fields fa (first half) and fb (second; < 0: zero)
  auto load = [&](cx<R>(&v)[E], int fa, int fb) {
    const int f = second ? fb : fa;
    const cx<R> *d = w + f * g.wfs + k;
#pragma unroll
    for (int c = 0; c < E; c++) v[c] = col && f >= 0 ? d[(long)(ty + TPP * c) * g.nfp] : zero<R>();
  };
  // field 2 and omega_x = I (ky w - kz v) of fields 1 and 2 (k_ypass, CURLX)
  auto load_w_ox = [&](cx<R>(&v)[E]) {
    const R kz = (R)k;
#pragma unroll
    for (int c = 0; c < E; c++) {
      const cx<R> *d = w + (long)(ty + TPP * c) * g.nfp + k;
      v[c] = col ? d[2 * g.wfs] : zero<R>();
      if (second && col) {
        const cx<R> vv = d[g.wfs], p = mk<R>(kz * vv.x, kz * vv.y);
        const R ky = (R)wave<N>(ty + TPP * c);
        v[c] = mk<R>(fm(-ky, v[c].y, p.y), fm(ky, v[c].x, -p.x));
      }
    }
  };
  // columns v -> physical rows z (X + I Y)
  auto to_physical = [&](cx<R>(&v)[E], cx<R>(&z)[E]) {
    fft_pencil<N, R, true>(v, ty, lds, ycol, tw);
#pragma unroll
    for (int c = 0; c < E; c++) lds[ycol(ty + TPP * c)] = v[c];
    __syncthreads();
#pragma unroll
    for (int c = 0; c < E; c++) {
      const int pos = tz + TPP * c, m = pos <= H ? pos : N - pos;
      const cx<R> x = lds[row * RS + m], y = lds[row * RS + NF + m];
      if (pos == 0 || pos == H) z[c] = mk<R>(x.x, y.x);
      else if (pos < H) z[c] = mk<R>(x.x - y.y, x.y + y.x);
      else z[c] = mk<R>(x.x + y.y, y.x - x.y);
    }
    __syncthreads();
    fft_pencil<N, R, true>(z, tz, lds, zrow, tw);
  };
  auto record = [&](int f, int c, R a) {
    if constexpr (REC) {
      if (live) rec[f * g.rs + at + TPP * c] = (double)a;
    }
  };

  R u[E], v[E], ww[E], ox[E], nz[E];
  cx<R> f1[E], a[E], z[E];
  if constexpr (MODE == 0) {
    load(a, 3, 4);
#pragma unroll
    for (int c = 0; c < E; c++) {
      u[c] = live ? (R)us[at + TPP * c] : (R)0;
      v[c] = live ? (R)us[g.rs + at + TPP * c] : (R)0;
      ww[c] = live ? (R)us[2 * g.rs + at + TPP * c] : (R)0;
    }
    to_physical(a, z);
    load(a, 5, -1);
    R oy[E];
#pragma unroll
    for (int c = 0; c < E; c++) {
      ox[c] = z[c].x * invn3;
      oy[c] = z[c].y * invn3;
    }
    to_physical(a, z);
#pragma unroll
    for (int c = 0; c < E; c++) z[c] = mk<R>(oy[c], z[c].x * invn3);
  } else {
    load(a, 0, 1);
    to_physical(a, z);
    load_w_ox(a);
#pragma unroll
    for (int c = 0; c < E; c++) {
      u[c] = z[c].x * invn3;
      v[c] = z[c].y * invn3;
    }
    to_physical(a, z);
    load(a, 4, 5);
#pragma unroll
    for (int c = 0; c < E; c++) {
      ww[c] = z[c].x * invn3;
      ox[c] = z[c].y * invn3;
    }
    to_physical(a, z);
#pragma unroll
    for (int c = 0; c < E; c++) {
      z[c] = mk<R>(z[c].x * invn3, z[c].y * invn3);
      if (MODE == 2 && live) {
        us[at + TPP * c] = (UR)u[c];
        us[g.rs + at + TPP * c] = (UR)v[c];
        us[2 * g.rs + at + TPP * c] = (UR)ww[c];
      }
    }
  }
  // u x omega (main.c:374-376)
#pragma unroll
  for (int c = 0; c < E; c++) {
    const R oy = z[c].x, oz = z[c].y;
    record(0, c, u[c]);
    record(1, c, v[c]);
    record(2, c, ww[c]);
    record(3, c, ox[c]);
    record(4, c, oy);
    record(5, c, oz);
    f1[c] = mk<R>(fm(v[c], oz, -(ww[c] * oy)), fm(ww[c], ox[c], -(u[c] * oz)));
    nz[c] = fm(u[c], oy, -(v[c] * ox[c]));
  }
  // r2c along z of (N_x, N_y) and N_z, kz < kmax, into columns [0, NK),
  // [NK, 2 NK) and [2 NK, 3 NK) of the plane
  fft_pencil<N, R, false>(f1, tz, lds, zrow, tw);
#pragma unroll
  for (int c = 0; c < E; c++) lds[zrow(tz + TPP * c)] = f1[c];
  __syncthreads();
  constexpr int EH = E / 2 + 1;  // positions tz + TPP*c < NK have c < EH
  cx<R> nx[EH], ny[EH];
#pragma unroll
  for (int c = 0; c < EH; c++) {
    const int pos = tz + TPP * c;
    if (pos < NK) {
      const cx<R> p = lds[zrow(pos)], m = lds[zrow(pos == 0 ? 0 : N - pos)];
      nx[c] = mk<R>((R)0.5 * (p.x + m.x), (R)0.5 * (p.y - m.y));
      ny[c] = mk<R>((R)0.5 * (p.y + m.y), -((R)0.5 * (p.x - m.x)));
    }
  }
  __syncthreads();
#pragma unroll
  for (int c = 0; c < E; c++) z[c] = mk<R>(nz[c], (R)0);
  fft_pencil<N, R, false>(z, tz, lds, zrow, tw);
#pragma unroll
  for (int c = 0; c < EH; c++) {
    const int pos = tz + TPP * c;
    if (pos < NK) {
      lds[row * RS + pos] = nx[c];
      lds[row * RS + NK + pos] = ny[c];
      lds[row * RS + 2 * NK + pos] = z[c];
    }
  }
  __syncthreads();
  // forward along y; the rows of the box are stored
#pragma unroll
  for (int c = 0; c < E; c++) a[c] = lds[ycol(ty + TPP * c)];
  __syncthreads();
  fft_pencil<N, R, false>(a, ty, lds, ycol, tw);
  if (q < 3 * NK) {
    cx<R> *d = w + (q / NK) * g.wfs + q % NK;
#pragma unroll
    for (int c = 0; c < E; c++)
      if (in_box(ty + TPP * c, N, NK)) d[(long)(ty + TPP * c) * g.nfp] = a[c];
  }
}

}  // namespace dnsk
