// adi_seg.hpp - device building blocks of the segmented ADI sweeps (grids up
// to 256): every element of a line in registers from its load to its store.
//
// A line of G points is cut into 16 segments of K = seg_len(G) elements, one
// segment per thread.  The system has one coefficient, so both Thomas
// recurrences need only cbet (q = i cs times a value is a swap and two
// products):
//   forward   y_k = cbet_k (r_k + i cs y_(k-1)),
//   backward  u_k = y_k + i cs cbet_k u_(k+1).
// Either one passes the value entering a segment on to the segment's end
// times the product P = prod (i cs cbet_k) over the segment, |P| < 1.  So
// each direction runs twice over the registers: once with nothing entering,
// whose end values give what enters every segment (from the H segments
// before it: the host's H makes the product over H segments smaller than
// 1e-25, two for the usual step lengths, at most 16), and once with that.
// Recomputing takes the 6 operations per element that a correction by a
// table of products would take, without the table.  A value that is not
// finite does not decay: where a segment's forward run ends with one, all 16
// segments are chained, so that it reaches the whole line as in a single
// recurrence.
//
// Step A's solution gets step B's explicit part at once, while the row's
// neighbours are in registers: the x sweep writes (1 + i cs d2x) u*, the y
// sweep adds the source and solves, and never looks at other columns.
//
// x sweep: 4 rows per wave on 16 lanes each.  The wave loads whole row pieces
// (64 adjacent cells per instruction; the rows above and below give d2y),
// and the right-hand sides go through LDS, wave-locally, into the segment
// layout and back.  One row per lane instead, as the segments lie in memory,
// touched 64 cache lines per instruction.
// y sweep: 16 columns per workgroup, so its loads and stores are row
// segments of 16 cells and thread (t, column) holds rows t K .. t K + K
// without any transpose; the end values cross waves through LDS.
// Floating-point contraction is off in each function body, as in
// adi_lines.hpp, so the single-field and the batch kernels round alike.
// A CU holds three or more workgroups of either, which overlap each other's
// memory latency.  Times: field_adi.hip, where they are launched.
#pragma once

#include "adi_lines.hpp"

#include <type_traits>

namespace g4 {
namespace adi {

constexpr int kSegs = 16;         // segments per line
constexpr int kSegLines = kAdiSegLines;  // lines per workgroup
constexpr int kSegThreads = 256;  // one per segment and line
constexpr int kSegMaxGrid = 256;

// Elements per segment for a grid: the smallest built length that covers it.
__host__ __device__ constexpr int seg_len(int G) {
  return G <= 64 ? 4 : (G <= 112 ? 7 : (G <= 128 ? 8 : (G <= 160 ? 10 : (G <= 208 ? 13 : 16))));
}
// Calls fn with the compile-time segment length of a grid.
template <class Fn>
__host__ __device__ __forceinline__ void with_seg_len(int G, Fn&& fn) {
  switch (seg_len(G)) {
    case 4: fn(std::integral_constant<int, 4>{}); break;
    case 7: fn(std::integral_constant<int, 7>{}); break;
    case 8: fn(std::integral_constant<int, 8>{}); break;
    case 10: fn(std::integral_constant<int, 10>{}); break;
    case 13: fn(std::integral_constant<int, 13>{}); break;
    default: fn(std::integral_constant<int, 16>{}); break;
  }
}

// Device table of a step length: cbet at [j * 16 + t] for element j of
// segment t (zero past the grid), the segment products P at [16 K + t], and
// {H, 0} at [16 K + 16].
__host__ __device__ constexpr int seg_table_size(int K) { return kSegs * K + kSegs + 1; }

// Segment pitch (odd, so the 16 segments of a row and the next row's spread
// over all banks) and row pitch of the x sweep's transpose buffer, scalars.
constexpr int seg_pitch(int K) { return K % 2 ? K : K + 1; }
constexpr int seg_row_pitch(int K) { return kSegs * seg_pitch(K); }
// LDS of a workgroup: the table, then the x sweep's buffer ([16 rows] of
// scalars) or the y sweep's end values ([2][16][16] complex) and sums.
constexpr size_t seg_lds_x(int K) {
  return sizeof(double2) * seg_table_size(K) + sizeof(double) * kSegLines * seg_row_pitch(K);
}
constexpr size_t seg_lds_y(int K) {
  return sizeof(double2) * (seg_table_size(K) + 2 * kSegs * kSegLines) + sizeof(double) * 4 * 8;
}

__device__ __forceinline__ void seg_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// v of the previous (next) lane of a row of 16 lanes; zero where there is none
template <int CTRL>
__device__ __forceinline__ double2 row_dpp(double2 v) {
  int r[4];
  const int* a = reinterpret_cast<const int*>(&v);
#pragma unroll
  for (int k = 0; k < 4; ++k) r[k] = __builtin_amdgcn_update_dpp(0, a[k], CTRL, 0xf, 0xf, true);
  double2 o;
  __builtin_memcpy(&o, r, sizeof(o));
  return o;
}
__device__ __forceinline__ double2 lane_prev(double2 v) { return row_dpp<0x111>(v); }  // row_shr:1
__device__ __forceinline__ double2 lane_next(double2 v) { return row_dpp<0x101>(v); }  // row_shl:1

// cb (r + i cs y)
__device__ __forceinline__ double2 seg_fwd(double2 cb, double2 r, double2 y, double cs) {
#pragma clang fp contract(off)
  const double qx = fma(-cs, y.y, r.x), qy = fma(cs, y.x, r.y);
  return make_double2(fma(cb.x, qx, -(cb.y * qy)), fma(cb.x, qy, cb.y * qx));
}
// y + i cs cb u
__device__ __forceinline__ double2 seg_bwd(double2 cb, double2 y, double2 u, double cs) {
#pragma clang fp contract(off)
  const double zx = -cs * u.y, zy = cs * u.x;
  return make_double2(fma(cb.x, zx, fma(-cb.y, zy, y.x)), fma(cb.x, zy, fma(cb.y, zx, y.y)));
}
__device__ __forceinline__ double2 cfma(double2 a, double2 p, double2 b) {  // a + p b
#pragma clang fp contract(off)
  return make_double2(fma(p.x, b.x, fma(-p.y, b.y, a.x)), fma(p.x, b.y, fma(p.y, b.x, a.y)));
}

// Whether v is not finite (or its components add up to no finite number).
__device__ __forceinline__ bool seg_bad(double2 v) { return !__builtin_isfinite(v.x + v.y); }

// H of the table, as a scalar (the loops over it are uniform).
__device__ __forceinline__ int seg_chain(const double2* tab, int K) {
  return __builtin_amdgcn_readfirstlane(static_cast<int>(tab[kSegs * K + kSegs].x));
}

// x sweep of rows 16 blk .. of one plane.  tab: the step's table in LDS; buf:
// the wave's rows of the transpose buffer.  sp: the slice's source inside rc.
template <class P, int K>
__device__ __forceinline__ void seg_x(const typename A2<P>::T* u, typename A2<P>::T* out, int G,
                                      double cs, const double2* tab,
                                      const typename A2<P>::T* sp, int4 rc, int blk,
                                      double* bufs) {
#pragma clang fp contract(off)
  using T2 = typename A2<P>::T;
  constexpr int E = sizeof(T2);
  constexpr int NI = (kSegs * K + kLane - 1) / kLane;  // row pieces of 64 cells
  constexpr int SP = seg_pitch(K), RP = seg_row_pitch(K);
  const int lane = threadIdx.x & (kLane - 1), wave = threadIdx.x / kLane;
  const int row0 = blk * kSegLines + 4 * wave;
  if (row0 >= G) return;
  const int g = lane / kSegs, t = lane % kSegs;
  double* buf = bufs + 4 * wave * RP;
  const int H = seg_chain(tab, K);
  const Rsrc ru = plane_rsrc(u, G, E);
  const Rsrc ro = plane_rsrc(out, G, E);
  const Rsrc rs = plane_rsrc(sp, G, E);
  // right-hand sides of the four rows, 64 adjacent cells per instruction
  double2 r[4][NI];
  {
    T2 c[6][NI];
#pragma unroll
    for (int q = 0; q < 6; ++q) {
      const int row = row0 - 1 + q;
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const int x = lane + kLane * i;
        c[q][i] = bload<0, T2>(ru, cell_off(row >= 0 && row < G && x < G, row, x, G, E));
      }
    }
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      double2 above = to_d(c[0][i]), cen = to_d(c[1][i]);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const double2 below = to_d(c[q + 2][i]);
        r[q][i] = rhs_of(cen, below, above, cs);
        above = cen;
        cen = below;
      }
    }
  }
  if (sp && row0 < rc.w && row0 + 4 > rc.y) {  // wave-uniform
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int x = lane + kLane * i;
      const bool xin = x >= rc.x && x < rc.z;
      T2 s[4];
#pragma unroll
      for (int q = 0; q < 4; ++q)
        s[q] = bload<0, T2>(rs, cell_off(xin && row0 + q >= rc.y && row0 + q < rc.w, row0 + q, x,
                                         G, E));
#pragma unroll
      for (int q = 0; q < 4; ++q) r[q][i] = zadd(r[q][i], to_d(s[q]));
    }
  }
  // into the segment layout: lane t of row g holds elements t K .. t K + K - 1
  double2 v[K];
  auto at = [&](int q, int x) { return q * RP + x + (x / K) * (SP - K); };
#pragma unroll
  for (int q = 0; q < 4; ++q)
#pragma unroll
    for (int i = 0; i < NI; ++i)
      if (kLane * (i + 1) <= kSegs * K || lane + kLane * i < kSegs * K)
        buf[at(q, lane + kLane * i)] = row0 + q < G ? r[q][i].x : 0.0;
  seg_lds_sync();
#pragma unroll
  for (int j = 0; j < K; ++j) v[j].x = buf[g * RP + t * SP + j];
  seg_lds_sync();
#pragma unroll
  for (int q = 0; q < 4; ++q)
#pragma unroll
    for (int i = 0; i < NI; ++i)
      if (kLane * (i + 1) <= kSegs * K || lane + kLane * i < kSegs * K)
        buf[at(q, lane + kLane * i)] = row0 + q < G ? r[q][i].y : 0.0;
  seg_lds_sync();
#pragma unroll
  for (int j = 0; j < K; ++j) v[j].y = buf[g * RP + t * SP + j];
  seg_lds_sync();
  // forward
  const double2 prod = tab[kSegs * K + t];
  double2 y = make_double2(0.0, 0.0);
#pragma unroll
  for (int j = 0; j < K; ++j) y = seg_fwd(tab[j * kSegs + t], v[j], y, cs);
  const int n = __any(seg_bad(y)) ? kSegs : H;  // segments to chain
  {
    double2 e = y;
    for (int h = 1; h < n; ++h) e = cfma(y, prod, lane_prev(e));
    y = lane_prev(e);
  }
#pragma unroll
  for (int j = 0; j < K; ++j) {
    y = seg_fwd(tab[j * kSegs + t], v[j], y, cs);
    v[j] = y;
  }
  // backward
  double2 w = make_double2(0.0, 0.0);
#pragma unroll
  for (int j = K - 1; j >= 0; --j) w = seg_bwd(tab[j * kSegs + t], v[j], w, cs);
  {
    double2 e = w;
    for (int h = 1; h < n; ++h) e = cfma(w, prod, lane_next(e));
    w = lane_next(e);
  }
  double2 right = w;  // u* of the element after this segment
#pragma unroll
  for (int j = K - 1; j >= 0; --j) {
    w = seg_bwd(tab[j * kSegs + t], v[j], w, cs);
    v[j] = w;
  }
  // the explicit part of step B, (1 + i cs d2x) u*
  {
    double2 left = lane_prev(v[K - 1]);
#pragma unroll
    for (int j = 0; j < K; ++j) {
      const double2 cen = v[j];
      v[j] = rhs_of(cen, j + 1 < K ? v[j + 1 < K ? j + 1 : 0] : right, left, cs);
      left = cen;
    }
  }
  // and back to row pieces
  if constexpr (sizeof(P) == 4) {
    float2* fb = reinterpret_cast<float2*>(buf);
#pragma unroll
    for (int j = 0; j < K; ++j) fb[g * RP + t * SP + j] = from_d<P>(v[j]);
    seg_lds_sync();
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const int x = lane + kLane * i;
        if (row0 + q < G && x < G) bstore<0>(ro, cell_off(true, row0 + q, x, G, E), fb[at(q, x)]);
      }
  } else {
#pragma unroll
    for (int j = 0; j < K; ++j) buf[g * RP + t * SP + j] = v[j].x;
    seg_lds_sync();
    double re[4][NI];
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const int x = lane + kLane * i;
        re[q][i] = x < kSegs * K ? buf[at(q, x)] : 0.0;
      }
    seg_lds_sync();
#pragma unroll
    for (int j = 0; j < K; ++j) buf[g * RP + t * SP + j] = v[j].y;
    seg_lds_sync();
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const int x = lane + kLane * i;
        if (row0 + q < G && x < G)
          bstore<0>(ro, cell_off(true, row0 + q, x, G, E), make_double2(re[q][i], buf[at(q, x)]));
      }
  }
}

// y sweep of columns 16 blk .. of one plane from the x sweep's output `in`;
// every thread of the workgroup takes part.  ends: LDS [2][16][16]; with
// STATS the block's field sums go to part[0..6] and the centre cell to
// centre[0..1] (red: LDS [4][8]).  With CLEAR the source cells this block read
// are then set to zero (the step's last reader of the source clears it for
// the next deposition); as a run-time switch it took registers that K = 16
// does not have (467 -> 542 us on 2048 planes without statistics).
template <class P, int K, bool STATS, bool CLEAR>
__device__ __forceinline__ void seg_y(const typename A2<P>::T* in, typename A2<P>::T* u, int G,
                                      double cs, const double2* tab,
                                      const typename A2<P>::T* sp, int4 rc, int blk,
                                      double2* ends, double* red, double* part, double* centre) {
#pragma clang fp contract(off)
  using T2 = typename A2<P>::T;
  constexpr int E = sizeof(T2);
  const int c = threadIdx.x % kSegLines, t = threadIdx.x / kSegLines;
  const int col = blk * kSegLines + c;
  const int row0 = t * K;
  const int H = seg_chain(tab, K);
  const Rsrc ri = plane_rsrc(in, G, E);
  const Rsrc ro = plane_rsrc(u, G, E);
  const Rsrc rs = plane_rsrc(sp, G, E);
  const bool cin = col < G;
  const bool src = sp && blk * kSegLines < rc.z && (blk + 1) * kSegLines > rc.x;  // uniform
  const bool scol = src && col >= rc.x && col < rc.z;
  double2 v[K];
  {
    T2 a[K];
#pragma unroll
    for (int j = 0; j < K; ++j)
      a[j] = bload<0, T2>(ri, cell_off(cin && row0 + j < G, row0 + j, col, G, E));
    if (src) {
      T2 s[K];
#pragma unroll
      for (int j = 0; j < K; ++j)
        s[j] = bload<0, T2>(rs, cell_off(scol && row0 + j >= rc.y && row0 + j < rc.w, row0 + j,
                                         col, G, E));
#pragma unroll
      for (int j = 0; j < K; ++j) v[j] = zadd(to_d(a[j]), to_d(s[j]));
    } else {
#pragma unroll
      for (int j = 0; j < K; ++j) v[j] = to_d(a[j]);
    }
  }
  // forward
  double2 y = make_double2(0.0, 0.0);
#pragma unroll
  for (int j = 0; j < K; ++j) y = seg_fwd(tab[j * kSegs + t], v[j], y, cs);
  ends[t * kSegLines + c] = y;
  static_assert(kSegThreads / kLane == 4);
  __shared__ int4 bad;
  reinterpret_cast<int*>(&bad)[threadIdx.x / kLane] = __any(seg_bad(y));
  __syncthreads();
  const int4 nf = bad;
  const int chain = __builtin_amdgcn_readfirstlane(nf.x | nf.y | nf.z | nf.w) ? kSegs : H;
  y = make_double2(0.0, 0.0);
  for (int h = chain; h >= 1; --h) {
    const int i = max(t - h, 0);
    const double2 n = cfma(ends[i * kSegLines + c], tab[kSegs * K + i], y);
    y.x = t >= h ? n.x : 0.0;
    y.y = t >= h ? n.y : 0.0;
  }
#pragma unroll
  for (int j = 0; j < K; ++j) {
    y = seg_fwd(tab[j * kSegs + t], v[j], y, cs);
    v[j] = y;
  }
  // backward
  double2 w = make_double2(0.0, 0.0);
#pragma unroll
  for (int j = K - 1; j >= 0; --j) w = seg_bwd(tab[j * kSegs + t], v[j], w, cs);
  double2* back = ends + kSegs * kSegLines;
  back[t * kSegLines + c] = w;
  __syncthreads();
  w = make_double2(0.0, 0.0);
  for (int h = chain; h >= 1; --h) {
    const int i = min(t + h, kSegs - 1);
    const double2 n = cfma(back[i * kSegLines + c], tab[kSegs * K + i], w);
    w.x = t + h < kSegs ? n.x : 0.0;
    w.y = t + h < kSegs ? n.y : 0.0;
  }
  const double shift = -0.5 * static_cast<double>(G - 1);
  const int icenter = (G * G - 1) / 2, crow = icenter / G, ccol = icenter % G;
  double sw = 0.0, s3 = 0.0, s4 = 0.0, s5 = 0.0, s6 = 0.0;
#pragma unroll
  for (int j = K - 1; j >= 0; --j) {
    w = seg_bwd(tab[j * kSegs + t], v[j], w, cs);
    const int row = row0 + j;
    const T2 o = from_d<P>(w);
    bstore<0>(ro, cell_off(cin && row < G, row, col, G, E), o);
    if constexpr (STATS) {  // rows and columns off the grid are zero
      const double re = o.x, im = o.y;
      const double wei = re * re + im * im;
      const double dy = row + shift;
      sw += wei;
      s3 += dy * wei;
      s4 += dy * dy * wei;
      s5 += re;
      s6 += im;
      if (row == crow && col == ccol) {
        centre[0] = re;
        centre[1] = im;
      }
    }
  }
  if (CLEAR && src) {
    T2 z;
    z.x = 0;
    z.y = 0;
#pragma unroll
    for (int j = 0; j < K; ++j)
      bstore<0>(rs, cell_off(scol && row0 + j >= rc.y && row0 + j < rc.w, row0 + j, col, G, E), z);
  }
  if constexpr (STATS) {
    const double dx = col + shift;
    const double acc[7] = {sw, dx * sw, dx * dx * sw, s3, s4, s5, s6};
#pragma unroll
    for (int q = 0; q < 7; ++q) {
      const double a = wave_total(acc[q]);
      if ((threadIdx.x & (kLane - 1)) == 0) red[(threadIdx.x / kLane) * 8 + q] = a;
    }
    __syncthreads();
    if (threadIdx.x < 7) {
      double a = 0.0;
      for (int i = 0; i < kSegThreads / kLane; ++i) a += red[i * 8 + threadIdx.x];
      part[threadIdx.x] = a;
    }
  }
}

}  // namespace adi
}  // namespace g4
