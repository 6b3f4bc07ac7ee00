// field_misc.hip - solver dispatch, slippage plane fill and field sums.
#include "kernels.hpp"

namespace g4 {

void adi_prepare(Field* f, double delz);
void adi_solve(Field* f, bool source_on, bool stats, bool clear);
void fft_prepare(Field* f, double delz);
void fft_solve(Field* f, bool source_on, bool stats, bool clear);

namespace {

constexpr int kStatTiles = 16;  // most tiles per plane of any ADI or standalone sums

// The end of a step: zero fill of the planes that slippage brought in
// (ControlCUDA.cpp:237-244) and, with raw, the field record of every slice
// from the solver's per-tile sums, in one launch.  In logical slice order
// (slice is in ring slot (is + first) % n, DiagnosticCUDA.cpp:320) the new
// planes are the first `front` and the last `back` slices; their records are
// zero.  Blocks below nrec take 32 slices each, 8 lanes per slice (lane k
// adds sum k over the tiles, in tile order; lane 7 copies the centre cell),
// the others zero planes.  ntile 0: stats holds the slices' sums themselves.
// Bound: launch latency.  Flag clear, plane fill, tile sums and slice order
// were four launches of ~4.5 us per step; the tile sums, one thread per
// slice, took 19 us at 4096 slices x 16 tiles and 33 us at 256 x 64.
template <class T2>
__global__ __launch_bounds__(256) void field_finish_kernel(T2* u, int64_t plane, int n, int first,
                                                           int front, int back, int nrec,
                                                           int per_plane, const double* stats,
                                                           int ntile, double* raw) {
  if (static_cast<int>(blockIdx.x) < nrec) {
    const int is = blockIdx.x * 32 + threadIdx.x / 8, k = threadIdx.x % 8;
    if (is >= n) return;
    const int p = (is + first) % n;
    const bool z = is < front || is >= n - back;
    double* o = raw + static_cast<int64_t>(is) * G4H_FIELD_RAW;
    double v = 0.0, c = 0.0;
    if (!z && ntile == 0) {
      v = stats[static_cast<int64_t>(p) * G4H_FIELD_RAW + k];
      if (k == 7) c = stats[static_cast<int64_t>(p) * G4H_FIELD_RAW + 8];
    } else if (!z && k < 7) {
      const double* t = stats + static_cast<int64_t>(p) * ntile * 8 + k;
      for (int i = 0; i < ntile; ++i) v += t[i * 8];
    } else if (!z) {
      const double* t = stats + static_cast<int64_t>(n) * ntile * 8 + 2 * p;
      v = t[0];
      c = t[1];
    }
    o[k] = v;
    if (k == 7) o[8] = c;
    return;
  }
  const int b = blockIdx.x - nrec, i = b / per_plane;
  const int is = i < front ? i : n - back + (i - front);
  T2* q = u + static_cast<int64_t>((is + first) % n) * plane;
  T2 z;
  z.x = 0;
  z.y = 0;
  for (int64_t e = (b % per_plane) * 256 + threadIdx.x; e < plane; e += 256 * per_plane) q[e] = z;
}

// Standalone per-plane field sums (g4_field_slice_reduce_kernel,
// DiagnosticCUDA.cpp:305-363) as per-tile sums in the solvers' layout:
// ntile workgroups per ring slot, whole rows per wave.  Bound: HBM (one
// read).  One workgroup per plane took 50 us for 48 planes of G = 151 FP64.
template <class T2>
__global__ __launch_bounds__(256) void plane_stats_kernel(const T2* u, int n, int G, int ntile,
                                                          double* partials) {
  __shared__ double red[4][8];
  const int p = blockIdx.x / ntile, tile = blockIdx.x % ntile;
  const int64_t plane = static_cast<int64_t>(G) * G;
  const T2* b = u + p * plane;
  const double shift = -0.5 * static_cast<double>(G - 1);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  double acc[7] = {0, 0, 0, 0, 0, 0, 0};
  for (int iy = tile * 4 + wave; iy < G; iy += 4 * ntile) {
    const T2* row = b + static_cast<int64_t>(iy) * G;
    const double dy = iy + shift;
    double rw = 0.0;
    for (int ix = lane; ix < G; ix += 64) {
      const T2 v = ld_stream(&row[ix]);
      const double re = v.x, im = v.y;
      const double wei = re * re + im * im;
      const double dx = ix + shift;
      rw += wei;
      acc[1] += dx * wei;
      acc[2] += dx * dx * wei;
      acc[5] += re;
      acc[6] += im;
    }
    acc[0] += rw;
    acc[3] += dy * rw;
    acc[4] += dy * dy * rw;
  }
#pragma unroll
  for (int k = 0; k < 7; ++k) {
    const double v = wave_total(acc[k]);
    if (lane == 0) red[wave][k] = v;
  }
  __syncthreads();
  if (threadIdx.x < 7) {
    double v = 0.0;
    for (int w = 0; w < 4; ++w) v += red[w][threadIdx.x];
    partials[(static_cast<int64_t>(p) * ntile + tile) * 8 + threadIdx.x] = v;
  }
  if (tile == 0 && threadIdx.x == 0) {
    double* c = partials + static_cast<int64_t>(n) * ntile * 8 + 2 * p;
    const T2 v = b[(plane - 1) / 2];
    c[0] = v.x;
    c[1] = v.y;
  }
}

// Streaming copy, 16 bytes per lane per iteration.
__global__ void copy16_kernel(const float4* __restrict__ src, float4* __restrict__ dst, int64_t n) {
  for (int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; i < n;
       i += static_cast<int64_t>(gridDim.x) * blockDim.x)
    dst[i] = src[i];
}

__global__ void reset_rect_kernel(int4* rect, int4* bbox, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) {
    rect[i] = make_int4(0, 0, 0, 0);
    bbox[i] = make_int4(0x7fffffff, 0x7fffffff, -1, -1);
  }
}

}  // namespace

// ceil(1024 / 64) line blocks of the lane sweeps, ceil(256 / 16) of the
// segmented ones and plane_stats_kernel's limit all come to 16.
void field_stats_reserve(Field* f) {
  const int ntile = f->kind == G4H_SOLVER_FFT ? std::max(kStatTiles, fft_stat_tiles(f)) : kStatTiles;
  const size_t n = static_cast<size_t>(f->nslice);
  const size_t need = n * (static_cast<size_t>(ntile) * 8 + 2);
  if (f->col_partials.size() < need) f->col_partials.alloc(f->ctx, need);
  if (f->kind == G4H_SOLVER_ADI && f->plane_stats.empty())
    f->plane_stats.alloc(f->ctx, n * G4H_FIELD_RAW);
}

double* field_partials(Field* f, int ntile) {
  field_stats_reserve(f);
  f->stats_ntile = ntile;
  return f->col_partials.get();
}

void ensure_source(Field* f) {
  const int64_t cells = f->cells();
  bool fresh = false;
  if (f->prec == G4H_FP64) {
    if (f->srcd.size() != static_cast<size_t>(cells)) {
      f->srcd.alloc(f->ctx, cells);
      G4_HIP(hipMemsetAsync(f->srcd.get(), 0, sizeof(double2) * cells, f->ctx->stream));
      fresh = true;
    }
  } else {
    if (f->srcf.size() != static_cast<size_t>(cells)) {
      f->srcf.alloc(f->ctx, cells);
      G4_HIP(hipMemsetAsync(f->srcf.get(), 0, sizeof(float2) * cells, f->ctx->stream));
      fresh = true;
    }
  }
  if (f->src_rect.size() != static_cast<size_t>(f->nslice)) {
    f->src_rect.alloc(f->ctx, f->nslice);
    f->dep_bbox.alloc(f->ctx, f->nslice);
    fresh = true;
  }
  if (fresh) field_reset_source(f);
}

bool source_needs_prepass(const Field* f, const Beam* b) {
  return !f->src_clear || f->src_epoch != b->epoch;
}

void source_deposited(Field* f, const Beam* b) {
  f->src_clear = false;
  f->src_epoch = b->epoch;
}

void field_reset_source(Field* f) {
  f->src_clear = false;
  f->src_epoch = 0;
  if (f->src_rect.empty()) return;
  f->ctx->launch(G4H_K_OTHER, [&] {
    hipLaunchKernelGGL(reset_rect_kernel, dim3((f->nslice + 255) / 256), dim3(256), 0,
                       f->ctx->stream, f->src_rect.get(), f->dep_bbox.get(), f->nslice);
  });
  // The source planes may hold stale values: clear them once.
  if (f->prec == G4H_FP64 && !f->srcd.empty())
    G4_HIP(hipMemsetAsync(f->srcd.get(), 0, sizeof(double2) * f->srcd.size(), f->ctx->stream));
  if (f->prec == G4H_MIXED && !f->srcf.empty())
    G4_HIP(hipMemsetAsync(f->srcf.get(), 0, sizeof(float2) * f->srcf.size(), f->ctx->stream));
}

void field_prepare_solver(Field* f, double delz) {
  if (f->kind == G4H_SOLVER_FFT)
    fft_prepare(f, delz);
  else
    adi_prepare(f, delz);
  f->solver_ready = true;
}

void field_solve(Field* f, bool source_on, bool stats, bool clear) {
  ensure_source(f);
  if (f->kind == G4H_SOLVER_FFT)
    fft_solve(f, source_on, stats, clear && source_on);
  else
    adi_solve(f, source_on, stats, clear && source_on);
  f->stats_valid = stats;
}

void field_plane_stats(Field* f) {
  // enough workgroups to fill the GPU from few planes, at least 4 rows each
  const int ntile =
      std::max(1, std::min({kStatTiles, (1024 + f->nslice - 1) / f->nslice, (f->ngrid + 3) / 4}));
  double* partials = field_partials(f, ntile);
  const dim3 grid(static_cast<unsigned>(f->nslice) * ntile);
  f->ctx->launch(G4H_K_OTHER, [&] {
    if (f->prec == G4H_FP64)
      hipLaunchKernelGGL(plane_stats_kernel<double2>, grid, dim3(256), 0, f->ctx->stream,
                         f->ud.get(), f->nslice, f->ngrid, ntile, partials);
    else
      hipLaunchKernelGGL(plane_stats_kernel<float2>, grid, dim3(256), 0, f->ctx->stream,
                         f->uf.get(), f->nslice, f->ngrid, ntile, partials);
  });
  f->stats_valid = true;
}

void field_finish(Field* f, const Shifted& z, double* d_raw) {
  require(!d_raw || f->stats_valid, "field statistics requested before they were computed");
  const int n = f->nslice;
  const int front = std::min(z.front, n), back = std::min(z.back, n - front);
  const int nrec = d_raw ? (n + 31) / 32 : 0;
  const int64_t plane = static_cast<int64_t>(f->ngrid) * f->ngrid;
  const int per_plane = static_cast<int>(std::min<int64_t>(256, (plane + 1023) / 1024));
  const int64_t blocks = nrec + static_cast<int64_t>(front + back) * per_plane;
  if (blocks == 0) return;
  const double* stats = f->stats_ntile == 0 ? f->plane_stats.get() : f->col_partials.get();
  f->ctx->launch(G4H_K_OTHER, [&] {
    if (f->prec == G4H_FP64)
      hipLaunchKernelGGL(field_finish_kernel<double2>, dim3(static_cast<unsigned>(blocks)),
                         dim3(256), 0, f->ctx->stream, f->ud.get(), plane, n, f->first, front,
                         back, nrec, per_plane, stats, f->stats_ntile, d_raw);
    else
      hipLaunchKernelGGL(field_finish_kernel<float2>, dim3(static_cast<unsigned>(blocks)),
                         dim3(256), 0, f->ctx->stream, f->uf.get(), plane, n, f->first, front,
                         back, nrec, per_plane, stats, f->stats_ntile, d_raw);
  });
}

void field_copy(Field* dst, const Field* src) {
  const size_t bytes = static_cast<size_t>(src->cells()) * (src->prec == G4H_FP64 ? 16 : 8);
  const int64_t n16 = static_cast<int64_t>(bytes / 16);
  const int blocks = static_cast<int>(std::min<int64_t>(8192, (n16 + 255) / 256));
  dst->ctx->launch(G4H_K_OTHER, [&] {
    hipLaunchKernelGGL(copy16_kernel, dim3(std::max(blocks, 1)), dim3(256), 0, dst->ctx->stream,
                       static_cast<const float4*>(src->data()), static_cast<float4*>(dst->data()),
                       n16);
  });
  dst->first = src->first;
  dst->accuslip = src->accuslip;
  dst->uploaded = true;
}

}  // namespace g4
