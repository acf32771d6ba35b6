// 3D fp64 spreading and interpolation as matrix products, for bins whose tile
// is at most 16 x 16 cells in x and y (plane_tiles()).
//
// The weight of a point is separable, so a plane z of the tile receives
// T_z[y][x] += sum_p (ky[p][y] kz[p][z] c_p) kx[p][x]: one v_mfma_f64_16x16x4
// per component and 4 points, the kernel weights padded to the 16-cell window
// by zeros. Interpolation contracts the same way:
// V[x][p] = sum_z sum_y G_z[y][x] (ky[p][y] kz[p][z]), 4 products per plane,
// component and 16 points, then a dot with kx[p].
// A subproblem's points are ordered by their first kernel plane
// (launch_plane_order), so the points that touch a plane are a range, and the
// planes of a subproblem are finished in order. In spreading each wave keeps two
// planes in registers; no tile is held in LDS, which carries the weights only.
//
// What bounds it: the matrix pipe, 64 clocks per product and SIMD; a point
// costs 2 ns / 4 products to spread, 2 ns 4 / 16 to interpolate: 72 clocks per
// CU at ns = 9. Counters at ns = 9: matrix pipe 50 % busy (both directions)
// beside the vector instructions that share the fp64 units; polynomial weights
// (es_device.hpp) instead of exp and sqrt took spreading from 303 to 272 us.
// The LDS-atomic kernels of spread_interp.hip pay 1458 64-bit atomics and 12
// conversion instructions per cell there. Measured, before -> after:
// spreading 1e6 points, 192 x 150 x 160 cells, ns = 9: 894 -> 272 us (the
// rounding of the sums is that of fp64 FMAs); 2e6 points, 262 x 262 x 72 cells,
// ns = 7: 775 -> 508 us. Interpolation, LDS kernel -> planes, 128^3 cells: ns = 9,
// 0.02 / 0.2 / 2 points per cell 218 / 223 / 1038 -> 42 / 133 / 872 us; ns = 12
// 940 / 960 / 2594 -> 92 / 168 / 1156 us; ns = 7 86 / 111 / 600 -> 29 / 101 / 717 us.
//
// Semantics as spread_interp.hip (reference
// src/neonufft/gpu/kernels/spreading_kernel.cu:588-660,
// interpolation_kernel.cu:193-319).
#include <algorithm>
#include <cfloat>

#include "es_device.hpp"

namespace nnf {

namespace {

using d4 = double __attribute__((ext_vector_type(4)));

constexpr int kPlaneThreads = 512;
constexpr int kPlaneWaves = kPlaneThreads / 64;
constexpr int kPlaneChunk = 128;  // points whose weights are in LDS at a time
constexpr int kPitch = 17;        // weights of one point and axis: 16, odd pitch
// readers step 16 points from any start: room past the chunk's end
constexpr int kPlaneRows = kPlaneChunk + 16;

__device__ inline int first_plane(uint32_t cell) { return unpack_cell<3>(cell, 2); }

// Kernel weights of a chunk of points. kx and ky are dense over the tile's 16
// cells; kz[p][z & 15] holds the NS planes of point p only, times the point's
// strength, the other entries are stale. zs[z] = points of the
// chunk that start below plane z; planes below zlast receive nothing from
// later chunks.
struct PlaneWeights {
  double kx[kPlaneRows * kPitch], ky[kPlaneRows * kPitch];
  Cplx<double> kz[kPlaneRows * kPitch];
  int zs[kMaxTilePlanes + 1];
  int zlast;
};

// One lane's point of a chunk, loaded ahead of its use: a wave holds 64 points,
// even waves the first half of the chunk, odd waves the second. (Separate
// variables: the choice between members of a struct goes through scratch.)
__device__ inline uint32_t chunk_point(const Subprob& sp, uint32_t base, int wave, int lane) {
  const uint32_t i = base + static_cast<uint32_t>((wave & 1) * 64 + lane);
  return sp.begin + min(i, sp.count - 1);
}

// before = cell of the point before p
__device__ inline void load_point(const PointRec<double, 3>* __restrict__ pts, uint32_t p,
                                  uint32_t begin, double& x, double& y, double& z, uint32_t& cell,
                                  uint32_t& before) {
  const PointRec<double, 3> r = pts[p];
  x = r.x[0];
  y = r.x[1];
  z = r.x[2];
  cell = r.cell;
  before = pts[max(p, begin + 1) - 1].cell;
}

// Fills the weights of a chunk of `cnt` points of strengths c. Wave = weights, lane = point, so every wave runs uniformly; the
// cells of kx and ky outside the kernel's window get their zeros.
template <int NS>
__device__ __forceinline__ void fill_weights(PlaneWeights& s, double px, double py, double pz,
                                             const Cplx<double>& c, uint32_t cell, uint32_t before,
                                             int cnt, int planes, int wave, int lane,
                                             const EsParams& es) {
  const int p = (wave & 1) * 64 + lane;
  const int r0 = unpack_cell<3>(cell, 0), r1 = unpack_cell<3>(cell, 1);
  const int r2 = first_plane(cell);
  // (axis, pair of pieces), the pairs of end pieces first: they cost the most
  for (int i = wave >> 1; i < 3 * ((NS + 1) / 2); i += kPlaneWaves / 2) {
    const int j = i / 3, d = i - 3 * j, j2 = NS - 1 - j;
    double lo, hi;
    es_pair<NS>(d == 0 ? px : (d == 1 ? py : pz), j, es, lo, hi);
    if (d == 0) {
      s.kx[p * kPitch + r0 + j] = lo;
      s.kx[p * kPitch + r0 + j2] = hi;
    } else if (d == 1) {
      s.ky[p * kPitch + r1 + j] = lo;
      s.ky[p * kPitch + r1 + j2] = hi;
    } else {
      s.kz[p * kPitch + ((r2 + j) & 15)] = Cplx<double>{lo * c.x, lo * c.y};
      s.kz[p * kPitch + ((r2 + j2) & 15)] = Cplx<double>{hi * c.x, hi * c.y};
    }
  }
  for (int i = wave >> 1; i < 2 * (16 - NS); i += kPlaneWaves / 2) {
    const int j = i >> 1;
    if (i & 1) {
      s.ky[p * kPitch + ((r1 + NS + j) & 15)] = 0.0;
    } else {
      s.kx[p * kPitch + ((r0 + NS + j) & 15)] = 0.0;
    }
  }
  if (wave < 2 && p < cnt) {
    for (int z = p == 0 ? 0 : first_plane(before) + 1; z <= r2; ++z) s.zs[z] = p;
    if (p == cnt - 1) {
      s.zlast = r2;
      for (int z = r2 + 1; z <= planes; ++z) s.zs[z] = cnt;
    }
  }
}

// Wave w owns the planes z = w (mod 8), two at a time: a point touches at most
// 12 consecutive planes, so at most two of a wave's planes are unfinished.
template <int NS>
__device__ __forceinline__ void plane_spread(const SpreadJob<double, 3>& job, const Subprob& sp,
                                             uint32_t sidx, const EsParams& es) {
  __shared__ PlaneWeights s;
  const BinGeom& g = job.g;
  const int t0 = g.tile[0], t1 = g.tile[1], t2 = g.tile[2];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int li = lane & 15, lk = lane >> 4;
  Cplx<double>* __restrict__ dst =
      job.tiles + static_cast<std::size_t>(sidx - job.sub_off) * tile_cells(g);

  d4 re[2] = {}, im[2] = {};
  int plane[2] = {wave, wave + kPlaneWaves};
  auto load_strength = [&](uint32_t p) {
    Cplx<double> c = job.in[job.perm ? job.perm[p] : p];
    if (job.pre) {
      const Cplx<double> q = job.pre[p];
      c = Cplx<double>{c.x * q.x - c.y * q.y, c.x * q.y + c.y * q.x};
    }
    return c;
  };
  uint32_t p = chunk_point(sp, 0, wave, lane);
  double px, py, pz;
  uint32_t cell, before;
  load_point(job.pts, p, sp.begin, px, py, pz, cell, before);
  Cplx<double> c = load_strength(p);
  for (uint32_t base = 0; base < sp.count; base += kPlaneChunk) {
    const int cnt = static_cast<int>(min(static_cast<uint32_t>(kPlaneChunk), sp.count - base));
    fill_weights<NS>(s, px, py, pz, c, cell, before, cnt, g.bin[2], wave, lane, es);
    __syncthreads();
    const bool last = base + kPlaneChunk >= sp.count;
    if (!last) {
      p = chunk_point(sp, base + kPlaneChunk, wave, lane);
      load_point(job.pts, p, sp.begin, px, py, pz, cell, before);
      c = load_strength(p);
    }
    const int zlast = __builtin_amdgcn_readfirstlane(s.zlast);
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      while (plane[k] < t2) {
        const int z = plane[k];
        const int lo = __builtin_amdgcn_readfirstlane(s.zs[max(z - NS + 1, 0)]);
        const int hi = __builtin_amdgcn_readfirstlane(s.zs[min(z + 1, g.bin[2])]);
        const double* kx = s.kx + (lo + lk) * kPitch + li;
        const double* ky = s.ky + (lo + lk) * kPitch + li;
        const Cplx<double>* kz = s.kz + (lo + lk) * kPitch + (z & 15);
        int n = hi - lo;
        // each step's weights are read one step ahead
        Cplx<double> wz = *kz;
        double wy = *ky, wx = *kx;
        for (; n >= 4; n -= 4) {
          const double a = wy * wz.x, b = wy * wz.y, x = wx;
          kx += 4 * kPitch;
          ky += 4 * kPitch;
          kz += 4 * kPitch;
          wz = *kz;
          wy = *ky;
          wx = *kx;
          re[k] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, x, re[k], 0, 0, 0);
          im[k] = __builtin_amdgcn_mfma_f64_16x16x4f64(b, x, im[k], 0, 0, 0);
        }
        if (n > 0) {
          const bool in = lk < n;
          wx = in ? wx : 0.0;
          const double a = in ? wy * wz.x : 0.0, b = in ? wy * wz.y : 0.0;
          re[k] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, wx, re[k], 0, 0, 0);
          im[k] = __builtin_amdgcn_mfma_f64_16x16x4f64(b, wx, im[k], 0, 0, 0);
        }
        if (!last && z >= zlast) break;
        // final: lane holds cells (x = li, y = 4 i + lk)
        if (li < t0) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int y = 4 * i + lk;
            if (y < t1) dst[(z * t1 + y) * t0 + li] = Cplx<double>{re[k][i], im[k][i]};
          }
        }
        re[k] = d4{0.0, 0.0, 0.0, 0.0};
        im[k] = d4{0.0, 0.0, 0.0, 0.0};
        plane[k] = z + 2 * kPlaneWaves;
      }
    }
    __syncthreads();
  }
}

template <int NS>
__global__ void __launch_bounds__(kPlaneThreads, 4)
    plane_spread_kernel(SpreadJob<double, 3> job, const Subprob* __restrict__ subs, uint32_t nsub,
                        EsParams es) {
  const uint32_t sidx = xcd_remap(blockIdx.x, nsub);
  plane_spread<NS>(job, subs[sidx], sidx, es);
}

template <int NS>
__global__ void __launch_bounds__(kPlaneThreads, 4)
    plane_spread_batch_kernel(const SpreadJob<double, 3>* __restrict__ jobs,
                              const Subprob* __restrict__ subs, uint32_t nsub, EsParams es) {
  const uint32_t sidx = xcd_remap(blockIdx.x, nsub);
  const Subprob sp = subs[sidx];
  const SpreadJob<double, 3> job = jobs[sp.job];
  plane_spread<NS>(job, sp, sidx, es);
}

// Interpolation. A wave takes 16 points in plane order and sums over all the
// planes they touch in the accumulators, so that the dot with kx and the sums
// across lanes are paid once per 16 points, and waves depend on no other wave.
// The planes come from the caches: neighbouring waves take neighbouring
// points, hence the same planes.
constexpr int kInterpWaves = 4;
constexpr int kInterpThreads = 64 * kInterpWaves;
constexpr int kInterpTake = 32;  // points whose weights a wave holds at a time

template <int NS>
__device__ __forceinline__ void plane_interp(const InterpJob<double, 3>& job, const Subprob& sp,
                                             const EsParams& es) {
  constexpr int kP = NS | 1;  // weights of one point and axis, odd pitch
  __shared__ double weights[kInterpWaves][3][kInterpTake * kP];
  const BinGeom& g = job.g;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int li = lane & 15, lk = lane >> 4;
  double* kx = weights[wave][0];
  double* ky = weights[wave][1];
  double* kz = weights[wave][2];

  int org[3], ext[3];
  {
    uint32_t bin = sp.bin;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const int o = static_cast<int>(bin % static_cast<uint32_t>(g.nbins[d])) * g.bin[d];
      bin /= static_cast<uint32_t>(g.nbins[d]);
      org[d] = o - NS / 2;
      ext[d] = min(g.bin[d], g.n[d] - o) + NS - 1;
    }
  }
  // Lane holds cells (x = li, y = 4 q + lk) of a plane. Cells past the bin's
  // extent repeat its edge: their weights are zero.
  const int gx = wrap_once(org[0] + min(li, ext[0] - 1), g.n[0]);
  std::size_t row[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int gy = wrap_once(org[1] + min(4 * q + lk, ext[1] - 1), g.n[1]);
    row[q] = static_cast<std::size_t>(gx) +
             static_cast<std::size_t>(g.n[0]) * static_cast<std::size_t>(gy);
  }
  const std::size_t area = static_cast<std::size_t>(g.n[0]) * static_cast<std::size_t>(g.n[1]);
  auto plane_at = [&](int z) {
    return job.grid + area * static_cast<std::size_t>(wrap_once(org[2] + z, g.n[2]));
  };

  // 16 or 32 points per wave and round, so that few points use every wave
  const uint32_t take = sp.count > 16 * kInterpWaves ? kInterpTake : 16;
  for (uint32_t base = wave * take; base < sp.count; base += kInterpWaves * take) {
    const int cnt = static_cast<int>(min(take, sp.count - base));
    // two lanes per point: one forms the weights of x, one those of y, both z
    const int own = lane & (kInterpTake - 1);
    const uint32_t mine = sp.begin + base + static_cast<uint32_t>(min(own, cnt - 1));
    const PointRec<double, 3> rec = job.pts[mine];
    const uint32_t to = job.perm[mine];
    const bool second = lane >= kInterpTake;
    const double x = second ? rec.x[1] : rec.x[0];
    double* w = (second ? ky : kx) + own * kP;
#pragma unroll 1
    for (int j = 0; j < (NS + 1) / 2; ++j) es_pair<NS>(x, j, es, w[j], w[NS - 1 - j]);
    w = kz + own * kP;
    const int end = second ? NS - 1 : 0;  // z: an end piece each
    w[end] = es_exact<NS>(rec.x[2], end, es);
#pragma unroll 1
    for (int j = 1; j < (NS + 1) / 2; ++j) es_pair<NS>(rec.x[2], j, es, w[j], w[NS - 1 - j]);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();

    for (int first = 0; first < cnt; first += 16) {
      const int i = first + li;  // this lane's point
      const bool in = i < cnt;
      const uint32_t cell = __shfl(rec.cell, i, 64);
      const int r0 = unpack_cell<3>(cell, 0), r1 = unpack_cell<3>(cell, 1);
      const int r2 = first_plane(cell);
      const int zbeg = __builtin_amdgcn_readlane(r2, 0);
      const int zend = __builtin_amdgcn_readlane(r2, min(15, cnt - 1 - first)) + NS;
      double wy[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int j = 4 * q + lk - r1;
        const double w = ky[i * kP + min(max(j, 0), NS - 1)];
        wy[q] = in && j >= 0 && j < NS ? w : 0.0;
      }
      d4 re = {}, im = {};
      // a plane's cells are loaded behind the products of the plane before
      Cplx<double> even[4], odd[4];
      auto load = [&](int z, Cplx<double> (&v)[4]) __attribute__((always_inline)) {
        const Cplx<double>* src = plane_at(z);
#pragma unroll
        for (int q = 0; q < 4; ++q) v[q] = src[row[q]];
      };
      auto add = [&](int z, const Cplx<double> (&v)[4]) __attribute__((always_inline)) {
        const int j = z - r2;
        double wz = kz[i * kP + min(max(j, 0), NS - 1)];
        wz = j >= 0 && j < NS ? wz : 0.0;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const double w = wy[q] * wz;
          re = __builtin_amdgcn_mfma_f64_16x16x4f64(v[q].x, w, re, 0, 0, 0);
          im = __builtin_amdgcn_mfma_f64_16x16x4f64(v[q].y, w, im, 0, 0, 0);
        }
      };
      load(zbeg, even);
      for (int z = zbeg; z < zend; z += 2) {
        if (z + 1 < zend) load(z + 1, odd);
        add(z, even);
        if (z + 1 >= zend) break;
        if (z + 2 < zend) load(z + 2, even);
        add(z + 1, odd);
      }
      // lane holds cells x = 4 q + lk of its point: dot with kx, over lk
      double sr = 0.0, si = 0.0;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int j = 4 * q + lk - r0;
        double w = kx[i * kP + min(max(j, 0), NS - 1)];
        w = j >= 0 && j < NS ? w : 0.0;
        sr = fma(w, re[q], sr);
        si = fma(w, im[q], si);
      }
      if (__any(!(fabs(sr) + fabs(si) <= DBL_MAX))) {
        // An infinity or NaN in a cell times a zero weight is NaN for all 16
        // points: each reads its own cells instead, lane lk the rows lk, lk + 4, ..
        sr = si = 0.0;
        for (int c = 0; in && c < NS; ++c) {
          const Cplx<double>* src = plane_at(r2 + c);
          for (int b = lk; b < NS; b += 4) {
            const std::size_t line = static_cast<std::size_t>(g.n[0]) *
                                     static_cast<std::size_t>(wrap_once(org[1] + r1 + b, g.n[1]));
            double tr = 0.0, ti = 0.0;
            for (int a = 0; a < NS; ++a) {
              const Cplx<double> v = src[line + wrap_once(org[0] + r0 + a, g.n[0])];
              tr = fma(kx[i * kP + a], v.x, tr);
              ti = fma(kx[i * kP + a], v.y, ti);
            }
            const double w = ky[i * kP + b] * kz[i * kP + c];
            sr = fma(w, tr, sr);
            si = fma(w, ti, si);
          }
        }
      }
      sr += __shfl_xor(sr, 16, 64);
      si += __shfl_xor(si, 16, 64);
      sr += __shfl_xor(sr, 32, 64);
      si += __shfl_xor(si, 32, 64);
      const uint32_t dst = __shfl(to, i, 64);
      if (lk == 0 && in) {
        if (job.post) {
          const Cplx<double> q = job.post[sp.begin + base + static_cast<uint32_t>(i)];
          const double tr = sr * q.x - si * q.y;
          si = sr * q.y + si * q.x;
          sr = tr;
        }
        job.out[dst] = Cplx<double>{sr, si};
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
}

// Part `part` of a subproblem: near-equal runs of whole 16-point groups, at least
// one group per wave; parts past the last point are empty. The launch takes all
// first parts, then all second ones: empty parts between full ones leave every
// other CU idle (128^3 cells, ns = 9, 0.02 points per cell: 66 us against 42).
__device__ inline bool split_subproblem(Subprob& sp, uint32_t part, uint32_t split) {
  const uint32_t run = max(16u * kInterpWaves, ((sp.count + split - 1) / split + 15u) & ~15u);
  if (part * run >= sp.count) return false;
  sp.begin += part * run;
  sp.count = min(run, sp.count - part * run);
  return true;
}

template <int NS>
__global__ void __launch_bounds__(kInterpThreads, 4)
    plane_interp_kernel(InterpJob<double, 3> job, const Subprob* __restrict__ subs, uint32_t nsub,
                        uint32_t split, EsParams es) {
  Subprob sp = subs[xcd_remap(blockIdx.x % nsub, nsub)];
  if (split_subproblem(sp, blockIdx.x / nsub, split)) plane_interp<NS>(job, sp, es);
}

template <int NS>
__global__ void __launch_bounds__(kInterpThreads, 4)
    plane_interp_batch_kernel(const InterpJob<double, 3>* __restrict__ jobs,
                              const Subprob* __restrict__ subs, uint32_t nsub, uint32_t split,
                              EsParams es) {
  Subprob sp = subs[xcd_remap(blockIdx.x % nsub, nsub)];
  if (!split_subproblem(sp, blockIdx.x / nsub, split)) return;
  const InterpJob<double, 3> job = jobs[sp.job];
  plane_interp<NS>(job, sp, es);
}

// Parts per subproblem: about 2048 workgroups of four waves fill the chip
// (four on a CU) twice. 64^3 cells at 0.5 points per cell, ns = 9 (192
// subproblems): 76 us in one part each, 50 in eight.
uint32_t interp_split(std::size_t nsub) {
  return static_cast<uint32_t>(std::min<std::size_t>(8, (2048 + nsub - 1) / nsub));
}

constexpr int kOrderThreads = 1024;
constexpr int kOrderPerThread = static_cast<int>(kMaxSubproblemPoints) / kOrderThreads;

// Counting sort of each subproblem's points by first kernel plane.
__global__ void __launch_bounds__(kOrderThreads)
    plane_order_kernel(const Subprob* __restrict__ subs, PointRec<double, 3>* __restrict__ pts,
                       uint32_t* __restrict__ perm) {
  __shared__ uint32_t cnt[kMaxTilePlanes];
  if (threadIdx.x < kMaxTilePlanes) cnt[threadIdx.x] = 0;
  __syncthreads();
  const Subprob sp = subs[blockIdx.x];
  PointRec<double, 3> rec[kOrderPerThread];
  uint32_t idx[kOrderPerThread], rank[kOrderPerThread];
#pragma unroll
  for (int k = 0; k < kOrderPerThread; ++k) {
    const uint32_t i = threadIdx.x + k * kOrderThreads;
    if (i < sp.count) {
      rec[k] = pts[sp.begin + i];
      idx[k] = perm[sp.begin + i];
      rank[k] = atomicAdd(&cnt[first_plane(rec[k].cell)], 1u);
    }
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < kOrderPerThread; ++k) {
    const uint32_t i = threadIdx.x + k * kOrderThreads;
    if (i < sp.count) {
      uint32_t pos = rank[k];
      for (int z = first_plane(rec[k].cell) - 1; z >= 0; --z) pos += cnt[z];
      pts[sp.begin + pos] = rec[k];
      perm[sp.begin + pos] = idx[k];
    }
  }
}

template <int NS>
void spread_ns(const SpreadJob<double, 3>& job, const Subprob* subs, std::size_t nsub,
               const EsParams& es, hipStream_t stream) {
  hipLaunchKernelGGL((plane_spread_kernel<NS>), dim3(static_cast<unsigned>(nsub)),
                     dim3(kPlaneThreads), 0, stream, job, subs, static_cast<uint32_t>(nsub), es);
  check_launch("plane_spread_kernel");
}

template <int NS>
void spread_batch_ns(const SpreadJob<double, 3>* jobs, const Subprob* subs, std::size_t nsub,
                     const EsParams& es, hipStream_t stream) {
  hipLaunchKernelGGL((plane_spread_batch_kernel<NS>), dim3(static_cast<unsigned>(nsub)),
                     dim3(kPlaneThreads), 0, stream, jobs, subs, static_cast<uint32_t>(nsub), es);
  check_launch("plane_spread_batch_kernel");
}

template <int NS>
void interp_ns(const InterpJob<double, 3>& job, const Subprob* subs, std::size_t nsub,
               const EsParams& es, hipStream_t stream) {
  const uint32_t split = interp_split(nsub);
  hipLaunchKernelGGL((plane_interp_kernel<NS>), dim3(static_cast<unsigned>(nsub) * split),
                     dim3(kInterpThreads), 0, stream, job, subs,
                     static_cast<uint32_t>(nsub), split, es);
  check_launch("plane_interp_kernel");
}

template <int NS>
void interp_batch_ns(const InterpJob<double, 3>* jobs, const Subprob* subs, std::size_t nsub,
                     const EsParams& es, hipStream_t stream) {
  const uint32_t split = interp_split(nsub);
  hipLaunchKernelGGL((plane_interp_batch_kernel<NS>), dim3(static_cast<unsigned>(nsub) * split),
                     dim3(kInterpThreads), 0, stream, jobs, subs,
                     static_cast<uint32_t>(nsub), split, es);
  check_launch("plane_interp_batch_kernel");
}

}  // namespace

#define NNF_PLANE_CASES(FN, ...)                                       \
  switch (ns) {                                                        \
    case 7: FN<7>(__VA_ARGS__); break;                                 \
    case 8: FN<8>(__VA_ARGS__); break;                                 \
    case 9: FN<9>(__VA_ARGS__); break;                                 \
    case 10: FN<10>(__VA_ARGS__); break;                               \
    case 11: FN<11>(__VA_ARGS__); break;                               \
    case 12: FN<12>(__VA_ARGS__); break;                               \
    default: throw neonufft::InternalError("n_spread not in [7, 12]"); \
  }

void launch_plane_spread(int ns, const SpreadJob<double, 3>& job, const Subprob* subs,
                         std::size_t nsub, const EsParams& es, hipStream_t stream) {
  if (nsub == 0) return;
  NNF_PLANE_CASES(spread_ns, job, subs, nsub, es, stream)
}

void launch_plane_spread_batch(int ns, const SpreadJob<double, 3>* jobs, const Subprob* subs,
                               std::size_t nsub, const EsParams& es, hipStream_t stream) {
  if (nsub == 0) return;
  NNF_PLANE_CASES(spread_batch_ns, jobs, subs, nsub, es, stream)
}

void launch_plane_interp(int ns, const InterpJob<double, 3>& job, const Subprob* subs,
                         std::size_t nsub, const EsParams& es, hipStream_t stream) {
  if (nsub == 0) return;
  NNF_PLANE_CASES(interp_ns, job, subs, nsub, es, stream)
}

void launch_plane_interp_batch(int ns, const InterpJob<double, 3>* jobs, const Subprob* subs,
                               std::size_t nsub, const EsParams& es, hipStream_t stream) {
  if (nsub == 0) return;
  NNF_PLANE_CASES(interp_batch_ns, jobs, subs, nsub, es, stream)
}

void launch_plane_order(const Subprob* subs, std::size_t nsub, PointRec<double, 3>* pts,
                        uint32_t* perm, hipStream_t stream) {
  if (nsub == 0) return;
  hipLaunchKernelGGL(plane_order_kernel, dim3(static_cast<unsigned>(nsub)), dim3(kOrderThreads), 0,
                     stream, subs, pts, perm);
  check_launch("plane_order_kernel");
}

}  // namespace nnf
