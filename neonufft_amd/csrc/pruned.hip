// Kernels of the pruned multi-dimensional FFT used by type 1 / type 2 plans
// in 2D and 3D.
//
// Type 1 keeps only N_d of the n_d frequencies per axis after the FFT, type 2
// starts from N_d nonzero entries per axis. Transforming one axis at a time
// with contiguous 1D rocFFT passes, and moving the next axis to the front with
// an LDS-tiled transpose that keeps only the retained entries (or expands
// them back with zeros), does a fraction of the full transform's work:
// 3D: x on n^3, y on n^2 N, z on n N^2 values; the reference instead runs the
// full in-place transform (src/neonufft/gpu/util/fft_grid.cpp:59-70) and then
// downsamples.
//
// Retained index j in [0, N) of an axis with n fine cells: fine index
// j < P ? j : j + n - N, mode k = j < P ? j : j - N, with P = N - N/2
// (mode_index.hpp).
#include <type_traits>

#include "kernels.hpp"
#include "mode_index.hpp"

namespace nnf {

namespace {

constexpr int kTile = 32;   // transpose tile edge
constexpr int kRowsPer = 8; // tile rows handled per pass by a 32 x 8 block

inline unsigned cap_slabs(std::size_t s) {
  return static_cast<unsigned>(s < 65535 ? (s ? s : 1) : 65535);
}

}  // namespace

// ---------------------------------------------------------------------------
// dst[s][c][r] = src[s][r][ret_fine(c)], r < R, c < Nc (retained of nc).
// Slab s = (hi, lo) with lo < lo_count; offsets hi * *_hi + lo * *_lo.
// ---------------------------------------------------------------------------
template <typename T>
__global__ void __launch_bounds__(kTile* kRowsPer)
    compact_transpose_kernel(const Cplx<T>* __restrict__ src, Cplx<T>* __restrict__ dst, int R,
                             int nc, int Nc, long long src_rs, long long dst_rs, int slabs,
                             int lo_count, long long src_hi, long long src_lo, long long dst_hi,
                             long long dst_lo) {
  __shared__ Cplx<T> tile[kTile][kTile + 1];
  const int c0 = blockIdx.x * kTile, r0 = blockIdx.y * kTile;
  for (int s = blockIdx.z; s < slabs; s += gridDim.z) {
    const long long sb = (s / lo_count) * src_hi + (s % lo_count) * src_lo;
    const long long db = (s / lo_count) * dst_hi + (s % lo_count) * dst_lo;
    const int c = c0 + threadIdx.x;
#pragma unroll
    for (int k = 0; k < kTile; k += kRowsPer) {
      const int r = r0 + threadIdx.y + k;
      if (r < R && c < Nc) tile[threadIdx.y + k][threadIdx.x] = src[sb + r * src_rs + ret_fine(c, nc, Nc)];
    }
    __syncthreads();
    const int r = r0 + threadIdx.x;
#pragma unroll
    for (int k = 0; k < kTile; k += kRowsPer) {
      const int cc = c0 + threadIdx.y + k;
      if (r < R && cc < Nc) dst[db + cc * dst_rs + r] = tile[threadIdx.x][threadIdx.y + k];
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// dst[s][r][f] = src[s][fine_ret(f)][r] for retained fine cells f < nf, else 0.
// ---------------------------------------------------------------------------
template <typename T>
__global__ void __launch_bounds__(kTile* kRowsPer)
    expand_transpose_kernel(const Cplx<T>* __restrict__ src, Cplx<T>* __restrict__ dst, int R,
                            int nf, int Nf, long long src_rs, long long dst_rs, int slabs,
                            int lo_count, long long src_hi, long long src_lo, long long dst_hi,
                            long long dst_lo) {
  __shared__ Cplx<T> tile[kTile][kTile + 1];
  const int f0 = blockIdx.x * kTile, r0 = blockIdx.y * kTile;
  for (int s = blockIdx.z; s < slabs; s += gridDim.z) {
    const long long sb = (s / lo_count) * src_hi + (s % lo_count) * src_lo;
    const long long db = (s / lo_count) * dst_hi + (s % lo_count) * dst_lo;
    // load src rows (retained index of fine cell f0 + ...) along r
    const int r = r0 + threadIdx.x;
#pragma unroll
    for (int k = 0; k < kTile; k += kRowsPer) {
      const int f = f0 + threadIdx.y + k;
      Cplx<T> v{T(0), T(0)};
      if (f < nf && r < R) {
        const int j = fine_ret(f, nf, Nf);
        if (j >= 0) v = src[sb + j * src_rs + r];
      }
      tile[threadIdx.y + k][threadIdx.x] = v;
    }
    __syncthreads();
    const int f = f0 + threadIdx.x;
#pragma unroll
    for (int k = 0; k < kTile; k += kRowsPer) {
      const int rr = r0 + threadIdx.y + k;
      if (rr < R && f < nf) dst[db + rr * dst_rs + f] = tile[threadIdx.x][threadIdx.y + k];
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// Type-1 output: the last FFT axis L is fastest in src, the x-retained axis
// is the row index. Slab = (member b, middle index m) for 3D (m = retained y),
// (b) for 2D. src[b][m][x'][l]: out_b[i0(x') st0 + i1(m) st1 + i2(l') st2] or,
// in 2D, out_b[i0(x') st0 + i1(l') st1], times the deconvolution factors.
// ---------------------------------------------------------------------------
template <typename T, int DIM>
__global__ void __launch_bounds__(kTile* kRowsPer)
    modes_out_kernel(const Cplx<T>* __restrict__ src, long long member_stride, Cplx<T>* single,
                     Cplx<T>* const* __restrict__ outs, int N0, int Nm, int nl, int Nl,
                     long long st0, long long stm, long long stl, const T* __restrict__ fs0,
                     const T* __restrict__ fsm, const T* __restrict__ fsl, int order_fft,
                     int slabs) {
  __shared__ Cplx<T> tile[kTile][kTile + 1];
  const int l0 = blockIdx.x * kTile, x0 = blockIdx.y * kTile;
  for (int s = blockIdx.z; s < slabs; s += gridDim.z) {
    const int b = DIM == 3 ? s / Nm : s;
    const int m = DIM == 3 ? s % Nm : 0;
    const Cplx<T>* sp = src + b * member_stride + (DIM == 3 ? static_cast<long long>(m) * N0 * nl : 0);
    Cplx<T>* out = outs ? outs[b] : single;
    // load [x'][l'] with l' along threadIdx.x (contiguous in src)
    const int l = l0 + threadIdx.x;
#pragma unroll
    for (int k = 0; k < kTile; k += kRowsPer) {
      const int x = x0 + threadIdx.y + k;
      if (x < N0 && l < Nl) tile[threadIdx.y + k][threadIdx.x] = sp[static_cast<long long>(x) * nl + ret_fine(l, nl, Nl)];
    }
    __syncthreads();
    const int x = x0 + threadIdx.x;
    T fm = T(1);
    long long om = 0;
    if (DIM == 3) {
      const int km = ret_mode(m, Nm);
      fm = fsm[km < 0 ? -km : km];
      om = static_cast<long long>(order_index(km, Nm, order_fft)) * stm;
    }
    if (x < N0) {
      const int kx = ret_mode(x, N0);
      const T fx = fs0[kx < 0 ? -kx : kx] * fm;
      const long long ox = static_cast<long long>(order_index(kx, N0, order_fft)) * st0 + om;
#pragma unroll
      for (int k = 0; k < kTile; k += kRowsPer) {
        const int ll = l0 + threadIdx.y + k;
        if (ll < Nl) {
          const int kl = ret_mode(ll, Nl);
          const T f = fx * fsl[kl < 0 ? -kl : kl];
          const Cplx<T> v = tile[threadIdx.x][threadIdx.y + k];
          out[ox + static_cast<long long>(order_index(kl, Nl, order_fft)) * stl] =
              Cplx<T>{v.x * f, v.y * f};
        }
      }
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// Type-2 input: the reverse of modes_out_kernel, with the last axis expanded
// to all nl fine cells (zeros outside the retained ones):
// dst[b][m][x'][f] = fs * in_b[...] for retained f, else 0.
// ---------------------------------------------------------------------------
template <typename T, int DIM>
__global__ void __launch_bounds__(kTile* kRowsPer)
    modes_in_kernel(const Cplx<T>* single, const Cplx<T>* const* __restrict__ ins,
                    Cplx<T>* __restrict__ dst, long long member_stride, int N0, int Nm, int nl,
                    int Nl, long long st0, long long stm, long long stl,
                    const T* __restrict__ fs0, const T* __restrict__ fsm,
                    const T* __restrict__ fsl, int order_fft, int slabs) {
  __shared__ Cplx<T> tile[kTile][kTile + 1];
  const int f0 = blockIdx.x * kTile, x0 = blockIdx.y * kTile;
  for (int s = blockIdx.z; s < slabs; s += gridDim.z) {
    const int b = DIM == 3 ? s / Nm : s;
    const int m = DIM == 3 ? s % Nm : 0;
    Cplx<T>* dp = dst + b * member_stride + (DIM == 3 ? static_cast<long long>(m) * N0 * nl : 0);
    const Cplx<T>* in = ins ? ins[b] : single;
    T fm = T(1);
    long long om = 0;
    if (DIM == 3) {
      const int km = ret_mode(m, Nm);
      fm = fsm[km < 0 ? -km : km];
      om = static_cast<long long>(order_index(km, Nm, order_fft)) * stm;
    }
    // load along x' (contiguous in the caller's array when st0 = 1)
    const int x = x0 + threadIdx.x;
#pragma unroll
    for (int k = 0; k < kTile; k += kRowsPer) {
      const int f = f0 + threadIdx.y + k;
      Cplx<T> v{T(0), T(0)};
      if (x < N0 && f < nl) {
        const int j = fine_ret(f, nl, Nl);
        if (j >= 0) {
          const int kx = ret_mode(x, N0), kl = ret_mode(j, Nl);
          const T fac = fm * fs0[kx < 0 ? -kx : kx] * fsl[kl < 0 ? -kl : kl];
          const Cplx<T> a = in[static_cast<long long>(order_index(kx, N0, order_fft)) * st0 + om +
                               static_cast<long long>(order_index(kl, Nl, order_fft)) * stl];
          v = Cplx<T>{a.x * fac, a.y * fac};
        }
      }
      tile[threadIdx.y + k][threadIdx.x] = v;
    }
    __syncthreads();
    const int f = f0 + threadIdx.x;
#pragma unroll
    for (int k = 0; k < kTile; k += kRowsPer) {
      const int xx = x0 + threadIdx.y + k;
      if (xx < N0 && f < nl) dp[static_cast<long long>(xx) * nl + f] = tile[threadIdx.x][threadIdx.y + k];
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// Small axes: the transform of an axis as a sum over its cells, joined to the
// step that moves or deconvolves its result, so an axis is one launch instead
// of a library FFT and a transpose. Small transforms are bound by their
// launches (~4 us each): 2000 points, 50 x 40 modes, type 1: 29.2 -> 25.2
// us; 4000 points, 24 x 20 x 16 modes, type 2: 30.9 -> 19.6 us.
// fp32 data; twiddles and sums in fp64, which keeps the error below the
// library FFT's whatever the length.
//
// A workgroup takes 16 lines x 16 / PARTS outputs, each sum in PARTS interleaved
// parts: one where the lines fill the chip (3D, 24 x 20 x 16 modes, type 2: 19.3
// us against 21.2 with four), four where they do not (2D, 50 x 40 modes, type 1:
// 25.9 us against 31.7 with one):
// out(r, o) = sum_i in(r, i) tw[(p0 + i step) mod n], where type 1 sums fine
// cells i for a retained frequency (p0 = 0, step = its fine index) and type 2
// the retained modes in ascending order for fine cell o (p0 = -(N/2) o, step = o).
// ---------------------------------------------------------------------------
constexpr int kDftLines = 16, kDftThreads = 256;

template <bool FORWARD, int PARTS, typename Load, typename Store>
__device__ inline void dft_lines(const double2* __restrict__ twg, int n, int N, int r0, int R,
                                 int o0, Load load, Store store) {
  __shared__ float2 in[kDftMaxLen * (kDftLines + 1)];
  __shared__ double2 tw[kDftMaxLen];
  const int len = FORWARD ? n : N, outs = FORWARD ? N : n;
  const int t = threadIdx.x;
  for (int i = t; i < n; i += kDftThreads) tw[i] = twg[i];
  // type 1 reads lines along their cells, type 2 along the rows
  for (int e = t; e < len * kDftLines; e += kDftThreads) {
    const int r = FORWARD ? e / len : e % kDftLines;
    const int i = FORWARD ? e - r * len : e / kDftLines;
    if (r0 + r < R) {
      const Cplx<float> v = load(r0 + r, i);
      in[i * (kDftLines + 1) + r] = float2{v.x, v.y};
    }
  }
  __syncthreads();
  const int r = t % kDftLines, part = (t / kDftLines) % PARTS;
  const int o = o0 + t / (kDftLines * PARTS);
  if (o >= outs) return;  // with all parts of its sums
  // lanes of rows past the end sum whatever the table holds and drop it
  int step, p;
  if (FORWARD) {
    step = ret_fine(o, n, N);
    p = (part * step) % n;
  } else {
    step = o;
    p = (part * step + n - ((N / 2) * o) % n) % n;
  }
  step = (PARTS * step) % n;
  double re = 0.0, im = 0.0;
#pragma unroll 8
  for (int i = part; i < len; i += PARTS) {
    const float2 v = in[i * (kDftLines + 1) + r];
    const double2 w = tw[p];
    re = fma(static_cast<double>(v.x), w.x, re);
    im = fma(static_cast<double>(v.x), w.y, im);
    re = fma(-static_cast<double>(v.y), w.y, re);
    im = fma(static_cast<double>(v.y), w.x, im);
    p += step;
    p -= p >= n ? n : 0;
  }
#pragma unroll
  for (int off = kDftLines; off < kDftLines * PARTS; off *= 2) {
    re += __shfl_xor(re, off, 64);
    im += __shfl_xor(im, off, 64);
  }
  if (part == 0 && r0 + r < R) {
    store(r0 + r, o, Cplx<float>{static_cast<float>(re), static_cast<float>(im)});
  }
}

// Retained index of the i-th retained mode in ascending order.
__device__ inline int ascending_ret(int i, int N) { return i < N / 2 ? i + N - N / 2 : i - N / 2; }

// compact_transpose_kernel after the FFT of its source lines.
template <int PARTS>
__global__ void __launch_bounds__(kDftThreads)
    dft_keep_kernel(const double2* __restrict__ tw, const Cplx<float>* __restrict__ src,
                    Cplx<float>* __restrict__ dst, int R, int n, int N, long long src_rs,
                    long long dst_rs, int lo_count, long long src_hi, long long src_lo,
                    long long dst_hi, long long dst_lo) {
  const int s = blockIdx.z;
  const Cplx<float>* sp = src + (s / lo_count) * src_hi + (s % lo_count) * src_lo;
  Cplx<float>* dp = dst + (s / lo_count) * dst_hi + (s % lo_count) * dst_lo;
  dft_lines<true, PARTS>(
      tw, n, N, blockIdx.y * kDftLines, R, blockIdx.x * (16 / PARTS),
      [&](int r, int i) { return sp[r * src_rs + i]; },
      [&](int r, int o, const Cplx<float>& v) { dp[o * dst_rs + r] = v; });
}

// expand_transpose_kernel followed by the FFT of its destination lines.
template <int PARTS>
__global__ void __launch_bounds__(kDftThreads)
    dft_expand_kernel(const double2* __restrict__ tw, const Cplx<float>* __restrict__ src,
                      Cplx<float>* __restrict__ dst, int R, int n, int N, long long src_rs,
                      long long dst_rs, int lo_count, long long src_hi, long long src_lo,
                      long long dst_hi, long long dst_lo) {
  const int s = blockIdx.z;
  const Cplx<float>* sp = src + (s / lo_count) * src_hi + (s % lo_count) * src_lo;
  Cplx<float>* dp = dst + (s / lo_count) * dst_hi + (s % lo_count) * dst_lo;
  dft_lines<false, PARTS>(
      tw, n, N, blockIdx.y * kDftLines, R, blockIdx.x * (16 / PARTS),
      [&](int r, int i) { return sp[ascending_ret(i, N) * src_rs + r]; },
      [&](int r, int o, const Cplx<float>& v) { dp[r * dst_rs + o] = v; });
}

// modes_out_kernel after the FFT of its source lines.
template <int DIM, int PARTS>
__global__ void __launch_bounds__(kDftThreads)
    dft_modes_out_kernel(const double2* __restrict__ tw, const Cplx<float>* __restrict__ src,
                         long long member_stride, Cplx<float>* single,
                         Cplx<float>* const* __restrict__ outs, int N0, int Nm, int nl, int Nl,
                         long long st0, long long stm, long long stl,
                         const float* __restrict__ fs0, const float* __restrict__ fsm,
                         const float* __restrict__ fsl, int order_fft) {
  const int s = blockIdx.z;
  const int b = DIM == 3 ? s / Nm : s, m = DIM == 3 ? s % Nm : 0;
  const Cplx<float>* sp =
      src + b * member_stride + (DIM == 3 ? static_cast<long long>(m) * N0 * nl : 0);
  Cplx<float>* out = outs ? outs[b] : single;
  float fm = 1.0f;
  if (DIM == 3) {
    const int km = ret_mode(m, Nm);
    fm = fsm[km < 0 ? -km : km];
    out += static_cast<long long>(order_index(km, Nm, order_fft)) * stm;
  }
  dft_lines<true, PARTS>(
      tw, nl, Nl, blockIdx.y * kDftLines, N0, blockIdx.x * (16 / PARTS),
      [&](int r, int i) { return sp[static_cast<long long>(r) * nl + i]; },
      [&](int r, int o, const Cplx<float>& v) {
        const int kx = ret_mode(r, N0), kl = ret_mode(o, Nl);
        const float f = fs0[kx < 0 ? -kx : kx] * fm * fsl[kl < 0 ? -kl : kl];
        out[static_cast<long long>(order_index(kx, N0, order_fft)) * st0 +
            static_cast<long long>(order_index(kl, Nl, order_fft)) * stl] =
            Cplx<float>{v.x * f, v.y * f};
      });
}

// modes_in_kernel followed by the FFT of its destination lines.
template <int DIM, int PARTS>
__global__ void __launch_bounds__(kDftThreads)
    dft_modes_in_kernel(const double2* __restrict__ tw, const Cplx<float>* single,
                        const Cplx<float>* const* __restrict__ ins, Cplx<float>* __restrict__ dst,
                        long long member_stride, int N0, int Nm, int nl, int Nl, long long st0,
                        long long stm, long long stl, const float* __restrict__ fs0,
                        const float* __restrict__ fsm, const float* __restrict__ fsl,
                        int order_fft) {
  const int s = blockIdx.z;
  const int b = DIM == 3 ? s / Nm : s, m = DIM == 3 ? s % Nm : 0;
  Cplx<float>* dp = dst + b * member_stride + (DIM == 3 ? static_cast<long long>(m) * N0 * nl : 0);
  const Cplx<float>* in = ins ? ins[b] : single;
  float fm = 1.0f;
  if (DIM == 3) {
    const int km = ret_mode(m, Nm);
    fm = fsm[km < 0 ? -km : km];
    in += static_cast<long long>(order_index(km, Nm, order_fft)) * stm;
  }
  dft_lines<false, PARTS>(
      tw, nl, Nl, blockIdx.y * kDftLines, N0, blockIdx.x * (16 / PARTS),
      [&](int r, int i) {
        const int kx = ret_mode(r, N0), kl = i - Nl / 2;
        const float f = fm * fs0[kx < 0 ? -kx : kx] * fsl[kl < 0 ? -kl : kl];
        const Cplx<float> a = in[static_cast<long long>(order_index(kx, N0, order_fft)) * st0 +
                                 static_cast<long long>(order_index(kl, Nl, order_fft)) * stl];
        return Cplx<float>{a.x * f, a.y * f};
      },
      [&](int r, int o, const Cplx<float>& v) { dp[static_cast<long long>(r) * nl + o] = v; });
}

namespace {
// fn(parts, grid) with four parts per sum while whole sums give fewer
// workgroups than there are CUs.
template <typename Fn>
void dft_launch(int rows, int outs, std::size_t slabs, Fn fn) {
  const unsigned groups = static_cast<unsigned>((rows + kDftLines - 1) / kDftLines);
  const unsigned z = static_cast<unsigned>(slabs);
  const unsigned whole = static_cast<unsigned>((outs + 15) / 16);
  if (static_cast<std::size_t>(whole) * groups * slabs < 256) {
    fn(std::integral_constant<int, 4>{}, dim3(static_cast<unsigned>((outs + 3) / 4), groups, z));
  } else {
    fn(std::integral_constant<int, 1>{}, dim3(whole, groups, z));
  }
}
}  // namespace

void launch_dft_move(bool keep, const double2* tw, const Cplx<float>* src, Cplx<float>* dst, int R,
                     int n, int N, long long src_rs, long long dst_rs, std::size_t slabs,
                     int lo_count, long long src_hi, long long src_lo, long long dst_hi,
                     long long dst_lo, hipStream_t stream) {
  if (!slabs || !R || !n || !N) return;
  dft_launch(R, keep ? N : n, slabs, [&](auto parts, dim3 grid) {
    constexpr int P = decltype(parts)::value;
    if (keep) {
      hipLaunchKernelGGL((dft_keep_kernel<P>), grid, dim3(kDftThreads), 0, stream, tw, src, dst, R,
                         n, N, src_rs, dst_rs, lo_count, src_hi, src_lo, dst_hi, dst_lo);
    } else {
      hipLaunchKernelGGL((dft_expand_kernel<P>), grid, dim3(kDftThreads), 0, stream, tw, src, dst,
                         R, n, N, src_rs, dst_rs, lo_count, src_hi, src_lo, dst_hi, dst_lo);
    }
  });
  check_launch("dft_move");
}

template <int DIM>
void launch_dft_modes_out(const double2* tw, const Cplx<float>* src, long long member_stride,
                          Cplx<float>* single, Cplx<float>* const* outs, int count, int N0, int Nm,
                          int nl, int Nl, long long st0, long long stm, long long stl,
                          const float* fs0, const float* fsm, const float* fsl, int order_fft,
                          hipStream_t stream) {
  const std::size_t slabs = static_cast<std::size_t>(count) * (DIM == 3 ? Nm : 1);
  if (!slabs) return;
  dft_launch(N0, Nl, slabs, [&](auto parts, dim3 grid) {
    hipLaunchKernelGGL((dft_modes_out_kernel<DIM, decltype(parts)::value>), grid,
                       dim3(kDftThreads), 0, stream, tw, src, member_stride, single, outs, N0, Nm,
                       nl, Nl, st0, stm, stl, fs0, fsm, fsl, order_fft);
  });
  check_launch("dft_modes_out_kernel");
}

template <int DIM>
void launch_dft_modes_in(const double2* tw, const Cplx<float>* single,
                         const Cplx<float>* const* ins, int count, Cplx<float>* dst,
                         long long member_stride, int N0, int Nm, int nl, int Nl, long long st0,
                         long long stm, long long stl, const float* fs0, const float* fsm,
                         const float* fsl, int order_fft, hipStream_t stream) {
  const std::size_t slabs = static_cast<std::size_t>(count) * (DIM == 3 ? Nm : 1);
  if (!slabs) return;
  dft_launch(N0, nl, slabs, [&](auto parts, dim3 grid) {
    hipLaunchKernelGGL((dft_modes_in_kernel<DIM, decltype(parts)::value>), grid,
                       dim3(kDftThreads), 0, stream, tw, single, ins, dst, member_stride, N0, Nm,
                       nl, Nl, st0, stm, stl, fs0, fsm, fsl, order_fft);
  });
  check_launch("dft_modes_in_kernel");
}

#define NNF_INST_DFT(DIM)                                                                        \
  template void launch_dft_modes_out<DIM>(const double2*, const Cplx<float>*, long long,          \
                                          Cplx<float>*, Cplx<float>* const*, int, int, int, int,  \
                                          int, long long, long long, long long, const float*,     \
                                          const float*, const float*, int, hipStream_t);          \
  template void launch_dft_modes_in<DIM>(const double2*, const Cplx<float>*,                      \
                                         const Cplx<float>* const*, int, Cplx<float>*, long long, \
                                         int, int, int, int, long long, long long, long long,     \
                                         const float*, const float*, const float*, int,           \
                                         hipStream_t);
NNF_INST_DFT(2)
NNF_INST_DFT(3)

// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------
template <typename T>
void launch_compact_transpose(const Cplx<T>* src, Cplx<T>* dst, int R, int nc, int Nc,
                              long long src_rs, long long dst_rs, std::size_t slabs, int lo_count,
                              long long src_hi, long long src_lo, long long dst_hi,
                              long long dst_lo, hipStream_t stream) {
  if (!slabs || !R || !Nc) return;
  const dim3 grid((Nc + kTile - 1) / kTile, (R + kTile - 1) / kTile, cap_slabs(slabs));
  hipLaunchKernelGGL((compact_transpose_kernel<T>), grid, dim3(kTile, kRowsPer), 0, stream, src,
                     dst, R, nc, Nc, src_rs, dst_rs, static_cast<int>(slabs), lo_count, src_hi,
                     src_lo, dst_hi, dst_lo);
  check_launch("compact_transpose_kernel");
}

template <typename T>
void launch_expand_transpose(const Cplx<T>* src, Cplx<T>* dst, int R, int nf, int Nf,
                             long long src_rs, long long dst_rs, std::size_t slabs, int lo_count,
                             long long src_hi, long long src_lo, long long dst_hi,
                             long long dst_lo, hipStream_t stream) {
  if (!slabs || !R || !nf) return;
  const dim3 grid((nf + kTile - 1) / kTile, (R + kTile - 1) / kTile, cap_slabs(slabs));
  hipLaunchKernelGGL((expand_transpose_kernel<T>), grid, dim3(kTile, kRowsPer), 0, stream, src,
                     dst, R, nf, Nf, src_rs, dst_rs, static_cast<int>(slabs), lo_count, src_hi,
                     src_lo, dst_hi, dst_lo);
  check_launch("expand_transpose_kernel");
}

template <typename T, int DIM>
void launch_modes_out(const Cplx<T>* src, long long member_stride, Cplx<T>* single,
                      Cplx<T>* const* outs, int count, int N0, int Nm, int nl, int Nl,
                      long long st0, long long stm, long long stl, const T* fs0, const T* fsm,
                      const T* fsl, int order_fft, hipStream_t stream) {
  const std::size_t slabs = static_cast<std::size_t>(count) * (DIM == 3 ? Nm : 1);
  const dim3 grid((Nl + kTile - 1) / kTile, (N0 + kTile - 1) / kTile, cap_slabs(slabs));
  hipLaunchKernelGGL((modes_out_kernel<T, DIM>), grid, dim3(kTile, kRowsPer), 0, stream, src,
                     member_stride, single, outs, N0, Nm, nl, Nl, st0, stm, stl, fs0, fsm, fsl,
                     order_fft, static_cast<int>(slabs));
  check_launch("modes_out_kernel");
}

template <typename T, int DIM>
void launch_modes_in(const Cplx<T>* single, const Cplx<T>* const* ins, int count, Cplx<T>* dst,
                     long long member_stride, int N0, int Nm, int nl, int Nl, long long st0,
                     long long stm, long long stl, const T* fs0, const T* fsm, const T* fsl,
                     int order_fft, hipStream_t stream) {
  const std::size_t slabs = static_cast<std::size_t>(count) * (DIM == 3 ? Nm : 1);
  const dim3 grid((nl + kTile - 1) / kTile, (N0 + kTile - 1) / kTile, cap_slabs(slabs));
  hipLaunchKernelGGL((modes_in_kernel<T, DIM>), grid, dim3(kTile, kRowsPer), 0, stream, single,
                     ins, dst, member_stride, N0, Nm, nl, Nl, st0, stm, stl, fs0, fsm, fsl,
                     order_fft, static_cast<int>(slabs));
  check_launch("modes_in_kernel");
}

#define NNF_INST_PRUNED_T(T)                                                                     \
  template void launch_compact_transpose<T>(const Cplx<T>*, Cplx<T>*, int, int, int, long long,   \
                                            long long, std::size_t, int, long long, long long,    \
                                            long long, long long, hipStream_t);                   \
  template void launch_expand_transpose<T>(const Cplx<T>*, Cplx<T>*, int, int, int, long long,    \
                                           long long, std::size_t, int, long long, long long,     \
                                           long long, long long, hipStream_t);
#define NNF_INST_PRUNED(T, DIM)                                                                  \
  template void launch_modes_out<T, DIM>(const Cplx<T>*, long long, Cplx<T>*, Cplx<T>* const*,    \
                                         int, int, int, int, int, long long, long long,           \
                                         long long, const T*, const T*, const T*, int,            \
                                         hipStream_t);                                            \
  template void launch_modes_in<T, DIM>(const Cplx<T>*, const Cplx<T>* const*, int, Cplx<T>*,     \
                                        long long, int, int, int, int, long long, long long,      \
                                        long long, const T*, const T*, const T*, int,             \
                                        hipStream_t);

NNF_INST_PRUNED_T(float)
NNF_INST_PRUNED_T(double)
NNF_INST_PRUNED(float, 2)
NNF_INST_PRUNED(float, 3)
NNF_INST_PRUNED(double, 2)
NNF_INST_PRUNED(double, 3)

}  // namespace nnf
