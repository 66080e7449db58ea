// Local H.psi and density kernels specialised to compile-time axis lengths, built on the
// two-level register FFT of fft_reg.hpp and the one-lane transforms of fft_lane.hpp. Same data
// layout and results as the generic kernels of fft.hip, which remain the path for every other
// grid. A grid takes them when two of its axes have one supported length (the plane, N x N) and
// the third (along the sticks, N1 planes) a supported length of its own: cubic grids, and those
// of cells elongated along one axis, whose plan then works in permuted axes.
//
// This header is compiled once per part of the length list (fft_fast_a.hip, ...): a part defines
// AMT_PART(X), its lengths, and AMT_PART_FN(name), the suffix of its three entry points.
#include "fft_fast.hpp"
#include "fft_lane.hpp"
#include "fft_reg.hpp"
#include "kernels.hpp"

namespace amt {
namespace {

constexpr int ceil_div(int a, int b) { return (a + b - 1) / b; }

template <typename C>
constexpr int stick_width() {
  return sizeof(C) == 16 ? 32 : 64;
}

// ----------------------------------------------------------------------- kernels
// Stick kernels run on a 1-D grid of 8 * nch * ceil(nkb / 8) workgroups. Workgroup w goes to
// XCD w % 8, and all nch stick chunks of band row kb get w % 8 = kb % 8, so every chunk of a
// band row runs on one XCD and its scattered sphere-order reads and writes of that row meet in
// one L2 instead of being fetched once per XCD.
__device__ __forceinline__ bool stick_block(int nch, int nkb, int& chunk, int& kb) {
  const int w = blockIdx.x, slot = w >> 3;
  chunk = slot % nch;
  kb = (slot / nch) * 8 + (w & 7);
  return kb < nkb;
}
inline unsigned stick_grid(int nch, int nkb) { return 8u * (unsigned)nch * (unsigned)((nkb + 7) / 8); }

template <int N, typename C, int W>
__global__ __launch_bounds__(256) void k_stick_inverse_n(const C* __restrict__ psi, C* __restrict__ sticks,
                                                         const int* __restrict__ stick_map, int smax, int npw_pad,
                                                         int nb, int k0, const C* __restrict__ tw, int nch,
                                                         int nkb) {
  constexpr int T2 = ceil_div(W * Split<N>::N1, 256);
  __shared__ C tile[N * W];
  const int tid = threadIdx.x;
  int chunk, kb;
  if (!stick_block(nch, nkb, chunk, kb)) return;
  const int k = k0 + kb / nb;
  const int s0 = chunk * W;
  const C* c = psi + (long long)kb * npw_pad;
  const int* mp = stick_map + (long long)k * N * smax;
  for (int e = tid; e < N * W; e += 256) {
    const int i = e / W, w = e % W, s = s0 + w;
    C v = cmake<C>(0, 0);
    if (s < smax) {
      const int g = mp[i * smax + s];
      if (g >= 0) v = c[g];
    }
    tile[e] = v;
  }
  __syncthreads();
  fft2<N, 1, T2, false>(tile, W, 1, W, nullptr, tw, tid, 256);
  C* out = sticks + (long long)kb * N * smax;
  for (int e = tid; e < N * W; e += 256) {
    const int i = e / W, w = e % W, s = s0 + w;
    if (s < smax) out[i * smax + s] = tile[e];
  }
}

template <int N, typename C, typename R, int W>
__global__ __launch_bounds__(256) void k_stick_forward_n(const C* __restrict__ sticks, const C* __restrict__ psi,
                                                         C* __restrict__ out, const int* __restrict__ stick_map,
                                                         const R* __restrict__ kin, const int* __restrict__ npw,
                                                         int smax, int npw_pad, int nb, int k0,
                                                         const C* __restrict__ tw, R scale, int nch, int nkb) {
  constexpr int T2 = ceil_div(W * Split<N>::N1, 256);
  __shared__ C tile[N * W];
  const int tid = threadIdx.x;
  int chunk, kb;
  if (!stick_block(nch, nkb, chunk, kb)) return;
  const int k = k0 + kb / nb;
  const int s0 = chunk * W;
  const C* in = sticks + (long long)kb * N * smax;
  for (int e = tid; e < N * W; e += 256) {
    const int i = e / W, w = e % W, s = s0 + w;
    tile[e] = (s < smax) ? in[i * smax + s] : cmake<C>(0, 0);
  }
  __syncthreads();
  fft2<N, -1, T2, false>(tile, W, 1, W, nullptr, tw, tid, 256);
  const int* mp = stick_map + (long long)k * N * smax;
  const C* cc = psi + (long long)kb * npw_pad;
  C* o = out + (long long)kb * npw_pad;
  const R* t = kin + (long long)k * npw_pad;
  if (npw && chunk == 0)  // the row's padding
    for (int g = npw[k] + tid; g < npw_pad; g += 256) o[g] = cmake<C>(0, 0);
  for (int e = tid; e < N * W; e += 256) {
    const int i = e / W, w = e % W, s = s0 + w;
    if (s < smax) {
      const int g = mp[i * smax + s];
      if (g >= 0) {
        const C x = cc[g];
        const C y = tile[e];
        o[g] = cmake<C>(t[g] * x.x + scale * y.x, t[g] * x.y + scale * y.y);
      }
    }
  }
}

// ----------------------------------------------------------------------- plane pieces
// Bit kk of a row's 128-bit stick mask, and the number of set bits below it.
__device__ __forceinline__ bool mask_bit(unsigned long long lo, unsigned long long hi, int kk) {
  return kk < 64 ? ((lo >> kk) & 1ull) : ((hi >> (kk - 64)) & 1ull);
}
__device__ __forceinline__ int mask_below(unsigned long long lo, unsigned long long hi, int kk) {
  return kk < 64 ? __popcll(lo & ((1ull << kk) - 1ull)) : __popcll(lo) + __popcll(hi & ((1ull << (kk - 64)) - 1ull));
}

// u[k1] *= w_N^{SIGN j2 k1} (tw = exp(-2 pi i m / N); j2 k1 < N for the four-step indices).
template <int N, int NA, int SIGN, typename C>
__device__ __forceinline__ void twiddle_row(C (&u)[NA], int j2, const C* __restrict__ tw) {
#pragma unroll
  for (int k1 = 1; k1 < NA; ++k1) {
    C w = tw[j2 * k1];
    if (SIGN > 0) w.y = -w.y;
    u[k1] = cmul(u[k1], w);
  }
}

// Local part of H.psi for one i-plane of one band row: the inverse 2D transform of the
// plane's sticks, times V_eff, and the forward 2D transform back onto the sticks. The length
// N = N1 N2 transforms are four-step (fft_reg.hpp) with these savings over a plain pair of
// 2D transforms:
//  * the sticks are read straight from the stick workspace by the first phase along k (the
//    row masks give each (j, k) its stick index), so the plane is never zeroed or scattered;
//  * along k only the rows j that hold sticks are transformed, and the first phase along j
//    reads the other rows as zeros;
//  * the second inverse phase along j, the V_eff multiply and the first forward phase along j
//    are one register pass: the forward transform uses the transposed split (N2 x N1), whose
//    first phase consumes exactly the N2 outputs one inverse task holds;
//  * the forward phase along j writes only rows that hold sticks, and the last phase along k
//    writes its outputs straight back to the sticks.
template <int N, typename C, typename R, int NTH>
__global__ __launch_bounds__(NTH) void k_plane_vloc_n(C* __restrict__ sticks, const int* __restrict__ rows,
                                                      const int* __restrict__ nrows,
                                                      const unsigned long long* __restrict__ rowmask,
                                                      const int* __restrict__ rowstart,
                                                      const unsigned long long* __restrict__ livemask,
                                                      const R* __restrict__ veff, int n1, int smax, int nb, int k0,
                                                      const C* __restrict__ tw) {
  constexpr int N1 = Split<N>::N1, N2 = Split<N>::N2;
  constexpr int TR = ceil_div(N * N1, NTH);  // rounds of the (row or column, k1) tasks
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  C* plane = reinterpret_cast<C*>(smem_raw);
  __shared__ int rl[(N + 3) / 4 * 4];  // sizes in multiples of 16 bytes keep the dynamic plane 16-byte aligned
  __shared__ int rs[(N + 3) / 4 * 4];
  __shared__ unsigned long long rm[2 * N];
  const int tid = threadIdx.x;
  const int i = blockIdx.x;
  const int kb = blockIdx.y;
  const int k = k0 + kb / nb;
  const int nr = nrows[k];
  const unsigned long long live_lo = livemask[2 * k], live_hi = livemask[2 * k + 1];
  C* st = sticks + ((long long)kb * n1 + i) * smax;
  for (int r = tid; r < nr; r += NTH) {
    const int j = rows[(long long)k * N + r];
    rl[r] = j;
    rs[r] = rowstart[(long long)k * N + j];
    rm[2 * r] = rowmask[((long long)k * N + j) * 2];
    rm[2 * r + 1] = rowmask[((long long)k * N + j) * 2 + 1];
  }
  __syncthreads();

  // 1. inverse along k, phase 1, rows with sticks: read the sticks, DFT_N1, twiddle
  for (int t = tid; t < nr * N2; t += NTH) {
    const int s = t / N2, j2 = t % N2;
    const unsigned long long lo = rm[2 * s], hi = rm[2 * s + 1];
    const C* src = st + rs[s];
    C u[N1];
#pragma unroll
    for (int n1 = 0; n1 < N1; ++n1) {
      const int kk = j2 + N2 * n1;
      u[n1] = mask_bit(lo, hi, kk) ? src[mask_below(lo, hi, kk)] : cmake<C>(0, 0);
    }
    small_dft<N1, 1>(u);
    twiddle_row<N, N1, 1>(u, j2, tw);
    C* row = plane + rl[s] * N;
#pragma unroll
    for (int k1 = 0; k1 < N1; ++k1) row[j2 + N2 * k1] = u[k1];
  }
  __syncthreads();
  // 2. inverse along k, phase 2 (in place: all reads, barrier, all writes)
  {
    C v[TR][N2];
#pragma unroll
    for (int q = 0; q < TR; ++q) {
      const int t = tid + q * NTH;
      if (t < nr * N1) {
        const C* row = plane + rl[t / N1] * N + N2 * (t % N1);
#pragma unroll
        for (int j2 = 0; j2 < N2; ++j2) v[q][j2] = row[j2];
        small_dft<N2, 1>(v[q]);
      }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < TR; ++q) {
      const int t = tid + q * NTH;
      if (t < nr * N1) {
        C* row = plane + rl[t / N1] * N + t % N1;
#pragma unroll
        for (int k2 = 0; k2 < N2; ++k2) row[N1 * k2] = v[q][k2];
      }
    }
  }
  __syncthreads();
  // 3. inverse along j, phase 1, every column; rows without sticks read as zeros
  for (int t = tid; t < N * N2; t += NTH) {
    const int c = t % N, j2 = t / N;
    C u[N1];
#pragma unroll
    for (int n1 = 0; n1 < N1; ++n1) {
      const int j = j2 + N2 * n1;
      u[n1] = mask_bit(live_lo, live_hi, j) ? plane[j * N + c] : cmake<C>(0, 0);
    }
    small_dft<N1, 1>(u);
    twiddle_row<N, N1, 1>(u, j2, tw);
#pragma unroll
    for (int k1 = 0; k1 < N1; ++k1) plane[(j2 + N2 * k1) * N + c] = u[k1];
  }
  __syncthreads();
  // 4. inverse along j phase 2, times V_eff, forward along j phase 1 of the transposed split
  //    (N = N2 x N1): task (c, k1) holds rows k1 + N1 m, m < N2, from the DFT to the twiddle.
  {
    const R* v = veff + (long long)i * N * N;
    C x[TR][N2];
#pragma unroll
    for (int q = 0; q < TR; ++q) {
      const int t = tid + q * NTH;
      if (t < N * N1) {
        const int c = t % N, k1 = t / N;
#pragma unroll
        for (int j2 = 0; j2 < N2; ++j2) x[q][j2] = plane[(N2 * k1 + j2) * N + c];
        small_dft<N2, 1>(x[q]);
#pragma unroll
        for (int m = 0; m < N2; ++m) x[q][m] = cscale(x[q][m], v[(k1 + N1 * m) * N + c]);
        small_dft<N2, -1>(x[q]);
        twiddle_row<N, N2, -1>(x[q], k1, tw);
      }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < TR; ++q) {
      const int t = tid + q * NTH;
      if (t < N * N1) {
        const int c = t % N, k1 = t / N;
#pragma unroll
        for (int m = 0; m < N2; ++m) plane[(k1 + N1 * m) * N + c] = x[q][m];
      }
    }
  }
  __syncthreads();
  // 5. forward along j, phase 2 of the transposed split: task (c, m) reads rows N1 m + k1,
  //    k1 < N1, and produces rows m + N2 p, p < N1; only rows with sticks are kept
  {
    constexpr int TC = ceil_div(N * N2, NTH);
    C y[TC][N1];
#pragma unroll
    for (int q = 0; q < TC; ++q) {
      const int t = tid + q * NTH;
      if (t < N * N2) {
        const int c = t % N, m = t / N;
#pragma unroll
        for (int k1 = 0; k1 < N1; ++k1) y[q][k1] = plane[(N1 * m + k1) * N + c];
        small_dft<N1, -1>(y[q]);
      }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < TC; ++q) {
      const int t = tid + q * NTH;
      if (t < N * N2) {
        const int c = t % N, m = t / N;
#pragma unroll
        for (int p = 0; p < N1; ++p) {
          const int j = m + N2 * p;
          if (mask_bit(live_lo, live_hi, j)) plane[j * N + c] = y[q][p];
        }
      }
    }
  }
  __syncthreads();
  // 6. forward along k, phase 1, rows with sticks
  for (int t = tid; t < nr * N2; t += NTH) {
    const int s = t / N2, j2 = t % N2;
    C* row = plane + rl[s] * N;
    C u[N1];
#pragma unroll
    for (int n1 = 0; n1 < N1; ++n1) u[n1] = row[j2 + N2 * n1];
    small_dft<N1, -1>(u);
    twiddle_row<N, N1, -1>(u, j2, tw);
#pragma unroll
    for (int k1 = 0; k1 < N1; ++k1) row[j2 + N2 * k1] = u[k1];
  }
  __syncthreads();
  // 7. forward along k, phase 2: outputs at k = k1 + N1 k2 go straight to their sticks
  for (int t = tid; t < nr * N1; t += NTH) {
    const int s = t / N1, k1 = t % N1;
    const C* row = plane + rl[s] * N + N2 * k1;
    C v[N2];
#pragma unroll
    for (int j2 = 0; j2 < N2; ++j2) v[j2] = row[j2];
    small_dft<N2, -1>(v);
    const unsigned long long lo = rm[2 * s], hi = rm[2 * s + 1];
    C* dst = st + rs[s];
#pragma unroll
    for (int k2 = 0; k2 < N2; ++k2) {
      const int kk = k1 + N1 * k2;
      if (mask_bit(lo, hi, kk)) dst[mask_below(lo, hi, kk)] = v[k2];
    }
  }
}

// sum_l w_l |u_l(r)|^2 over the bands of one chunk of the list, on one i-plane: the inverse 2D
// transform of each band's plane as in k_plane_vloc_n (sticks read through the row masks, rows
// without sticks read as zeros along j), and the second phase along j squares its outputs into
// FP64 accumulators held by the task that computes them (task (c, k1) always owns rows
// k1 + N1 m of column c), so the transformed plane is never written back.
template <int N, typename C>
__global__ __launch_bounds__(512) void k_density_plane_n(const C* __restrict__ sticks, const int* __restrict__ rows,
                                                         const int* __restrict__ nrows,
                                                         const unsigned long long* __restrict__ rowmask,
                                                         const int* __restrict__ rowstart,
                                                         const unsigned long long* __restrict__ livemask,
                                                         const int* __restrict__ band_list,
                                                         const double* __restrict__ band_weight, int nlist,
                                                         int chunk, int n1, int smax, int nb, int k0,
                                                         const C* __restrict__ tw, double* __restrict__ part) {
  constexpr int NTH = 512;
  constexpr int NP = N * N;
  constexpr int N1 = Split<N>::N1, N2 = Split<N>::N2;
  constexpr int TR = ceil_div(N * N1, NTH);
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  C* plane = reinterpret_cast<C*>(smem_raw);
  __shared__ int rl[(N + 3) / 4 * 4];  // sizes in multiples of 16 bytes keep the dynamic plane 16-byte aligned
  __shared__ int rs[(N + 3) / 4 * 4];
  __shared__ unsigned long long rm[2 * N];
  const int tid = threadIdx.x;
  const int i = blockIdx.x;
  const int ch = blockIdx.y;
  double acc[TR][N2];
#pragma unroll
  for (int q = 0; q < TR; ++q)
#pragma unroll
    for (int m = 0; m < N2; ++m) acc[q][m] = 0.0;
  const int l0 = ch * chunk;
  const int l1 = (l0 + chunk < nlist) ? l0 + chunk : nlist;
  for (int l = l0; l < l1; ++l) {
    const int kb = band_list[l];
    const double wgt = band_weight[l];
    const int k = k0 + kb / nb;
    const int nr = nrows[k];
    const unsigned long long live_lo = livemask[2 * k], live_hi = livemask[2 * k + 1];
    const C* st = sticks + ((long long)kb * n1 + i) * smax;
    for (int r = tid; r < nr; r += NTH) {
      const int j = rows[(long long)k * N + r];
      rl[r] = j;
      rs[r] = rowstart[(long long)k * N + j];
      rm[2 * r] = rowmask[((long long)k * N + j) * 2];
      rm[2 * r + 1] = rowmask[((long long)k * N + j) * 2 + 1];
    }
    __syncthreads();
    // inverse along k, phase 1 (sticks read through the row masks)
    for (int t = tid; t < nr * N2; t += NTH) {
      const int s = t / N2, j2 = t % N2;
      const unsigned long long lo = rm[2 * s], hi = rm[2 * s + 1];
      const C* src = st + rs[s];
      C u[N1];
#pragma unroll
      for (int n1 = 0; n1 < N1; ++n1) {
        const int kk = j2 + N2 * n1;
        u[n1] = mask_bit(lo, hi, kk) ? src[mask_below(lo, hi, kk)] : cmake<C>(0, 0);
      }
      small_dft<N1, 1>(u);
      twiddle_row<N, N1, 1>(u, j2, tw);
      C* row = plane + rl[s] * N;
#pragma unroll
      for (int k1 = 0; k1 < N1; ++k1) row[j2 + N2 * k1] = u[k1];
    }
    __syncthreads();
    // inverse along k, phase 2 (in place)
    {
      C v[TR][N2];
#pragma unroll
      for (int q = 0; q < TR; ++q) {
        const int t = tid + q * NTH;
        if (t < nr * N1) {
          const C* row = plane + rl[t / N1] * N + N2 * (t % N1);
#pragma unroll
          for (int j2 = 0; j2 < N2; ++j2) v[q][j2] = row[j2];
          small_dft<N2, 1>(v[q]);
        }
      }
      __syncthreads();
#pragma unroll
      for (int q = 0; q < TR; ++q) {
        const int t = tid + q * NTH;
        if (t < nr * N1) {
          C* row = plane + rl[t / N1] * N + t % N1;
#pragma unroll
          for (int k2 = 0; k2 < N2; ++k2) row[N1 * k2] = v[q][k2];
        }
      }
    }
    __syncthreads();
    // inverse along j, phase 1 (rows without sticks read as zeros)
    for (int t = tid; t < N * N2; t += NTH) {
      const int c = t % N, j2 = t / N;
      C u[N1];
#pragma unroll
      for (int n1 = 0; n1 < N1; ++n1) {
        const int j = j2 + N2 * n1;
        u[n1] = mask_bit(live_lo, live_hi, j) ? plane[j * N + c] : cmake<C>(0, 0);
      }
      small_dft<N1, 1>(u);
      twiddle_row<N, N1, 1>(u, j2, tw);
#pragma unroll
      for (int k1 = 0; k1 < N1; ++k1) plane[(j2 + N2 * k1) * N + c] = u[k1];
    }
    __syncthreads();
    // inverse along j, phase 2, squared into the accumulators
#pragma unroll
    for (int q = 0; q < TR; ++q) {
      const int t = tid + q * NTH;
      if (t < N * N1) {
        const int c = t % N, k1 = t / N;
        C x[N2];
#pragma unroll
        for (int j2 = 0; j2 < N2; ++j2) x[j2] = plane[(N2 * k1 + j2) * N + c];
        small_dft<N2, 1>(x);
#pragma unroll
        for (int m = 0; m < N2; ++m) acc[q][m] += wgt * ((double)x[m].x * (double)x[m].x + (double)x[m].y * (double)x[m].y);
      }
    }
    __syncthreads();  // the next band overwrites the plane and the row lists
  }
  double* out = part + ((long long)ch * n1 + i) * NP;
#pragma unroll
  for (int q = 0; q < TR; ++q) {
    const int t = tid + q * NTH;
    if (t < N * N1) {
      const int c = t % N, k1 = t / N;
#pragma unroll
      for (int m = 0; m < N2; ++m) out[(k1 + N1 * m) * N + c] = acc[q][m];
    }
  }
}

// ----------------------------------------------------------------------- one-lane plane kernel
// The sphere of the bands has half the radius of the density's, for which the grid is made, so
// of N rows (and of N columns of a row) only those within H = N/4 + 1 of zero, modulo N, hold
// sticks: 2 H + 1 rows ("narrow" plans; the extra one covers k-point shifts). They are kept in
// compressed slots 0 .. 2 H.
template <int N>
struct Prune {
  static constexpr int H = lane_half_width(N), ROWS = 2 * H + 1, LD = N | 1;
  static constexpr bool live(int j) { return j <= H || j >= N - H; }
  static constexpr int slot(int j) { return j <= H ? j : j - (N - ROWS); }
};

// LDS reads of other lanes' values stay behind the writes before them: the wavefront's LDS
// operations execute in order, only the compiler has to keep them so.
__device__ __forceinline__ void wave_lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}
// value of another lane of the quad (DPP quad_perm)
template <int CTRL>
__device__ __forceinline__ float quad_perm(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xf, 0xf, true));
}
template <int CTRL>
__device__ __forceinline__ double quad_perm(double v) {
  return __hiloint2double(__builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xf, 0xf, true),
                          __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xf, 0xf, true));
}
// Length-N transforms of one row or column by P neighbouring lanes (P = 1 or 4), M = N / P
// points in each lane's registers. Inverse: lane p computes outputs P q + p from the live inputs
// at slot(j) * stride:
//   y_p[j] = w_N^{p j} sum_s i^{p s} x[j + s M] (P = 4),  u[P q + p] = DFT_M(y_p)[q],
// of whose P terms at most two are live. tw holds w_N^{p j} at p M + j.
template <int N, int P, typename C, typename Get>
__device__ __forceinline__ void pruned_inverse(C (&y)[N / P], const Get& get, int p, const C* tw) {
  using R = decltype(C::x);
  using Pr = Prune<N>;
  constexpr int M = N / P;
  static_assert(P == 1 || P == 4, "one lane per row or a quad");
  // i^(p s) of the P = 4 first step for s = 1 (its conjugate for s = 3), (-1)^p for s = 2
  const R cr = p == 0 ? (R)1 : p == 2 ? (R)-1 : (R)0, ci = p == 1 ? (R)1 : p == 3 ? (R)-1 : (R)0;
  const R sg = p & 1 ? (R)-1 : (R)1;
  static_for<M>([&](auto j_) {
    constexpr int j = j_;
    C v = cmake<C>(0, 0);
    if constexpr (Pr::live(j)) v = get(j_);
    if constexpr (P == 4) {
      if constexpr (Pr::live(j + M)) {
        const C x = get(std::integral_constant<int, j + M>{});
        v = cmake<C>(v.x + (cr * x.x - ci * x.y), v.y + (cr * x.y + ci * x.x));
      }
      if constexpr (Pr::live(j + 2 * M)) {
        const C x = get(std::integral_constant<int, j + 2 * M>{});
        v = cmake<C>(v.x + sg * x.x, v.y + sg * x.y);
      }
      if constexpr (Pr::live(j + 3 * M)) {
        const C x = get(std::integral_constant<int, j + 3 * M>{});
        v = cmake<C>(v.x + (cr * x.x + ci * x.y), v.y + (cr * x.y - ci * x.x));
      }
    }
    if constexpr (P > 1 && j > 0) {
      const C w = tw[p * M + j];
      v = cmake<C>(v.x * w.x + v.y * w.y, v.y * w.x - v.x * w.y);
    }
    y[j] = v;
  });
  lane_dft<M, 1>(y);
}
// Forward: lane p holds u[P q + p]; its DFT_M, times w_N^{-p k}, is combined across the P lanes by
// quad permutations, after which each lane holds the outputs s M + k of one s and hands the live
// ones to put(k, value) with put = range(s).
template <int N, int P, typename C, typename Range>
__device__ __forceinline__ void pruned_forward(C (&y)[N / P], const Range& range, int p, const C* tw) {
  using R = decltype(C::x);
  using Pr = Prune<N>;
  constexpr int M = N / P;
  lane_dft<M, -1>(y);
  if constexpr (P > 1) {
    const R sa = p >= 2 ? (R)-1 : (R)1, sb = p & 1 ? (R)-1 : (R)1;
    const R c3 = p == 3 ? (R)0 : (R)1, s3 = p == 3 ? (R)1 : (R)0;
    static_for<M>([&](auto k_) {
      constexpr int k = k_;
      if constexpr (k > 0) y[k] = cmul(y[k], tw[p * M + k]);
      const R zx = quad_perm<0x4E>(y[k].x) + sa * y[k].x, zy = quad_perm<0x4E>(y[k].y) + sa * y[k].y;  // lanes 2 3 0 1
      const R rx = zx * c3 - zy * s3, ry = zy * c3 + zx * s3;                                          // lane 3: times i
      y[k].x = quad_perm<0xB1>(rx) + sb * rx;  // lanes 1 0 3 2
      y[k].y = quad_perm<0xB1>(ry) + sb * ry;
    });
  }
  const int s = p == 0 ? 0 : p == 1 ? 2 : p == 2 ? 3 : 1;
  const auto put = range(s);
  static_for<M>([&](auto k_) {
    constexpr int k = k_;
    constexpr unsigned mask = (Pr::live(k) ? 1u : 0u) | (P > 1 && Pr::live(k + M) ? 2u : 0u) |
                              (P > 1 && Pr::live(k + 2 * M) ? 4u : 0u) | (P > 1 && Pr::live(k + 3 * M) ? 8u : 0u);
    if constexpr (P == 1) {
      if constexpr (mask != 0) put(k_, y[k]);
    } else {
      if ((mask >> s) & 1u) put(k_, y[k]);
    }
  });
}

// Both on LDS rows or columns in compressed slots. Outputs s M + k of one s lie at slot s M + k (the
// low end of the range) or s M + k - (N - ROWS) (the high end); for P = 1 both ends are met.
template <int N, int P, typename C>
__device__ __forceinline__ void slots_inverse(C (&y)[N / P], const C* base, int stride, int p, const C* tw) {
  pruned_inverse<N, P>(y, [&](auto j) { return base[Prune<N>::slot(j) * stride]; }, p, tw);
}
template <int N, int P, typename C>
__device__ __forceinline__ void slots_forward(C (&y)[N / P], C* base, int stride, int p, const C* tw) {
  using Pr = Prune<N>;
  constexpr int M = N / P;
  pruned_forward<N, P>(
      y,
      [&](int s) {
        C* out = base + (P == 1 ? 0 : s * M <= Pr::H ? s * M : s * M - (N - Pr::ROWS)) * stride;
        return [out, stride](auto k, C v) { out[(P == 1 ? Pr::slot(k) : (int)k) * stride] = v; };
      },
      p, tw);
}

// Local part of H.psi for one i-plane of one band row, as k_plane_vloc_n, with every transform in
// registers: LDS holds only the live rows ((2 H + 1) x N instead of N x N elements: the FP64 plane
// of 108^2, 187 KB, becomes 102 KB), each row and column is read and written once per direction
// (about 2 plane volumes of LDS traffic instead of 8) and all twiddles inside a lane are literals.
// Phases, one barrier each: sticks -> compressed slots; rows inverse; columns inverse, V_eff,
// forward; rows forward; slots -> sticks. Planes are dealt to the XCDs by i mod 8, so the bands
// of one plane read V_eff from one L2.
//
// Measured (MI355X, per launch): FP32 84^3, 160 bands 320 us against 369 for the four-step kernel,
// 108^3, 440 bands 1.92 against 2.62 ms, 42^3, 1024 bands 199 against 223 us; FP64 108^3, 45 bands
// 0.42 ms where whole-grid transforms took 5.9 ms. What bounds it: VALU issue for one lane per row
// (a third of the lanes idle at N = 42), the waits around five barriers with four. Which lengths
// take it, and both sides' times: lane_count().
template <int N, int P, typename C, typename R, int NTH, int WAVES>
__global__ __launch_bounds__(NTH, WAVES) void k_plane_lane_n(C* __restrict__ sticks, const int* __restrict__ stick_jk,
                                                             const int* __restrict__ nsticks,
                                                             const R* __restrict__ veff, int n1, int smax, int nb,
                                                             int k0, int nkb, const C* __restrict__ tw) {
  using Pr = Prune<N>;
  constexpr int M = N / P, ROWS = Pr::ROWS, LD = Pr::LD;
  constexpr int IT = (ROWS * ROWS + NTH - 1) / NTH;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  C* plane = reinterpret_cast<C*>(smem_raw);
  __shared__ C twl[P > 1 ? N : 1];
  const int tid = threadIdx.x;
  const int id = blockIdx.x, x = id & 7, q8 = id >> 3;
  const int i = x + 8 * (q8 / nkb), kb = q8 % nkb;
  if (i >= n1) return;
  const int k = k0 + kb / nb, S = nsticks[k];
  const int* jk = stick_jk + (long long)k * smax;
  C* st = sticks + ((long long)kb * n1 + i) * smax;
  int at[IT];
  C in[IT];
  static_for<IT>([&](auto u_) {
    constexpr int u = u_;
    const int s = tid + u * NTH;
    at[u] = s < S ? jk[s] : 0;
    in[u] = s < S ? st[s] : cmake<C>(0, 0);
  });
  if constexpr (P > 1) {
    for (int e = tid; e < N; e += NTH) twl[e] = tw[(e / M) * (e % M)];
  }
  for (int e = tid; e < ROWS * ROWS; e += NTH) plane[e / ROWS * LD + e % ROWS] = cmake<C>(0, 0);
  __syncthreads();
  static_for<IT>([&](auto u_) {
    constexpr int u = u_;
    if (tid + u * NTH < S) {
      const int j = at[u] / N, c = at[u] % N;
      at[u] = (j <= Pr::H ? j : j - (N - ROWS)) * LD + (c <= Pr::H ? c : c - (N - ROWS));
      plane[at[u]] = in[u];
    }
  });
  __syncthreads();
  {
    C y[M];
    for (int t = tid; t < ROWS * P; t += NTH) {
      const int p = t % P;
      C* row = plane + (t / P) * LD;
      slots_inverse<N, P>(y, row, 1, p, twl);
      wave_lds_order();
      static_for<M>([&](auto q_) { row[P * q_ + p] = y[q_]; });
    }
    __syncthreads();
    for (int t = tid; t < N * P; t += NTH) {
      const int p = t % P, c = t / P;
      C* col = plane + c;
      slots_inverse<N, P>(y, col, LD, p, twl);
      const R* v = veff + ((long long)i * N + p) * N + c;
      static_for<M>([&](auto q_) { y[q_] = cscale(y[q_], v[P * q_ * N]); });
      slots_forward<N, P>(y, col, LD, p, twl);
    }
    __syncthreads();
    for (int t = tid; t < ROWS * P; t += NTH) {
      const int p = t % P;
      C* row = plane + (t / P) * LD;
      static_for<M>([&](auto q_) { y[q_] = row[P * q_ + p]; });
      wave_lds_order();
      slots_forward<N, P>(y, row, 1, p, twl);
    }
  }
  __syncthreads();
  static_for<IT>([&](auto u_) {
    constexpr int u = u_;
    if (tid + u * NTH < S) st[tid + u * NTH] = plane[at[u]];
  });
}
// ----------------------------------------------------------------------- launchers

// Where the one-lane kernel is used, its lanes per row and its workgroup (one pass over the rows).
template <int N, typename R>
struct FourStepFits {  // one whole plane and its row tables in 160 KB
  static constexpr bool value = (long long)N * N * 2 * (int)sizeof(R) + 24LL * N <= 160 * 1024;
};
template <int N, typename R>
struct LanePlane {
  static constexpr bool fp64 = sizeof(R) == 8;
  static constexpr int lanes = lane_count(N, fp64);
  static constexpr bool use = lanes > 0;
  // One wavefront per plane with one lane per row (no barrier waits); four with four lanes, or
  // eight where LDS holds one plane per CU. (A workgroup of six leaves SIMDs uneven: 84^2 FP32
  // 511 us against 322.)
  static constexpr int threads = lanes == 1 ? 64 : fp64 && N > 100 ? 512 : 256;
  // Wavefronts per SIMD that the registers are held to: by the LDS of a plane with four lanes, and
  // for one lane 4 up to the length whose row just fits 128 registers, 3 up to 60, 2 in FP64. The
  // lengths next to a step spill (FP32 10 to 48 registers at 44, 45 and 48, 24 to 61 at 55, 56 and 60) and
  // are still ahead of the four-step kernel where lane_count() has them.
  static constexpr int waves = lanes == 1 ? (fp64 ? 2 : N <= 48 ? 4 : 3) : fp64 && N > 100 ? 1 : 2;
};

template <int N, typename R, int W>
int stick_pass(const Plan& p, int pass, const void* psi_, void* hpsi_, void* sticks_, int nb, int k0, int nkb,
               hipStream_t s) {
  using C = typename Cplx<R>::T;
  constexpr int prec = sizeof(R) == 8 ? kFP64 : kFP32;
  const int a = p.axis[0];
  const C* tw = prec == kFP64 ? (const C*)p.d_tw64[a] : (const C*)p.d_tw32[a];
  const R* kin = prec == kFP64 ? (const R*)p.d_kin64 : (const R*)p.d_kin32;
  const int nch = (p.smax + W - 1) / W;
  const dim3 grid(stick_grid(nch, nkb));
  if (pass == kStickInverse)
    hipLaunchKernelGGL((k_stick_inverse_n<N, C, W>), grid, dim3(256), 0, s, static_cast<const C*>(psi_),
                       static_cast<C*>(sticks_), p.d_stick_map, p.smax, p.npw_pad, nb, k0, tw, nch, nkb);
  else
    hipLaunchKernelGGL((k_stick_forward_n<N, C, R, W>), grid, dim3(256), 0, s, static_cast<const C*>(sticks_),
                       static_cast<const C*>(psi_), static_cast<C*>(hpsi_), p.d_stick_map, kin,
                       pass == kStickForwardPad ? p.d_npw : nullptr, p.smax, p.npw_pad,
                       nb, k0, tw, (R)(1.0 / ((double)p.n1 * p.n2 * p.n3)), nch, nkb);
  return hipGetLastError() != hipSuccess ? 1 : 0;
}

template <int N, typename R>
int stick_t(const Plan& p, int pass, const void* psi, void* hpsi, void* sticks, int nb, int k0, int nkb,
            hipStream_t s) {
  constexpr int prec = sizeof(R) == 8 ? kFP64 : kFP32;
  constexpr int W = stick_width<typename Cplx<R>::T>();
  return p.fast_stick_w[prec] == W / 2  // the launch shape the plan holds (autotuner)
             ? stick_pass<N, R, W / 2>(p, pass, psi, hpsi, sticks, nb, k0, nkb, s)
             : stick_pass<N, R, W>(p, pass, psi, hpsi, sticks, nb, k0, nkb, s);
}

template <int N, typename R>
int plane_t(const Plan& p, void* sticks_, const void* veff_, int nb, int k0, int nkb, hipStream_t s) {
  using C = typename Cplx<R>::T;
  constexpr int prec = sizeof(R) == 8 ? kFP64 : kFP32;
  C* sticks = static_cast<C*>(sticks_);
  const R* veff = static_cast<const R*>(veff_);
  const int a = p.axis[1], n1 = p.dim(0);
  const C* tw = prec == kFP64 ? (const C*)p.d_tw64[a] : (const C*)p.d_tw32[a];
  if constexpr (LanePlane<N, R>::use) {
    if (p.narrow) {
      using L = LanePlane<N, R>;
      constexpr size_t lds = (size_t)Prune<N>::ROWS * Prune<N>::LD * sizeof(C);
      hipLaunchKernelGGL((k_plane_lane_n<N, L::lanes, C, R, L::threads, L::waves>),
                         dim3(8u * (unsigned)((n1 + 7) / 8) * (unsigned)nkb), dim3(L::threads), lds, s, sticks, p.d_stick_jk,
                         p.d_nsticks, veff, n1, p.smax, nb, k0, nkb, tw);
      return hipGetLastError() != hipSuccess ? 1 : 0;
    }
  }
  if constexpr (FourStepFits<N, R>::value) {
    const size_t plds = (size_t)N * N * sizeof(C);
    if (p.plane_nth[prec] == 512)
      hipLaunchKernelGGL((k_plane_vloc_n<N, C, R, 512>), dim3(n1, nkb), dim3(512), plds, s, sticks, p.d_rows,
                         p.d_nrows, p.d_rowmask, p.d_rowstart, p.d_livemask, veff, n1, p.smax, nb, k0, tw);
    else
      hipLaunchKernelGGL((k_plane_vloc_n<N, C, R, 256>), dim3(n1, nkb), dim3(256), plds, s, sticks, p.d_rows,
                         p.d_nrows, p.d_rowmask, p.d_rowstart, p.d_livemask, veff, n1, p.smax, nb, k0, tw);
    return hipGetLastError() != hipSuccess ? 1 : 0;
  }
  return 1;  // not reached: such a plan takes the full-grid route
}

template <int N, typename R>
int density_t(const Plan& p, const void* sticks, int nb, int k0, const int* list, const double* weight, int nlist,
              int chunk, double* part, hipStream_t s) {
  using C = typename Cplx<R>::T;
  if constexpr (FourStepFits<N, R>::value) {
    const int a = p.axis[1], n1 = p.dim(0), nchunk = (nlist + chunk - 1) / chunk;
    const C* tw = sizeof(R) == 8 ? (const C*)p.d_tw64[a] : (const C*)p.d_tw32[a];
    hipLaunchKernelGGL((k_density_plane_n<N, C>), dim3(n1, nchunk), dim3(512), (size_t)N * N * sizeof(C), s,
                       static_cast<const C*>(sticks), p.d_rows, p.d_nrows, p.d_rowmask, p.d_rowstart, p.d_livemask,
                       list, weight, nlist, chunk, n1, p.smax, nb, k0, tw, part);
    return hipGetLastError() != hipSuccess ? 1 : 0;
  }
  return 1;  // not reached: such a plan takes the full-grid route
}

}  // namespace

// The part's lengths: -1 for any other.
int AMT_PART_FN(fast_stick)(const Plan& p, int prec, int pass, const void* psi, void* hpsi, void* sticks, int nb,
                            int k0, int nkb, hipStream_t s) {
  switch (p.dim(0)) {
#define AMT_CASE(N)                                                                     \
  case N:                                                                               \
    return prec == kFP64 ? stick_t<N, double>(p, pass, psi, hpsi, sticks, nb, k0, nkb, s) \
                         : stick_t<N, float>(p, pass, psi, hpsi, sticks, nb, k0, nkb, s);
    AMT_PART(AMT_CASE)
#undef AMT_CASE
    default:
      return -1;
  }
}

int AMT_PART_FN(fast_plane)(const Plan& p, int prec, void* sticks, const void* veff, int nb, int k0, int nkb,
                            hipStream_t s) {
  switch (p.dim(1)) {
#define AMT_CASE(N)                                                              \
  case N:                                                                        \
    return prec == kFP64 ? plane_t<N, double>(p, sticks, veff, nb, k0, nkb, s) \
                         : plane_t<N, float>(p, sticks, veff, nb, k0, nkb, s);
    AMT_PART(AMT_CASE)
#undef AMT_CASE
    default:
      return -1;
  }
}

int AMT_PART_FN(fast_density)(const Plan& p, int prec, const void* sticks, int nb, int k0, const int* list,
                              const double* weight, int nlist, int chunk, double* part, hipStream_t s) {
  switch (p.dim(1)) {
#define AMT_CASE(N)                                                                                     \
  case N:                                                                                               \
    return prec == kFP64 ? density_t<N, double>(p, sticks, nb, k0, list, weight, nlist, chunk, part, s) \
                         : density_t<N, float>(p, sticks, nb, k0, list, weight, nlist, chunk, part, s);
    AMT_PART(AMT_CASE)
#undef AMT_CASE
    default:
      return -1;
  }
}

}  // namespace amt
