// Cholesky factorisation of small Hermitian Gram matrices and the inverse of the factor (FP64
// complex), and the Loewdin series of a nearly orthonormal block's Gram matrix: what the
// Davidson's orthonormalisation needs between two matrix products.
//
// G = L L^H in 32 x 32 blocks; the result is L^{-1} (its product with the block is orthonormal),
// the trace of G (= ||L||_F^2) and the column sums of |L^{-1}|^2, from which the caller bounds the
// singular values. Launches: k_chol_load takes the Hermitian part of the raw product and factors
// the first diagonal block; k_chol_step(j) gives every trailing block (i, k) its own workgroup,
// which forms L_ij and L_kj = A W_j^H (W = inverse of the diagonal factor; recomputing them per
// workgroup replaces a grid-wide wait between panel and update), subtracts L_ij L_kj^H, and, in
// the workgroup of the next diagonal block, factors that one too; k_chol_inverse runs one block
// column of L^{-1} per workgroup. Block products run on v_mfma_f64_16x16x4, one 16 x 16 quarter
// per wavefront. A diagonal block is factored and inverted together (factor_block).
//
// What bounds it: the chain of launches and diagonal blocks (a 160-row matrix is 16 MFLOP).
// Measured on MI355X, host call to result, against potrf + trsm of the library: 18 us at up to 32
// rows (40-143), 67 at 96 (274), 127 at 160 (476), 239 at 256 (744), 655 at 512 (1640); with the
// diagonal blocks updated in LDS instead of registers 198 at 160 rows. The Loewdin series, one
// launch for eight: 12 us at 64 rows, 19 at 160. The lead shrinks with the rows (3.7 to 2.5), as
// the library's larger products fill the chip; above 512 its route is kept.
#include "kernels.hpp"

namespace amt {
namespace {

constexpr int CB = 32;           // block size
constexpr int CT = 256;          // threads: four wavefronts, one 16 x 16 quarter of a block each
typedef double doublex4 __attribute__((ext_vector_type(4)));
struct Tile {
  double2 v[CB][CB + 1];
};

__device__ __forceinline__ double2 conj2(double2 a) { return make_double2(a.x, -a.y); }

// One wavefront's quarter of A op(B): element q of lane l is at row r0 + l / 16 + 4 q, column
// c0 + l % 16 (op: conj(B)^T with kConjT, else B).
template <bool kConjT>
__device__ __forceinline__ void block_product(const Tile& a, const Tile& b, doublex4& re, doublex4& im) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = (wave >> 1) * 16 + (lane & 15), c = (wave & 1) * 16 + (lane & 15);
#pragma unroll
  for (int ks = 0; ks < CB / 4; ++ks) {
    const int k = 4 * ks + (lane >> 4);
    const double2 x = a.v[r][k];
    const double2 y = kConjT ? conj2(b.v[c][k]) : b.v[k][c];
    re = __builtin_amdgcn_mfma_f64_16x16x4f64(x.x, y.x, re, 0, 0, 0);
    im = __builtin_amdgcn_mfma_f64_16x16x4f64(x.x, y.y, im, 0, 0, 0);
    re = __builtin_amdgcn_mfma_f64_16x16x4f64(-x.y, y.y, re, 0, 0, 0);
    im = __builtin_amdgcn_mfma_f64_16x16x4f64(x.y, y.x, im, 0, 0, 0);
  }
}
template <typename F>
__device__ __forceinline__ void each_of_quarter(const doublex4& re, const doublex4& im, F&& f) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int q = 0; q < 4; ++q)
    f((wave >> 1) * 16 + (lane >> 4) + 4 * q, (wave & 1) * 16 + (lane & 15), make_double2(re[q], im[q]));
}
__device__ __forceinline__ void load_tile(Tile& t, const double2* src, int ld) {
  for (int e = threadIdx.x; e < CB * CB; e += CT) t.v[e / CB][e % CB] = src[(long long)(e / CB) * ld + e % CB];
}

// w = inverse of the Cholesky factor of a (its lower triangle is read). `bad` (LDS) becomes
// 1 + base + c at the first pivot that is not positive. Elements stay in registers: slot (r, k)
// holds a_rk until step k has used its column and the unscaled w_rk from then on, so that step c
// shares with all threads only p = a_cc, the column a_rc (r > c) and the row w_ck (k < c): one
// array of 32 values, two copies in turn, one barrier a step.
__device__ __forceinline__ void factor_block(const Tile& a, Tile& w, int base, int* bad) {
  __shared__ double2 shared[2][CB];
  __shared__ double pivot[CB];
  constexpr int kRows = CT / CB;  // rows between the slots of one thread
  const int k = threadIdx.x % CB, r0 = threadIdx.x / CB;
  double2 v[CB / kRows];
  __syncthreads();
#pragma unroll
  for (int u = 0; u < CB / kRows; ++u) v[u] = a.v[r0 + u * kRows][k];
#pragma unroll
  for (int cu = 0; cu < CB / kRows; ++cu)
    for (int cr = 0; cr < kRows; ++cr) {
      const int c = cu * kRows + cr;
      double2* sh = shared[c & 1];
      if (k == c) {
#pragma unroll
        for (int u = cu; u < CB / kRows; ++u)
          if (r0 + u * kRows >= c) sh[r0 + u * kRows] = v[u];
      } else if (r0 == cr && k < c) {
        sh[k] = v[cu];
      }
      __syncthreads();
      const double p = sh[c].x, ip = 1.0 / p;
      if (threadIdx.x == 0) {
        if (!(p > 0.0) && *bad == 0) *bad = 1 + base + c;
        pivot[c] = p;
      }
      // a_rk -= a_rc conj(a_kc) / p;  w_rk -= a_rc w_ck / p, with w_cc = 1 and w_rc = 0 so far
      double2 x = sh[k];
      if (k > c) x.y = -x.y;
      if (k == c) x = make_double2(1.0, 0.0);
#pragma unroll
      for (int u = cu; u < CB / kRows; ++u) {
        const int r = r0 + u * kRows;
        if (r <= c) continue;
        const double2 s = sh[r], l = make_double2(s.x * ip, s.y * ip);
        const double2 o = k == c ? make_double2(0.0, 0.0) : v[u];
        v[u] = make_double2(o.x - (l.x * x.x - l.y * x.y), o.y - (l.x * x.y + l.y * x.x));
      }
    }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < CB / kRows; ++u) {  // rows over sqrt(p_r); zero above the diagonal
    const int r = r0 + u * kRows;
    const double is = 1.0 / sqrt(pivot[r]);
    w.v[r][k] = k < r ? make_double2(v[u].x * is, v[u].y * is) : make_double2(k == r ? is : 0.0, 0.0);
  }
  __syncthreads();
}

// Workspace of one matrix: A [np][np] (lower blocks), L [np][np] (blocks below the diagonal), W
// [nblk][CB][CB], flags (one int); np = CB nblk.
struct CholWs {
  double2 *a, *l, *w;
  int* bad;
};
__host__ __device__ inline size_t chol_ws_elems(int nblk) {
  return 2 * (size_t)nblk * nblk * CB * CB + (size_t)nblk * CB * CB + 1;
}
__device__ __forceinline__ CholWs chol_ws(void* ws, int nblk, int batch) {
  double2* base = static_cast<double2*>(ws) + (size_t)batch * chol_ws_elems(nblk);
  const size_t nn = (size_t)nblk * nblk * CB * CB;
  return {base, base + nn, base + 2 * nn, reinterpret_cast<int*>(base + 2 * nn + (size_t)nblk * CB * CB)};
}
// row and column of the e-th block of a lower triangle
__device__ __forceinline__ void lower_block(int e, int& i, int& k) {
  i = 0;
  while ((i + 1) * (i + 2) / 2 <= e) ++i;
  k = e - i * (i + 1) / 2;
}

// A = (G + G^H) / 2 with the identity past `used` rows; block (0, 0) is factored.
template <typename C>
__global__ __launch_bounds__(CT) void k_chol_load(const C* __restrict__ g, int n, int nblk,
                                                  const int* __restrict__ used, void* __restrict__ ws) {
  __shared__ Tile a, w;
  __shared__ int bad;
  const int b = blockIdx.y, m = used ? used[b] : n, np = nblk * CB;
  int i, k;
  lower_block(blockIdx.x, i, k);
  const CholWs s = chol_ws(ws, nblk, b);
  const C* src = g + (long long)b * n * n;
  for (int e = threadIdx.x; e < CB * CB; e += CT) {
    const int r = i * CB + e / CB, c = k * CB + e % CB;
    double2 v = make_double2(r == c ? 1.0 : 0.0, 0.0);
    if (r < m && c < m) {
      const C x = src[(long long)r * n + c], y = src[(long long)c * n + r];
      v = make_double2(0.5 * ((double)x.x + (double)y.x), 0.5 * ((double)x.y - (double)y.y));
    }
    a.v[e / CB][e % CB] = v;
    if (blockIdx.x > 0) s.a[(long long)r * np + c] = v;
  }
  if (blockIdx.x > 0) return;
  if (threadIdx.x == 0) bad = 0;
  __syncthreads();
  factor_block(a, w, 0, &bad);
  for (int e = threadIdx.x; e < CB * CB; e += CT) s.w[e] = w.v[e / CB][e % CB];
  if (threadIdx.x == 0) *s.bad = bad;
}

__global__ __launch_bounds__(CT) void k_chol_step(int j, int nblk, void* __restrict__ ws) {
  __shared__ Tile w, x, li, lk;
  __shared__ int bad;
  const int np = nblk * CB;
  int i, k;
  lower_block(blockIdx.x, i, k);
  i += j + 1;
  k += j + 1;
  const CholWs s = chol_ws(ws, nblk, blockIdx.y);
  load_tile(w, s.w + (size_t)j * CB * CB, CB);
  load_tile(x, s.a + (long long)i * CB * np + j * CB, np);
  __syncthreads();
  doublex4 re = {0, 0, 0, 0}, im = {0, 0, 0, 0};
  block_product<true>(x, w, re, im);
  each_of_quarter(re, im, [&](int r, int c, double2 v) { li.v[r][c] = v; });
  if (i == k) {
    each_of_quarter(re, im, [&](int r, int c, double2 v) { s.l[(long long)(i * CB + r) * np + j * CB + c] = v; });
  } else {
    __syncthreads();
    load_tile(x, s.a + (long long)k * CB * np + j * CB, np);
    __syncthreads();
    re = {0, 0, 0, 0};
    im = {0, 0, 0, 0};
    block_product<true>(x, w, re, im);
    each_of_quarter(re, im, [&](int r, int c, double2 v) { lk.v[r][c] = v; });
  }
  __syncthreads();
  re = {0, 0, 0, 0};
  im = {0, 0, 0, 0};
  block_product<true>(li, i == k ? li : lk, re, im);
  double2* a = s.a + (long long)i * CB * np + k * CB;
  const bool next = i == j + 1 && k == j + 1;
  each_of_quarter(re, im, [&](int r, int c, double2 v) {
    const double2 o = a[(long long)r * np + c];
    const double2 d = make_double2(o.x - v.x, o.y - v.y);
    if (next)
      x.v[r][c] = d;
    else
      a[(long long)r * np + c] = d;
  });
  if (!next) return;
  if (threadIdx.x == 0) bad = *s.bad;
  __syncthreads();
  factor_block(x, w, (j + 1) * CB, &bad);
  for (int e = threadIdx.x; e < CB * CB; e += CT) s.w[(size_t)(j + 1) * CB * CB + e] = w.v[e / CB][e % CB];
  if (threadIdx.x == 0) *s.bad = bad;
}

// Block column j of X = L^{-1}: X_jj = W_j, X_ij = -W_i sum_{k < i} L_ik X_kj (X in A's workspace).
// stats of a matrix: status, trace of G's used part, then sum |X|^2 of each block column.
template <typename C>
__global__ __launch_bounds__(CT) void k_chol_inverse(const C* __restrict__ g, int n, int nblk,
                                                     const int* __restrict__ used, void* __restrict__ ws,
                                                     C* __restrict__ linv, double* __restrict__ stats) {
  __shared__ Tile t1, t2;
  __shared__ double red[CT / 64];
  const int j = blockIdx.x, b = blockIdx.y, m = used ? used[b] : n, np = nblk * CB;
  const CholWs s = chol_ws(ws, nblk, b);
  C* out = linv + (long long)b * n * n;
  double sum = 0.0;
  auto emit = [&](int r, int c, double2 v) {  // r, c in the whole matrix
    if (r >= n || c >= n) return;
    out[(long long)r * n + c] = cmake<C>((decltype(C::x))v.x, (decltype(C::x))v.y);
    if (r < m && c < m) sum += v.x * v.x + v.y * v.y;
  };
  for (int i = 0; i < j; ++i)
    for (int e = threadIdx.x; e < CB * CB; e += CT) emit(i * CB + e / CB, j * CB + e % CB, make_double2(0.0, 0.0));
  for (int e = threadIdx.x; e < CB * CB; e += CT) {
    const double2 v = s.w[(size_t)j * CB * CB + e];
    s.a[(long long)(j * CB + e / CB) * np + j * CB + e % CB] = v;
    emit(j * CB + e / CB, j * CB + e % CB, v);
  }
  for (int i = j + 1; i < nblk; ++i) {
    doublex4 re = {0, 0, 0, 0}, im = {0, 0, 0, 0};
    for (int k = j; k < i; ++k) {
      __syncthreads();  // the tiles of the product before, and X_kj written by this workgroup
      load_tile(t1, s.l + (long long)i * CB * np + k * CB, np);
      load_tile(t2, s.a + (long long)k * CB * np + j * CB, np);
      __syncthreads();
      block_product<false>(t1, t2, re, im);
    }
    __syncthreads();
    each_of_quarter(re, im, [&](int r, int c, double2 v) { t2.v[r][c] = v; });
    load_tile(t1, s.w + (size_t)i * CB * CB, CB);
    __syncthreads();
    re = {0, 0, 0, 0};
    im = {0, 0, 0, 0};
    block_product<false>(t1, t2, re, im);
    each_of_quarter(re, im, [&](int r, int c, double2 v) {
      v = make_double2(-v.x, -v.y);
      s.a[(long long)(i * CB + r) * np + j * CB + c] = v;
      emit(i * CB + r, j * CB + c, v);
    });
  }
  for (int off = 32; off > 0; off >>= 1) sum += __shfl_down(sum, off, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = sum;
  __syncthreads();
  if (threadIdx.x == 0) {
    double* st = stats + (long long)b * (nblk + 2);
    st[2 + j] = red[0] + red[1] + red[2] + red[3];
    if (j == 0) st[0] = (double)*s.bad;
  }
  if (j != 0) return;
  double tr = 0.0;  // trace of G's used part
  for (int r = threadIdx.x; r < m; r += CT) tr += (double)g[(long long)b * n * n + (long long)r * n + r].x;
  for (int off = 32; off > 0; off >>= 1) tr += __shfl_down(tr, off, 64);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = tr;
  __syncthreads();
  if (threadIdx.x == 0) stats[(long long)b * (nblk + 2) + 1] = red[0] + red[1] + red[2] + red[3];
}

// the larger of two values, NaN if either is
__device__ __forceinline__ double larger(double a, double b) { return b > a || b != b ? b : a; }

// rot = I - E/2 + 3 E^2 / 8 with E = (G + G^H)/2 - I, and the largest |component| of E per block row.
template <typename C>
__global__ __launch_bounds__(CT) void k_lowdin(const C* __restrict__ g, int n, int nblk, C* __restrict__ rot,
                                               double* __restrict__ emax) {
  __shared__ Tile t1, t2;
  __shared__ double red[CT / 64];
  const int i = blockIdx.x / nblk, j = blockIdx.x % nblk;
  auto element = [&](int r, int c) {
    double2 v = make_double2(0.0, 0.0);
    if (r < n && c < n) {
      const C x = g[(long long)r * n + c], y = g[(long long)c * n + r];
      v = make_double2(0.5 * ((double)x.x + (double)y.x) - (r == c ? 1.0 : 0.0), 0.5 * ((double)x.y - (double)y.y));
    }
    return v;
  };
  doublex4 re = {0, 0, 0, 0}, im = {0, 0, 0, 0};
  double big = 0.0;
  for (int k = 0; k < nblk; ++k) {
    __syncthreads();
    for (int e = threadIdx.x; e < CB * CB; e += CT) {
      const double2 a = element(i * CB + e / CB, k * CB + e % CB);
      t1.v[e / CB][e % CB] = a;
      t2.v[e / CB][e % CB] = element(k * CB + e / CB, j * CB + e % CB);
      if (j == 0) {
        big = larger(big, fabs(a.x));
        big = larger(big, fabs(a.y));
      }
    }
    __syncthreads();
    block_product<false>(t1, t2, re, im);
  }
  each_of_quarter(re, im, [&](int r, int c, double2 v) {
    r += i * CB;
    c += j * CB;
    if (r >= n || c >= n) return;
    const double2 e = element(r, c);
    rot[(long long)r * n + c] = cmake<C>((decltype(C::x))((r == c ? 1.0 : 0.0) - 0.5 * e.x + 0.375 * v.x),
                                         (decltype(C::x))(-0.5 * e.y + 0.375 * v.y));
  });
  if (j != 0) return;
  for (int off = 32; off > 0; off >>= 1) big = larger(big, __shfl_down(big, off, 64));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = big;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int q = 1; q < CT / 64; ++q) big = larger(big, red[q]);
    emax[i] = big;
  }
}

int failed(const char* what) {
  const hipError_t e = hipGetLastError();
  if (e == hipSuccess) return 0;
  set_error(std::string(what) + " launch: " + hipGetErrorString(e));
  return 1;
}

template <typename C>
int chol_t(const C* g, int n, const int* used, int batch, C* linv, double* stats, void* ws, hipStream_t s) {
  const int nblk = (n + CB - 1) / CB;
  hipLaunchKernelGGL(k_chol_load<C>, dim3(nblk * (nblk + 1) / 2, batch), dim3(CT), 0, s, g, n, nblk, used, ws);
  for (int j = 0; j + 1 < nblk; ++j) {
    const int t = nblk - 1 - j;
    hipLaunchKernelGGL(k_chol_step, dim3(t * (t + 1) / 2, batch), dim3(CT), 0, s, j, nblk, ws);
  }
  hipLaunchKernelGGL(k_chol_inverse<C>, dim3(nblk, batch), dim3(CT), 0, s, g, n, nblk, used, ws, linv, stats);
  return failed("chol_inverse");
}

}  // namespace

int chol_blocks(int n) { return (n + CB - 1) / CB; }
size_t chol_workspace_bytes(int n, int batch) { return (size_t)batch * chol_ws_elems(chol_blocks(n)) * sizeof(double2); }

int launch_chol_inverse(int prec, int n, const void* g, const int* used, int batch, void* linv, double* stats, void* ws,
                        hipStream_t s) {
  return prec == kFP64 ? chol_t(static_cast<const double2*>(g), n, used, batch, static_cast<double2*>(linv), stats, ws, s)
                       : chol_t(static_cast<const float2*>(g), n, used, batch, static_cast<float2*>(linv), stats, ws, s);
}

int launch_lowdin(int prec, int n, const void* g, void* rot, double* emax, hipStream_t s) {
  const int nblk = chol_blocks(n);
  if (prec == kFP64)
    hipLaunchKernelGGL(k_lowdin<double2>, dim3(nblk * nblk), dim3(CT), 0, s, (const double2*)g, n, nblk, (double2*)rot, emax);
  else
    hipLaunchKernelGGL(k_lowdin<float2>, dim3(nblk * nblk), dim3(CT), 0, s, (const float2*)g, n, nblk, (float2*)rot, emax);
  return failed("lowdin");
}

}  // namespace amt
