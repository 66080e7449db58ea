// Complex GEMM on the CDNA matrix cores (MFMA), FP32 and FP64.
//
// C = alpha * A op(B) + beta * C with row-major interleaved-complex operands and real
// alpha, beta. op = 0 (NN): B is K x N. op = 1 (NC): B is N x K and conj(B)^T is
// used -- the projector contraction <beta|psi> and every subspace overlap is of this
// form, with the reduction along the contiguous plane-wave axis of both operands.
//
// Complex arithmetic runs on the real matrix cores with Gauss's three-product form:
//   P1 += A_re B_re,  P2 += A_im B_im,  P3 += (A_re + A_im)(B_re + B_im)
//   C_re = P1 - P2,   C_im = P3 - P1 - P2
// i.e. three v_mfma_*_16x16x4 per 16x16x4 complex step instead of four (measured 12-27 %
// faster on every projector and subspace shape, with the same error against an FP64
// product: 2-6e-7 relative in FP32).
// The FP32 and FP64 instructions share one operand layout, so one template serves
// both on the input side: lane l supplies A[l % 16][l / 16] and B[l / 16][l % 16]. The
// accumulator differs (measured on gfx950): accumulator element q of lane l is
// D[4 (l / 16) + q][l % 16] for FP32 and D[l / 16 + 4 q][l % 16] for FP64.
//
// Tiling: a 256-thread workgroup computes 16 W rows x 64 columns, W = 1..5 (7 in FP32 without second
// sums, 4 in FP64 with them: registers) chosen for the row count (plan_gemm): each of the four wavefronts
// owns 16 columns and all 16 W rows, so 8 bands compute 16 rows, 45 compute 48 and 160 compute 160,
// where fixed 64-row tiles computed 64, 64 and 192. K advances 128 bytes of a row at a time (16 complex64, 8
// complex128) through two LDS buffers: the next tile's 16-byte global loads are issued before
// this tile's MFMAs and stored after them, one barrier per tile. Rows past M are clamped to the
// last row and columns of an NN product past N to the last ones (their results are not stored),
// so whole K tiles load without a test: a test per element had put a wait between the loads.
// Only the last, partial K tile of a chunk tests each element.
//
// LDS holds A (and B of an NC product, whose rows run along K too) as rows of 144 bytes: eight
// 16-byte chunks and 16 bytes of padding, which spreads the 16 rows that a fragment read touches
// over all banks. One 16-byte read gives a lane its fragment of one MFMA step in FP64 and of two
// in FP32: lane group g = lane / 16 reads chunk 4 p + g, i.e. the K index of step (p, s) is
// (4 p + g) * (16 / sizeof(C)) + s; any order of K is the same sum as long as A and B agree. B of
// an NN product stays [k][column], read 8 (16) bytes at a time from rows of 72 (64) elements.
//
// Accumulation over a long K is two-level: the MFMA's FP32 accumulators cover 64 to 256 of K
// (inner_sums()) and are then added into FP64 registers, so the rounding error of a long contraction
// (subspace overlaps over ~10^5 plane waves) grows with that length, not with K. One FP32 accumulator over
// all of K = 81k left relative errors of ~6e-5 in the Gram matrices of a 440-band Davidson,
// enough to stall an SCF. The additions cost 2 to 5 % of a product; split partials are summed in
// FP64 too. FP64 products of a middling K have second sums of the same kind.
//
// What bounds it: the matrix cores. Of a wavefront's cycles on 440 x 3852 x 40 000 (FP32, NC) 81 %
// are MFMA at the 2.14 GHz the chip holds under them. Measured (TFLOP/s at 8 real flops per
// complex multiply-add; in brackets 64- and 80-row tiles with a test per element):
//   FP32 160 x 1152 x 37073 NC 135 (118), 160 x 37073 x 1152 NN 128 (90), 640 x 160 x 37073 NC
//   122 (100), 45 x 3852 x 80989 NC 127 (84), 440 x 80989 x 3852 NN 149 (113), 440 x 3852 x 80989
//   NC 150 (107); FP64 160 x 1152 x 37073 NC 73 (46), its NN 76 (53), 45 x 3852 x 80989 NC 65 (39).
#include <array>
#include <climits>
#include <cmath>
#include <map>
#include <mutex>
#include <type_traits>

#include "kernels.hpp"

namespace amt {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef double doublex4 __attribute__((ext_vector_type(4)));

template <typename R>
struct Mfma;
template <>
struct Mfma<float> {
  using acc_t = floatx4;
  static __device__ __forceinline__ acc_t mma(float a, float b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lane, int q) { return (lane >> 4) * 4 + q; }
};
template <>
struct Mfma<double> {
  using acc_t = doublex4;
  static __device__ __forceinline__ acc_t mma(double a, double b, acc_t c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lane, int q) { return (lane >> 4) + 4 * q; }
};

constexpr int BN = 64;            // columns of a tile
constexpr int kChunks = 8;        // 16-byte chunks of one operand row and K tile

template <typename R>
struct Vec16;  // 16 bytes of a row: two complex64 or one complex128
template <>
struct Vec16<float> {
  typedef float T __attribute__((ext_vector_type(4)));
  typedef float U __attribute__((ext_vector_type(4), aligned(8)));  // rows start at any element
};
template <>
struct Vec16<double> {
  typedef double T __attribute__((ext_vector_type(2)));
  typedef double U __attribute__((ext_vector_type(2), aligned(16)));
};

template <typename R, int OP, bool kTwoLevel, int W>
__global__ __launch_bounds__(256, 2) void k_zgemm(int M, int N, int K, int kchunk, int nsplit,
                                               const typename Cplx<R>::T* __restrict__ A, long long lda,
                                               long long sA, const typename Cplx<R>::T* __restrict__ B,
                                               long long ldb, long long sB, typename Cplx<R>::T* __restrict__ Cm,
                                               long long ldc, long long sC, R alpha, R beta,
                                               typename Cplx<R>::T* __restrict__ part, int mfast, int flush_tiles) {
  using C = typename Cplx<R>::T;
  using acc_t = typename Mfma<R>::acc_t;
  using V = typename Vec16<R>::T;
  using VU = typename Vec16<R>::U;
  constexpr int E = 16 / sizeof(C);        // elements per chunk, MFMA steps per fragment read
  constexpr int BK = kChunks * E;          // K per tile
  constexpr int ROWS = 16 * W;
  constexpr int NA = (ROWS + 31) / 32;     // A chunks per thread
  constexpr int NB = 2;                    // B chunks per thread (64 x 8, or BK x 64 / E)
  constexpr int CPR = BN / E;              // chunks per K row of an NN product's B tile
  constexpr int LDB = sizeof(C) == 8 ? BN + 8 : BN;  // elements per K row of it in LDS
  constexpr int BSZ = OP == 0 ? BK * LDB * (int)sizeof(C) / 16 : BN * (kChunks + 1);
  __shared__ V As[2][ROWS][kChunks + 1];
  __shared__ V Bs[2][BSZ];
  // XCD-aware order: workgroups are handed to the 8 XCDs round-robin by linear id, so
  // logical tile t = (id % 8) * (T8 / 8) + id / 8 gives each XCD a contiguous run of tiles
  // that share an operand panel in its L2: the N-tiles of one M-tile and K-chunk (A panel),
  // or with mfast the M-tiles of one N-tile (B panel; NN products with few M-tiles).
  const unsigned gx = gridDim.x, gy = gridDim.y, gxy = gridDim.x * gridDim.y;
  const unsigned T = gxy * gridDim.z, T8 = T & ~7u;
  const unsigned id = blockIdx.x + gx * blockIdx.y + gxy * blockIdx.z;
  const unsigned tl = id < T8 ? (id & 7u) * (T8 >> 3) + (id >> 3) : id;
  const unsigned txy = tl % gxy;
  const int bz = (int)(tl / gxy);
  const int batch = bz / nsplit, split = bz % nsplit;
  const int m0 = (int)(mfast ? txy % gy : txy / gx) * ROWS, n0 = (int)(mfast ? txy / gy : txy % gx) * BN;
  const int kbeg = split * kchunk;
  const int kend = (kbeg + kchunk < K) ? kbeg + kchunk : K;
  A += (long long)batch * sA;
  B += (long long)batch * sB;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l15 = lane & 15, grp = lane >> 4;
  acc_t p1[W], p2[W], p3[W];  // Gauss's three products
#pragma unroll
  for (int a = 0; a < W; ++a)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      p1[a][q] = 0;
      p2[a][q] = 0;
      p3[a][q] = 0;
    }
  // C_re and C_im of one accumulator element; conj(B) turns the signs of the P2 terms
  auto re_of = [](auto t1, auto t2) { return OP == 0 ? t1 - t2 : t1 + t2; };
  auto im_of = [](auto t1, auto t2, auto t3) { return OP == 0 ? t3 - t1 - t2 : t3 - t1 + t2; };
  // second-level FP64 sums of the accumulators (two-level form only)
  double sumr[kTwoLevel ? W : 1][4], sumi[kTwoLevel ? W : 1][4];
  auto flush = [&]() {
    if constexpr (kTwoLevel) {
#pragma unroll
      for (int a = 0; a < W; ++a)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const double t1 = p1[a][q], t2 = p2[a][q], t3 = p3[a][q];
          sumr[a][q] += re_of(t1, t2);
          sumi[a][q] += im_of(t1, t2, t3);
          p1[a][q] = 0;
          p2[a][q] = 0;
          p3[a][q] = 0;
        }
    }
  };
  if constexpr (kTwoLevel) {
#pragma unroll
    for (int a = 0; a < W; ++a)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        sumr[a][q] = 0.0;
        sumi[a][q] = 0.0;
      }
  }
  // A chunk (row, c): id = tid + 256 u, row = id / 8, c = id % 8. The first K tile's addresses.
  const C* pa[NA];
#pragma unroll
  for (int u = 0; u < NA; ++u) {
    const int row = m0 + tid / kChunks + 32 * u;
    pa[u] = A + (long long)(row < M ? row : M - 1) * lda + kbeg + (tid % kChunks) * E;
  }
  const C* pb[NB];
#pragma unroll
  for (int u = 0; u < NB; ++u) {
    if constexpr (OP == 0) {
      const int e = tid + 256 * u, k = e / CPR, c = n0 + (e % CPR) * E;
      pb[u] = B + (long long)(kbeg + k) * ldb + c;
    } else {
      const int col = n0 + tid / kChunks + 32 * u;
      pb[u] = B + (long long)(col < N ? col : N - 1) * ldb + kbeg + (tid % kChunks) * E;
    }
  }
  const long long stepb = OP == 0 ? (long long)BK * ldb : BK;
  // Column chunks of an NN tile past N read the last E columns instead; one that starts at the
  // last column (FP32, N - n0 odd) finds it in its second element.
  bool last_col[NB];
#pragma unroll
  for (int u = 0; u < NB; ++u) {
    const int c = n0 + ((tid + 256 * u) % CPR) * E;
    last_col[u] = OP == 0 && E == 2 && N >= E && c == N - 1;
    if (OP == 0 && c > N - E && N >= E) pb[u] -= c - (N - E);
  }
  V ra[NA], rb[NB];
  // whole K tile: no test, so the loads of a tile are all in flight together
  auto gload = [&]() {
#pragma unroll
    for (int u = 0; u < NA; ++u) {
      if (ROWS % 32 == 0 || u < NA - 1 || tid < 128) ra[u] = *reinterpret_cast<const VU*>(pa[u]);
      pa[u] += BK;
    }
#pragma unroll
    for (int u = 0; u < NB; ++u) {
      rb[u] = *reinterpret_cast<const VU*>(pb[u]);
      pb[u] += stepb;
    }
  };
  // the last K tile of a chunk (and every tile of a one-column FP32 NN product): element by
  // element, zeros past kend
  auto gload_tail = [&](int k0) {
    const int left = kend - k0 - (tid % kChunks) * E;  // elements of this thread's row chunk that exist
    auto some = [](const C* q, int have) {
      V v;
#pragma unroll
      for (int e = 0; e < E; ++e) {
        C x = cmake<C>(0, 0);
        if (e < have) x = q[e];
        v[2 * e] = x.x;
        v[2 * e + 1] = x.y;
      }
      return v;
    };
#pragma unroll
    for (int u = 0; u < NA; ++u) {
      if (ROWS % 32 == 0 || u < NA - 1 || tid < 128) ra[u] = some(pa[u], left);
      pa[u] += BK;
    }
#pragma unroll
    for (int u = 0; u < NB; ++u) {
      if constexpr (OP == 0) {
        const int e = tid + 256 * u, c = n0 + (e % CPR) * E;
        rb[u] = some(pb[u], k0 + e / CPR < kend ? (N >= E ? E : N - c) : 0);
      } else {
        rb[u] = some(pb[u], left);
      }
      pb[u] += stepb;
    }
  };
  auto sstore = [&](int buf) {
#pragma unroll
    for (int u = 0; u < NA; ++u)
      if (ROWS % 32 == 0 || u < NA - 1 || tid < 128) As[buf][tid / kChunks + 32 * u][tid % kChunks] = ra[u];
#pragma unroll
    for (int u = 0; u < NB; ++u) {
      if constexpr (OP == 0) {
        const int e = tid + 256 * u;
        V v = rb[u];
        if constexpr (E == 2) {
          v[0] = last_col[u] ? v[2] : v[0];
          v[1] = last_col[u] ? v[3] : v[1];
        }
        Bs[buf][(e / CPR) * (LDB / E) + e % CPR] = v;
      } else {
        Bs[buf][(tid / kChunks + 32 * u) * (kChunks + 1) + tid % kChunks] = rb[u];
      }
    }
  };
  // the fragments of steps (p, 0 .. E - 1) and their MFMAs
  struct Frag {
    V a[W], b;
  };
  auto fragments = [&](Frag& f, int buf, int p) {
#pragma unroll
    for (int r = 0; r < W; ++r) f.a[r] = As[buf][r * 16 + l15][p * 4 + grp];
    if constexpr (OP == 0) {
      const C* bs = reinterpret_cast<const C*>(&Bs[buf][0]) + (p * 4 + grp) * E * LDB + wave * 16 + l15;
#pragma unroll
      for (int s = 0; s < E; ++s) {
        const C b = bs[s * LDB];
        f.b[2 * s] = b.x;
        f.b[2 * s + 1] = b.y;
      }
    } else {
      f.b = Bs[buf][(wave * 16 + l15) * (kChunks + 1) + p * 4 + grp];
    }
  };
  auto products = [&](const Frag& f) {
#pragma unroll
    for (int s = 0; s < E; ++s) {
      const R bx = f.b[2 * s], by = f.b[2 * s + 1], bz2 = OP == 0 ? bx + by : bx - by;
#pragma unroll
      for (int r = 0; r < W; ++r) {
        const R ax = f.a[r][2 * s], ay = f.a[r][2 * s + 1];
        p1[r] = Mfma<R>::mma(ax, bx, p1[r]);
        p2[r] = Mfma<R>::mma(ay, by, p2[r]);
        p3[r] = Mfma<R>::mma(ax + ay, bz2, p3[r]);
      }
    }
  };
  const int nt = kbeg < kend ? (kend - kbeg + BK - 1) / BK : 0;                 // K tiles
  const int nfull = OP == 0 && N < E ? 0 : (kbeg < kend ? (kend - kbeg) / BK : 0);  // of which whole
  auto gload_tile = [&](int tile) {
    if (tile < nfull)
      gload();
    else if (tile < nt)
      gload_tail(kbeg + tile * BK);
  };
  // A tile's turn: its first fragments are in f0 and the next tile's values in ra, rb. The next
  // tile goes to the other buffer and its successor's loads are issued; the barrier that makes it
  // visible and the read of its first fragments lie between the two halves of the MFMAs.
  Frag f0, f1;
  int buf = 0, tile = 0, until_flush = flush_tiles;
  auto step = [&](auto load, bool more) {
    fragments(f1, buf, 1);
    if (more) sstore(buf ^ 1);
    load();
    products(f0);
    __syncthreads();
    buf ^= 1;
    if (more) fragments(f0, buf, 0);
    products(f1);
    ++tile;
    if constexpr (kTwoLevel) {
      if (--until_flush == 0) {
        flush();
        until_flush = flush_tiles;
      }
    }
  };
  if (nt > 0) {
    gload_tile(0);
    sstore(0);
    gload_tile(1);
    __syncthreads();
    fragments(f0, 0, 0);
    while (tile + 2 < nfull) step(gload, true);
    while (tile < nt) step([&] { gload_tile(tile + 2); }, tile + 1 < nt);
  }
  flush();
#pragma unroll
  for (int r = 0; r < W; ++r)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int row = m0 + r * 16 + Mfma<R>::row(lane, q);
      const int col = n0 + wave * 16 + l15;
      if (row < M && col < N) {
        C v;
        if constexpr (kTwoLevel)
          v = cmake<C>((R)sumr[r][q], (R)sumi[r][q]);
        else
          v = cmake<C>(re_of(p1[r][q], p2[r][q]), im_of(p1[r][q], p2[r][q], p3[r][q]));
        if (part) {
          part[(((long long)batch * nsplit + split) * M + row) * N + col] = v;
        } else {
          C* dst = Cm + (long long)batch * sC + (long long)row * ldc + col;
          C o = cmake<C>(alpha * v.x, alpha * v.y);
          if (beta != (R)0) {
            const C old = *dst;
            o.x += beta * old.x;
            o.y += beta * old.y;
          }
          *dst = o;
        }
      }
    }
}

// Sum of the split partials in FP64: each output element is summed by kReduceGroups threads
// (splits g, g + kReduceGroups, ...) whose partial sums are added in a fixed order, so a
// product's result does not depend on scheduling; 32 consecutive elements per group keep the
// loads of one split contiguous.
constexpr int kReduceGroups = 8, kReduceCols = 32;

template <typename R>
__global__ __launch_bounds__(kReduceGroups * kReduceCols) void k_splitk_reduce(
    int M, int N, int nsplit, const typename Cplx<R>::T* __restrict__ part, typename Cplx<R>::T* __restrict__ Cm,
    long long ldc, long long sC, R alpha, R beta) {
  using C = typename Cplx<R>::T;
  __shared__ double red[kReduceGroups][kReduceCols][2];
  const int g = threadIdx.x / kReduceCols, el = threadIdx.x % kReduceCols;
  const long long mn = (long long)M * N;
  const long long e = (long long)blockIdx.x * kReduceCols + el;
  const int batch = blockIdx.y;
  double sr = 0, si = 0;
  if (e < mn) {
    const C* p = part + (long long)batch * nsplit * mn + e;
#pragma unroll 4
    for (int s = g; s < nsplit; s += kReduceGroups) {
      const C v = p[(long long)s * mn];
      sr += v.x;
      si += v.y;
    }
  }
  red[g][el][0] = sr;
  red[g][el][1] = si;
  __syncthreads();
  if (g != 0 || e >= mn) return;
  for (int q = 1; q < kReduceGroups; ++q) {
    sr += red[q][el][0];
    si += red[q][el][1];
  }
  const int row = (int)(e / N), col = (int)(e % N);
  C* dst = Cm + (long long)batch * sC + (long long)row * ldc + col;
  C o = cmake<C>((R)(alpha * sr), (R)(alpha * si));
  if (beta != (R)0) {
    const C old = *dst;
    o.x += beta * old.x;
    o.y += beta * old.y;
  }
  *dst = o;
}

// ----------------------------------------------------------------------- choices
static std::mutex g_split_mutex;
static std::map<std::array<int, 6>, int> g_split_table;

static std::array<int, 6> split_key(int prec, int op, int m, int n, int k, int batch) {
  return {prec, op, (m + 63) / 64, (n + 63) / 64, (k + 255) / 256, batch};
}

// Longest K that one accumulator covers without second sums, and K between the additions into them
// beyond it. A product's rounding grows with the accumulator's length, so the length follows
// from the shape and not from the split that happens to be fastest:
//   NC (overlaps, projections: K the plane waves): 256; up to 4096 of K 128, as a few splits of at
//     most 256 that divide such a K are shorter than that themselves; 64 for outputs of 512 tiles of
//     64 x 64 and more, whose K is not split at all.
//   NN (rotations, projector applications): 128 beyond 256 of K, 64 beyond 1024. Outputs of 512
//     tiles of 80 x 64 and more keep one accumulator up to 1024: the rotations of a whole subspace,
//     bound by the matrix cores (160 x 37 073 x 480: 154 us, with additions every 64 of K 168).
// Measured with random operands: the projector applications 40 x 9300 x 288, 58 x 13 900 x 432 and
// 80 x 18 500 x 576 are off by 2.8, 2.8 and 2.9e-7 in 15.2, 32.5 and 59.7 us, with one accumulator
// over all of K by 4.4, 5.3 and 6.1e-7 in 14.7, 31.7 and 55.3, with additions every 64 of K by 2.1e-7
// in 15.5, 33.4 and 61.0. NC products of K > 4096 with additions every 64: 2.1e-7 for 3.9e-7, 3 to 8 %
// slower.
// FP64: 192, then additions every 160 of K, where the output has fewer than 512 tiles of 80 x 64 and
// K is 257 to 1024 (NN) or 16 384 (NC). Past these the products of a whole subspace and the
// projections of 10^5 plane waves, bound by the matrix cores, keep one accumulator per split. Error
// (1e-16) and time, with single accumulators and so: NN 58 x 13 900 x 432 10.4 in 56.2 us and 5.9 in
// 57.2, 80 x 18 500 x 576 10.3 in 109 and 5.4 in 112, 80 x 18 500 x 1000 15.7 in 188 and 5.7 in 202;
// NC 5 of 19 x 1381 x 355 8.7 in 20.9 and 5.5 in 21.5, 16 of 64 x 144 x 4954 8.8 in 118 and 6.1 in
// 121, 4 of 40 x 288 x 9300 7.9 in 73.5 and 5.8 in 76.6.
struct InnerSums {
  int limit, flush;
};
static InnerSums inner_sums(int prec, int op, int m, int n, int k, int batch) {
  auto tiles = [&](int rows) { return (long long)((m + rows - 1) / rows) * ((n + BN - 1) / BN) * batch; };
  if (prec == kFP64) return {k > 256 && k <= (op == 0 ? 1024 : 16384) && tiles(80) < 512 ? 192 : INT_MAX, 160};
  if (op == 0) return {k <= 256 || (k <= 1024 && tiles(80) >= 512) ? 1024 : 0, k <= 1024 ? 128 : 64};
  const int flush = k > 1024 && tiles(64) >= 512 ? 64 : k > 4096 ? 256 : 128;
  return {k <= 256 ? 256 : flush, flush};
}
constexpr int kMinChunk = 64;
// FP32 NC products with both output sides at least this are left alone by the split tuning.
constexpr int kBigSide = 256;

// Tile rows in 16s, widest kernel of each kind (registers: two wavefronts per SIMD).
constexpr int kMaxW = 7, kMaxWLong = 5, kMaxW64 = 5, kMaxW64Long = 4;

struct GemmPlan {
  int w;        // rows of a tile in 16s
  int ns;       // K splits
  int kchunk;   // K per split, a multiple of the K tile
  bool two;     // second-level sums
  int flush;    // K tiles between them
};

static bool split_is_tunable(int prec, int op, int m, int n, int k) {
  return !(prec == kFP32 && op == 1 && m >= kBigSide && n >= kBigSide && k > 0);
}

// W and the split along K, by the time a plan takes in units of one 16-row K tile of one
// workgroup (0.18 us: 12 MFMAs of 32 or 6 of 64 cycles in each wavefront):
//   (ceil(workgroups / 256 CUs) + 0.8) * (K tiles + 2) * (W + 0.35)  + the partials' traffic,
// the 2 standing for a workgroup's start and end, the 0.35 for a tile's work beside its rows
// (barrier, B operand) and the 0.8 for the last workgroups of a CU, which have fewer wavefronts
// beside them to hide their waits (so a few long workgroups per CU lose to more, shorter ones).
// The first factor is what uneven rounds cost: 160 x 37 073 x 1152 (580
// column tiles) in 32-row tiles fills its last round better than in 80-row ones. Against a sweep
// of every W and split the choice is within 5 % on the Si8, Si64 and Si214 shapes.
// No split lengthens an accumulator past inner_sums(): 3.7-4.1e-7 (relative norm, random operands) on
// every NC shape above, where single accumulators over 256 to 1024 of K gave 4.1 to 7.9e-7.
static GemmPlan plan_gemm(int prec, int op, int m, int n, int k, int batch) {
  const int csize = prec == kFP64 ? 16 : 8, bk = kChunks * 16 / csize;
  const double cols = (double)((n + BN - 1) / BN) * batch, out = (double)m * n * batch * csize;
  const InnerSums sums = inner_sums(prec, op, m, n, k, batch);
  GemmPlan best{1, 1, bk, false, sums.flush / bk};
  double best_cost = 1e300;
  int lo = 1, hi = (k + kMinChunk - 1) / kMinChunk;
  hi = hi > 256 ? 256 : hi < 1 ? 1 : hi;
  if (split_is_tunable(prec, op, m, n, k)) {
    std::lock_guard<std::mutex> lock(g_split_mutex);
    auto it = g_split_table.find(split_key(prec, op, m, n, k, batch));
    if (it != g_split_table.end()) lo = hi = it->second < hi ? it->second : hi;
  }
  const auto widest = [&](bool two) { return prec == kFP64 ? (two ? kMaxW64Long : kMaxW64) : two ? kMaxWLong : kMaxW; };
  double rows[kMaxW + 1];
  for (int w = 1; w <= kMaxW; ++w) rows[w] = (double)((m + 16 * w - 1) / (16 * w)) * cols;
  for (int want = lo; want <= hi; want += 1 + want / 8) {
    int kchunk = ((k + want - 1) / want + bk - 1) / bk * bk;
    if (kchunk < bk) kchunk = bk;
    const int ns = k > 0 ? (k + kchunk - 1) / kchunk : 1;
    if (best_cost < 1e300 && (long long)batch * ns > 65535) break;
    const bool two = (op == 1 || prec == kFP64 ? kchunk : k) > sums.limit;
    const double tiles = kchunk / bk + 2, extra = ns > 1 ? 20.0 + 2.0 * out * ns / 1.3e6 : 0.0;
    for (int w = 1; w <= widest(two); ++w) {
      const double cost =
          (std::ceil(rows[w] * ns / 256.0) + 0.8) * tiles * (w + 0.35) * (two && prec == kFP32 ? 1.1 : 1.0) + extra;
      if (cost < best_cost) {
        best_cost = cost;
        best.w = w;
        best.ns = ns;
        best.kchunk = kchunk;
        best.two = two;
      }
    }
  }
  return best;
}

int set_zgemm_split(int prec, int op, int m, int n, int k, int batch, int split) {
  if (split < 0 || split > 256) {
    set_error("zgemm split must be 0 (heuristic) .. 256");
    return 1;
  }
  if (!split_is_tunable(prec, op, m, n, k)) return 2;
  std::lock_guard<std::mutex> lock(g_split_mutex);
  const auto key = split_key(prec, op, m, n, k, batch);
  if (split == 0)
    g_split_table.erase(key);
  else
    g_split_table[key] = split;
  return 0;
}

size_t zgemm_workspace_bytes(int prec, int op, int m, int n, int k, int batch) {
  const GemmPlan g = plan_gemm(prec, op, m, n, k, batch);
  if (g.ns <= 1) return 0;
  const size_t c = prec == kFP64 ? 16 : 8;
  return (size_t)batch * g.ns * m * n * c;
}

// Splits summed and contracted in one launch, for small products: out = P D with P the sum of the
// partials (FP64 sums rounded to R, as k_splitk_reduce stores them) and D real, block-diagonal
// over atoms. A workgroup takes, of one row, the columns whose atom block starts in its
// kDijCols: with blocks of up to 33 columns it sums at most kDijPass columns, each summed by one
// workgroup only, and keeps them in LDS. Bound by the launch and one chain of loads: 5.9 us for
// 8 x 36 in 12 splits, where k_splitk_reduce and k_dij take 4 and 5.4 and a gap between them (H.psi
// of 2 atoms 37 -> 31 us with the fill of H.psi gone as well). Past one workgroup per CU the two
// kernels, with more wavefronts in flight, win: 7.7 + 6.1 us against 35-44 for 16 x 64 x 144, 17.3 +
// 6.2 against 45 for 160 x 1152.
constexpr long long kDijFuse = 256;  // workgroups
constexpr int kDijCols = 96, kDijPass = 128, kDijGroups = kReduceGroups / 2;

template <typename R>
__global__ __launch_bounds__(kDijGroups * kDijPass) void k_splitk_dij(
    int M, int N, int nsplit, const typename Cplx<R>::T* __restrict__ part, const R* __restrict__ D, long long sD,
    const int* __restrict__ blk_start, const int* __restrict__ blk_len, typename Cplx<R>::T* __restrict__ out,
    long long sO) {
  using C = typename Cplx<R>::T;
  __shared__ double red[kReduceGroups][kDijPass][2];
  __shared__ C sum[kDijPass];
  __shared__ int reach[kDijPass / 64];
  const int g = threadIdx.x / kDijPass, el = threadIdx.x % kDijPass;
  const int row = blockIdx.y, batch = blockIdx.z, first = blockIdx.x * kDijCols;
  const long long mn = (long long)M * N;
  const C* p = part + (long long)batch * nsplit * mn + (long long)row * N;
  for (int w0 = first; w0 < N; w0 += kDijPass) {  // a second window for longer blocks only
    if (w0 > first && blk_start[w0] >= first + kDijCols) break;
    const int col = w0 + el;
    const int j0 = col < N ? blk_start[col] : N;
    const bool own = col < N && j0 >= first && j0 < first + kDijCols;
    const int j1 = own ? j0 + blk_len[col] : 0;
    int hi = j1;
    for (int o = 32; o > 0; o >>= 1) hi = max(hi, __shfl_xor(hi, o, 64));
    if (g == 0 && (el & 63) == 0) reach[el >> 6] = hi;
    __syncthreads();
    for (int q = 0; q < kDijPass / 64; ++q) hi = max(hi, reach[q]);
    const R* d = D + batch * sD + col;
    R sr = 0, si = 0;
    for (int base = first; base < hi; base += kDijPass) {  // columns any owned block may hold
      const int c = base + el;
      double xr = 0, xi = 0, yr = 0, yi = 0;  // k_splitk_reduce's groups g and g + kDijGroups
      if (c < hi)
#pragma unroll 4
        for (int s = g; s < nsplit; s += kReduceGroups) {
          const C v = p[(long long)s * mn + c];
          const C u = s + kDijGroups < nsplit ? p[(long long)(s + kDijGroups) * mn + c] : cmake<C>(0, 0);
          xr += v.x;
          xi += v.y;
          yr += u.x;
          yi += u.y;
        }
      red[g][el][0] = xr;
      red[g][el][1] = xi;
      red[g + kDijGroups][el][0] = yr;
      red[g + kDijGroups][el][1] = yi;
      __syncthreads();
      if (g == 0) {
        for (int q = 1; q < kReduceGroups; ++q) {
          xr += red[q][el][0];
          xi += red[q][el][1];
        }
        sum[el] = cmake<C>((R)xr, (R)xi);
      }
      __syncthreads();
      if (g == 0 && own)
#pragma unroll 4
        for (int j = max(j0, base); j < min(j1, base + kDijPass); ++j) {
          const R dj = d[(long long)j * N];
          sr += sum[j - base].x * dj;
          si += sum[j - base].y * dj;
        }
      __syncthreads();
    }
    if (g == 0 && own) out[batch * sO + (long long)row * N + col] = cmake<C>(sr, si);
    __syncthreads();
  }
}

int launch_dij(int prec, const void* P, const void* D, const int* blk_start, const int* blk_len, void* out, int nrow,
               int nproj, long long sP, long long sD, long long sO, int batch, hipStream_t s);

template <typename R>
static int zgemm_t(int op, int m, int n, int k, double alpha, const void* a, long long lda, long long sa,
                   const void* b, long long ldb, long long sb, double beta, void* c, long long ldc, long long sc,
                   int batch, void* ws, size_t ws_bytes, hipStream_t s, const DijArgs* dij = nullptr) {
  using C = typename Cplx<R>::T;
  if (m <= 0 || n <= 0 || batch <= 0) return 0;
  const GemmPlan g = plan_gemm(std::is_same<R, double>::value ? kFP64 : kFP32, op, m, n, k, batch);
  const int ns = g.ns, kchunk = g.kchunk;
  const size_t need = ns > 1 ? (size_t)batch * ns * m * n * sizeof(C) : 0;
  C* part = nullptr;
  if (ns > 1) {
    if (ws == nullptr || ws_bytes < need) {
      set_error("zgemm: split-K workspace too small (" + std::to_string(ws_bytes) + " < " + std::to_string(need) +
                ")");
      return 1;
    }
    part = static_cast<C*>(ws);
  }
  if ((long long)batch * ns > 65535) {
    set_error("zgemm: batch x split exceeds the grid limit");
    return 1;
  }
  const dim3 grid((n + BN - 1) / BN, (m + 16 * g.w - 1) / (16 * g.w), batch * ns);
  const int mfast = op == 0 && grid.y > 1 && grid.x >= grid.y;
  C* const p = ns > 1 ? part : nullptr;
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(256), 0, s, m, n, k, kchunk, ns, (const C*)a, lda, sa, (const C*)b, ldb, sb,
                       (C*)c, ldc, sc, (R)alpha, (R)beta, p, mfast, g.flush);
  };
#define AMT_W(TWO, W)                \
  case W:                            \
    if (op == 0)                     \
      launch(k_zgemm<R, 0, TWO, W>); \
    else                             \
      launch(k_zgemm<R, 1, TWO, W>); \
    break;
  if constexpr (std::is_same<R, float>::value) {
    if (g.two) {
      switch (g.w) { AMT_W(true, 1) AMT_W(true, 2) AMT_W(true, 3) AMT_W(true, 4) AMT_W(true, 5) }
    } else {
      switch (g.w) {
        AMT_W(false, 1) AMT_W(false, 2) AMT_W(false, 3) AMT_W(false, 4) AMT_W(false, 5) AMT_W(false, 6)
        AMT_W(false, 7)
      }
    }
  } else {
    if (g.two) {
      switch (g.w) { AMT_W(true, 1) AMT_W(true, 2) AMT_W(true, 3) AMT_W(true, 4) }
    } else {
      switch (g.w) { AMT_W(false, 1) AMT_W(false, 2) AMT_W(false, 3) AMT_W(false, 4) AMT_W(false, 5) }
    }
  }
#undef AMT_W
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    set_error(std::string("zgemm launch: ") + hipGetErrorString(e));
    return 1;
  }
  const bool fuse = dij && ns > 1 && (long long)((n + kDijCols - 1) / kDijCols) * m * batch <= kDijFuse;
  if (fuse) {
    hipLaunchKernelGGL((k_splitk_dij<R>), dim3((n + kDijCols - 1) / kDijCols, m, batch),
                       dim3(kDijGroups * kDijPass), 0, s, m, n, ns, (const C*)part, (const R*)dij->d, dij->sd,
                       dij->blk_start, dij->blk_len, (C*)dij->out, dij->so);
    e = hipGetLastError();
    if (e != hipSuccess) {
      set_error(std::string("zgemm contraction launch: ") + hipGetErrorString(e));
      return 1;
    }
  } else if (ns > 1) {
    const long long mn = (long long)m * n;
    hipLaunchKernelGGL((k_splitk_reduce<R>), dim3((unsigned)((mn + kReduceCols - 1) / kReduceCols), batch),
                       dim3(kReduceGroups * kReduceCols), 0, s, m, n, ns, (const C*)part, (C*)c, ldc, sc, (R)alpha,
                       (R)beta);
    e = hipGetLastError();
    if (e != hipSuccess) {
      set_error(std::string("zgemm reduce launch: ") + hipGetErrorString(e));
      return 1;
    }
  }
  if (dij && !fuse)
    return launch_dij(std::is_same<R, double>::value ? kFP64 : kFP32, c, dij->d, dij->blk_start, dij->blk_len, dij->out,
                      m, n, sc, dij->sd, dij->so, batch, s);
  return 0;
}

int launch_zgemm(int prec, int op, int m, int n, int k, double alpha, const void* a, long long lda, long long sa,
                 const void* b, long long ldb, long long sb, double beta, void* c, long long ldc, long long sc,
                 int batch, void* ws, size_t ws_bytes, hipStream_t s) {
  return prec == kFP64 ? zgemm_t<double>(op, m, n, k, alpha, a, lda, sa, b, ldb, sb, beta, c, ldc, sc, batch, ws,
                                         ws_bytes, s)
                       : zgemm_t<float>(op, m, n, k, alpha, a, lda, sa, b, ldb, sb, beta, c, ldc, sc, batch, ws,
                                        ws_bytes, s);
}

int launch_zgemm_dij(int prec, int m, int n, int k, const void* a, long long lda, long long sa, const void* b,
                     long long ldb, long long sb, void* proj, const DijArgs& dij, int batch, void* ws, size_t ws_bytes,
                     hipStream_t s) {
  return prec == kFP64 ? zgemm_t<double>(1, m, n, k, 1.0, a, lda, sa, b, ldb, sb, 0.0, proj, n, (long long)m * n, batch,
                                         ws, ws_bytes, s, &dij)
                       : zgemm_t<float>(1, m, n, k, 1.0, a, lda, sa, b, ldb, sb, 0.0, proj, n, (long long)m * n, batch,
                                        ws, ws_bytes, s, &dij);
}

}  // namespace amt
