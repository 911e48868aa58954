// Strided-batched FP64 GEMM on the matrix cores (v_mfma_f64_16x16x4f64),
// column-major like BLAS:  C[g] = alpha op(A[g]) op(B[g]) + beta C[g].
// Used by the Schwarz local factorisations (updates of block columns and of
// what lies right of a panel, the blocked triangular solves), whose operands
// are blocks of 64 to 512 columns of matrices up to tens of thousands of rows,
// and by the FMM's compression.
//
// One workgroup (4 wavefronts) computes a 64 x 64 tile of C; each wavefront a
// 32 x 32 quarter as 2 x 2 blocks of 16 x 16.  The k dimension is staged in
// LDS 16 at a time (op(A) as [k][m], op(B) as [k][n]), the next stage's
// global loads issued before the current stage's products.  The products are
// formed transposed (C^T = op(B)^T op(A)^T): lane l supplies op(B)[k][n] as
// the A fragment and op(A)[m][k] as the B fragment (A fragment: row l % 16,
// k l / 16; B fragment: k l / 16, column l % 16), so accumulator register v
// of lane l holds C[m = l % 16][n = l / 16 + 4 v] and the 16 lanes of a
// group store 16 consecutive rows of a column (128 contiguous bytes).
//
// lower_only skips the tiles that lie strictly above the diagonal (a
// symmetric trailing update whose upper triangle is never read).  C may be A
// or B where a workgroup's tile reads only the rows or columns
// that it writes (one tile across the other dimension): all its loads come
// before its stores.  In large batches all tiles of one matrix run on one XCD
// (blocks go to the 8 XCDs round robin), whose L2 then holds the operand they
// share; a few matrices would leave XCDs idle that way.
#include "common.hpp"
#include "solvers.hpp"

namespace {

typedef double f64x4 __attribute__((ext_vector_type(4)));

constexpr int kT = 64;   // tile side
constexpr int kK = 16;   // k per LDS stage
constexpr int kLd = kT + 1;

template <bool TA, bool TB>
__global__ __launch_bounds__(256) void k_dgemm(int M, int N, int K, double alpha,
                                               const double *A, int lda, int64_t sA,
                                               const double *B, int ldb, int64_t sB, double beta,
                                               double *C, int ldc, int64_t sC, int tiles_m,
                                               int tiles, int batch, int xcds, int from_c,
                                               int lower_only) {
  __shared__ double As[kK][kLd];  // op(A)[m][k] stored [k][m]
  __shared__ double Bs[kK][kLd];  // op(B)[k][n] stored [k][n]
  const int q = int(blockIdx.x) / xcds;
  const int g = (q / tiles) * xcds + int(blockIdx.x) % xcds;
  if (g >= batch) return;  // uniform over the workgroup
  const int tm = (q % tiles) % tiles_m, tn = (q % tiles) / tiles_m;
  const int m0 = tm * kT, n0 = tn * kT;
  if (lower_only && m0 + kT - 1 < n0) return;  // uniform over the workgroup
  A += int64_t(g) * sA;
  B += int64_t(g) * sB;
  C += int64_t(g) * sC;
  const int t = threadIdx.x;
  const int lane = t & 63, wave = t >> 6;
  const int wm = (wave & 1) * 32, wn = (wave >> 1) * 32;

  // global -> register staging of one k stage: 4 elements of each operand
  // per thread, coalesced along the operand's contiguous dimension
  double ra[4], rb[4];
  auto load = [&](int k0) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      int m, k;
      if (!TA) { m = t & 63; k = (t >> 6) + 4 * i; }   // A[m + k lda], m fastest
      else { k = t & 15; m = (t >> 4) + 16 * i; }       // A[k + m lda], k fastest
      const int gm = m0 + m, gk = k0 + k;
      double v = 0.0;
      if (gm < M && gk < K) v = TA ? A[int64_t(gm) * lda + gk] : A[int64_t(gk) * lda + gm];
      ra[i] = v;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      int n, k;
      if (!TB) { k = t & 15; n = (t >> 4) + 16 * i; }   // B[k + n ldb], k fastest
      else { n = t & 63; k = (t >> 6) + 4 * i; }        // B[n + k ldb], n fastest
      const int gn = n0 + n, gk = k0 + k;
      double v = 0.0;
      if (gn < N && gk < K) v = TB ? B[int64_t(gk) * ldb + gn] : B[int64_t(gn) * ldb + gk];
      rb[i] = v;
    }
  };
  auto store = [&]() {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (!TA) As[(t >> 6) + 4 * i][t & 63] = ra[i];
      else As[t & 15][(t >> 4) + 16 * i] = ra[i];
      if (!TB) Bs[t & 15][(t >> 4) + 16 * i] = rb[i];
      else Bs[(t >> 6) + 4 * i][t & 63] = rb[i];
    }
  };

  f64x4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f64x4{0.0, 0.0, 0.0, 0.0};

  const int kl = lane >> 4, rl = lane & 15;
  // acc[i][j][v] = C[m = m0 + wm + 16 i + rl][n = n0 + wn + 16 j + kl + 4 v].
  // from_c: the sums start from beta C / alpha (alpha is 1 or -1), so that an
  // update that nearly cancels C rounds at the size of what is left of it, not
  // at the size of the whole product
  if (from_c) {
    const double f = beta * alpha;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int gm = m0 + wm + 16 * i + rl;
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int gn = n0 + wn + 16 * j + kl + 4 * v;
          if (gm < M && gn < N) acc[i][j][v] = f * C[int64_t(gn) * ldc + gm];
        }
    }
  }
  load(0);
  for (int k0 = 0; k0 < K; k0 += kK) {
    __syncthreads();
    store();
    __syncthreads();
    if (k0 + kK < K) load(k0 + kK);
#pragma unroll
    for (int ks = 0; ks < kK / 4; ++ks) {
      const int k = ks * 4 + kl;
      double fa[2], fb[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) fa[j] = Bs[k][wn + j * 16 + rl];  // op(B)^T rows = n
#pragma unroll
      for (int i = 0; i < 2; ++i) fb[i] = As[k][wm + i * 16 + rl];  // op(A)^T cols = m
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(fa[j], fb[i], acc[i][j], 0, 0, 0);
    }
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int gm = m0 + wm + 16 * i + rl;
    if (gm >= M) continue;
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int gn = n0 + wn + 16 * j + kl + 4 * v;
        if (gn >= N) continue;
        double *c = C + int64_t(gn) * ldc + gm;
        const double r = alpha * acc[i][j][v];
        *c = beta == 0.0 || from_c ? r : r + beta * *c;
      }
  }
}

}  // namespace

namespace abh {

void dgemm_strided_batched(hipStream_t st, bool ta, bool tb, int m, int n, int k, double alpha,
                           const double *A, int lda, int64_t sA, const double *B, int ldb,
                           int64_t sB, double beta, double *C, int ldc, int64_t sC, int batch,
                           bool from_c, bool lower_only) {
  if (m <= 0 || n <= 0 || batch <= 0) return;
  ABH_REQUIRE(k >= 0 && lda >= 1 && ldb >= 1 && ldc >= m, ABH_ERR_INVALID_ARG,
              "dgemm: bad leading dimension");
  ABH_REQUIRE(!from_c || alpha == 1.0 || alpha == -1.0, ABH_ERR_INVALID_ARG,
              "dgemm: alpha must be 1 or -1");
  ABH_REQUIRE(batch <= 65535, ABH_ERR_INVALID_ARG, "dgemm: batch too large");
  const int tm = int(ceil_div(m, kT)), tn = int(ceil_div(n, kT));
  if (k == 0) {
    // C = beta C: the product is empty
    ABH_REQUIRE(beta == 1.0, ABH_ERR_INVALID_ARG, "dgemm: k == 0 needs beta == 1");
    return;
  }
  const int tiles = tm * tn, xcds = batch >= 64 ? 8 : 1;
  const int64_t blocks = int64_t(tiles) * (ceil_div(batch, xcds) * xcds);
  ABH_REQUIRE(blocks < (int64_t(1) << 31), ABH_ERR_INVALID_ARG, "dgemm: too many tiles");
  const dim3 grid{unsigned(blocks)};
  if (!ta && !tb)
    k_dgemm<false, false><<<grid, 256, 0, st>>>(m, n, k, alpha, A, lda, sA, B, ldb, sB, beta, C,
                                                 ldc, sC, tm, tiles, batch, xcds, from_c,
                                                 lower_only);
  else if (!ta && tb)
    k_dgemm<false, true><<<grid, 256, 0, st>>>(m, n, k, alpha, A, lda, sA, B, ldb, sB, beta, C,
                                                ldc, sC, tm, tiles, batch, xcds, from_c,
                                                lower_only);
  else if (ta && !tb)
    k_dgemm<true, false><<<grid, 256, 0, st>>>(m, n, k, alpha, A, lda, sA, B, ldb, sB, beta, C,
                                                ldc, sC, tm, tiles, batch, xcds, from_c,
                                                lower_only);
  else
    k_dgemm<true, true><<<grid, 256, 0, st>>>(m, n, k, alpha, A, lda, sA, B, ldb, sB, beta, C,
                                               ldc, sC, tm, tiles, batch, xcds, from_c,
                                               lower_only);
  check_launch();
}

}  // namespace abh
