// Q Z for the complex Hermitian eigendecomposition: the reflectors of the
// Householder reduction (trd_step_c, zhetrd's lower storage) applied to the
// tridiagonal eigenvectors in compact-WY blocks on the FP64 matrix cores.
//
// Q = H_0 H_1 ... with H_k = I - tau_k v_k v_k^H, v_k(k + 1) = 1 and
// v_k(k + 2 ..) in row k of S.  QB reflectors form I - V T V^H; eigenvectors
// are rows x of X, so a block (last to first) is W = X conj(V)^T, U = W T^T,
// X -= U V.  Complex products run as real ones on interleaved data: with
// B[2i][2p] = B[2i + 1][2p + 1] = Re v, B[2i + 1][2p] = -B[2i][2p + 1] = Im v,
// W = X B and X -= U B^T (8 flops per complex multiply-add, none wasted).
#include <algorithm>

#include "common.hpp"

namespace jv {

namespace {

typedef double dx4 __attribute__((ext_vector_type(4)));

constexpr int QB = 64;             // reflectors per block
constexpr int QC = 2 * QB;         // real columns of W and U
constexpr int QM = 64;             // eigenvectors per workgroup
constexpr int QK = 16;             // real depth per LDS stage
constexpr int QAS = QK + 2, QBS = QC + 2;  // LDS pitches (two-way conflicts at most)

struct QArgs {
  const cd* S;      // reflectors
  int n;
  cd* X;            // [n][n] eigenvectors (rows)
  double* part;     // partial products [split][rows][QC]
  const double* U;  // [n][QC]
};

// v_k(i), zero for reflectors past the last (k > n - 2) and rows past n.
__device__ inline cd q_v(const QArgs& a, int k, int i) {
  const cd s = a.S[(int64_t)min(k, a.n - 1) * a.n + min(i, a.n - 1)];
  if (k > a.n - 2 || i >= a.n || i <= k) return {0.0, 0.0};
  return i == k + 1 ? cd{1.0, 0.0} : s;
}

// MODE 0: W of block k0 (workgroup: QM eigenvectors x one slice of the rows i);
// MODE 1: V^H V of every block (blockIdx.x: block, its V as the left operand);
// MODE 2: X -= U B^T (workgroup: QM eigenvectors x QB entries, depth QC).
// Four waves of 64 x 32 real outputs (4 x 2 blocks of 16 x 16 x 4); the next
// stage's operands load into registers while the matrix cores work on this
// one's.  2112 x 2112: 8.6 ms of library products, 2.2 ms of triangular solves
// and 1.5 ms of copies and small products before (rocSOLVER zunmtr, 13.5 ms
// with its gaps); here 1.24 (W), 0.72 (U), 1.54 (update) and 0.11 ms (T).
template <int MODE>
__global__ void __launch_bounds__(256, 2) q_gemm(QArgs a, int k0) {
  __shared__ double As[2][QM * QAS];
  __shared__ double Bs[2][QK * QBS];
  const int t = threadIdx.x, lane = t % WAVE, w = t / WAVE, n = a.n;
  if (MODE == 1) k0 = blockIdx.x * QB;
  const int i0 = k0 + 1;
  const int m0 = MODE == 1 ? 0 : blockIdx.x * QM;
  int beg = 0, end = QC / QK;  // stages
  if (MODE != 2) {
    const int stages = (n - i0 + QK / 2 - 1) / (QK / 2), per = (stages + (int)gridDim.y - 1) / (int)gridDim.y;
    beg = blockIdx.y * per;
    end = min(stages, beg + per);
  }
  cd ra[2], rb[2];
  auto load = [&](int st) {
    if constexpr (MODE == 2) {
      const double* u = a.U + (int64_t)min(m0 + t / 4, n - 1) * QC + st * QK + (t % 4) * 4;
      ra[0] = {u[0], u[1]};
      ra[1] = {u[2], u[3]};
      const int k = k0 + st * (QK / 2) + t / 32, i = i0 + blockIdx.y * QB + (t % 32) * 2;
#pragma unroll
      for (int e = 0; e < 2; ++e) rb[e] = q_v(a, k, i + e);
    } else {
      const int i = i0 + st * (QK / 2) + (t % 4) * 2;
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        rb[e] = q_v(a, k0 + t / 4, i + e);
        if constexpr (MODE == 1) {
          ra[e] = rb[e];
        } else {
          // rows past n are multiplied by zero reflector entries
          ra[e] = a.X[(int64_t)min(m0 + t / 4, n - 1) * n + min(i + e, n - 1)];
        }
      }
    }
  };
  auto store = [&](int buf) {
    double* as = As[buf] + (t / 4) * QAS + (t % 4) * 4;
    as[0] = ra[0].re;
    as[1] = ra[0].im;
    as[2] = ra[1].re;
    as[3] = ra[1].im;
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      if constexpr (MODE == 2) {
        double* b = Bs[buf] + (size_t)(2 * (t / 32)) * QBS + 2 * ((t % 32) * 2 + e);
        b[0] = rb[e].re;
        b[1] = rb[e].im;
        b[QBS] = -rb[e].im;
        b[QBS + 1] = rb[e].re;
      } else {
        double* b = Bs[buf] + (size_t)(2 * ((t % 4) * 2 + e)) * QBS + 2 * (t / 4);
        b[0] = rb[e].re;
        b[1] = -rb[e].im;
        b[QBS] = rb[e].im;
        b[QBS + 1] = rb[e].re;
      }
    }
  };
  dx4 acc[4][2];
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int q = 0; q < 2; ++q) acc[r][q] = dx4{0.0, 0.0, 0.0, 0.0};
  if (beg < end) {
    load(beg);
    store(0);
  }
  __syncthreads();
  for (int st = beg; st < end; ++st) {
    const int buf = (st - beg) & 1;
    if (st + 1 < end) load(st + 1);
#pragma unroll
    for (int kk = 0; kk < QK; kk += 4) {
      double fa[4], fb[2];
#pragma unroll
      for (int r = 0; r < 4; ++r) fa[r] = As[buf][(r * 16 + lane % 16) * QAS + kk + lane / 16];
#pragma unroll
      for (int q = 0; q < 2; ++q) fb[q] = Bs[buf][(kk + lane / 16) * QBS + w * 32 + q * 16 + lane % 16];
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int q = 0; q < 2; ++q) acc[r][q] = __builtin_amdgcn_mfma_f64_16x16x4f64(fa[r], fb[q], acc[r][q], 0, 0, 0);
    }
    if (st + 1 < end) store(buf ^ 1);
    __syncthreads();
  }
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int row = r * 16 + 4 * j + lane / 16, col = w * 32 + q * 16 + lane % 16;
        if constexpr (MODE == 2) {
          const int i = i0 + blockIdx.y * QB + col / 2;
          if (m0 + row < n && i < n) ((double*)a.X)[((int64_t)(m0 + row) * n + i) * 2 + col % 2] -= acc[r][q][j];
        } else {
          const int64_t rows = MODE == 1 ? (int64_t)gridDim.x * QB : (int64_t)gridDim.x * QM;
          const int64_t at = (MODE == 1 ? (int64_t)blockIdx.x * QB : m0) + row;
          a.part[((int64_t)blockIdx.y * rows + at) * QC + col] = acc[r][q][j];
        }
      }
}

// T of every block (forward, columnwise, as LAPACK's zlarft): T_jj = tau_j,
// T[0:j, j] = -tau_j T[0:j, 0:j] (V^H v_j)[0:j].  A workgroup per block, four
// threads per row; T is written transposed ([column][row], for q_u's reads).
__global__ void __launch_bounds__(256) q_t(const double* __restrict__ part, int splits, const cd* __restrict__ tau, int n,
                                           cd* __restrict__ Tt) {
  extern __shared__ double lds[];
  cd* T = (cd*)lds;          // [row][QB + 1]
  cd* G = T + QB * (QB + 1);  // [j][q] = v_q^H v_j
  const int t = threadIdx.x, p = t / 4, sl = t % 4, b = blockIdx.x;
  const int64_t rows = (int64_t)gridDim.x * QB;
  for (int e = t; e < QB * QB; e += 256) {
    cd s = {0.0, 0.0};
    for (int k = 0; k < splits; ++k) {
      const double* g = part + ((k * rows + (int64_t)b * QB + e / QB) * QC) + 2 * (e % QB);
      s = s + cd{g[0], g[1]};
    }
    G[e] = s;
    T[e / QB * (QB + 1) + e % QB] = {0.0, 0.0};
  }
  __syncthreads();
  for (int j = 0; j < QB; ++j) {
    const int k = b * QB + j;
    const cd tj = k <= n - 2 ? tau[k] : cd{0.0, 0.0};
    cd s = {0.0, 0.0};
    for (int q = sl; q < j; q += 4) s = s + T[p * (QB + 1) + q] * G[j * QB + q];
    for (int m = 1; m < 4; m *= 2) {
      s.re += __shfl_xor(s.re, m);
      s.im += __shfl_xor(s.im, m);
    }
    if (sl == 0) T[p * (QB + 1) + j] = p < j ? cd{-1.0, 0.0} * (tj * s) : (p == j ? tj : cd{0.0, 0.0});
    __syncthreads();
  }
  for (int e = t; e < QB * QB; e += 256) Tt[(int64_t)b * QB * QB + e] = T[e % QB * (QB + 1) + e / QB];
}

// U = W T^T of one block: 16 eigenvectors per workgroup, the slices of W summed
// in slice order.
__global__ void __launch_bounds__(256) q_u(const double* __restrict__ part, int splits, int64_t rows,
                                           const cd* __restrict__ Tt, int n, double* __restrict__ U) {
  __shared__ cd W[16][QB];
  const int t = threadIdx.x, r0 = blockIdx.x * 16;
  for (int e = t; e < 16 * QB; e += 256) {
    const int64_t at = ((int64_t)(r0 + e / QB)) * QC + 2 * (e % QB);
    cd s = {0.0, 0.0};
    for (int k = 0; k < splits; ++k) {
      const double* g = part + (int64_t)k * rows * QC + at;
      s = s + cd{g[0], g[1]};
    }
    W[e / QB][e % QB] = s;
  }
  __syncthreads();
  const int p = t % QB, rr = t / QB * 4;
  cd u[4] = {};
  for (int q = 0; q < QB; ++q) {
    const cd x = Tt[q * QB + p];  // T[p][q], zero below the diagonal
#pragma unroll
    for (int k = 0; k < 4; ++k) u[k] = u[k] + x * W[rr + k][q];
  }
#pragma unroll
  for (int k = 0; k < 4; ++k)
    if (r0 + rr + k < n) {
      double* o = U + (int64_t)(r0 + rr + k) * QC + 2 * p;
      o[0] = u[k].re;
      o[1] = u[k].im;
    }
}

constexpr int WS_Q_PART = 122, WS_Q_U = 123, WS_Q_T = 124;
// Slices of the depth: about 1.5 workgroups per CU, each at least eight stages.
int q_splits(int tiles, int n) { return std::max(1, std::min((384 + tiles - 1) / tiles, (n + 63) / 64)); }

}  // namespace

// X <- Q X for the n x n eigenvectors in the rows of X, reflectors in S, tau
// (n - 1 complex) as trd_step_c leaves them.
int herm_apply_q(const double* S, const double* tau, int n, double* X, hipStream_t st) {
  const int nblk = (n - 1 + QB - 1) / QB, mt = (n + QM - 1) / QM;
  const int ks = q_splits(mt, n), kg = q_splits(nblk, n);
  const size_t pw = (size_t)ks * mt * QM * QC, pg = (size_t)kg * nblk * QB * QC;
  double* part = (double*)workspace(sizeof(double) * std::max(pw, pg), WS_Q_PART);
  double* U = (double*)workspace(sizeof(double) * (size_t)n * QC, WS_Q_U);
  cd* Tt = (cd*)workspace(sizeof(cd) * (size_t)nblk * QB * QB, WS_Q_T);
  if (!part || !U || !Tt) return fail(JV_E_NOMEM, "eigh: workspace allocation failed");
  QArgs a = {(const cd*)S, n, (cd*)X, part, U};
  hipLaunchKernelGGL(q_gemm<1>, dim3((unsigned)nblk, (unsigned)kg), dim3(256), 0, st, a, 0);
  JV_LAUNCH_CHECK("q_gemm (V^H V)");
  const size_t lds = sizeof(cd) * (QB * (QB + 1) + QB * QB);
  hipError_t e = hipFuncSetAttribute((const void*)q_t, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e != hipSuccess) return hip_fail(e, "hipFuncSetAttribute(q_t)");
  hipLaunchKernelGGL(q_t, dim3((unsigned)nblk), dim3(256), lds, st, part, kg, (const cd*)tau, n, Tt);
  JV_LAUNCH_CHECK("q_t");
  for (int b = nblk - 1; b >= 0; --b) {
    const int k0 = b * QB, len = n - k0 - 1;
    const int s = std::max(1, std::min(ks, (len + 63) / 64));
    hipLaunchKernelGGL(q_gemm<0>, dim3((unsigned)mt, (unsigned)s), dim3(256), 0, st, a, k0);
    JV_LAUNCH_CHECK("q_gemm (W)");
    hipLaunchKernelGGL(q_u, dim3((unsigned)((n + 15) / 16)), dim3(256), 0, st, part, s, (int64_t)mt * QM,
                       Tt + (size_t)b * QB * QB, n, U);
    JV_LAUNCH_CHECK("q_u");
    hipLaunchKernelGGL(q_gemm<2>, dim3((unsigned)mt, (unsigned)((len + QB - 1) / QB)), dim3(256), 0, st, a, k0);
    JV_LAUNCH_CHECK("q_gemm (update)");
  }
  return JV_OK;
}

}  // namespace jv
