// The per-edge ("bucketed") ICTD tensor product of the reference's native extension on gfx950: the
// operations of molecular_force_field._C_ictd_tp (csrc/ictd_tp.cpp:498-522, CUDA half
// csrc/ictd_tp_cuda.cu) for the arguments its CUDA path takes (fp32 and fp64, mul_in2 == 1):
//
//   project:  y[b][p][k][i] = sum_{m,n} a[b][i][m] v[b][n] U[m*m2 + n][p*K + k]
//   mix:      out[b][o][k]  = sum_p g[b][p] sum_i y[b][p][k][i] W[p][o][i]
//
// and the transposes of both with respect to every argument (the einsum semantics of
// models/ictd_irreps_cuda.py:169-288).  B is the batch (edges), I = mul_in1, O = mul_out, K = kdim,
// PK = P*K.  Layouts: a [B][I][m1], v [B][1][m2], U [m1*m2][PK], y [B][P][K][I], W [P][O][I],
// g [B][P], out [B][O][K].
//
// The projections contract over at most 9 x 9 components and run on the VALU, one wave per batch
// element with the factor ub[m][pk] = sum_n v[n] U[m*m2+n][pk] formed once per element in LDS (the
// gradient of v alone on the matrix cores).  The channel mixes are GEMMs over (b, k) rows: fp64 on
// v_mfma_f64_16x16x4_f64 (MI355X runs fp64 matrix and vector FMAs at the same peak, the MFMA form keeps the
// operand reuse of the tile); fp32 up to 128 channels with the weights resident in LDS and split-fp16
// products, otherwise, and for the weight gradient, on v_mfma_f32_16x16x4_f32.  Every kernel writes or,
// with `acc`, adds to its output, so the double-backward sums of the reference (csrc/ictd_tp_cuda.cu:528-533,
// 796-802) are the same kernels run two or three times.  Sums over the batch (the gradients of U and W)
// go through per-block partial sums and a reduction in a fixed order: results are deterministic.

#include <algorithm>

#include "common.h"
#include "fsctep.h"

namespace fsc {
namespace bucket {

constexpr int MAXM = 9;     // 2l + 1 for l <= 4
constexpr int MAXPK = 64;   // P * K handled by one lane each in the U/b transposes
constexpr int UREG = 32;    // per-lane U-gradient entries: m1 * m2 * PK <= 64 * UREG
constexpr int IC = 32;      // channels per staging chunk of the U/b transposes

struct Dims {
  int64_t B;
  int I, m1, m2, P, K, O;
};

typedef double d4 __attribute__((ext_vector_type(4)));

// Sixteen bytes at any float's address (one access all the same): the operations take operands and outputs of any
// alignment, views at an odd offset among them.
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
__device__ __forceinline__ f4 ld4u(const float* p) { return *reinterpret_cast<const f4u*>(p); }
__device__ __forceinline__ void st4u(float* p, const f4& v) { *reinterpret_cast<f4u*>(p) = v; }

// One 16-deep K step of a 16 x 16 output tile for either element type.  Both MFMAs take lane l's operands
// as A[l%16][l/16] and B[l/16][l%16]; their results differ in layout: register j of lane l holds
// D[4*(l/16) + j][l%16] for v_mfma_f32_16x16x4_f32 and D[l/16 + 4*j][l%16] for v_mfma_f64_16x16x4_f64
// (checked on gfx950).  row(q, j) gives the tile row of result register j in lane group q.
template <typename T>
struct Mma;
template <>
struct Mma<float> {
  using V = f4;
  static __device__ __forceinline__ V zero() { return V{0.f, 0.f, 0.f, 0.f}; }
  static __device__ __forceinline__ V mma(const V& a, const V& b, V c) { return mfma_k16(a, b, c); }
  static __device__ __forceinline__ V ld(const float* p) { return ld4u(p); }
  static __device__ __forceinline__ int row(int q, int j) { return 4 * q + j; }
};
template <>
struct Mma<double> {
  using V = d4;
  static __device__ __forceinline__ V zero() { return V{0.0, 0.0, 0.0, 0.0}; }
  static __device__ __forceinline__ V mma(const V& a, const V& b, V c) {
    c = __builtin_amdgcn_mfma_f64_16x16x4f64(a.x, b.x, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f64_16x16x4f64(a.y, b.y, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f64_16x16x4f64(a.z, b.z, c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a.w, b.w, c, 0, 0, 0);
  }
  static __device__ __forceinline__ V ld(const double* p) { return V{p[0], p[1], p[2], p[3]}; }
  static __device__ __forceinline__ int row(int q, int j) { return q + 4 * j; }
};

// Factor of the projection for element b, padded to MAXM rows: ub[m][pk] = sum_n v[b][n] U[m*m2+n][pk] for
// m < m1 and zero for m1 <= m < MAXM (us: U in LDS), so that the contractions below run over MAXM rows with
// no branch (a branch per row would make every product wait for all outstanding stores).
template <typename T>
__device__ __forceinline__ void form_ub(const Dims& d, int PK, const T* __restrict__ v, const T* us, T* ub, int64_t b,
                                        bool ok, int lane) {
  T vb[MAXM];   // v[b][n], zero past m2: all loads issued together (one wait)
#pragma unroll
  for (int n = 0; n < MAXM; ++n) {
    const T x = v[(ok ? b : 0) * d.m2 + min(n, d.m2 - 1)];
    vb[n] = (ok && n < d.m2) ? x : T(0);
  }
  for (int idx = lane; idx < MAXM * PK; idx += 64) {
    const int m = idx / PK, pk = idx - m * PK;
    const int mc = min(m, d.m1 - 1);
    T s = 0;
#pragma unroll
    for (int n = 0; n < MAXM; ++n) s += vb[n] * us[(mc * d.m2 + min(n, d.m2 - 1)) * PK + pk];
    ub[idx] = m < d.m1 ? s : T(0);
  }
}

template <typename T>
__device__ __forceinline__ void put(T* p, T v, int acc) { *p = acc ? *p + v : v; }

// TA false: y[b][pk][i] (+)= sum_m a[b][i][m] ub[m][pk]        (src = a, dst = y)
// TA true:  grad_a[b][i][m] (+)= sum_pk gy[b][pk][i] ub[m][pk]  (src = gy, dst = grad_a)
// Four waves per block, one batch element per wave per step; U staged in LDS once per block.  Lane i holds
// its a row (MAXM values, zero past m1; the loads clamp their index) or its gy values eight at a time.
template <typename T, bool TA, bool ACC>
__global__ __launch_bounds__(256) void project_kernel(Dims d, const T* __restrict__ src, const T* __restrict__ v,
                                                      const T* __restrict__ U, T* __restrict__ dst) {
  extern __shared__ __align__(16) char smraw[];
  T* sm = reinterpret_cast<T*>(smraw);
  const int PK = d.P * d.K, MN = d.m1 * d.m2;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  T* us = sm;
  T* ub = sm + MN * PK + wave * MAXM * PK;
  for (int idx = threadIdx.x; idx < MN * PK; idx += 256) us[idx] = U[idx];
  __syncthreads();
  // the trip count is the same for every wave of the block (barriers inside)
  for (int64_t b0 = (int64_t)blockIdx.x * 4; b0 < d.B; b0 += (int64_t)gridDim.x * 4) {
    const int64_t b = b0 + wave;
    const bool ok = b < d.B;
    form_ub(d, PK, v, us, ub, b, ok, lane);
    __syncthreads();
    if (ok) {   // wave-uniform
      for (int i = lane; i < d.I; i += 64) {
        if constexpr (!TA) {
          const T* ar = src + (b * d.I + i) * d.m1;
          T av[MAXM];
#pragma unroll
          for (int m = 0; m < MAXM; ++m) {
            const T x = ar[min(m, d.m1 - 1)];
            av[m] = m < d.m1 ? x : T(0);
          }
          T* yo = dst + b * PK * d.I + i;
          for (int pk = 0; pk < PK; ++pk) {
            T s = 0;
#pragma unroll
            for (int m = 0; m < MAXM; ++m) s += av[m] * ub[m * PK + pk];
            if constexpr (ACC) s += yo[(int64_t)pk * d.I];
            yo[(int64_t)pk * d.I] = s;
          }
        } else {
          const T* gp = src + b * PK * d.I + i;
          T sa[MAXM];
#pragma unroll
          for (int m = 0; m < MAXM; ++m) sa[m] = 0;
          for (int pk0 = 0; pk0 < PK; pk0 += 8) {
            T g8[8];
            int pc[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
              pc[j] = min(pk0 + j, PK - 1);
              const T x = gp[(int64_t)pc[j] * d.I];
              g8[j] = pk0 + j < PK ? x : T(0);
            }
#pragma unroll
            for (int j = 0; j < 8; ++j)
#pragma unroll
              for (int m = 0; m < MAXM; ++m) sa[m] += g8[j] * ub[m * PK + pc[j]];
          }
          T* o = dst + (b * d.I + i) * d.m1;
#pragma unroll
          for (int m = 0; m < MAXM; ++m)
            if (m < d.m1) {
              T val = sa[m];
              if constexpr (ACC) val += o[m];
              o[m] = val;
            }
        }
      }
    }
    __syncthreads();
  }
}

// Transposes with respect to v and U, through T_b[m][pk] = sum_i a[b][i][m] gy[b][pk][i]:
//   grad_v[b][n] (+)= sum_{m,pk} U[m*m2+n][pk] T_b[m][pk]                      (DO_V)
//   grad_U[m*m2+n][pk] = sum_b v[b][n] T_b[m][pk]: per-block partial sums upart  (DO_U)
// Lane pk forms column pk of T over channel chunks staged in LDS (gy transposed, padded rows); the lane
// keeps its U-gradient entries (m1*m2*PK <= 64*UREG) in registers over the block's elements.
template <typename T, bool DO_V, bool DO_U>
__global__ __launch_bounds__(256) void project_t_kernel(Dims d, const T* __restrict__ gy, const T* __restrict__ a,
                                                        const T* __restrict__ v, const T* __restrict__ U,
                                                        T* __restrict__ grad_v, int acc, T* __restrict__ upart) {
  extern __shared__ __align__(16) char smraw[];
  T* sm = reinterpret_cast<T*>(smraw);
  const int PK = d.P * d.K, MN = d.m1 * d.m2;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int per_wave = IC * d.m1 + IC * (PK + 1) + d.m1 * PK;
  T* us = sm;
  T* as = sm + MN * PK + wave * per_wave;   // [IC][m1]
  T* gs = as + IC * d.m1;                   // [IC][PK + 1]
  T* ts = gs + IC * (PK + 1);               // [m1][PK]
  if constexpr (DO_V) {
    for (int idx = threadIdx.x; idx < MN * PK; idx += 256) us[idx] = U[idx];
  }
  T ureg[UREG];
#pragma unroll
  for (int j = 0; j < UREG; ++j) ureg[j] = 0;
  __syncthreads();
  for (int64_t b0 = (int64_t)blockIdx.x * 4; b0 < d.B; b0 += (int64_t)gridDim.x * 4) {
    const int64_t b = b0 + wave;
    const bool ok = b < d.B;
    T tacc[MAXM];
#pragma unroll
    for (int m = 0; m < MAXM; ++m) tacc[m] = 0;
    for (int i0 = 0; i0 < d.I; i0 += IC) {
      const int ic = min(IC, d.I - i0);
      for (int idx = lane; idx < IC * d.m1; idx += 64)
        as[idx] = (ok && idx < ic * d.m1) ? a[(b * d.I + i0) * d.m1 + idx] : T(0);
      for (int idx = lane; idx < PK * IC; idx += 64) {
        const int pk = idx / IC, ii = idx - pk * IC;
        gs[ii * (PK + 1) + pk] = (ok && ii < ic) ? gy[(b * PK + pk) * d.I + i0 + ii] : T(0);
      }
      __syncthreads();
      if (lane < PK) {
        for (int ii = 0; ii < ic; ++ii) {
          const T gv = gs[ii * (PK + 1) + lane];
#pragma unroll
          for (int m = 0; m < MAXM; ++m)
            if (m < d.m1) tacc[m] += as[ii * d.m1 + m] * gv;
        }
      }
      __syncthreads();
    }
    if (lane < PK) {
#pragma unroll
      for (int m = 0; m < MAXM; ++m)
        if (m < d.m1) ts[m * PK + lane] = tacc[m];
    }
    __syncthreads();
    if constexpr (DO_V) {
      if (ok && lane < d.m2) {
        T s = 0;
        for (int m = 0; m < d.m1; ++m)
          for (int pk = 0; pk < PK; ++pk) s += us[(m * d.m2 + lane) * PK + pk] * ts[m * PK + pk];
        put(grad_v + b * d.m2 + lane, s, acc);
      }
    }
    if constexpr (DO_U) {
      if (ok) {
#pragma unroll
        for (int j = 0; j < UREG; ++j) {
          const int idx = lane + 64 * j;
          if (idx < MN * PK) {
            const int mn = idx / PK, pk = idx - mn * PK;
            const int m = mn / d.m2, n = mn - m * d.m2;
            ureg[j] += v[b * d.m2 + n] * ts[m * PK + pk];
          }
        }
      }
    }
    __syncthreads();
  }
  if constexpr (DO_U) {
    // the four waves' sums, added in a fixed order, are the block's partial sums
    T* red = sm;   // [4][MN * PK] (the host sizes the LDS for it)
#pragma unroll
    for (int j = 0; j < UREG; ++j) {
      const int idx = lane + 64 * j;
      if (idx < MN * PK) red[wave * MN * PK + idx] = ureg[j];
    }
    __syncthreads();
    for (int idx = threadIdx.x; idx < MN * PK; idx += 256)
      upart[(int64_t)blockIdx.x * MN * PK + idx] =
          ((red[idx] + red[MN * PK + idx]) + red[2 * MN * PK + idx]) + red[3 * MN * PK + idx];
  }
}

// grad_v alone: grad_v[b][n] (+)= sum_{m,pk} U[m*m2+n][pk] T_b[m][pk].  One wave per element forms T_b on the
// matrix cores (rows m padded to 16, NT tiles of 16 columns pk, K = channels), so gy and a are read once from
// global memory and nothing but U is staged; the general kernel above moves both through LDS and keeps one lane
// a column busy.  The lane's partial sums of the m2 outputs are added over the wave by halving exchanges (8
// outputs: 4 + 2 + 1 + 3 shuffles).  60,011 elements, 128 channels, m1 7, PK 7 (0.43 GB read): 440 -> 110 us on
// average over the lmax 3 buckets, 4 TB/s.  Channels in whole 4-vectors: I % 4 == 0, 16-byte aligned gy.
template <typename T, int NT>
__global__ __launch_bounds__(256) void project_tv_kernel(Dims d, const T* __restrict__ gy, const T* __restrict__ a,
                                                         const T* __restrict__ U, T* __restrict__ grad_v, int acc) {
  using M = Mma<T>;
  using V = typename M::V;
  extern __shared__ __align__(16) char smraw[];
  T* us = reinterpret_cast<T*>(smraw);   // [m2][16][16*NT], zero past m1 and PK
  const int PK = d.P * d.K;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, q = lane >> 4;
  for (int idx = threadIdx.x; idx < d.m2 * 256 * NT; idx += 256) {
    const int pk = idx % (16 * NT), nm = idx / (16 * NT), m = nm & 15, n = nm >> 4;
    us[idx] = (m < d.m1 && pk < PK) ? U[(m * d.m2 + n) * PK + pk] : T(0);
  }
  __syncthreads();
  const bool rv = r < d.m1;
  for (int64_t b = (int64_t)blockIdx.x * 4 + wave; b < d.B; b += (int64_t)gridDim.x * 4) {
    V t[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) t[j] = M::zero();
    const T* ab = a + b * d.I * d.m1 + (rv ? r : 0);
    const T* gb = gy + b * PK * d.I;
#pragma unroll 2
    for (int i0 = 0; i0 < d.I; i0 += 16) {
      const bool iv = i0 + 4 * q < d.I;   // the channel tail enters as zeros on both sides
      const int ic = iv ? i0 + 4 * q : 0;
      V av, bv[NT];
#pragma unroll
      for (int s = 0; s < 4; ++s) av[s] = ab[(ic + s) * d.m1];
#pragma unroll
      for (int j = 0; j < NT; ++j) bv[j] = M::ld(gb + (int64_t)min(16 * j + r, PK - 1) * d.I + ic);
#pragma unroll
      for (int s = 0; s < 4; ++s) av[s] = iv && rv ? av[s] : T(0);
#pragma unroll
      for (int j = 0; j < NT; ++j) {
#pragma unroll
        for (int s = 0; s < 4; ++s) bv[j][s] = iv ? bv[j][s] : T(0);
        t[j] = M::mma(av, bv[j], t[j]);
      }
    }
    for (int n0 = 0; n0 < d.m2; n0 += 8) {
      T s[8];
#pragma unroll
      for (int n = 0; n < 8; ++n) {
        s[n] = 0;
        if (n0 + n < d.m2) {
          const T* un = us + (n0 + n) * 256 * NT + r;
#pragma unroll
          for (int jj = 0; jj < 4; ++jj)
#pragma unroll
            for (int j = 0; j < NT; ++j) {
              const T uv = un[M::row(q, jj) * 16 * NT + 16 * j];
              // rows past m1 hold 0 * gy and columns past PK repeat column PK - 1: left out, not multiplied
              // by zero, so that an infinite input stays in its own sums
              s[n] += (M::row(q, jj) < d.m1 && 16 * j + r < PK) ? uv * t[j][jj] : T(0);
            }
        }
      }
#pragma unroll
      for (int k = 4; k > 0; k >>= 1) {   // lane bits 5, 4, 3 choose the half of the outputs it keeps
        const int off = 8 * k;
        const bool hi = lane & off;
#pragma unroll
        for (int n = 0; n < 4; ++n)
          if (n < k) {
            const T mine = hi ? s[n + k] : s[n], other = hi ? s[n] : s[n + k];
            s[n] = mine + __shfl_xor(other, off, 64);
          }
      }
#pragma unroll
      for (int off = 4; off > 0; off >>= 1) s[0] += __shfl_xor(s[0], off, 64);
      const int n = n0 + (lane >> 3);
      if ((lane & 7) == 0 && n < d.m2) put(grad_v + b * d.m2 + n, s[0], acc);
    }
  }
}

// out[idx] (+)= sum over parts of part[p][idx], in a fixed order: 8 groups of threads take every eighth part,
// their sums are added in order.  A thread per output walked up to 4096 parts one load after another in 64
// blocks (P O I = 16,384 outputs, 2048 parts: 282 us); 32 outputs a block keep 128-byte reads and 8 chains a
// block in flight.
template <typename T>
__global__ __launch_bounds__(256) void sum_parts_kernel(int64_t n, int nparts, const T* __restrict__ part,
                                                        T* __restrict__ out, int acc) {
  __shared__ T red[8][32];
  const int c = threadIdx.x & 31, grp = threadIdx.x >> 5;
  for (int64_t i0 = (int64_t)blockIdx.x * 32; i0 < n; i0 += (int64_t)gridDim.x * 32) {
    const int64_t idx = i0 + c;
    T s = 0;
    if (idx < n) {
#pragma unroll 8
      for (int p = grp; p < nparts; p += 8) s += part[(int64_t)p * n + idx];
    }
    red[grp][c] = s;
    __syncthreads();
    if (grp == 0 && idx < n) {
#pragma unroll
      for (int k = 1; k < 8; ++k) s += red[k][c];
      put(out + idx, s, acc);
    }
    __syncthreads();
  }
}
unsigned sum_parts_grid(int64_t n) { return (unsigned)std::min<int64_t>((n + 31) / 32, 4096); }

// ---------------------------------------------------------------- channel mix (MFMA), every wave for itself
// All of fp64, whose operands are twice as large; of fp32 the sizes that fill neither a slice nor the chip (mix_sliced
// and the entry points), the other fp32 forms are further down.
// Rows are the (b, k) pairs R = b*K + k.  A wave takes two 16-row tiles and eight 16-column tiles; lane
// (r, q) of an MFMA supplies A[r][4q..4q+3] and B[4q..4q+3][r] for a 16-deep K step and ends with
// D[4q + j][r] in result register j (common.h).

// out[b][o][k] (+)= sum_p g[b][p] sum_i y[b][p][k][i] W[p][o][i]   (K = (p, i); grid: 128 rows x 128 columns)
// TG: the per-path dot with the output gradient instead, grad_g[b][p] (+)= sum_{k,o} go[b][o][k]
// sum_i y[b][p][k][i] W[p][o][i] (grid: batch groups of 128/K elements x paths, all columns per block).
template <typename T, bool TG>
__global__ __launch_bounds__(256) void mix_kernel(Dims d, const T* __restrict__ y, const T* __restrict__ W,
                                                  const T* __restrict__ g, const T* __restrict__ go,
                                                  T* __restrict__ out, int acc) {
  using M = Mma<T>;
  using V = typename M::V;
  // fp32 requests the next K step's operands before the current products (two register sets); fp64,
  // whose operand sets are twice as large, works one step at a time
  constexpr bool PF = sizeof(T) == 4;
  __shared__ T rs[128];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, q = lane >> 4;
  const int K = d.K, P = d.P, I = d.I, O = d.O;
  const int64_t R = d.B * K;
  // TG: the block's rows are whole batch elements bb0 .. bb0 + BB - 1 (rows never straddle two blocks)
  const int BB = 128 / K;
  const int64_t bb0 = (int64_t)blockIdx.x * BB;
  const int64_t rbeg = TG ? bb0 * K : (int64_t)blockIdx.x * 128;
  const int64_t rend = TG ? std::min<int64_t>((bb0 + BB) * K, R) : R;
  const int p_only = TG ? (int)blockIdx.y : -1;
  int64_t rb[2];
  int rk[2];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int64_t row = rbeg + wave * 32 + 16 * t + r;
    const int64_t rr = row < rend ? row : 0;
    rb[t] = rr / K;
    rk[t] = (int)(rr - rb[t] * K);
  }
  T rowsum[2][4];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int j = 0; j < 4; ++j) rowsum[t][j] = 0;
  const int ocb_beg = TG ? 0 : (int)blockIdx.y * 128, ocb_end = TG ? O : std::min(O, ocb_beg + 128);
  for (int o0 = ocb_beg; o0 < ocb_end; o0 += 128) {
    V accm[2][8];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int j = 0; j < 8; ++j) accm[t][j] = M::zero();
    bool cv[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) cv[j] = o0 + 16 * j + r < O;
    // K steps (path p, channels i0 .. i0 + 15) in order.  Loads are unconditional at clamped addresses and
    // nothing reads them before the products: rows and columns past the end accumulate values that are never
    // stored, and the channel tail (I % 16) is cut by a zero scale on the A rows, applied with the gate when
    // the step is multiplied.
    const int pb = TG ? p_only : 0, pe = TG ? p_only + 1 : P;
    const int nis = (I + 15) / 16, nst = (pe - pb) * nis;
    int oc[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) oc[j] = cv[j] ? o0 + 16 * j + r : 0;
    auto load = [&](int st, V (&av)[2], T (&gs)[2], V (&bw)[8]) {
      const int p = pb + st / nis, ii = (st % nis) * 16 + 4 * q;
      const bool iv = ii < I;   // I % 4 == 0: the whole 4-vector is in range
      const int ic = iv ? ii : 0;
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        gs[t] = TG ? T(1) : g[rb[t] * P + p];
        if (!iv) gs[t] = 0;
        av[t] = M::ld(y + ((rb[t] * P + p) * K + rk[t]) * I + ic);
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) bw[j] = M::ld(W + ((int64_t)p * O + oc[j]) * I + ic);
    };
    auto mma = [&](const V (&av)[2], const T (&gs)[2], const V (&bw)[8]) {
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const V a = av[t] * gs[t];
#pragma unroll
        for (int j = 0; j < 8; ++j) accm[t][j] = M::mma(a, bw[j], accm[t][j]);
      }
    };
    if constexpr (PF) {
      V a0[2], b0[8], a1[2], b1[8];
      T g0[2], g1[2];
      if (nst > 0) load(0, a0, g0, b0);
      for (int st = 0; st < nst; st += 2) {
        if (st + 1 < nst) load(st + 1, a1, g1, b1);
        __builtin_amdgcn_sched_barrier(0);
        mma(a0, g0, b0);
        if (st + 1 < nst) {
          if (st + 2 < nst) load(st + 2, a0, g0, b0);
          __builtin_amdgcn_sched_barrier(0);
          mma(a1, g1, b1);
        }
      }
    } else {
      for (int st = 0; st < nst; ++st) {
        V a0[2], b0[8];
        T g0[2];
        load(st, a0, g0, b0);
        mma(a0, g0, b0);
      }
    }
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) {
        const int64_t row = rbeg + wave * 32 + 16 * t + M::row(q, jj);
        if (row >= rend) continue;
        const int64_t b = row / K;
        const int k = (int)(row - b * K);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          if (!cv[j]) continue;
          const int o = o0 + 16 * j + r;
          if constexpr (TG) rowsum[t][jj] += accm[t][j][jj] * go[(b * O + o) * K + k];
          else put(out + (b * O + o) * K + k, accm[t][j][jj], acc);
        }
      }
  }
  if constexpr (TG) {
    // row sums over the 16 column lanes, then over the K rows of each batch element
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) {
        T s = rowsum[t][jj];
#pragma unroll
        for (int off = 1; off < 16; off <<= 1) s += __shfl_xor(s, off, 64);
        if (r == 0) rs[wave * 32 + 16 * t + M::row(q, jj)] = s;
      }
    __syncthreads();
    if (threadIdx.x < BB) {
      const int64_t b = bb0 + threadIdx.x;
      if (b < d.B) {
        T s = 0;
        for (int k = 0; k < K; ++k) s += rs[threadIdx.x * K + k];
        put(out + b * P + p_only, s, acc);
      }
    }
  }
}

// Wt[p][i][o] = W[p][o][i]
template <typename T>
__global__ void transpose_w_kernel(int P, int O, int I, const T* __restrict__ W, T* __restrict__ Wt) {
  const int64_t n = (int64_t)P * O * I;
  for (int64_t idx = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; idx < n; idx += (int64_t)gridDim.x * blockDim.x) {
    const int o = (int)(idx % O);
    const int64_t pi = idx / O;
    const int i = (int)(pi % I), p = (int)(pi / I);
    Wt[idx] = W[((int64_t)p * O + o) * I + i];
  }
}

// grad_y[b][p][k][i] (+)= g[b][p] sum_o go[b][o][k] W[p][o][i]: rows (b, k), columns i, K = o; grid: 128 rows x
// (path, 128-column block).  B from the transposed weights Wt[p][i][o] (4-vectors along o).
template <typename T>
__global__ __launch_bounds__(256) void mix_ty_kernel(Dims d, const T* __restrict__ go, const T* __restrict__ Wt,
                                                     const T* __restrict__ g, T* __restrict__ gy, int acc) {
  using M = Mma<T>;
  using V = typename M::V;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, q = lane >> 4;
  const int K = d.K, P = d.P, I = d.I, O = d.O;
  const int64_t R = d.B * K;
  const int nib = (I + 127) / 128;
  const int p = (int)blockIdx.y / nib, i0c = ((int)blockIdx.y % nib) * 128;
  int64_t rb[2];
  int rk[2];
  bool rv[2];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int64_t row = (int64_t)blockIdx.x * 128 + wave * 32 + 16 * t + r;
    rv[t] = row < R;
    const int64_t rr = rv[t] ? row : 0;
    rb[t] = rr / K;
    rk[t] = (int)(rr - rb[t] * K);
  }
  bool cv[8];
  const T* wr[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int i = i0c + 16 * j + r;
    cv[j] = i < I;
    wr[j] = Wt + ((int64_t)p * I + (cv[j] ? i : 0)) * O;
  }
  V accm[2][8];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int j = 0; j < 8; ++j) accm[t][j] = M::zero();
  for (int o0 = 0; o0 < O; o0 += 16) {
    const int oo = o0 + 4 * q;
    const bool ov = oo < O;   // O % 4 == 0
    V av[2], bw[8];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const T* gp = go + (rb[t] * O + oo) * K + rk[t];
#pragma unroll
      for (int s = 0; s < 4; ++s) av[t][s] = (ov && rv[t]) ? gp[(int64_t)s * K] : T(0);
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) bw[j] = (ov && cv[j]) ? M::ld(wr[j] + oo) : M::zero();
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int j = 0; j < 8; ++j) accm[t][j] = M::mma(av[t], bw[j], accm[t][j]);
  }
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int jj = 0; jj < 4; ++jj) {
      const int64_t row = (int64_t)blockIdx.x * 128 + wave * 32 + 16 * t + M::row(q, jj);
      if (row >= R) continue;
      const int64_t b = row / K;
      const int k = (int)(row - b * K);
      const T gate = g[b * P + p];
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (cv[j]) put(gy + ((b * P + p) * K + k) * I + i0c + 16 * j + r, accm[t][j][jj] * gate, acc);
    }
}

// Partial sums of grad_W[p][o][i] = sum_{(b,k)} g[b][p] go[b][o][k] y[b][p][k][i] over a range of rows:
// part[s][p][o][i].  M = o, N = i, K = rows (b, k), 16 rows per MFMA step; block (split s, path p, 128 x 128
// output tile): wave w takes o tiles 2w, 2w + 1 and all eight i tiles.
template <typename T>
__global__ __launch_bounds__(256) void mix_tw_kernel(Dims d, const T* __restrict__ go, const T* __restrict__ y,
                                                     const T* __restrict__ g, int64_t rows_per_split,
                                                     T* __restrict__ part) {
  using M = Mma<T>;
  using V = typename M::V;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, q = lane >> 4;
  const int K = d.K, P = d.P, I = d.I, O = d.O;
  const int64_t R = d.B * K;
  const int s = blockIdx.x, p = blockIdx.y;
  const int nib = (I + 127) / 128;
  const int o0c = ((int)blockIdx.z / nib) * 128, i0c = ((int)blockIdx.z % nib) * 128;
  const int64_t r0 = (int64_t)s * rows_per_split, r1 = std::min(R, r0 + rows_per_split);
  V accm[2][8];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int j = 0; j < 8; ++j) accm[t][j] = M::zero();
  bool ovt[2], ivt[8];
#pragma unroll
  for (int t = 0; t < 2; ++t) ovt[t] = o0c + wave * 32 + 16 * t + r < O;
#pragma unroll
  for (int j = 0; j < 8; ++j) ivt[j] = i0c + 16 * j + r < I;
  for (int64_t rr0 = r0; rr0 < r1; rr0 += 16) {
    // K step: rows rr0 + 4q + u (u = 0..3) for this lane group
    T gv[4];
    int64_t yoff[4], goff[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int64_t row = rr0 + 4 * q + u;
      const bool ok = row < r1;
      const int64_t rw = ok ? row : r0;
      const int64_t b = rw / K;
      const int k = (int)(rw - b * K);
      gv[u] = ok ? g[b * P + p] : T(0);
      yoff[u] = ((b * P + p) * K + k) * I;
      goff[u] = b * O * K + k;
    }
    V av[2], bw[8];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int o = o0c + wave * 32 + 16 * t + r;
#pragma unroll
      for (int u = 0; u < 4; ++u) av[t][u] = ovt[t] ? go[goff[u] + (int64_t)o * K] * gv[u] : T(0);
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int i = i0c + 16 * j + r;
#pragma unroll
      for (int u = 0; u < 4; ++u) bw[j][u] = ivt[j] ? y[yoff[u] + i] : T(0);
    }
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int j = 0; j < 8; ++j) accm[t][j] = M::mma(av[t], bw[j], accm[t][j]);
  }
  T* ps = part + ((int64_t)s * P + p) * O * I;
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int jj = 0; jj < 4; ++jj) {
      const int o = o0c + wave * 32 + 16 * t + M::row(q, jj);
      if (o >= O) continue;
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (ivt[j]) ps[(int64_t)o * I + i0c + 16 * j + r] = accm[t][j][jj];
    }
}

// ---------------------------------------------------------------- channel mix, fp32
// The fp32 forms are bound by the fp32 matrix rate (157 TFLOP/s).  These take any size; the resident kernels further
// down are the faster ones for the sizes they hold.  A block of four waves takes 128 rows x 128 columns, wave w the
// rows 32w .. 32w+31.  The column operand (weights, [column][contraction]) is common to the four waves and goes
// through LDS 32 contraction steps at a time, rows padded to 36 floats (conflict-free 16-byte reads); the next slice
// and the wave's own rows are requested a slice (4096 MFMA cycles) ahead.  60,011 elements, K 7, 128 x 128 channels
// (13.8 GFLOP, y and out 0.43 GB): forward 279 -> 260 us, gate gradient 485 -> 272, input gradient 309 -> 171
// (81 TFLOP/s) against every wave reading the weights from L2 itself.
constexpr int KS = 32;          // contraction steps per slice
constexpr int WPAD = KS + 4;
constexpr int OPAD = 132;       // row stride of an output slice [32 columns][128 rows]; 32 * OPAD <= 128 * WPAD

// The block's share of a weight slice in flight: 128 columns x 32 steps, four 16-byte pieces a thread.  Pieces past
// the matrix are cleared when they are stored: a select beside the load would wait for it.
struct WSlice {
  f4 v[4];
  __device__ __forceinline__ static bool inside(int s, int ncol, int nk, int c0, int k0) {
    return c0 + (int)(threadIdx.x >> 3) + 32 * s < ncol && k0 + 4 * (int)(threadIdx.x & 7) < nk;
  }
  __device__ __forceinline__ void load(const float* __restrict__ w, int ncol, int nk, int c0, int k0) {
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int c = c0 + (threadIdx.x >> 3) + 32 * s, k = k0 + 4 * (threadIdx.x & 7);
      v[s] = ld4u(w + (inside(s, ncol, nk, c0, k0) ? (int64_t)c * nk + k : 0));
    }
  }
  __device__ __forceinline__ f4 piece(int s, int ncol, int nk, int c0, int k0) const {
    return inside(s, ncol, nk, c0, k0) ? v[s] : f4{0.f, 0.f, 0.f, 0.f};
  }
};

// The products of one slice: a[h][t] holds the contraction steps 16h + 4q .. + 3 of row tile t.
__device__ __forceinline__ void mma_slice(const f4 (&a)[2][2], const float* ws, int r, int q, f4 (&accm)[2][8]) {
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const f4 b = ld4(ws + (16 * j + r) * WPAD + 16 * h + 4 * q);
#pragma unroll
      for (int t = 0; t < 2; ++t) accm[t][j] = mfma_k16(a[h][t], b, accm[t][j]);
    }
}

// out[b][o][k] (+)= sum_p g[b][p] sum_i y[b][p][k][i] W[p][o][i]; grid: 128 rows x 128 columns o.
// TG: grad_g[b][p] (+)= sum_{k,o} go[b][o][k] sum_i y[b][p][k][i] W[p][o][i]; grid: 128/K whole elements x
// paths, every column by the same block.
template <bool TG>
__global__ __launch_bounds__(256, 3) void mix32_kernel(Dims d, const float* __restrict__ y, const float* __restrict__ W,
                                                       const float* __restrict__ g, const float* __restrict__ go,
                                                       float* __restrict__ out, int acc) {
  __shared__ float ws[128 * WPAD];
  __shared__ float rs[128];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, q = lane >> 4;
  const int K = d.K, P = d.P, I = d.I, O = d.O;
  const uint32_t R = (uint32_t)(d.B * K);   // below 2^31 (checked): 32-bit row arithmetic, a 64-bit division by K
  const int BB = 128 / K;                   // for each of a lane's rows took a third of the kernel
  const uint32_t bb0 = blockIdx.x * BB;
  const uint32_t rbeg = TG ? bb0 * K : blockIdx.x * 128;
  const uint32_t rend = TG ? std::min((bb0 + BB) * (uint32_t)K, R) : std::min(rbeg + 128, R);
  int64_t yb[2], rb[2];   // the lane's rows: offset of y at path 0, element
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const uint32_t row = rbeg + wave * 32 + 16 * t + r;
    const uint32_t rr = row < rend ? row : rbeg;
    rb[t] = rr / (uint32_t)K;
    yb[t] = (rb[t] * P * K + (rr - (uint32_t)rb[t] * K)) * I;
  }
  const int ns = (I + KS - 1) / KS;
  const int pb = TG ? (int)blockIdx.y : 0, pe = TG ? pb + 1 : P;
  const int ob = TG ? 0 : (int)blockIdx.y * 128, oe = TG ? O : std::min(O, ob + 128);
  float rowsum[2][4];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int j = 0; j < 4; ++j) rowsum[t][j] = 0.f;
  for (int o0 = ob; o0 < oe; o0 += 128) {
    f4 accm[2][8];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int j = 0; j < 8; ++j) accm[t][j] = f4{0.f, 0.f, 0.f, 0.f};
    // the slices of every path in order: position (p, s)
    WSlice w;
    f4 an[2][2];
    float gn[2];
    auto request = [&](int p, int s) {
      w.load(W + (int64_t)p * O * I, O, I, o0, s * KS);
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        gn[t] = TG ? 1.f : g[rb[t] * P + p];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int i = s * KS + 16 * h + 4 * q;
          an[h][t] = ld4u(y + yb[t] + (int64_t)p * K * I + (i < I ? i : 0));
        }
      }
    };
    request(pb, 0);
    int p = pb, s = 0;
    while (p < pe) {
      f4 a[2][2];
      __syncthreads();   // the previous slice is read
#pragma unroll
      for (int u = 0; u < 4; ++u)
        st4(ws + ((threadIdx.x >> 3) + 32 * u) * WPAD + 4 * (threadIdx.x & 7), w.piece(u, O, I, o0, s * KS));
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          a[h][t] = an[h][t] * gn[t];
          if (s * KS + 16 * h + 4 * q >= I) a[h][t] = f4{0.f, 0.f, 0.f, 0.f};
        }
      int p1 = p, s1 = s + 1;
      if (s1 == ns) { s1 = 0; ++p1; }
      if (p1 < pe) request(p1, s1);
      __syncthreads();
      mma_slice(a, ws, r, q, accm);
      p = p1;
      s = s1;
    }
    if constexpr (TG) {
      // loads at clamped addresses, so that they are all in flight together
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) {
          const uint32_t row = std::min<uint32_t>(rbeg + wave * 32 + 16 * t + 4 * q + jj, rend - 1);
          const uint32_t b = row / (uint32_t)K;
          const float* gp = go + (int64_t)b * O * K + (row - b * K);
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const int o = o0 + 16 * j + r;
            const float gv = gp[(int64_t)std::min(o, O - 1) * K];
            rowsum[t][jj] += o < O ? accm[t][j][jj] * gv : 0.f;
          }
        }
    } else {
      // out[b][o][k] holds an element's rows side by side: a store per register would write 4 bytes every 4K.
      // 32 columns at a time pass through LDS, [column][row], and leave in runs of 32 K floats an element.  A
      // thread's values are 256 apart in (element, column, k), reached by carries: dividing for each of them took
      // 5 to 15 us of a launch.
      const uint32_t nrow = rend - rbeg, b0 = rbeg / (uint32_t)K, nb = (rend - 1) / (uint32_t)K - b0 + 1;
      const uint32_t dc = 256u / (uint32_t)K, dk = 256u - dc * K;
      const uint32_t c1 = threadIdx.x / (uint32_t)K, k1 = threadIdx.x - c1 * K;
#pragma unroll
      for (int sl = 0; sl < 4; ++sl) {
        const int oc = std::min(32, O - o0 - 32 * sl);   // columns of the slice
        if (oc <= 0) break;                               // the same for every thread
        __syncthreads();
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int jh = 0; jh < 2; ++jh)
            st4(ws + (16 * jh + r) * OPAD + wave * 32 + 16 * t + 4 * q, accm[t][2 * sl + jh]);
        __syncthreads();
        uint32_t bi = c1 >> 5, c = c1 & 31, k = k1;
#pragma unroll 4
        while (bi < nb) {
          const int32_t lr = (int32_t)((b0 + bi) * K + k - rbeg);
          if (lr >= 0 && lr < (int32_t)nrow && (int)c < oc)
            put(out + ((int64_t)(b0 + bi) * O + o0 + 32 * sl + c) * K + k, ws[c * OPAD + lr], acc);
          k += dk;
          c += dc;
          if (k >= (uint32_t)K) { k -= K; ++c; }
          bi += c >> 5;
          c &= 31;
        }
      }
    }
  }
  if constexpr (TG) {
    // row sums over the 16 column lanes, then over the K rows of each batch element
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) {
        float v = rowsum[t][jj];
#pragma unroll
        for (int off = 1; off < 16; off <<= 1) v += __shfl_xor(v, off, 64);
        if (r == 0) rs[wave * 32 + 16 * t + 4 * q + jj] = v;
      }
    __syncthreads();
    if (threadIdx.x < BB) {
      const int64_t b = (int64_t)bb0 + threadIdx.x;
      if (b < d.B) {
        float v = 0.f;
        for (int k = 0; k < K; ++k) v += rs[threadIdx.x * K + k];
        put(out + b * P + pb, v, acc);
      }
    }
  }
}

// grad_y[b][p][k][i] (+)= g[b][p] sum_o go[b][o][k] W[p][o][i]; grid: 128 rows x (path, 128 columns i), column
// operand Wt[p][i][o].  Column 8r + j of the block is column r of tile j, so that a lane stores 8 channels in
// a row.
__global__ __launch_bounds__(256, 3) void mix32_ty_kernel(Dims d, const float* __restrict__ go,
                                                          const float* __restrict__ Wt, const float* __restrict__ g,
                                                          float* __restrict__ gy, int acc) {
  __shared__ float ws[128 * WPAD];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, q = lane >> 4;
  const int K = d.K, P = d.P, I = d.I, O = d.O;
  const uint32_t R = (uint32_t)(d.B * K);
  const int nib = (I + 127) / 128;
  const int p = (int)blockIdx.y / nib, i0 = ((int)blockIdx.y % nib) * 128;
  const uint32_t rbeg = blockIdx.x * 128;
  int64_t gb[2];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const uint32_t row = rbeg + wave * 32 + 16 * t + r;
    const uint32_t rr = row < R ? row : 0, b = rr / (uint32_t)K;
    gb[t] = (int64_t)b * O * K + (rr - b * K);
  }
  f4 accm[2][8];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int j = 0; j < 8; ++j) accm[t][j] = f4{0.f, 0.f, 0.f, 0.f};
  WSlice w;
  f4 an[2][2];
  auto request = [&](int k0) {
    w.load(Wt + (int64_t)p * I * O, I, O, i0, k0);
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int o = k0 + 16 * h + 4 * q;
        const float* gp = go + gb[t] + (int64_t)(o < O ? o : 0) * K;
#pragma unroll
        for (int u = 0; u < 4; ++u) an[h][t][u] = gp[(int64_t)u * K];
      }
  };
  request(0);
  for (int k0 = 0; k0 < O; k0 += KS) {
    f4 a[2][2];
    __syncthreads();
    // columns re-ordered on the way into LDS: row 16j + r of the slice is column 8r + j
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int c = (threadIdx.x >> 3) + 32 * s;
      st4(ws + (16 * (c & 7) + (c >> 3)) * WPAD + 4 * (threadIdx.x & 7), w.piece(s, I, O, i0, k0));
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        a[h][t] = an[h][t];
        if (k0 + 16 * h + 4 * q >= O) a[h][t] = f4{0.f, 0.f, 0.f, 0.f};
      }
    if (k0 + KS < O) request(k0 + KS);
    __syncthreads();
    mma_slice(a, ws, r, q, accm);
  }
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int jj = 0; jj < 4; ++jj) {
      const uint32_t row = rbeg + wave * 32 + 16 * t + 4 * q + jj;
      if (row >= R) continue;
      const uint32_t b = row / (uint32_t)K;
      const float gate = g[(int64_t)b * P + p];
      float* o = gy + (((int64_t)b * P + p) * K + (row - b * K)) * I + i0 + 8 * r;
#pragma unroll
      for (int hh = 0; hh < 2; ++hh)
        if (i0 + 8 * r + 4 * hh < I) {   // I % 4 == 0
          f4 v = {accm[t][4 * hh][jj], accm[t][4 * hh + 1][jj], accm[t][4 * hh + 2][jj], accm[t][4 * hh + 3][jj]};
          v = v * gate;
          if (acc) v = ld4u(o + 4 * hh) + v;
          st4u(o + 4 * hh, v);
        }
    }
}

// Partial sums of grad_W[p][o][i] = sum_{(b,k)} g[b][p] go[b][o][k] y[b][p][k][i] over a range of rows.  Block
// (split, path, 16 T x 16 T tile; T 2, 4 or 8 by the channels); both operands go through LDS 256 / T rows at a time
// (each read from memory once a block instead of once a wave), the next rows in flight meanwhile: a thread's four
// pieces of y and sixteen values of go are only gated or cleared when they are stored.  Wave w takes a quarter of
// the tile.  60,011 elements, K 7, 128 x 128: 333 us with each wave loading its own operands, 252 with gates and
// bounds applied beside the loads, 190 now; 20,011 elements at 64 x 64 on 128 x 128 tiles 98, now 28.
template <int T>
__global__ __launch_bounds__(256, 3) void mix32_tw_kernel(Dims d, const float* __restrict__ go,
                                                          const float* __restrict__ y, const float* __restrict__ g,
                                                          int64_t rows_per_split, float* __restrict__ part) {
  constexpr int W = 16 * T, RS = 256 / T, WT = T / 2;
  constexpr int TPAD = W + 16;   // row stride of the staged rows: the four rows of an MFMA step on distinct banks
  __shared__ __align__(16) float gs[RS * TPAD];
  __shared__ __align__(16) float ys[RS * TPAD];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, q = lane >> 4;
  const int K = d.K, P = d.P, I = d.I, O = d.O;
  const uint32_t R = (uint32_t)(d.B * K);
  const int s = blockIdx.x, p = blockIdx.y;
  const int nib = (I + W - 1) / W;
  const int o0 = ((int)blockIdx.z / nib) * W, i0 = ((int)blockIdx.z % nib) * W;
  const uint32_t r0 = (uint32_t)(s * rows_per_split), r1 = (uint32_t)std::min<int64_t>(R, r0 + rows_per_split);
  const int wo = 16 * WT * (wave >> 1), wi = 16 * WT * (wave & 1);
  f4 accm[WT][WT];
#pragma unroll
  for (int t = 0; t < WT; ++t)
#pragma unroll
    for (int j = 0; j < WT; ++j) accm[t][j] = f4{0.f, 0.f, 0.f, 0.f};
  f4 yn[4];
  float gn[16], gate[16];
  const int ycol = 4 * (threadIdx.x % (4 * T)), yrow = threadIdx.x / (4 * T);   // rows yrow + (64 / T) u
  const int ocol = threadIdx.x % W;                                             // rows orow .. orow + 15
  const int orow = 16 * (T >= 4 ? __builtin_amdgcn_readfirstlane(threadIdx.x / W) : threadIdx.x / W);
  const bool yok = i0 + ycol < I, ook = o0 + ocol < O;
  auto request = [&](uint32_t rr) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const uint32_t row = std::min(rr + yrow + (64 / T) * u, r1 - 1), b = row / (uint32_t)K;
      yn[u] = ld4u(y + (((int64_t)b * P + p) * K + (row - b * K)) * I + (yok ? i0 + ycol : 0));
    }
    // go: 16 rows of one column; the element and row in it advance without divisions
    const uint32_t first = std::min(rr + orow, r1 - 1);
    uint32_t b = first / (uint32_t)K, k = first - b * K;
    const float* gc = go + (int64_t)(ook ? o0 + ocol : 0) * K;
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      gn[u] = gc[(int64_t)b * O * K + k];
      gate[u] = g[(int64_t)b * P + p];
      if (rr + orow + u + 1 < r1 && ++k == (uint32_t)K) { k = 0; ++b; }
    }
  };
  request(r0);
  for (uint32_t rr = r0; rr < r1; rr += RS) {
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int row = yrow + (64 / T) * u;
      st4(ys + row * TPAD + ycol, yok && rr + row < r1 ? yn[u] : f4{0.f, 0.f, 0.f, 0.f});
    }
#pragma unroll
    for (int u = 0; u < 16; ++u) gs[(orow + u) * TPAD + ocol] = ook && rr + orow + u < r1 ? gn[u] * gate[u] : 0.f;
    if (rr + RS < r1) request(rr + RS);
    __syncthreads();
    const int nrow = std::min<int>(RS, r1 - rr);   // the rows past it hold zeros
#pragma unroll 8
    for (int k4 = 0; k4 < nrow; k4 += 4) {
      float a[WT], b[WT];
#pragma unroll
      for (int t = 0; t < WT; ++t) a[t] = gs[(k4 + q) * TPAD + wo + 16 * t + r];
#pragma unroll
      for (int j = 0; j < WT; ++j) b[j] = ys[(k4 + q) * TPAD + wi + 16 * j + r];
#pragma unroll
      for (int t = 0; t < WT; ++t)
#pragma unroll
        for (int j = 0; j < WT; ++j) accm[t][j] = mfma16x16x4(a[t], b[j], accm[t][j]);
    }
  }
  float* ps = part + ((int64_t)s * P + p) * O * I;
#pragma unroll
  for (int t = 0; t < WT; ++t)
#pragma unroll
    for (int jj = 0; jj < 4; ++jj) {
      const int o = o0 + wo + 16 * t + 4 * q + jj;
      if (o >= O) continue;
#pragma unroll
      for (int j = 0; j < WT; ++j) {
        const int i = i0 + wi + 16 * j + r;
        if (i < I) ps[(int64_t)o * I + i] = accm[t][j][jj];
      }
    }
}

// ---------------------------------------------------------------- channel mix, fp32, whole weight matrix resident
// For at most 16 T input and output channels (T 2, 4, 8) one path's weight matrix fits in LDS (70 KB at 128
// channels, two blocks a CU): it is staged once a block, and the four waves then walk row tiles of their own with
// no barrier, the next tile's rows in flight during the products.  The products are split-fp16 (common.h): each column
// of the product (an output channel's weights, or an input channel's in the gradients) is scaled by the power of two of
// its own largest weight and staged as two fp16 planes, each row by the power of two of its own largest value (both
// undone on the result), 3 MFMAs of 16 cycles a 32-deep step against 8 of 32 on the fp32 MFMA, which bound the
// fp32 form of these kernels.  Error against 64 bits, 3,011 elements, outputs / gradients of the
// gates: 1.5e-7 / 2.5e-7 at 128 channels, 1.1e-7 / 1.9e-7 at 32 (fp32 MFMA: 2.1e-7 / 2.9e-7, 1.2e-7 / 3.2e-7), whatever
// the rows' and the channels' magnitudes (one scale for the whole matrix left a channel 1e-10 below the largest with
// 4e-2 of error); within one row or channel an entry keeps 2^-39 of the largest.  A row or channel with a non-finite
// entry gives non-finite results and leaves the others' alone.
// A tile is EB = 32 / K whole batch elements (row e K + k), so that a tile's outputs are contiguous.
// 60,011 elements, K 7, 128 x 128, sliced kernels / resident with fp32 products / this: forward 260 / 214 / 118 us,
// gate gradient 272 / 210 / 165, input gradient 171 + 5 / 190 / 168 (the last two read go in 4-byte pieces, element
// columns 4 K apart, and wait for them); 20,011 at 64 x 64: 54 / 34 / 27, 51 / 36 / 27, 41 + 5 / 38 / 35.
struct TileRow {   // element of the tile and row in it; the rows past EB K repeat the first
  int el, k;
  bool ok;
};
// v / K for 0 <= v <= 512 and K <= 32 with mg = 65536 / K + 1 (the excess v / 65536 stays below 1 / K)
__device__ __forceinline__ int div_k(int v, uint32_t mg) { return (int)(((uint32_t)v * mg) >> 16); }
__device__ __forceinline__ TileRow tile_row(int rho, int K, uint32_t mg, int EB) {
  const int el = div_k(rho, mg);
  const bool ok = el < EB;
  return {ok ? el : 0, ok ? rho - el * K : 0, ok};
}

__device__ __forceinline__ float finite_abs(float v) { return fabsf(v) <= 3.402823466e38f ? fabsf(v) : 0.f; }

// k with max |x| 2^k in [2^13, 2^14) for the largest finite |x| of a row or column (0 where that is 0), at most 127:
// below 2^-113 the scaled values are multiples of 2^-22 all the same, so nothing is lost.
__device__ __forceinline__ int split_exponent(float mx) {
  if (!(mx > 0.f)) return 0;
  int e;
  frexpf(mx, &e);   // mx = f 2^e, f in [0.5, 1)
  return min(14 - e, 127);
}
__device__ __forceinline__ float pow2_of(int k) { return __int_as_float((k + 127) << 23); }   // -126 <= k <= 127

// The factor gate 2^e of a row of results as a float and, in e, the exponent left over, 0 unless it is beyond 2^+-60.
// A result's factor is the product of a row's, a column's and a gate's, which taken together can leave the range where
// the result does not; its sum of scaled products lies in 2^-48 .. 2^35, so the float may be applied first.
__device__ __forceinline__ float row_factor(float gate, int& e) {
  int eg;
  const float m = frexpf(gate, &eg);
  const int all = e + eg, part = min(max(all, -60), 60);
  e = all - part;
  return m * pow2_of(part);
}

// The largest v >= 0 of each group of G = 8, 16 or 32 consecutive lanes, in all of them, without LDS (shuffles for each
// of a thread's 16 rows cost 3 us a launch at 128 channels).
template <int CTRL>
__device__ __forceinline__ float dpp_max(float v) {
  return fmaxf(v, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xF, 0xF, true)));
}
template <int G>
__device__ __forceinline__ float group_max(float v) {
  v = dpp_max<0xB1>(v);    // lanes 1 0 3 2 of each four
  v = dpp_max<0x4E>(v);    // lanes 2 3 0 1
  v = dpp_max<0x141>(v);   // mirrored eight
  if constexpr (G >= 16) v = dpp_max<0x140>(v);   // mirrored sixteen
  if constexpr (G >= 32) {   // rows 0 and 1, 2 and 3 of sixteen lanes
    typedef unsigned u2 __attribute__((ext_vector_type(2)));
    const unsigned x = __float_as_uint(v);
    const u2 w = __builtin_bit_cast(u2, __builtin_amdgcn_permlane16_swap(x, x, false, false));
    v = fmaxf(__uint_as_float(w.x), __uint_as_float(w.y));
  }
  return v;
}

// The matrix W [O][I] in LDS as two fp16 planes, zero beyond its size: ws[plane][o][i], or transposed (TRANS) with
// column i of the product in row 16 (i % T) + i / T, so that a lane's T tiles are T consecutive columns.  Each column
// of the product (row o, or column i, of W) is scaled by the power of two of its own largest finite entry; ex[row of
// ws] is the exponent that undoes it.  Ends with a barrier.
template <int T, bool TRANS>
__device__ __forceinline__ void stage_matrix(const float* __restrict__ W, int O, int I,
                                             _Float16 (&ws)[2][16 * T][16 * T + 8], int (&ex)[16 * T],
                                             float (&red)[TRANS ? 4 : 1][16 * T]) {
  typedef _Float16 h4 __attribute__((ext_vector_type(4)));
  constexpr int NP = T * T / 4;
  const int i = 4 * (threadIdx.x % (4 * T));   // the thread's four columns; rows o of piece s below
  auto row = [&](int s) { return (int)(threadIdx.x + 256 * s) / (4 * T); };
  f4 v[NP];
#pragma unroll
  for (int s = 0; s < NP; ++s) v[s] = ld4u(W + (row(s) < O && i < I ? (int64_t)row(s) * I + i : 0));
#pragma unroll
  for (int s = 0; s < NP; ++s)
    if (!(row(s) < O && i < I)) v[s] = f4{0.f, 0.f, 0.f, 0.f};
  float sc[TRANS ? 4 : NP];   // the scale of column i + u (TRANS) or of row(s)
  if constexpr (TRANS) {
    float mx[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < 4; ++u) {
#pragma unroll
      for (int s = 0; s < NP; ++s) mx[u] = fmaxf(mx[u], finite_abs(v[s][u]));
#pragma unroll
      for (int off = 32; off >= 4 * T; off >>= 1) mx[u] = fmaxf(mx[u], __shfl_xor(mx[u], off, 64));
    }
    if ((threadIdx.x & 63) < 4 * T) st4(&red[threadIdx.x >> 6][i], f4{mx[0], mx[1], mx[2], mx[3]});
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int k = split_exponent(fmaxf(fmaxf(red[0][i + u], red[1][i + u]), fmaxf(red[2][i + u], red[3][i + u])));
      sc[u] = pow2_of(k);
      if (threadIdx.x < 4 * T) ex[16 * ((i + u) % T) + (i + u) / T] = -k;
    }
  } else {
    int ks[NP];
#pragma unroll
    for (int s = 0; s < NP; ++s) {   // 4 T consecutive lanes hold a row
      const float m4 =
          fmaxf(fmaxf(finite_abs(v[s][0]), finite_abs(v[s][1])), fmaxf(finite_abs(v[s][2]), finite_abs(v[s][3])));
      ks[s] = split_exponent(group_max<4 * T>(m4));
      sc[s] = pow2_of(ks[s]);
    }
    if (i == 0) {
#pragma unroll
      for (int s = 0; s < NP; ++s) ex[row(s)] = -ks[s];
    }
  }
#pragma unroll
  for (int s = 0; s < NP; ++s) {
    const int o = row(s);
    h4 h, l;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const float x = v[s][u] * sc[TRANS ? u : s];
      h[u] = (_Float16)x;
      l[u] = (_Float16)(x - (float)h[u]);
    }
    if constexpr (TRANS) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        ws[0][16 * ((i + u) % T) + (i + u) / T][o] = h[u];
        ws[1][16 * ((i + u) % T) + (i + u) / T][o] = l[u];
      }
    } else {
      *reinterpret_cast<h4*>(&ws[0][o][i]) = h;
      *reinterpret_cast<h4*>(&ws[1][o][i]) = l;
    }
  }
  __syncthreads();
}

// MODE 0: out[b][o][k] (+)= g[b] sum_i y[b][k][i] W[o][i]  (one path; src = y)
// MODE 1: grad_g[b][p] (+)= sum_{k,i} y[b][p][k][i] u[b][k][i], u = sum_o go[b][o][k] W[p][o][i]  (path blockIdx.y,
//         src = go; contracting over o first meets y, whose rows are contiguous, after the products)
// MODE 2: grad_y[b][p][k][i] (+)= g[b][p] u[b][k][i]  (path blockIdx.y, src = go)
template <int T, int MODE>
__global__ __launch_bounds__(256, 2) void mix32_resident_kernel(Dims d, int EB, const float* __restrict__ src,
                                                                const float* __restrict__ W,
                                                                const float* __restrict__ g,
                                                                const float* __restrict__ y, float* __restrict__ dst,
                                                                int acc) {
  constexpr int BLD = 36, HS = T / 2;   // HS: 32-deep contraction steps
  __shared__ __align__(16) _Float16 ws[2][16 * T][16 * T + 8];
  __shared__ __align__(16) float red[MODE != 0 ? 4 : 1][16 * T];
  __shared__ int ex[16 * T];   // undoes the scale of a column of the product
  __shared__ __align__(16) float tr[MODE == 2 ? 1 : 4][MODE == 0 ? 16 * BLD : 32];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, q = lane >> 4;
  const int K = d.K, P = d.P, I = d.I, O = d.O, p = MODE == 0 ? 0 : (int)blockIdx.y;
  stage_matrix<T, MODE != 0>(W + (int64_t)p * O * I, O, I, ws, ex, red);
  const int nk = MODE != 0 ? O : I;                                   // contraction length
  const int64_t sstride = MODE != 0 ? (int64_t)O * K : (int64_t)K * I;   // an element of src
  const uint32_t mg = 65536u / (uint32_t)K + 1;
  const TileRow ar[2] = {tile_row(r, K, mg, EB), tile_row(16 + r, K, mg, EB)};
  const int64_t ntiles = (d.B + EB - 1) / EB, tstep = (int64_t)gridDim.x * 4;
  f4 a[2][T];   // the lane's rows: contraction steps 32 h + 8 q + 4 e .. + 3 in a[.][2 h + e]
  float gt[2] = {1.f, 1.f};
  auto request = [&](int64_t tile) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int64_t b = std::min<int64_t>(tile * EB + ar[t].el, d.B - 1);
      if constexpr (MODE == 0) gt[t] = g[b];
      const float* sp = src + b * sstride + (MODE != 0 ? ar[t].k : ar[t].k * I);
#pragma unroll
      for (int h = 0; h < T; ++h) {
        const int k = 32 * (h >> 1) + 8 * q + 4 * (h & 1), kc = k < nk ? k : 0;
        if constexpr (MODE != 0) {
#pragma unroll
          for (int u = 0; u < 4; ++u) a[t][h][u] = sp[(int64_t)(kc + u) * K];
        } else {
          a[t][h] = ld4u(sp + kc);
        }
      }
    }
  };
  int64_t tile = (int64_t)blockIdx.x * 4 + wave;
  if (tile >= ntiles) return;   // no barrier follows
  request(tile);
  for (; tile < ntiles; tile += tstep) {
    // the rows split, each by the power of two of its largest finite value (its values sit in four lanes); er undoes it
    h8 xh[2][HS], xl[2][HS];
    int er[2];
    float fr[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      float mx = 0.f;
#pragma unroll
      for (int h = 0; h < T; ++h) {
        if (32 * (h >> 1) + 8 * q + 4 * (h & 1) >= nk) a[t][h] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int u = 0; u < 4; ++u) mx = fmaxf(mx, finite_abs(a[t][h][u]));
      }
      mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
      mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
      const int kr = split_exponent(mx);
      const float sr = pow2_of(kr);
#pragma unroll
      for (int h = 0; h < HS; ++h) {
        const float v[8] = {a[t][2 * h][0],     a[t][2 * h][1],     a[t][2 * h][2],     a[t][2 * h][3],
                            a[t][2 * h + 1][0], a[t][2 * h + 1][1], a[t][2 * h + 1][2], a[t][2 * h + 1][3]};
        split2h(v, sr, xh[t][h], xl[t][h]);
      }
      er[t] = -kr;
      if constexpr (MODE == 0) fr[t] = row_factor(gt[t], er[t]);
    }
    __builtin_amdgcn_sched_barrier(0);
    request(std::min(tile + tstep, ntiles - 1));
    __builtin_amdgcn_sched_barrier(0);
    f4 accm[2][T];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int j = 0; j < T; ++j) accm[t][j] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int h = 0; h < HS; ++h)
#pragma unroll
      for (int j = 0; j < T; ++j) {
        const h8 wh = *reinterpret_cast<const h8*>(&ws[0][16 * j + r][32 * h + 8 * q]);
        const h8 wl = *reinterpret_cast<const h8*>(&ws[1][16 * j + r][32 * h + 8 * q]);
#pragma unroll
        for (int t = 0; t < 2; ++t) accm[t][j] = mfma_x3(xh[t][h], xl[t][h], wh, wl, accm[t][j]);
      }
    int ew[T];
#pragma unroll
    for (int j = 0; j < T; ++j) ew[j] = ex[16 * j + r];
    const int64_t b0 = tile * EB;
    const int nel = (int)std::min<int64_t>(EB, d.B - b0);
    uint32_t mge = mg;
    asm volatile("" : "+s"(mge));   // row indices are formed anew for each tile, not held across the products
    // result register jj of lane group q is row 4 q + jj of the tile: its exponent and gate are held by lane 4 q + jj
    if constexpr (MODE == 0) {
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) {
          const float f = __shfl(fr[t], 4 * q + jj, 64);
#pragma unroll
          for (int j = 0; j < T; ++j) accm[t][j][jj] = ldexpf(accm[t][j][jj] * f, ew[j]);
        }
      if (__ballot(er[0] | er[1])) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int jj = 0; jj < 4; ++jj) {
            const int e = __shfl(er[t], 4 * q + jj, 64);
#pragma unroll
            for (int j = 0; j < T; ++j) accm[t][j][jj] = ldexpf(accm[t][j][jj], e);
          }
      }
      // out[b][o][k] holds an element's rows side by side: 16 columns at a time turn through LDS and leave in runs
      // of 16 K floats an element (a store per register would write 4 bytes every 4 K)
      float* ob = dst + b0 * O * K;
      int lo[8], oo[8], cc[8];   // place in LDS, place in the output and column of the lane's 8 values of a slice
      {
        const int run = 16 * K;
        int el = div_k(lane >> 4, mge), rem = lane - el * run, c = div_k(rem, mge), k = rem - c * K;
        const int dk = 64 - div_k(64, mge) * K, dc = div_k(64, mge);
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          lo[u] = c * BLD + el * K + k;
          oo[u] = (el * O + c) * K + k;
          cc[u] = el < nel ? c : 1 << 20;
          k += dk;   // 64 values on, with carries
          c += dc;
          if (k >= K) { k -= K; ++c; }
          while (c >= 16) { c -= 16; ++el; }
        }
      }
#pragma unroll
      for (int j = 0; j < T; ++j) {
        __builtin_amdgcn_wave_barrier();   // the LDS operations of a wave are in order
#pragma unroll
        for (int t = 0; t < 2; ++t) st4(&tr[wave][r * BLD + 16 * t + 4 * q], accm[t][j]);
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int u = 0; u < 8; ++u)
          if (cc[u] + 16 * j < O) put(ob + oo[u] + 16 * j * K, tr[wave][lo[u]], acc);
      }
    } else if constexpr (MODE == 1) {
      float rowsum[8];
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) {
          // the row's exponent is undone on its sum (the row at most 1 until then): y W is in range where go W need
          // not be
#pragma unroll
          for (int j = 0; j < T; ++j) accm[t][j][jj] = ldexpf(accm[t][j][jj], ew[j] - 14);
          const TileRow w = tile_row(16 * t + 4 * q + jj, K, mge, EB);
          const float* yp = y + (((b0 + (w.el < nel ? w.el : 0)) * P + p) * K + w.k) * I;
          float v = 0.f;
          if constexpr (T >= 4) {
#pragma unroll
            for (int hh = 0; hh < T / 4; ++hh) {
              const bool iv = T * r + 4 * hh < I;   // I % 4 == 0
              const f4 yv = ld4u(yp + (iv ? T * r + 4 * hh : 0));
#pragma unroll
              for (int u = 0; u < 4; ++u) v += iv ? accm[t][4 * hh + u][jj] * yv[u] : 0.f;
            }
          } else {
#pragma unroll
            for (int j = 0; j < T; ++j) {
              const int i = T * r + j;
              const float yv = yp[std::min(i, I - 1)];
              v += i < I ? accm[t][j][jj] * yv : 0.f;
            }
          }
          rowsum[4 * t + jj] = ldexpf(v, __shfl(er[t], 4 * q + jj, 64) + 14);
          if (jj & 1) __builtin_amdgcn_sched_barrier(0);   // two rows of y in flight, not all eight (registers)
        }
      // over the 16 column lanes by halving exchanges: lane bits 3, 2, 1 choose the half of the rows kept
#pragma unroll
      for (int n = 4, off = 8; n > 0; n >>= 1, off >>= 1) {
        const bool hi = lane & off;
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (i < n) {
            const float mine = hi ? rowsum[i + n] : rowsum[i], other = hi ? rowsum[i] : rowsum[i + n];
            rowsum[i] = mine + __shfl_xor(other, off, 64);
          }
      }
      rowsum[0] += __shfl_xor(rowsum[0], 1, 64);
      const int i8 = (lane >> 1) & 7;   // 4 t + jj of the row this lane holds
      __builtin_amdgcn_wave_barrier();
      if (!(lane & 1)) tr[wave][16 * (i8 >> 2) + 4 * q + (i8 & 3)] = rowsum[0];
      __builtin_amdgcn_wave_barrier();
      if (lane < nel) {
        float v = 0.f;
        for (int k = 0; k < K; ++k) v += tr[wave][lane * K + k];
        put(dst + (b0 + lane) * P + p, v, acc);
      }
    } else {
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) {
          const int e0 = __shfl(er[t], 4 * q + jj, 64);
          const TileRow w = tile_row(16 * t + 4 * q + jj, K, mge, EB);
          if (!w.ok || w.el >= nel) continue;
          const int64_t b = b0 + w.el;
          int e = e0;
          const float f = row_factor(g[b * P + p], e);
          float* o = dst + ((b * P + p) * K + w.k) * I + T * r;
          if constexpr (T >= 4) {
#pragma unroll
            for (int hh = 0; hh < T / 4; ++hh)
              if (T * r + 4 * hh < I) {   // I % 4 == 0
                f4 v;
#pragma unroll
                for (int u = 0; u < 4; ++u) v[u] = ldexpf(accm[t][4 * hh + u][jj] * f, e + ew[4 * hh + u]);
                if (acc) v = ld4u(o + 4 * hh) + v;
                st4u(o + 4 * hh, v);
              }
          } else {
#pragma unroll
            for (int j = 0; j < T; ++j)
              if (T * r + j < I) put(o + j, ldexpf(accm[t][j][jj] * f, e + ew[j]), acc);
          }
        }
    }
  }
}

// ---------------------------------------------------------------- host side
int check_dims(const Dims& d, bool proj) {
  FSC_CHECK_ARG(d.B >= 0 && d.I > 0 && d.P > 0 && d.K > 0, "bucket op: sizes must be positive");
  FSC_CHECK_ARG(d.B * d.K < (1LL << 31) && d.B * (int64_t)d.P * d.K * d.I < (1LL << 46), "bucket op: batch too large");
  if (proj) {
    FSC_CHECK_ARG(d.m1 > 0 && d.m1 <= MAXM && d.m2 > 0 && d.m2 <= MAXM, "bucket projection: m1 and m2 must be in 1..9");
    FSC_CHECK_ARG(d.P * d.K <= MAXPK, "bucket projection: P*kdim must be <= 64");
  } else {
    FSC_CHECK_ARG(d.O > 0 && d.I % 4 == 0 && d.O % 4 == 0, "bucket channel mix: mul_in1 and mul_out must be multiples of 4");
    FSC_CHECK_ARG(d.K <= 128, "bucket channel mix: kdim must be <= 128");
  }
  return 0;
}

unsigned batch_grid(int64_t B) { return (unsigned)std::max<int64_t>(1, std::min<int64_t>((B + 3) / 4, 4096)); }

size_t proj_t_lds(const Dims& d, bool do_u, size_t elem) {
  const int PK = d.P * d.K, MN = d.m1 * d.m2;
  const size_t main = (size_t)(MN * PK + 4 * (IC * d.m1 + IC * (PK + 1) + d.m1 * PK)) * elem;
  return do_u ? std::max(main, (size_t)4 * MN * PK * elem) : main;
}

// Tile width of the resident form, 0 where it does not apply: channels within one matrix of 128 x 128, an element's K
// rows within a tile of 32.  Whole elements leave rows of a tile empty (15 of 32 at K 17), which costs less than the
// other forms.  210,000 rows, resident / others, us, forward, input gradient, gate gradient: 128 channels, K 16 51 / 97,
// 55 / 80, 56 / 116, K 17 65 / 102, 75 / 82, 88 / 133, K 11 60 / 100, 78 / 83, 84 / 121; 64 channels, K 17 35 / 55,
// 33 / 49, 38 / 64; 32 channels, K 17 18 / 31, 20 / 33, 35 / 39.
int resident_width(const Dims& d) {
  const int c = std::max(d.I, d.O);
  if (d.K > 32 || c > 128) return 0;
  return c <= 32 ? 2 : c <= 64 ? 4 : 8;
}

// The forward slice by slice: enough workgroups that the slices' barriers are covered by other blocks, and channels
// that leave less than half of the last 32-step slice empty.  Against every wave for itself (mix_kernel), us, three
// paths: 128 channels, K 7, 55 workgroups 41 / 44, K 17, 133: 46 / 47, K 5, 391: 82 / 76, K 7, 547: 121 / 103; 144
// channels, K 64, 1,000 workgroups: 161 / 175; 4 channels, K 7, 547: 19 / 25.
bool mix_sliced(const Dims& d, int64_t workgroups) { return workgroups >= 320 && (d.I % 32 == 0 || d.I % 32 > 16); }

template <int MODE>
void launch_resident(const Dims& d, int t, const float* src, const float* w, const float* g, const float* y, float* dst,
                     int acc, hipStream_t st) {
  const int eb = 32 / d.K;
  const int64_t blocks = ((d.B + eb - 1) / eb + 3) / 4, paths = MODE == 0 ? 1 : d.P;
  // as many blocks as are resident at once: the matrix is staged once in each
  const int64_t cap = std::max<int64_t>(1, (t == 8 ? 512 : t == 4 ? 1024 : 2048) / paths);
  const dim3 grid((unsigned)std::min(blocks, cap), (unsigned)paths);
  if (t == 8)
    mix32_resident_kernel<8, MODE><<<grid, 256, 0, st>>>(d, eb, src, w, g, y, dst, acc);
  else if (t == 4)
    mix32_resident_kernel<4, MODE><<<grid, 256, 0, st>>>(d, eb, src, w, g, y, dst, acc);
  else
    mix32_resident_kernel<2, MODE><<<grid, 256, 0, st>>>(d, eb, src, w, g, y, dst, acc);
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

template <typename T>
size_t project_tv_lds(const Dims& d) { return (size_t)d.m2 * 256 * ((d.P * d.K + 15) / 16) * sizeof(T); }
// whole aligned 4-vectors of channels, and the padded factor within 64 KB (only fp64 at m2 9, PK > 48 exceeds it)
template <typename T>
bool project_tv_ok(const Dims& d, const T* gy) {
  return d.I % 4 == 0 && aligned16(gy) && project_tv_lds<T>(d) <= 65536;
}

template <typename T>
void launch_project_tv(const Dims& d, const T* gy, const T* a, const T* u, T* grad_v, int acc, hipStream_t st) {
  const int nt = (d.P * d.K + 15) / 16;
  const size_t lds = project_tv_lds<T>(d);
  const unsigned grid = std::min(batch_grid(d.B), 2048u);   // resident at once: the factor is staged once a block
  if (nt == 1)
    project_tv_kernel<T, 1><<<grid, 256, lds, st>>>(d, gy, a, u, grad_v, acc);
  else if (nt == 2)
    project_tv_kernel<T, 2><<<grid, 256, lds, st>>>(d, gy, a, u, grad_v, acc);
  else if (nt == 3)
    project_tv_kernel<T, 3><<<grid, 256, lds, st>>>(d, gy, a, u, grad_v, acc);
  else
    project_tv_kernel<T, 4><<<grid, 256, lds, st>>>(d, gy, a, u, grad_v, acc);
}

// ---------------------------------------------------------------- entry points, for T = float and double
template <typename T>
int project(int64_t B, int32_t I, int32_t m1, int32_t m2, int32_t P, int32_t K, const T* a, const T* v, const T* u,
            T* y, int32_t accumulate, hipStream_t st) {
  const Dims d{B, I, m1, m2, P, K, 0};
  if (check_dims(d, true)) return 1;
  if (B == 0) return 0;
  const size_t lds = (size_t)(m1 * m2 * P * K + 4 * MAXM * P * K) * sizeof(T);
  if (accumulate)
    project_kernel<T, false, true><<<batch_grid(B), 256, lds, st>>>(d, a, v, u, y);
  else
    project_kernel<T, false, false><<<batch_grid(B), 256, lds, st>>>(d, a, v, u, y);
  return check_launch("bucket project") ? 2 : 0;
}

template <typename T>
int project_transpose_a(int64_t B, int32_t I, int32_t m1, int32_t m2, int32_t P, int32_t K, const T* grad_y,
                        const T* v, const T* u, T* grad_a, int32_t accumulate, hipStream_t st) {
  const Dims d{B, I, m1, m2, P, K, 0};
  if (check_dims(d, true)) return 1;
  if (B == 0) return 0;
  const size_t lds = (size_t)(m1 * m2 * P * K + 4 * MAXM * P * K) * sizeof(T);
  if (accumulate)
    project_kernel<T, true, true><<<batch_grid(B), 256, lds, st>>>(d, grad_y, v, u, grad_a);
  else
    project_kernel<T, true, false><<<batch_grid(B), 256, lds, st>>>(d, grad_y, v, u, grad_a);
  return check_launch("bucket project_transpose_a") ? 2 : 0;
}

int project_workspace(int64_t B, int32_t I, int32_t m1, int32_t m2, int32_t P, int32_t K, int64_t* workspace_elems) {
  const Dims d{B, I, m1, m2, P, K, 0};
  if (check_dims(d, true)) return 1;
  FSC_CHECK_ARG((int64_t)m1 * m2 * P * K <= 64 * UREG, "bucket projection: m1*m2*P*kdim must be <= 2048");
  *workspace_elems = (int64_t)batch_grid(B) * m1 * m2 * P * K;
  return 0;
}

template <typename T>
int project_transpose_vu(int64_t B, int32_t I, int32_t m1, int32_t m2, int32_t P, int32_t K, const T* grad_y,
                         const T* a, const T* v, const T* u, T* grad_v, T* grad_u, int32_t accumulate, T* workspace,
                         hipStream_t st) {
  const Dims d{B, I, m1, m2, P, K, 0};
  if (check_dims(d, true)) return 1;
  FSC_CHECK_ARG(grad_v || grad_u, "bucket project_transpose: nothing requested");
  const int64_t mnpk = (int64_t)m1 * m2 * P * K;
  if (grad_u) FSC_CHECK_ARG(mnpk <= 64 * UREG && workspace, "bucket projection: m1*m2*P*kdim must be <= 2048");
  const unsigned grid = batch_grid(B);
  if (B > 0) {
    const size_t lds = proj_t_lds(d, grad_u != nullptr, sizeof(T));
    if (grad_v && grad_u)
      project_t_kernel<T, true, true><<<grid, 256, lds, st>>>(d, grad_y, a, v, u, grad_v, accumulate, workspace);
    else if (grad_v && project_tv_ok<T>(d, grad_y))
      launch_project_tv<T>(d, grad_y, a, u, grad_v, accumulate, st);
    else if (grad_v)
      project_t_kernel<T, true, false><<<grid, 256, lds, st>>>(d, grad_y, a, v, u, grad_v, accumulate, nullptr);
    else
      project_t_kernel<T, false, true><<<grid, 256, lds, st>>>(d, grad_y, a, v, u, nullptr, 0, workspace);
    if (check_launch("bucket project_transpose")) return 2;
  }
  if (grad_u) {
    // (no elements: a sum over zero parts, which writes zeros or leaves an accumulated output unchanged)
    sum_parts_kernel<T><<<sum_parts_grid(mnpk), 256, 0, st>>>(mnpk, B > 0 ? (int)grid : 0, workspace, grad_u, accumulate);
    if (check_launch("bucket project_transpose_u reduce")) return 2;
  }
  return 0;
}

template <typename T>
int mix(int64_t B, int32_t P, int32_t K, int32_t I, int32_t O, const T* y, const T* w, const T* gates, T* out,
        int32_t accumulate, hipStream_t st) {
  const Dims d{B, I, 0, 0, P, K, O};
  if (check_dims(d, false)) return 1;
  if (B == 0) return 0;
  const dim3 grid((unsigned)((B * K + 127) / 128), (unsigned)((O + 127) / 128));
  if constexpr (std::is_same_v<T, float>) {
    const int t = P == 1 ? resident_width(d) : 0;   // several paths add up in one product: below
    if (t) {
      launch_resident<0>(d, t, y, w, gates, nullptr, out, accumulate, st);
      return check_launch("bucket mix") ? 2 : 0;
    }
    if (mix_sliced(d, (int64_t)grid.x * grid.y)) {
      mix32_kernel<false><<<grid, 256, 0, st>>>(d, y, w, gates, nullptr, out, accumulate);
      return check_launch("bucket mix") ? 2 : 0;
    }
  }
  mix_kernel<T, false><<<grid, 256, 0, st>>>(d, y, w, gates, nullptr, out, accumulate);
  return check_launch("bucket mix") ? 2 : 0;
}

template <typename T>
int mix_transpose_g(int64_t B, int32_t P, int32_t K, int32_t I, int32_t O, const T* grad_out, const T* y, const T* w,
                    T* grad_g, int32_t accumulate, hipStream_t st) {
  const Dims d{B, I, 0, 0, P, K, O};
  if (check_dims(d, false)) return 1;
  if (B == 0) return 0;
  const int BB = 128 / K;
  const dim3 grid((unsigned)((B + BB - 1) / BB), (unsigned)P);
  if constexpr (std::is_same_v<T, float>) {
    if (const int t = resident_width(d)) {
      launch_resident<1>(d, t, grad_out, w, nullptr, y, grad_g, accumulate, st);
      return check_launch("bucket mix_transpose_g") ? 2 : 0;
    }
    // at most half a slice of channels in a launch that does not fill the chip: every wave for itself (4 channels, K 64,
    // one path, 64 elements: 8.2 us against 9.4; 1,000 elements in 500 workgroups: 15 against 13)
    if (d.I > 16 || (int64_t)grid.x * grid.y > 160) {
      mix32_kernel<true><<<grid, 256, 0, st>>>(d, y, w, nullptr, grad_out, grad_g, accumulate);
      return check_launch("bucket mix_transpose_g") ? 2 : 0;
    }
  }
  mix_kernel<T, true><<<grid, 256, 0, st>>>(d, y, w, nullptr, grad_out, grad_g, accumulate);
  return check_launch("bucket mix_transpose_g") ? 2 : 0;
}

// Tile of the weight gradient (16 T channels a side; the fp64 kernel's is 128 whatever T) and its row splits: about
// 768 blocks, three a CU, of at least 64 rows (256 rows a split left 700 elements on 3 to 20 blocks: 57 us, 13 now).
// The same for fp64, against 2,048 blocks of at least 256 rows: 60,011 elements, K 7, 128 channels 1,307 -> 682 us (fewer
// parts to add), 700 elements, K 3 72 -> 25, 20,011 elements of 32 channels, K 5 233 -> 142.
int mix_tw_tile(int32_t I, int32_t O) {
  const int c = std::max(I, O);
  return c <= 32 ? 2 : c <= 64 ? 4 : 8;
}
int64_t mix_tw_splits(int64_t B, int32_t P, int32_t K, int32_t I, int32_t O, int64_t* rows_per_split) {
  const int64_t R = std::max<int64_t>(B * K, 1);
  const int64_t tiles = (int64_t)P * ((O + 127) / 128) * ((I + 127) / 128);
  const int64_t want = std::max<int64_t>(1, 768 / tiles);
  int64_t rps = std::max<int64_t>(64, (R + want - 1) / want);
  rps = (rps + 31) / 32 * 32;
  *rows_per_split = rps;
  return (R + rps - 1) / rps;
}

int mix_workspace(int64_t B, int32_t P, int32_t K, int32_t I, int32_t O, int64_t* workspace_elems) {
  const Dims d{B, I, 0, 0, P, K, O};
  if (check_dims(d, false)) return 1;
  int64_t rps;
  const int64_t ns = mix_tw_splits(B, P, K, I, O, &rps);
  *workspace_elems = std::max<int64_t>(ns * P * (int64_t)O * I, (int64_t)P * O * I);
  return 0;
}

template <typename T>
int mix_transpose_y(int64_t B, int32_t P, int32_t K, int32_t I, int32_t O, const T* grad_out, const T* w,
                    const T* gates, T* grad_y, int32_t accumulate, T* workspace, hipStream_t st) {
  const Dims d{B, I, 0, 0, P, K, O};
  if (check_dims(d, false)) return 1;
  if (B == 0) return 0;
  if constexpr (std::is_same_v<T, float>) {
    if (const int t = resident_width(d)) {
      launch_resident<2>(d, t, grad_out, w, gates, nullptr, grad_y, accumulate, st);
      return check_launch("bucket mix_transpose_y") ? 2 : 0;
    }
  }
  const int64_t nw = (int64_t)P * O * I;
  transpose_w_kernel<T><<<(unsigned)std::min<int64_t>((nw + 255) / 256, 4096), 256, 0, st>>>(P, O, I, w, workspace);
  if (check_launch("bucket transpose_w")) return 2;
  const dim3 grid((unsigned)((B * K + 127) / 128), (unsigned)(P * ((I + 127) / 128)));
  // at most 16 channels on both sides leave most of a slice and of a lane's eight columns empty: every wave for itself
  // (16 channels, K 64, 20,000 elements: 107 us against 138)
  if constexpr (std::is_same_v<T, float>)
    if (std::max(I, O) > 16) {
      mix32_ty_kernel<<<grid, 256, 0, st>>>(d, grad_out, workspace, gates, grad_y, accumulate);
      return check_launch("bucket mix_transpose_y") ? 2 : 0;
    }
  mix_ty_kernel<T><<<grid, 256, 0, st>>>(d, grad_out, workspace, gates, grad_y, accumulate);
  return check_launch("bucket mix_transpose_y") ? 2 : 0;
}

template <typename T>
int mix_transpose_w(int64_t B, int32_t P, int32_t K, int32_t I, int32_t O, const T* grad_out, const T* y,
                    const T* gates, T* grad_w, int32_t accumulate, T* workspace, hipStream_t st) {
  const Dims d{B, I, 0, 0, P, K, O};
  if (check_dims(d, false)) return 1;
  const int64_t nw = (int64_t)P * O * I;
  if (B == 0) {   // a sum over zero parts
    sum_parts_kernel<T><<<sum_parts_grid(nw), 256, 0, st>>>(nw, 0, workspace, grad_w, accumulate);
    return check_launch("bucket mix_transpose_w") ? 2 : 0;
  }
  int64_t rps;
  const int64_t ns = mix_tw_splits(B, P, K, I, O, &rps);
  const dim3 grid((unsigned)ns, (unsigned)P, (unsigned)(((O + 127) / 128) * ((I + 127) / 128)));
  if constexpr (std::is_same_v<T, float>)
    switch (mix_tw_tile(I, O)) {
      case 2: mix32_tw_kernel<2><<<grid, 256, 0, st>>>(d, grad_out, y, gates, rps, workspace); break;
      case 4: mix32_tw_kernel<4><<<grid, 256, 0, st>>>(d, grad_out, y, gates, rps, workspace); break;
      default: mix32_tw_kernel<8><<<grid, 256, 0, st>>>(d, grad_out, y, gates, rps, workspace);
    }
  else
    mix_tw_kernel<T><<<grid, 256, 0, st>>>(d, grad_out, y, gates, rps, workspace);
  if (check_launch("bucket mix_transpose_w")) return 2;
  sum_parts_kernel<T><<<sum_parts_grid(nw), 256, 0, st>>>(nw, (int)ns, workspace, grad_w, accumulate);
  return check_launch("bucket mix_transpose_w reduce") ? 2 : 0;
}

}  // namespace bucket
}  // namespace fsc

// ===================================================================== C ABI
// fsc_bucket_<op> takes float arrays, fsc_bucket_<op>_f64 double arrays; workspaces are counted in
// elements of the op's type.
using namespace fsc;

#define FSC_BUCKET_ABI(SUF, T)                                                                                        \
  extern "C" int fsc_bucket_project##SUF(int64_t B, int32_t I, int32_t m1, int32_t m2, int32_t P, int32_t K,        \
                                         const T* a, const T* v, const T* u, T* y, int32_t accumulate,               \
                                         hipStream_t st) {                                                          \
    return bucket::project<T>(B, I, m1, m2, P, K, a, v, u, y, accumulate, st);                                      \
  }                                                                                                                  \
  extern "C" int fsc_bucket_project_transpose_a##SUF(int64_t B, int32_t I, int32_t m1, int32_t m2, int32_t P,       \
                                                     int32_t K, const T* grad_y, const T* v, const T* u, T* grad_a,  \
                                                     int32_t accumulate, hipStream_t st) {                          \
    return bucket::project_transpose_a<T>(B, I, m1, m2, P, K, grad_y, v, u, grad_a, accumulate, st);                \
  }                                                                                                                  \
  extern "C" int fsc_bucket_project_transpose_vu##SUF(int64_t B, int32_t I, int32_t m1, int32_t m2, int32_t P,      \
                                                      int32_t K, const T* grad_y, const T* a, const T* v,           \
                                                      const T* u, T* grad_v, T* grad_u, int32_t accumulate,         \
                                                      T* workspace, hipStream_t st) {                               \
    return bucket::project_transpose_vu<T>(B, I, m1, m2, P, K, grad_y, a, v, u, grad_v, grad_u, accumulate,         \
                                           workspace, st);                                                          \
  }                                                                                                                  \
  extern "C" int fsc_bucket_mix##SUF(int64_t B, int32_t P, int32_t K, int32_t I, int32_t O, const T* y, const T* w, \
                                     const T* gates, T* out, int32_t accumulate, hipStream_t st) {                  \
    return bucket::mix<T>(B, P, K, I, O, y, w, gates, out, accumulate, st);                                         \
  }                                                                                                                  \
  extern "C" int fsc_bucket_mix_transpose_g##SUF(int64_t B, int32_t P, int32_t K, int32_t I, int32_t O,             \
                                                 const T* grad_out, const T* y, const T* w, T* grad_g,              \
                                                 int32_t accumulate, hipStream_t st) {                              \
    return bucket::mix_transpose_g<T>(B, P, K, I, O, grad_out, y, w, grad_g, accumulate, st);                       \
  }                                                                                                                  \
  extern "C" int fsc_bucket_mix_transpose_y##SUF(int64_t B, int32_t P, int32_t K, int32_t I, int32_t O,             \
                                                 const T* grad_out, const T* w, const T* gates, T* grad_y,          \
                                                 int32_t accumulate, T* workspace, hipStream_t st) {                \
    return bucket::mix_transpose_y<T>(B, P, K, I, O, grad_out, w, gates, grad_y, accumulate, workspace, st);        \
  }                                                                                                                  \
  extern "C" int fsc_bucket_mix_transpose_w##SUF(int64_t B, int32_t P, int32_t K, int32_t I, int32_t O,             \
                                                 const T* grad_out, const T* y, const T* gates, T* grad_w,          \
                                                 int32_t accumulate, T* workspace, hipStream_t st) {                \
    return bucket::mix_transpose_w<T>(B, P, K, I, O, grad_out, y, gates, grad_w, accumulate, workspace, st);        \
  }

FSC_BUCKET_ABI(, float)
FSC_BUCKET_ABI(_f64, double)
#undef FSC_BUCKET_ABI

extern "C" int fsc_bucket_project_workspace(int64_t B, int32_t I, int32_t m1, int32_t m2, int32_t P, int32_t K,
                                            int64_t* workspace_floats) {
  return bucket::project_workspace(B, I, m1, m2, P, K, workspace_floats);
}

extern "C" int fsc_bucket_mix_workspace(int64_t B, int32_t P, int32_t K, int32_t I, int32_t O, int64_t* workspace_floats) {
  return bucket::mix_workspace(B, P, K, I, O, workspace_floats);
}
