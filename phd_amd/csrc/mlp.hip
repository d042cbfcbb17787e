// mlp.hip -- BF16 matrix-core kernels of the chemistry surrogate MLP
// (12 -> 256 -> 256 -> 256 -> 10, GELU) for CDNA4 (gfx950): forward with
// fused bias + GELU, backward (data and weight gradients, bias sums),
// loss gradient and Adam.  Operands are BF16 (raw 16-bit storage),
// accumulation FP32 on v_mfma_f32_16x16x32_bf16.  The surrogate has no
// counterpart in the reference; it replaces PSR_CHEMKIN/DVODE substeps
// (chemkin/psr_chemkin.f:1) for the cells its error indicator accepts.
#include "izem_ctx.h"

#include <stdint.h>

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
// four floats where the caller's pointer need not be 16-byte aligned
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
typedef uint16_t u16;

#define MT 128  // tile rows (M)
#define NT 64   // tile columns (N)
#define KT 64   // tile depth (K), two MFMA 16x16x32 per wave sub-tile
#define KSL 32  // granularity of a split-K slice
#define LDT 72  // LDS row stride in bf16 (144 B: 16-byte aligned rows)

enum {
  EPI_F32 = 0,
  EPI_BIAS_GELU = 1,
  EPI_BIAS_F32 = 2,
  EPI_GELU_BWD = 3,
  EPI_GELU_ONLY = 5,  // inference: gelu(AB + bias) as bf16, no pre-activation kept
  EPI_PARTIAL = 4
};

__device__ inline float bf2f(u16 h) { return __uint_as_float(((unsigned)h) << 16); }
__device__ inline u16 f2bf(float f) {
  // round to nearest even: one v_cvt_pk_bf16_f32 on gfx950
  return __builtin_bit_cast(u16, (__bf16)f);
}
// erf by Abramowitz & Stegun, Handbook of Mathematical Functions, 7.1.26:
// erf(x) = 1 - t (a1 + t (a2 + t (a3 + t (a4 + t a5)))) exp(-x^2) with
// t = 1 / (1 + p x), absolute error below 1.5e-7 for x >= 0, odd extension.
// Branch-free: the library erff takes a different polynomial on either side
// of |x| = 1 and a wave whose lanes straddle it runs both; its extra accuracy
// is lost in the BF16 activations anyway.
__device__ inline float erf_as(float x) {
  const float a = fabsf(x);
  const float t = __builtin_amdgcn_rcpf(1.0f + 0.3275911f * a);
  const float poly =
      t * (0.254829592f + t * (-0.284496736f + t * (1.421413741f + t * (-1.453152027f +
                                                                         t * 1.061405429f))));
  return copysignf(1.0f - poly * __expf(-a * a), x);
}
// z Phi(z) = max(z, 0) - |z| q(|z|) with the normal tail q(x) = 2^P(x), P a
// polynomial fitted to log2 q on [0, 6.5] with the weight x q: |z| q is within
// 4e-8 of the tail term everywhere (tests/test_mlp_cpu.py), and z Phi(z) within
// that and half an ulp of the result (the erf form above: 7e-7).  P's
// leading coefficient is negative, so q goes to 0 beyond 6.5.  Ten operations and
// one exponential where the erf form takes twenty, a reciprocal and an
// exponential: the activations bind k_mlp_fused as much as the products.
// The finite bound keeps inf for z = inf; a NaN in z comes through q (the
// median is the maximum and the minimum without a canonicalising move first).
__device__ inline float gelu(float z) {
  const float x = fabsf(z);
  float p = -1.7058535205505265e-06f;
  p = fmaf(p, x, 2.5302828325801663e-05f);
  p = fmaf(p, x, -0.00011573545561732734f);
  p = fmaf(p, x, -0.0003194422878719516f);
  p = fmaf(p, x, 0.0073265519719698385f);
  p = fmaf(p, x, -0.052707288790111675f);
  p = fmaf(p, x, -0.4591193039890919f);
  p = fmaf(p, x, -1.1511221964207652f);
  p = fmaf(p, x, -0.9999989806607171f);
  const float inf = __builtin_inff(), big = 3.402823466e38f;
  return fmaf(-fabsf(__builtin_amdgcn_fmed3f(z, -inf, big)), __builtin_amdgcn_exp2f(p),
              __builtin_amdgcn_fmed3f(z, 0.0f, inf));
}
__device__ inline float gelu_d(float z) {
  return 0.5f * (1.0f + erf_as(z * 0.70710678118654752f)) +
         z * 0.39894228040143268f * __expf(-0.5f * z * z);
}

// An R x 64 tile (rows r0.., depth k0..) of the logical matrix X[R][Kd], in
// registers between its load from memory and its store to lds[r][k], so that
// the next tile's loads are in flight during the products of this one.
// TR = 0: X stored row-major X[r*ld + k] (k contiguous), 16 bytes a load;
// TR = 1: X stored transposed X[k*ld + r] (r contiguous): four 8-byte rows of
// a 4 x 4 block, transposed in registers, so that the store has four depths
// of a row in 8 bytes.  Out-of-range elements are zero; a matrix whose rows
// are not aligned for the wide load is read element by element.
template <int TR, int R>
struct Tile {
  static constexpr int P = TR == 0 ? R / 32 : R / 64;  // passes of the 256 threads
  uint4 q[TR == 0 ? P : 2 * P];
  // TR = 1: a wave takes 8 x 8 blocks (32 rows, 32 depths): its loads are 64
  // contiguous bytes, and its stores, 144 bytes apart in rows and 8 in depths,
  // meet each bank twice in 64 lanes (32 row blocks by 2: sixteen times, and
  // the stores then bound the product of two transposed operands)
  static __device__ inline int row(int p, int t) {
    return ((p * 4 + (t >> 6)) % (R / 32)) * 32 + (t & 7) * 4;
  }
  static __device__ inline int depth(int p, int t) {
    return ((p * 4 + (t >> 6)) / (R / 32)) * 32 + ((t >> 3) & 7) * 4;
  }
  __device__ inline void load(const u16 *__restrict__ X, long ld, int rows, int Kd, int r0,
                              int k0) {
    const int t = threadIdx.x;
    if constexpr (TR == 0) {
      const bool wide = (ld & 7) == 0 && (((uintptr_t)X) & 15) == 0;
#pragma unroll
      for (int p = 0; p < P; p++) {
        const int gr = r0 + p * 32 + (t >> 3), gk = k0 + (t & 7) * 8;
        if (wide && gr < rows && gk + 7 < Kd) {
          q[p] = *(const uint4 *)(X + (long)gr * ld + gk);
        } else {
          u16 v[8];
#pragma unroll
          for (int i = 0; i < 8; i++)
            v[i] = (gr < rows && gk + i < Kd) ? X[(long)gr * ld + gk + i] : 0;
          q[p] = make_uint4(v[0] | (unsigned)v[1] << 16, v[2] | (unsigned)v[3] << 16,
                            v[4] | (unsigned)v[5] << 16, v[6] | (unsigned)v[7] << 16);
        }
      }
    } else {
      const bool wide = (ld & 3) == 0 && (((uintptr_t)X) & 7) == 0;
#pragma unroll
      for (int p = 0; p < P; p++) {
        const int gr = r0 + row(p, t), gk = k0 + depth(p, t);
        uint2 a[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
          if (wide && gk + j < Kd && gr + 3 < rows) {
            a[j] = *(const uint2 *)(X + (long)(gk + j) * ld + gr);
          } else {
            u16 v[4];
#pragma unroll
            for (int i = 0; i < 4; i++)
              v[i] = (gk + j < Kd && gr + i < rows) ? X[(long)(gk + j) * ld + gr + i] : 0;
            a[j] = make_uint2(v[0] | (unsigned)v[1] << 16, v[2] | (unsigned)v[3] << 16);
          }
        }
        q[2 * p] = make_uint4(a[0].x, a[1].x, a[2].x, a[3].x);
        q[2 * p + 1] = make_uint4(a[0].y, a[1].y, a[2].y, a[3].y);
      }
    }
  }
  __device__ inline void store(u16 (*lds)[LDT]) const {
    const int t = threadIdx.x;
    if constexpr (TR == 0) {
#pragma unroll
      for (int p = 0; p < P; p++) *(uint4 *)&lds[p * 32 + (t >> 3)][(t & 7) * 8] = q[p];
    } else {
#pragma unroll
      for (int p = 0; p < P; p++) {
        const int r = row(p, t), k = depth(p, t);
#pragma unroll
        for (int h = 0; h < 2; h++) {
          const uint4 w = q[2 * p + h];  // rows r + 2h, r + 2h + 1 at depths k..k+3
          *(uint2 *)&lds[r + 2 * h][k] =
              make_uint2((w.x & 0xffffu) | w.y << 16, (w.z & 0xffffu) | w.w << 16);
          *(uint2 *)&lds[r + 2 * h + 1][k] =
              make_uint2(w.x >> 16 | (w.y & 0xffff0000u), w.z >> 16 | (w.w & 0xffff0000u));
        }
      }
    }
  }
};

// C[M][N] = A[M][K] . B[K][N] (+ epilogue).  A: TA = 0 row-major, 1 stored
// as [K][M]; B: TB = 0 stored as [N][K] (weights transposed), 1 stored as
// [K][N].  Block: 256 threads = 4 waves on a 128 x 64 tile, each wave a
// 64 x 32 quarter as 4 x 2 MFMA 16x16x32 accumulators.  Split-K: slice z
// takes K range [z * kslice, (z + 1) * kslice) and (EPI_PARTIAL) writes its
// partial product to Cf + z * M * ldcf.  These products are bound by their
// operands' and results' traffic (a batch of 65536 rows against 256 x 256
// weights): what matters is that loads stay in flight, hence the tile held in
// registers across the products, and 128 rows so that a row block of A is read
// by N / 64 blocks only.  The weights (or B) are the first operand of the
// matrix instruction, so that a lane ends with four consecutive columns of a
// row: 16-byte stores of FP32, 8-byte ones of BF16 where the rows allow it.
// Per product at 65536 x 256 x 256, from a 64 x 64 x 32 tile staged element by
// element: forward 40 -> 33 us, backward 50 -> 38, split-K weight gradient
// 58 -> 34, of 28, 28 and 14 at the rate of a copy.
template <int TA, int TB, int EPI>
__global__ void __launch_bounds__(256)
k_gemm(int M, int N, int K, const u16 *__restrict__ A, long lda, const u16 *__restrict__ B,
       long ldb, const float *__restrict__ bias, const float *__restrict__ aux, long ldaux,
       float *__restrict__ Cf, long ldcf, u16 *__restrict__ Cb, long ldcb, int kslice) {
  __shared__ __attribute__((aligned(16))) u16 As[MT][LDT];
  __shared__ __attribute__((aligned(16))) u16 Bs[NT][LDT];
  // workgroups go to the 8 XCDs in turn: the blocks that share a large operand
  // (the column tiles of a row tile of A; all tiles of a split-K slice) are 8
  // apart, hence on one XCD, and read it from its L2 after the first of them
  const int nt = (N + NT - 1) / NT, mt = (M + MT - 1) / MT;
  const int per = EPI == EPI_PARTIAL ? nt * mt : nt;
  const int grp = blockIdx.x / (8 * per) * 8 + blockIdx.x % 8, mem = blockIdx.x / 8 % per;
  const int z = EPI == EPI_PARTIAL ? grp : 0;
  const int m0 = (EPI == EPI_PARTIAL ? mem / nt : grp) * MT, n0 = mem % nt * NT;
  const int kb = z * kslice, ke = min(K, kb + kslice);
  if (m0 >= M || kb >= K) return;  // the last groups of 8 may be short
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int wm = w >> 1, wn = w & 1;
  f32x4 acc[4][2];
#pragma unroll
  for (int i = 0; i < 4; i++)
#pragma unroll
    for (int j = 0; j < 2; j++) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
  // a lane has row m0 + wm 64 + i 16 + lr and columns nb + j 16 .. + 3
  const int lr = lane & 15, nb = n0 + wn * 32 + (lane >> 4) * 4;
  if (EPI == EPI_BIAS_GELU || EPI == EPI_BIAS_F32 || EPI == EPI_GELU_ONLY) {
    // the bias starts the sum, as in k_mlp_fused
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int n = nb + j * 16 + r;
        const float b0 = n < N ? bias[n] : 0.f;
#pragma unroll
        for (int i = 0; i < 4; i++) acc[i][j][r] = b0;
      }
  }
  // the pre-activations of the backward epilogue, in flight during the product
  f32x4 pre[4][2];
  if (EPI == EPI_GELU_BWD) {
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
      for (int j = 0; j < 2; j++) {
        const int m = m0 + wm * 64 + i * 16 + lr, n = nb + j * 16;
        const float *x = aux + (long)m * ldaux + n;
        if (m < M && n + 3 < N) {
          pre[i][j] = *(const f32x4u *)x;
        } else {
#pragma unroll
          for (int r = 0; r < 4; r++) pre[i][j][r] = (m < M && n + r < N) ? x[r] : 0.f;
        }
      }
  }
  Tile<TA, MT> ta;
  Tile<TB == 0 ? 0 : 1, NT> tb;
  ta.load(A, lda, M, ke, m0, kb);
  tb.load(B, ldb, N, ke, n0, kb);
  for (int k0 = kb; k0 < ke; k0 += KT) {
    ta.store(As);
    tb.store(Bs);
    __syncthreads();
    if (k0 + KT < ke) {
      ta.load(A, lda, M, ke, m0, k0 + KT);
      tb.load(B, ldb, N, ke, n0, k0 + KT);
    }
#pragma unroll
    for (int h = 0; h < KT / 32; h++) {
      const int kc = h * 32 + (lane >> 4) * 8;
      bf16x8 af[4], bfr[2];
#pragma unroll
      for (int i = 0; i < 4; i++)
        af[i] = __builtin_bit_cast(bf16x8,
                                   *(const uint4 *)&As[wm * 64 + i * 16 + (lane & 15)][kc]);
#pragma unroll
      for (int j = 0; j < 2; j++)
        bfr[j] = __builtin_bit_cast(bf16x8,
                                    *(const uint4 *)&Bs[wn * 32 + j * 16 + (lane & 15)][kc]);
#pragma unroll
      for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bfr[j], af[i], acc[i][j], 0, 0, 0);
    }
    __syncthreads();
  }
  float *Cz = Cf;
  if (EPI == EPI_PARTIAL) Cz = Cf + (long)z * M * ldcf;
  const bool wideb = (ldcb & 3) == 0 && (((uintptr_t)Cb) & 7) == 0;
#pragma unroll
  for (int i = 0; i < 4; i++)
#pragma unroll
    for (int j = 0; j < 2; j++) {
      const int m = m0 + wm * 64 + i * 16 + lr, n = nb + j * 16;
      if (m >= M || n >= N) continue;
      const f32x4 a = acc[i][j];
      if (EPI != EPI_GELU_ONLY && EPI != EPI_GELU_BWD) {
        float *c = Cz + (long)m * ldcf + n;
        if (n + 3 < N) {
          *(f32x4u *)c = a;
        } else {
#pragma unroll
          for (int r = 0; r < 3; r++)
            if (n + r < N) c[r] = a[r];
        }
      }
      if (EPI == EPI_BIAS_GELU || EPI == EPI_GELU_ONLY || EPI == EPI_GELU_BWD) {
        u16 v[4];
#pragma unroll
        for (int r = 0; r < 4; r++)
          v[r] = f2bf(EPI == EPI_GELU_BWD ? a[r] * gelu_d(pre[i][j][r]) : gelu(a[r]));
        u16 *c = Cb + (long)m * ldcb + n;
        if (wideb && n + 3 < N) {
          *(uint2 *)c = make_uint2(v[0] | (unsigned)v[1] << 16, v[2] | (unsigned)v[3] << 16);
        } else {
#pragma unroll
          for (int r = 0; r < 4; r++)
            if (n + r < N) c[r] = v[r];
        }
      }
    }
}

// out[i] = sum over s of part[s * n + i] (fixed order: deterministic)
__global__ void k_sum_slices(long n, int ns, const float *__restrict__ part,
                             float *__restrict__ out) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  // loads sixteen at a time, added in order
  float s = 0.f;
#pragma unroll 16
  for (int z = 0; z < ns; z++) s += part[(long)z * n + i];
  out[i] = s;
}

// column sums of a BF16 matrix G[M][N] over row slices: part[s][n]
__global__ void k_colsum(int M, int N, const u16 *__restrict__ G, long ld, int rows,
                         float *__restrict__ part) {
  const int n = blockIdx.x * blockDim.x + threadIdx.x;
  const int s = blockIdx.y;
  if (n >= N) return;
  const int r0 = s * rows, r1 = min(M, r0 + rows);
  float a = 0.f;
  for (int r = r0; r < r1; r++) a += bf2f(G[(long)r * ld + n]);
  part[(long)s * N + n] = a;
}

// the same for N and ld multiples of 8 (16-byte rows of 8 columns): each
// thread sums 8 columns of every (1024 / (N / 8))-th row of its slice, and
// the row groups of a block are added in a fixed order, so the sums do
// not depend on timing.  The callers' slices are few (64): 1024 threads and
// four loads in flight each keep enough of the chip's memory busy.
#define CS_T 1024
__global__ void __launch_bounds__(CS_T) k_colsum8(int M, int N, const u16 *__restrict__ G, long ld,
                                                  int rows, float *__restrict__ part) {
  __shared__ float red[CS_T * 8];
  const int cpr = N / 8;               // 16-byte chunks per row
  const int rg = CS_T / cpr;           // rows per block iteration
  const int t = threadIdx.x;
  const int ch = t % cpr, g = t / cpr;
  const int s = blockIdx.x;
  const int r0 = s * rows, r1 = min(M, r0 + rows);
  float a[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  if (g < rg) {
#pragma unroll 4
    for (int r = r0 + g; r < r1; r += rg) {
      const uint4 w = *reinterpret_cast<const uint4 *>(G + (long)r * ld + ch * 8);
      const unsigned u[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
      for (int q = 0; q < 4; q++) {
        a[2 * q] += __uint_as_float(u[q] << 16);
        a[2 * q + 1] += __uint_as_float(u[q] & 0xffff0000u);
      }
    }
  }
  // column-major so that the threads below read consecutive words
#pragma unroll
  for (int q = 0; q < 8; q++) red[q * CS_T + t] = a[q];
  __syncthreads();
  // thread (column, chunk) adds the row groups in order
  if (t < N) {
    const int q = t / cpr, c = t % cpr;
    float sum = 0.f;
    for (int gg = 0; gg < rg; gg++) sum += red[q * CS_T + gg * cpr + c];
    part[(long)s * N + c * 8 + q] = sum;
  }
}

// Adam (Kingma & Ba 2015) on an FP32 master matrix P[rows][cols] (row-major)
// with gradient G, moments m, v; writes BF16 copies P^T (ldt) and P (ldw)
// when given.  Step t >= 1.
__global__ void k_adam(int rows, int cols, float *__restrict__ P, const float *__restrict__ G,
                       float *__restrict__ m, float *__restrict__ v, float lr, float b1, float b2,
                       float eps, float c1, float c2, u16 *__restrict__ Pt, long ldt,
                       u16 *__restrict__ Pw, long ldw) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (long)rows * cols) return;
  const float g = G[i];
  const float mi = b1 * m[i] + (1.f - b1) * g;
  const float vi = b2 * v[i] + (1.f - b2) * g * g;
  m[i] = mi;
  v[i] = vi;
  const float p = P[i] - lr * (mi * c1) / (sqrtf(vi * c2) + eps);
  P[i] = p;
  const int r = (int)(i / cols), c = (int)(i % cols);
  if (Pt) Pt[(long)c * ldt + r] = f2bf(p);
  if (Pw) Pw[(long)r * ldw + c] = f2bf(p);
}

// write BF16 copies of an FP32 matrix (initialisation)
__global__ void k_to_bf16(int rows, int cols, const float *__restrict__ P, u16 *__restrict__ Pt,
                          long ldt, u16 *__restrict__ Pw, long ldw) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (long)rows * cols) return;
  const int r = (int)(i / cols), c = (int)(i % cols);
  if (Pt) Pt[(long)c * ldt + r] = f2bf(P[i]);
  if (Pw) Pw[(long)r * ldw + c] = f2bf(P[i]);
}

// mean-square loss over nout of the ldp output columns: dY = 2 (pred -
// target) / (B nout) as BF16 (padding columns zero); loss sum of squares
// accumulated into *loss (one atomic per block)
__global__ void k_mse(int Bn, int nout, int npad, const float *__restrict__ pred, long ldp,
                      const float *__restrict__ tgt, long ldt, float scale,
                      u16 *__restrict__ dY, long ldd, float *__restrict__ loss) {
  __shared__ float red[4];
  // a thread keeps its column: the block walks the rows, 256 / npad at a time
  // (npad <= 256) or one by one
  float sq = 0.f;
  const int w = npad < 256 ? npad : 256, rpb = 256 / w;
  const int j0 = threadIdx.x % w, rr = threadIdx.x / w;
  if (rr < rpb) {
    for (int j = j0; j < npad; j += w)
#pragma unroll 4
      for (long b = (long)blockIdx.x * rpb + rr; b < Bn; b += (long)gridDim.x * rpb) {
        float g = 0.f;
        if (j < nout) {
          const float d = pred[b * ldp + j] - tgt[b * ldt + j];
          sq += d * d;
          g = 2.f * d * scale;
        }
        dY[b * ldd + j] = f2bf(g);
      }
  }
  for (int off = 32; off > 0; off >>= 1) sq += __shfl_xor(sq, off, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = sq;
  __syncthreads();
  if (threadIdx.x == 0) {
    float s = 0.f;
    for (int q = 0; q < (int)(blockDim.x >> 6); q++) s += red[q];
    atomicAdd(loss, s);
  }
}

// ------------------------------------------------------------------ C ABI
// groups of k_gemm's block order: as many as fill all 8 XCDs
static unsigned gemm_groups(int g) { return ((unsigned)g + 7u) / 8u * 8u; }

#define LAUNCH_GEMM(TA_, TB_, EPI_)                                                           \
  hipLaunchKernelGGL((k_gemm<TA_, TB_, EPI_>), grid, dim3(256), 0, ctx->stream, M, N, K,      \
                     (const u16 *)A, lda, (const u16 *)B, ldb, bias, aux, ldaux, Cf, ldcf,     \
                     (u16 *)Cb, ldcb, kslice)

template <int EPI>
static void gemm_dispatch(izem_ctx *ctx, dim3 grid, int ta, int tb, int M, int N, int K,
                          const void *A, long lda, const void *B, long ldb, const float *bias,
                          const float *aux, long ldaux, float *Cf, long ldcf, void *Cb,
                          long ldcb, int kslice) {
  if (!ta && !tb) LAUNCH_GEMM(0, 0, EPI);
  else if (!ta && tb) LAUNCH_GEMM(0, 1, EPI);
  else if (ta && !tb) LAUNCH_GEMM(1, 0, EPI);
  else LAUNCH_GEMM(1, 1, EPI);
}

extern "C" int izem_mlp_gemm(izem_ctx *ctx, int ta, int tb, int epi, int M, int N, int K,
                             const void *A, long lda, const void *B, long ldb,
                             const float *bias, const float *aux, long ldaux, float *Cf,
                             long ldcf, void *Cb, long ldcb) {
  if (!ctx || !A || !B || M <= 0 || N <= 0 || K <= 0 || epi < 0 || epi > 5 || epi == 4)
    return IZEM_E_ARG;
  if ((epi == EPI_BIAS_GELU || epi == EPI_BIAS_F32 || epi == EPI_GELU_ONLY) && !bias)
    return IZEM_E_ARG;
  if ((epi == EPI_BIAS_GELU || epi == EPI_GELU_BWD || epi == EPI_GELU_ONLY) && !Cb)
    return IZEM_E_ARG;
  if (epi == EPI_GELU_BWD && !aux) return IZEM_E_ARG;
  if ((epi == EPI_F32 || epi == EPI_BIAS_GELU || epi == EPI_BIAS_F32) && !Cf) return IZEM_E_ARG;
  const dim3 grid(gemm_groups((M + MT - 1) / MT) * ((N + NT - 1) / NT));
  const int ks = ((K + KSL - 1) / KSL) * KSL;
  int pk = iz_prof_begin(ctx, IZP_OTHER);
  switch (epi) {
    case EPI_F32: gemm_dispatch<EPI_F32>(ctx, grid, ta, tb, M, N, K, A, lda, B, ldb, bias, aux, ldaux, Cf, ldcf, Cb, ldcb, ks); break;
    case EPI_BIAS_GELU: gemm_dispatch<EPI_BIAS_GELU>(ctx, grid, ta, tb, M, N, K, A, lda, B, ldb, bias, aux, ldaux, Cf, ldcf, Cb, ldcb, ks); break;
    case EPI_BIAS_F32: gemm_dispatch<EPI_BIAS_F32>(ctx, grid, ta, tb, M, N, K, A, lda, B, ldb, bias, aux, ldaux, Cf, ldcf, Cb, ldcb, ks); break;
    case EPI_GELU_ONLY: gemm_dispatch<EPI_GELU_ONLY>(ctx, grid, ta, tb, M, N, K, A, lda, B, ldb, bias, aux, ldaux, Cf, ldcf, Cb, ldcb, ks); break;
    default: gemm_dispatch<EPI_GELU_BWD>(ctx, grid, ta, tb, M, N, K, A, lda, B, ldb, bias, aux, ldaux, Cf, ldcf, Cb, ldcb, ks); break;
  }
  iz_prof_end(ctx, pk);
  IZ_CHECK(hipGetLastError());
  return IZEM_OK;
}

extern "C" int izem_mlp_gemm_splitk(izem_ctx *ctx, int ta, int tb, int M, int N, int K,
                                    const void *A, long lda, const void *B, long ldb,
                                    int nslices, float *work, float *C) {
  if (!ctx || !A || !B || !work || !C || M <= 0 || N <= 0 || K <= 0 || nslices < 1)
    return IZEM_E_ARG;
  int ks = (K + nslices - 1) / nslices;
  ks = ((ks + KSL - 1) / KSL) * KSL;
  const int nz = (K + ks - 1) / ks;
  const dim3 grid(gemm_groups(nz) * ((N + NT - 1) / NT) * ((M + MT - 1) / MT));
  const float *nul = nullptr;
  gemm_dispatch<EPI_PARTIAL>(ctx, grid, ta, tb, M, N, K, A, lda, B, ldb, nul, nul, 0, work,
                             N, nullptr, 0, ks);
  const long n = (long)M * N;
  hipLaunchKernelGGL(k_sum_slices, dim3(iz_blocks(n, 256)), dim3(256), 0, ctx->stream, n, nz,
                     work, C);
  IZ_CHECK(hipGetLastError());
  return IZEM_OK;
}

extern "C" int izem_mlp_colsum(izem_ctx *ctx, int M, int N, const void *G, long ld,
                               int nslices, float *work, float *out) {
  if (!ctx || !G || !work || !out || M <= 0 || N <= 0 || nslices < 1) return IZEM_E_ARG;
  const int rows = (M + nslices - 1) / nslices;
  const int ns = (M + rows - 1) / rows;
  if (N % 8 == 0 && ld % 8 == 0 && N <= 256 && ((uintptr_t)G & 15) == 0)
    hipLaunchKernelGGL(k_colsum8, dim3(ns), dim3(CS_T), 0, ctx->stream, M, N, (const u16 *)G, ld,
                       rows, work);
  else
    hipLaunchKernelGGL(k_colsum, dim3((N + 255) / 256, ns), dim3(256), 0, ctx->stream, M, N,
                       (const u16 *)G, ld, rows, work);
  hipLaunchKernelGGL(k_sum_slices, dim3(iz_blocks(N, 256)), dim3(256), 0, ctx->stream, (long)N,
                     ns, work, out);
  IZ_CHECK(hipGetLastError());
  return IZEM_OK;
}

extern "C" int izem_mlp_adam(izem_ctx *ctx, int rows, int cols, float *P, const float *G,
                             float *m, float *v, float lr, float b1, float b2, float eps,
                             int step, void *Pt, long ldt, void *Pw, long ldw) {
  if (!ctx || !P || !G || !m || !v || rows <= 0 || cols <= 0 || step < 1) return IZEM_E_ARG;
  const float c1 = 1.f / (1.f - powf(b1, (float)step));
  const float c2 = 1.f / (1.f - powf(b2, (float)step));
  const long n = (long)rows * cols;
  hipLaunchKernelGGL(k_adam, dim3(iz_blocks(n, 256)), dim3(256), 0, ctx->stream, rows, cols, P,
                     G, m, v, lr, b1, b2, eps, c1, c2, (u16 *)Pt, ldt, (u16 *)Pw, ldw);
  IZ_CHECK(hipGetLastError());
  return IZEM_OK;
}

extern "C" int izem_mlp_to_bf16(izem_ctx *ctx, int rows, int cols, const float *P, void *Pt,
                                long ldt, void *Pw, long ldw) {
  if (!ctx || !P || rows <= 0 || cols <= 0) return IZEM_E_ARG;
  const long n = (long)rows * cols;
  hipLaunchKernelGGL(k_to_bf16, dim3(iz_blocks(n, 256)), dim3(256), 0, ctx->stream, rows, cols,
                     P, (u16 *)Pt, ldt, (u16 *)Pw, ldw);
  IZ_CHECK(hipGetLastError());
  return IZEM_OK;
}

extern "C" int izem_mlp_mse(izem_ctx *ctx, int Bn, int nout, int npad, const float *pred,
                            long ldp, const float *tgt, long ldt, void *dY, long ldd,
                            float *loss) {
  if (!ctx || !pred || !tgt || !dY || !loss || Bn <= 0 || nout <= 0 || npad < nout)
    return IZEM_E_ARG;
  const long n = (long)Bn * npad;
  const float scale = 1.f / ((float)Bn * (float)nout);
  // a few blocks per CU: one same-address atomic per block
  hipLaunchKernelGGL(k_mse, dim3(iz_blocks_capped(ctx, n, 256, 2)), dim3(256), 0, ctx->stream,
                     Bn, nout, npad,
                     pred, ldp, tgt, ldt, scale, (u16 *)dY, ldd, loss);
  IZ_CHECK(hipGetLastError());
  return IZEM_OK;
}

// -------------------------------------------------------------------
// Fused inference: all four layers of the surrogate for a tile of 128
// cells in one block.  The activations stay in one LDS buffer (128 x 256
// BF16), overwritten in place: every wave reads the whole input tile, so
// the block synchronises once after the products and once after the
// epilogue has written the layer's output.  The weights are read as MFMA
// operands straight from L2 (every block uses the same 273 KB), the
// fragments of the next 32-deep slice loaded while the current one is in
// the matrix cores.  Persistent grid over row tiles.  Weights Wt_l are
// stored [N][K] (the B operand of a 16x16x32 MFMA is then one 16-byte load
// per lane); layer widths K = 32 | 256 | 256 | 256, N = 256 | 256 | 256 | 64.
// Bound by the vector unit's activations beside the products: 2^20 cells take
// 630 us (520 TFLOP/s; 840 us with the erf form, one BF16 and one LDS write per
// element); 64 rows with 3 or 4 waves per SIMD instead of 128 with 2: 790, 825.
// -------------------------------------------------------------------
#define FX 264  // LDS row stride of an activation tile (bf16): 528 B, 16-byte aligned

template <int K, int N, bool LAST, int RB>
__device__ __forceinline__ void fused_layer(u16 (*X)[FX], const u16 *__restrict__ Wt,
                                   const float *__restrict__ b, float *__restrict__ pred,
                                   int row0, int M) {
  constexpr int NW = N / 4;        // columns per wave
  constexpr int CB = NW / 16;      // 16-column blocks per wave
  constexpr int KS = K / 32;       // 32-deep slices
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  // accumulators transposed (weights as the first operand): a lane has one
  // row m and four consecutive columns, which it stores at once
  f32x4 acc[RB][CB];
#pragma unroll
  for (int j = 0; j < CB; j++) {
    const f32x4 bj = *(const f32x4u *)(b + w * NW + j * 16 + (lane >> 4) * 4);
#pragma unroll
    for (int i = 0; i < RB; i++) acc[i][j] = bj;
  }
  const u16 *wrow[CB];
#pragma unroll
  for (int j = 0; j < CB; j++)
    wrow[j] = Wt + (long)(w * NW + j * 16 + (lane & 15)) * K + (lane >> 4) * 8;
  bf16x8 bcur[CB];
#pragma unroll
  for (int j = 0; j < CB; j++) bcur[j] = __builtin_bit_cast(bf16x8, *(const uint4 *)wrow[j]);
#pragma unroll 1
  for (int ks = 0; ks < KS; ks++) {
    const int k0 = ks * 32;
    // next slice's weight fragments, in flight during this slice's products
    bf16x8 bnext[CB];
    if (ks + 1 < KS) {
#pragma unroll
      for (int j = 0; j < CB; j++)
        bnext[j] = __builtin_bit_cast(bf16x8, *(const uint4 *)(wrow[j] + k0 + 32));
    }
#pragma unroll
    for (int i = 0; i < RB; i++) {
      const uint4 q = *(const uint4 *)&X[i * 16 + (lane & 15)][k0 + (lane >> 4) * 8];
      const bf16x8 af = __builtin_bit_cast(bf16x8, q);
#pragma unroll
      for (int j = 0; j < CB; j++)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bcur[j], af, acc[i][j], 0, 0, 0);
    }
    if (ks + 1 < KS) {
#pragma unroll
      for (int j = 0; j < CB; j++) bcur[j] = bnext[j];
    }
  }
  if (!LAST) __syncthreads();  // every wave has read the input tile
#pragma unroll
  for (int i = 0; i < RB; i++)
#pragma unroll
    for (int j = 0; j < CB; j++) {
      const int m = i * 16 + (lane & 15), n = w * NW + j * 16 + (lane >> 4) * 4;
      const f32x4 z = acc[i][j];
      if (LAST) {
        if (row0 + m < M) *(f32x4u *)(pred + (long)(row0 + m) * N + n) = z;
      } else {
        ushort4 q;
        q.x = f2bf(gelu(z[0]));
        q.y = f2bf(gelu(z[1]));
        q.z = f2bf(gelu(z[2]));
        q.w = f2bf(gelu(z[3]));
        *(ushort4 *)&X[m][n] = q;
      }
    }
  if (!LAST) __syncthreads();  // the output tile is complete
}

// resident 256-thread blocks per CU (one wave per SIMD each)
#ifndef IZ_MLP_WAVES
#define IZ_MLP_WAVES 2
#endif
// rows of an activation tile (16 per row block)
#ifndef IZ_MLP_ROWS
#define IZ_MLP_ROWS 128
#endif

__global__ void __attribute__((amdgpu_flat_work_group_size(256, 256),
                               amdgpu_waves_per_eu(IZ_MLP_WAVES, IZ_MLP_WAVES)))
k_mlp_fused(int M, const u16 *__restrict__ X, const u16 *__restrict__ W0,
            const u16 *__restrict__ W1, const u16 *__restrict__ W2, const u16 *__restrict__ W3,
            const float *__restrict__ b0, const float *__restrict__ b1,
            const float *__restrict__ b2, const float *__restrict__ b3,
            float *__restrict__ pred) {
  constexpr int R = IZ_MLP_ROWS, RB = R / 16;
  __shared__ __attribute__((aligned(16))) u16 A[R][FX];
  const int ntiles = (M + R - 1) / R;
  for (int tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
    const int row0 = tile * R;
    // input tile: R rows x 32 features (16 B per thread and pass)
#pragma unroll
    for (int p = 0; p < R / 64; p++) {
      const int t = threadIdx.x, r = p * 64 + (t >> 2), c = (t & 3) * 8;
      uint4 q = make_uint4(0, 0, 0, 0);
      if (row0 + r < M) q = *(const uint4 *)(X + (long)(row0 + r) * 32 + c);
      *(uint4 *)&A[r][c] = q;
    }
    __syncthreads();
    fused_layer<32, 256, false, RB>(A, W0, b0, nullptr, row0, M);
#pragma unroll 1
    for (int l = 0; l < 2; l++)
      fused_layer<256, 256, false, RB>(A, l ? W2 : W1, l ? b2 : b1, nullptr, row0, M);
    fused_layer<256, 64, true, RB>(A, W3, b3, pred, row0, M);
    __syncthreads();  // the next tile's input overwrites A
  }
}

extern "C" int izem_mlp_infer(izem_ctx *ctx, int M, const void *X, const void *const *Wt,
                              const float *const *b, float *pred) {
  if (!ctx || M <= 0 || !X || !Wt || !b || !pred) return IZEM_E_ARG;
  for (int l = 0; l < 4; l++)
    if (!Wt[l] || !b[l] || (((uintptr_t)Wt[l]) & 15)) return IZEM_E_ARG;
  if (((uintptr_t)X) & 15) return IZEM_E_ARG;
  const long ntiles = (M + IZ_MLP_ROWS - 1) / IZ_MLP_ROWS;
  long g = (long)ctx->ncu * IZ_MLP_WAVES;
  if (g > ntiles) g = ntiles;
  int pk = iz_prof_begin(ctx, IZP_CHEM);
  hipLaunchKernelGGL(k_mlp_fused, dim3((unsigned)g), dim3(256), 0, ctx->stream, M,
                     (const u16 *)X, (const u16 *)Wt[0], (const u16 *)Wt[1], (const u16 *)Wt[2],
                     (const u16 *)Wt[3], b[0], b[1], b[2], b[3], pred);
  iz_prof_end(ctx, pk);
  IZ_CHECK(hipGetLastError());
  return IZEM_OK;
}
