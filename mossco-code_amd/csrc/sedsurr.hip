// sedsurr.hip -- the spin-up surrogate (include/sedsurr.h) on gfx950.
//
// A multilayer perceptron trained and evaluated with hand-written kernels:
//   k_gemm     bf16 x bf16 -> fp32 on the MFMA units (v_mfma_f32_32x32x16
//              bf16), 64 x 64 block tiles, four waves of 32 x 32, operands
//              staged through LDS: the forward product H W with its epilogues
//              (bias + GELU storing the pre-activation; bias only; bias, the
//              squared error and its gradient in bf16)
//   k_bwd      the data gradient dZ W^T (with the GELU' product) and the weight
//              gradient H^T dZ of a layer in one launch, by the same tiles; the
//              bias gradients (column sums of dZ) are the row of a ones column
//              appended to the left operand, and a product over many rows is
//              split into slices, summed in a fixed order by their reader
//   k_adam     Adam on the fp32 master parameters, writing the bf16 copy, with
//              the next step's gather and the step's loss in blocks of its own
//   k_gather   minibatch rows of the resident training set, bf16 inputs
//   k_set_params, k_get_params  between the caller's and the padded layout
// Layer widths are padded on the device (inputs to 32, outputs to a
// multiple of 64) with zero weights, which keeps the products exact and the
// padded parameters at zero through training.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "sedcol.h"
#include "sedsurr.h"

namespace ss {

using bf16 = unsigned short;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// fp32 -> bf16, round to nearest even (NaN kept quiet)
__host__ __device__ inline bf16 to_bf16(float f)
{
  unsigned u = __builtin_bit_cast(unsigned, f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (bf16)((u >> 16) | 0x40u);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (bf16)(u >> 16);
}
__host__ __device__ inline float from_bf16(bf16 b) { return __builtin_bit_cast(float, (unsigned)b << 16); }

// GELU, tanh form: 0.5 z (1 + tanh(c (z + a z^3))), c = sqrt(2/pi), a = 0.044715
constexpr float kGc = 0.7978845608028654f, kGa = 0.044715f;
__device__ inline float tanh_e(float u) { return 1.0f - 2.0f / (expf(2.0f * u) + 1.0f); }
__device__ inline float gelu(float z)
{
  const float t = tanh_e(kGc * (z + kGa * z * z * z));
  return 0.5f * z * (1.0f + t);
}
__device__ inline float gelu_grad(float z)
{
  const float t = tanh_e(kGc * (z + kGa * z * z * z));
  return 0.5f * (1.0f + t) + 0.5f * z * (1.0f - t * t) * kGc * (1.0f + 3.0f * kGa * z * z);
}

constexpr int BM = 64, BN = 64, BK = 64;
enum { EPI_F32 = 0, EPI_BIAS = 1, EPI_BIAS_GELU = 2, EPI_GELU_GRAD = 3, EPI_LOSS = 4 };

struct Epi {
  float *out_f;       // fp32 output (EPI_F32, EPI_BIAS; pre-activation for EPI_BIAS_GELU; squared
                      // errors per block for EPI_LOSS)
  int ldo;
  long long zstride;  // EPI_F32 with split k: distance between the slices' outputs
  bf16 *out_h;        // bf16 output (EPI_BIAS_GELU activation, EPI_GELU_GRAD and EPI_LOSS dZ)
  int ldh;
  const float *bias;  // EPI_BIAS, EPI_BIAS_GELU
  const float *zin;   // EPI_GELU_GRAD: pre-activation of the layer below; EPI_LOSS: targets
  int ldz;
  float scale;        // EPI_LOSS: dZ = scale (output - target) over the first n_out columns
  int n_out;
};

// eight consecutive bf16 of a row-major array, or zeros.  Every leading
// dimension is a multiple of 32 and every array starts on a 16-byte boundary, so
// a group of eight is inside or outside as a whole and its load is aligned.
__device__ __forceinline__ uint4 load8(const bf16 *__restrict__ p, bool ok)
{
  uint4 v = make_uint4(0u, 0u, 0u, 0u);
  if (ok) v = *reinterpret_cast<const uint4 *>(p);
  return v;
}
__device__ inline bf16 elem8(const uint4 &w, int j)
{
  const unsigned u = j < 2 ? w.x : j < 4 ? w.y : j < 6 ? w.z : w.w;
  return (bf16)((j & 1) ? (u >> 16) : (u & 0xffffu));
}

// Tiles of both operands in LDS with k contiguous (A as [m][k], B as [n][k]),
// double buffered.  Rows of 128 bytes without padding; the 16-byte chunk c of
// row r sits at c ^ swz(r), so that the lanes of an operand read (32
// consecutive rows, one chunk) and of a transposing write (rows 8 apart) meet
// different banks: with rows padded to 144 bytes those writes met in fours.
struct Tiles {
  bf16 a[2][BM][BK], b[2][BN][BK];
};
__device__ __forceinline__ int swz(int r) { return ((r >> 3) ^ (r >> 1)) & 7; }
// the element at (r, k) of a tile
__device__ __forceinline__ bf16 *at(bf16 (&t)[64][BK], int r, int k)
{
  return &t[r][((((k >> 3) ^ swz(r)) << 3)) | (k & 7)];
}

// One 64 x 64 tile (bx, by) of C (M x N) = op(A) (M x K) op(B) (K x N);
// op(A)(m,k) = TA ? A[k lda + m] : A[m lda + k], op(B)(k,n) = TB ? B[n ldb + k] :
// B[k ldb + n].  Out-of-range rows, columns and k are loaded as zero and not
// stored.  Slice z takes k in [z kchunk, (z+1) kchunk) and (EPI_F32) writes its
// partial product at out_f + z zstride.
//
// With k contiguous in LDS a lane's MFMA operand (8 consecutive k of one row or
// column) is one 16-byte LDS read.  v_mfma_f32_32x32x16_bf16: lane l supplies
// row (A) / column (B) l % 32 at k = 8 (l / 32) + 0..7.  A tile is four MFMAs per
// wave, so the products here are bound by the latency of their loads and by what
// surrounds the k loop: kDepth tiles are in flight in registers, the double buffer
// leaves one barrier per tile, and the code is kept short.  The MFMAs accumulate k
// in increasing order of 16-wide steps, whatever the depth.  Mean time of the
// three hidden layers' forward products of 4096 rows (32, 512, 512 -> 512) and of
// a hidden layer's backward pass (2 x 2.1 GFLOP):
//   one tile in flight, rows padded to 144 bytes         13.9 us   34.6 us (two launches)
//   four tiles, the backward pass in one launch          14.2      29.6
//   ... chunks exchanged instead of padding              13.5      26.3
//   ... two tiles (106 instead of 134 registers)         13.2      23.7
//   ... whole 16-byte loads, rolled epilogue, XCD order  10.6      19.0
constexpr int kDepth = 2;
static_assert(kDepth % 2 == 0, "the two buffers alternate");
template <bool TA, bool TB, int EPI>
__device__ __forceinline__ void gemm_tile(Tiles &S, int bx, int by, int z, int M, int N, int K, int kchunk,
                                          const bf16 *__restrict__ A, int lda, const bf16 *__restrict__ B, int ldb,
                                          const Epi &e, int ones_row)
{
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int bm = by * BM, bn = bx * BN;
  const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
  const int kb0 = z * kchunk;
  const int kend = min(K, kb0 + kchunk);
  f32x16 acc;
#pragma unroll
  for (int v = 0; v < 16; ++v) acc[v] = 0.0f;
  const int r = lane & 31, q8 = (lane >> 5) * 8;

  // This thread's share of a 64 x 64 tile of each operand: eight consecutive k
  // of the rows tid / 8 + 32 h, h = 0, 1, or, for an operand stored k-major (TA
  // for A, !TB for B), which is transposed on its way into LDS, the same eight m
  // (or n) at two consecutive k (k even), so that every tile element pair
  // (m, k..k+1) is one 4-byte LDS write.
  uint4 ra[kDepth][2], rb[kDepth][2];
  const int c8 = (tid % 8) * 8, r8 = tid / 8;
  auto fetch = [&](uint4 (&va)[2], uint4 (&vb)[2], int k0) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (TA) {
        const int m = bm + c8, k = k0 + 2 * r8 + h;
        // row ones_row of op(A) is all ones: the product's row ones_row is then
        // the column sums of op(B)
        va[h] = load8(A + (size_t)k * lda + m, k < kend && m < ones_row);
        if (m == ones_row && k < kend) va[h].x = 0x3F80u;  // bf16 1.0
      } else {
        const int m = bm + r8 + 32 * h, k = k0 + c8;
        va[h] = load8(A + (size_t)m * lda + k, k < kend && m < M);
      }
      if (TB) {
        const int n = bn + r8 + 32 * h, k = k0 + c8;
        vb[h] = load8(B + (size_t)n * ldb + k, k < kend && n < N);
      } else {
        const int n = bn + c8, k = k0 + 2 * r8 + h;
        vb[h] = load8(B + (size_t)k * ldb + n, k < kend && n < ldb);
      }
    }
  };
  auto pair = [](const uint4 &lo, const uint4 &hi, int j) {
    return (unsigned)elem8(lo, j) | ((unsigned)elem8(hi, j) << 16);
  };
  auto stage = [&](int buf, const uint4 (&va)[2], const uint4 (&vb)[2]) {
    if (TA) {
#pragma unroll
      for (int j = 0; j < 8; ++j) *reinterpret_cast<unsigned *>(at(S.a[buf], c8 + j, 2 * r8)) = pair(va[0], va[1], j);
    } else {
#pragma unroll
      for (int h = 0; h < 2; ++h) *reinterpret_cast<uint4 *>(at(S.a[buf], r8 + 32 * h, c8)) = va[h];
    }
    if (TB) {
#pragma unroll
      for (int h = 0; h < 2; ++h) *reinterpret_cast<uint4 *>(at(S.b[buf], r8 + 32 * h, c8)) = vb[h];
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) *reinterpret_cast<unsigned *>(at(S.b[buf], c8 + j, 2 * r8)) = pair(vb[0], vb[1], j);
    }
  };

#pragma unroll
  for (int u = 0; u < kDepth; ++u)
    if (kb0 + u * BK < kend) fetch(ra[u], rb[u], kb0 + u * BK);
  for (int k0 = kb0; k0 < kend; k0 += kDepth * BK) {
#pragma unroll
    for (int u = 0; u < kDepth; ++u) {
      const int ku = k0 + u * BK;
      if (ku < kend) {
        const int buf = u & 1;
        stage(buf, ra[u], rb[u]);
        __syncthreads();
        if (ku + kDepth * BK < kend) fetch(ra[u], rb[u], ku + kDepth * BK);
#pragma unroll
        for (int kk = 0; kk < BK; kk += 16) {
          const bf16x8 a = *reinterpret_cast<const bf16x8 *>(at(S.a[buf], wm + r, kk + q8));
          const bf16x8 b = *reinterpret_cast<const bf16x8 *>(at(S.b[buf], wn + r, kk + q8));
          acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc, 0, 0, 0);
        }
      }
    }
  }
  // The result goes through LDS, so that the epilogue is one rolled loop over
  // four columns per thread with 16-byte loads and stores.  In the accumulator of
  // the 32 x 32 product a lane holds column (lane & 31), register v holds row
  // 8 (v / 4) + 4 (lane / 32) + v % 4.
  __syncthreads();  // the tiles are done with
  float (*C)[BN + 4] = reinterpret_cast<float (*)[BN + 4]>(&S);
#pragma unroll
  for (int v = 0; v < 16; ++v) C[wm + 8 * (v >> 2) + (lane >> 5) * 4 + (v & 3)][wn + r] = acc[v];
  __syncthreads();
  float sq = 0.0f;  // EPI_LOSS: the thread's squared errors
  if constexpr (EPI == EPI_BIAS) {
    // any width and any alignment of the output
    const int col = bn + lane;
    const float bias = col < N ? e.bias[col] : 0.0f;
    for (int row = wave; row < BM; row += 4)
      if (bm + row < M && col < N) e.out_f[(size_t)(bm + row) * e.ldo + col] = C[row][lane] + bias;
  } else {
    const int c4 = (tid % 16) * 4, col = bn + c4;
    float4 bias = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if constexpr (EPI == EPI_BIAS_GELU || EPI == EPI_LOSS)
      if (col < N) bias = *reinterpret_cast<const float4 *>(e.bias + col);
#pragma unroll 1
    for (int t = tid / 16; t < BM; t += 16) {
      const int row = bm + t;
      if (row >= M || col >= N) break;
      const float4 x4 = *reinterpret_cast<const float4 *>(&C[t][c4]);
      float x[4] = {x4.x + bias.x, x4.y + bias.y, x4.z + bias.z, x4.w + bias.w};
      if constexpr (EPI == EPI_F32) {
        *reinterpret_cast<float4 *>(e.out_f + z * e.zstride + (size_t)row * e.ldo + col) = x4;
      } else {
        if constexpr (EPI == EPI_BIAS_GELU) {
          *reinterpret_cast<float4 *>(e.out_f + (size_t)row * e.ldo + col) = make_float4(x[0], x[1], x[2], x[3]);
#pragma unroll
          for (int j = 0; j < 4; ++j) x[j] = gelu(x[j]);
        } else {
          const float4 z4 = *reinterpret_cast<const float4 *>(e.zin + (size_t)row * e.ldz + col);
          const float zs[4] = {z4.x, z4.y, z4.z, z4.w};
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            if constexpr (EPI == EPI_GELU_GRAD) {
              x[j] *= gelu_grad(zs[j]);
            } else {
              const float d = col + j < e.n_out ? x[j] - zs[j] : 0.0f;
              sq += d * d;
              x[j] = e.scale * d;
            }
          }
        }
        const unsigned lo = to_bf16(x[0]) | ((unsigned)to_bf16(x[1]) << 16);
        const unsigned hi = to_bf16(x[2]) | ((unsigned)to_bf16(x[3]) << 16);
        *reinterpret_cast<uint2 *>(e.out_h + (size_t)row * e.ldh + col) = make_uint2(lo, hi);
      }
    }
  }
  if constexpr (EPI == EPI_LOSS) {
    // the block's squared errors, in a fixed order: lanes by halves, then the
    // four waves
    __syncthreads();  // the results are done with
    float *red = reinterpret_cast<float *>(&S);
    red[tid] = sq;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
      if (tid < w) red[tid] += red[tid + w];
      __syncthreads();
    }
    if (tid == 0) e.out_f[by * ((N + BN - 1) / BN) + bx] = red[0];
  }
}

// Blocks go to the eight XCDs in turn, each with an L2 of its own: block i of n
// takes tile xcd_order(i, n), which hands every XCD one run of consecutive tiles.
// With the column tiles counted fastest, a run shares its rows of the left
// operand, and in k_bwd the gradients' slices of the batch.
__device__ __forceinline__ int xcd_order(int i, int n)
{
  const int x = i & 7, q = n >> 3, rest = n & 7;
  return x * q + min(x, rest) + (i >> 3);
}

template <int EPI>
__global__ __launch_bounds__(256) void k_gemm(int M, int N, int K, const bf16 *__restrict__ A, int lda,
                                              const bf16 *__restrict__ B, int ldb, Epi e)
{
  __shared__ __attribute__((aligned(16))) Tiles S;
  const int nx = gridDim.x, t = xcd_order(blockIdx.y * nx + blockIdx.x, nx * gridDim.y);
  gemm_tile<false, false, EPI>(S, t % nx, t / nx, 0, M, N, K, K, A, lda, B, ldb, e, -1);
}

// Both products of a layer's backward pass, which need the same dZ and not each
// other: the first nd blocks make tiles of dZ W^T (with GELU'), the others those
// of [H_in, 1]^T dZ.  Neither product fills the device to its end alone.
struct Bwd {
  const bf16 *dz, *w, *hin;
  int b, win, wout, kchunk, ndx, nd, nwx, nwy, ng;  // ndx, nwx, nwy: tiles per row / column; nd, ng: blocks
  Epi d, g;
};
__global__ __launch_bounds__(256) void k_bwd(Bwd p)
{
  __shared__ __attribute__((aligned(16))) Tiles S;
  int i = blockIdx.x;
  if (i < p.nd) {
    i = xcd_order(i, p.nd);
    gemm_tile<false, true, EPI_GELU_GRAD>(S, i % p.ndx, i / p.ndx, 0, p.b, p.win, p.wout, p.wout, p.dz, p.wout, p.w,
                                          p.wout, p.d, -1);
  } else {
    i = xcd_order(i - p.nd, p.ng);
    const int z = i / (p.nwx * p.nwy), t = i % (p.nwx * p.nwy);
    gemm_tile<true, false, EPI_F32>(S, t % p.nwx, t / p.nwx, z, p.win + 1, p.wout, p.b, p.kchunk, p.hin, p.win, p.dz,
                                    p.wout, p.g, p.win);
  }
}

// rows of the fp32 sets (or of X itself when rows is null) into padded
// batch buffers: Xb bf16 (b x kin, zero beyond n_in), Yb fp32 (b x nout_p);
// one wave per row, block blk of 256 threads
struct Gather {
  const float *X, *Y;
  const int *rows;
  int n_in, n_out, b, kin, nout_p;
  bf16 *Xb;
  float *Yb;
};
__device__ __forceinline__ void gather_rows(const Gather &q, int blk)
{
  const int i = blk * 4 + (int)(threadIdx.x >> 6), l = threadIdx.x & 63;
  if (i >= q.b) return;
  const long long src = q.rows ? q.rows[i] : i;
  for (int j = l; j < q.kin; j += 64) q.Xb[(size_t)i * q.kin + j] = j < q.n_in ? to_bf16(q.X[src * q.n_in + j]) : (bf16)0;
  if (q.Yb)
    for (int j = l; j < q.nout_p; j += 64)
      q.Yb[(size_t)i * q.nout_p + j] = j < q.n_out ? q.Y[src * q.n_out + j] : 0.0f;
}
__global__ __launch_bounds__(256) void k_gather(Gather q) { gather_rows(q, blockIdx.x); }

// out[0] = sum(part[0..n-1]) * scale (one block)
__device__ __forceinline__ void sum_parts(const float *part, int n, float scale, float *out)
{
  __shared__ float red[256];
  float s = 0.0f;
  for (int i = threadIdx.x; i < n; i += 256) s += part[i];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[0] = red[0] * scale;
}
// Split-k slices of the weight gradients, summed by their reader: layer l's
// parameters [woff, woff + welems) take their gradient from nz slices at
// part + pofs (slice z at + z welems) when nz > 1, else from g
constexpr int kMaxLayers = 17;  // n_layers <= 16 hidden layers + the output layer
struct Slices {
  int nl;
  long long woff[kMaxLayers], welems[kMaxLayers], pofs[kMaxLayers];
  int nz[kMaxLayers];
};

// The end of a training step in one launch: Adam in the first na blocks, four
// parameters per thread (every layer's part starts and ends at a multiple of 64
// floats), the next step's batch in the blocks after them, and the loss of this
// step in the last one (13.4 + 5.6 + 4.4 us in launches of their own, 11.2 us
// together; the parameters, moments and slices are 40 MB).
struct Step {
  float *w;
  const float *g;
  float *m, *v;
  bf16 *wb;
  long long n;
  float lr, b1, b2, eps, bc1, bc2;
  const float *part;  // split-k slices
  int na, ng;         // blocks of Adam and of the gather (0: none)
  const float *lpart;
  int nlpart;
  float lscale;
  float *loss;
  Gather next;
};
__global__ __launch_bounds__(256) void k_adam(Step p, Slices sl)
{
  if ((int)blockIdx.x >= p.na) {
    const int i = (int)blockIdx.x - p.na;
    if (i < p.ng) gather_rows(p.next, i);
    else sum_parts(p.lpart, p.nlpart, p.lscale, p.loss);
    return;
  }
  const long long i = 4 * (blockIdx.x * 256ll + threadIdx.x);
  if (i >= p.n) return;
  int l = 0;
  while (l + 1 < sl.nl && i >= sl.woff[l + 1]) ++l;
  float4 gi;
  if (sl.nz[l] > 1) {
    // the slices in order
    gi = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    const float *q = p.part + sl.pofs[l] + (i - sl.woff[l]);
    const long long step = sl.welems[l];
    const int nz = sl.nz[l];
#pragma unroll 8
    for (int z = 0; z < nz; ++z) {
      const float4 t = *reinterpret_cast<const float4 *>(q + z * step);
      gi.x += t.x;
      gi.y += t.y;
      gi.z += t.z;
      gi.w += t.w;
    }
  } else {
    gi = *reinterpret_cast<const float4 *>(p.g + i);
  }
  const float4 m4 = *reinterpret_cast<const float4 *>(p.m + i), v4 = *reinterpret_cast<const float4 *>(p.v + i);
  const float4 w4 = *reinterpret_cast<const float4 *>(p.w + i);
  float gs[4] = {gi.x, gi.y, gi.z, gi.w}, ms[4] = {m4.x, m4.y, m4.z, m4.w}, vs[4] = {v4.x, v4.y, v4.z, v4.w};
  float ws[4] = {w4.x, w4.y, w4.z, w4.w};
  unsigned hb[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    ms[k] = p.b1 * ms[k] + (1.0f - p.b1) * gs[k];
    vs[k] = p.b2 * vs[k] + (1.0f - p.b2) * gs[k] * gs[k];
    ws[k] = ws[k] - p.lr * (ms[k] / p.bc1) / (sqrtf(vs[k] / p.bc2) + p.eps);
    hb[k] = to_bf16(ws[k]);
  }
  *reinterpret_cast<float4 *>(p.m + i) = make_float4(ms[0], ms[1], ms[2], ms[3]);
  *reinterpret_cast<float4 *>(p.v + i) = make_float4(vs[0], vs[1], vs[2], vs[3]);
  *reinterpret_cast<float4 *>(p.w + i) = make_float4(ws[0], ws[1], ws[2], ws[3]);
  *reinterpret_cast<uint2 *>(p.wb + i) = make_uint2(hb[0] | (hb[1] << 16), hb[2] | (hb[3] << 16));
}

// The caller's parameter vector (layers' W and b without padding) to the padded
// device layout with its bf16 copy, or back.  Layer l's entries are fi rows of
// fo weights and the row of biases, at flat + fofs, on the device rows of fop
// at woff (fip rows, then the biases); the rest of a padded layer stays zero.
struct Layers {
  int nl;
  int fi[kMaxLayers], fo[kMaxLayers], fip[kMaxLayers], fop[kMaxLayers];
  long long fofs[kMaxLayers], woff[kMaxLayers];
};
__global__ __launch_bounds__(256) void k_set_params(Layers L, const float *__restrict__ flat, float *w, bf16 *wb,
                                                    float *m, float *v)
{
  const int l = blockIdx.y;
  const int fop = L.fop[l];
  const int n = (L.fip[l] + 1) * fop;
  for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
    const int r = i / fop, c = i - r * fop;
    const int src = r < L.fi[l] ? r : r == L.fip[l] ? L.fi[l] : -1;  // the biases follow the padded rows
    const float x = src >= 0 && c < L.fo[l] ? flat[L.fofs[l] + (long long)src * L.fo[l] + c] : 0.0f;
    const long long o = L.woff[l] + i;
    w[o] = x;
    wb[o] = to_bf16(x);
    m[o] = 0.0f;
    v[o] = 0.0f;
  }
}
// sl (or null): the gradient instead, layers split over k as the sum of their
// slices in order; the last block then sums the loss
__global__ __launch_bounds__(256) void k_get_params(Layers L, const float *__restrict__ w, float *__restrict__ flat,
                                                    int grad, Slices sl, const float *__restrict__ part,
                                                    const float *lpart, int nlpart, float lscale, float *loss)
{
  const int l = blockIdx.y;
  if (l == L.nl) {
    if (blockIdx.x == 0) sum_parts(lpart, nlpart, lscale, loss);
    return;
  }
  const int fo = L.fo[l], n = (L.fi[l] + 1) * fo;
  const int nz = grad ? sl.nz[l] : 1;
  for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
    const int r = i / fo, c = i - r * fo;
    const long long j = (long long)(r < L.fi[l] ? r : L.fip[l]) * L.fop[l] + c;
    float x;
    if (nz > 1) {
      x = 0.0f;
#pragma unroll 8
      for (int z = 0; z < nz; ++z) x += part[sl.pofs[l] + z * sl.welems[l] + j];
    } else {
      x = w[L.woff[l] + j];
    }
    flat[L.fofs[l] + i] = x;
  }
}

}  // namespace ss

using ss::bf16;

namespace {

thread_local std::string g_err;

int fail(int code, const std::string &msg)
{
  g_err = msg;
  return code;
}

#define HIPOK(call)                                                                  \
  do {                                                                               \
    hipError_t e_ = (call);                                                          \
    if (e_ != hipSuccess)                                                            \
      return fail(SEDCOL_EHIP, std::string(#call) + ": " + hipGetErrorString(e_));   \
  } while (0)

inline int round_up(int x, int m) { return (x + m - 1) / m * m; }

}  // namespace

// Makes the handle's device current for the duration of one entry point and
// restores the caller's current device afterwards: a handle belongs to the
// device that was current at sedsurr_create.
struct DeviceScope {
  int prev = -1, dev;
  explicit DeviceScope(int d) : dev(d)
  {
    if (hipGetDevice(&prev) != hipSuccess) prev = -1;
    if (prev != dev) (void)hipSetDevice(dev);
  }
  ~DeviceScope()
  {
    if (prev >= 0 && prev != dev) (void)hipSetDevice(prev);
  }
  DeviceScope(const DeviceScope &) = delete;
  DeviceScope &operator=(const DeviceScope &) = delete;
};

struct sedsurr_handle {
  int device = 0;  // current at sedsurr_create; every call runs on it
  sedsurr_shape s{};
  int kin = 0, nout_p = 0, nl = 0;  // padded input width, padded output width, weight layers
  std::vector<int> fi, fo, fip, fop;    // logical and padded fan-in / fan-out per layer
  std::vector<long long> woff, boff;    // offsets of W_l and b_l in the padded flat vector
  long long np_pad = 0, np = 0;         // padded and logical parameter counts
  float *w = nullptr, *g = nullptr, *m = nullptr, *v = nullptr;
  bf16 *wb = nullptr;
  bf16 *xb = nullptr;                   // max_batch x kin
  std::vector<bf16 *> hs;               // hidden activations, max_batch x n_hidden
  std::vector<float *> zs;              // pre-activations
  float *yb = nullptr;                  // max_batch x nout_p
  bf16 *dz0 = nullptr, *dz1 = nullptr;  // max_batch x max(n_hidden, nout_p)
  float *part = nullptr;                // squared errors per block, then the loss of sedsurr_loss_grad
  float *kpart_all = nullptr;           // split-k partial weight gradients, one region per layer
  std::vector<long long> kpofs;         // offset of layer l's region in kpart_all
  ss::Slices slices{};                  // the slices of the last backward pass
  ss::Layers layers{};                  // padded and caller's layouts of the parameters
  float *flat = nullptr;                // np: parameters or gradient in the caller's layout
  float *h_loss = nullptr;              // pinned: the loss of sedsurr_loss_grad
  float *loss = nullptr;                // per-step losses of a train call
  int loss_cap = 0;
  float *X = nullptr, *Y = nullptr;     // training set
  long long ndata = 0;
  int *rows = nullptr;
  long long rows_cap = 0;
  float *xin = nullptr, *yin = nullptr; // staging of loss_grad / predict inputs
  float *ydev = nullptr;                // sedsurr_predict_device output (ydev_rows x n_out)
  int64_t ydev_rows = 0;
  long long step = 0;                   // Adam steps taken
  hipStream_t st = nullptr;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  double last_ms = 0.0;
  int last_launches = 0;
};

namespace {

constexpr int kMaxSplit = 8;     // k slices of a weight-gradient product
constexpr int kParamBlocks = 256;  // blocks per layer of the parameter copies

template <int EPI>
void gemm(sedsurr_handle *h, int M, int N, int K, const bf16 *A, int lda, const bf16 *B, int ldb, ss::Epi e,
          int *launches)
{
  dim3 grid((N + ss::BN - 1) / ss::BN, (M + ss::BM - 1) / ss::BM);
  hipLaunchKernelGGL(ss::k_gemm<EPI>, grid, dim3(256), 0, h->st, M, N, K, A, lda, B, ldb, e);
  ++*launches;
}

// k slices of the weight-gradient product of a batch of b rows: enough to
// give the device about 512 blocks, each slice at least 256 rows
int split_for(int M, int N, int b)
{
  const int tiles = ((M + ss::BM - 1) / ss::BM) * ((N + ss::BN - 1) / ss::BN);
  int s = 1;
  while (s < kMaxSplit && tiles * s < 512 && b / (2 * s) >= 256) s *= 2;
  return s;
}

// width of the activation entering layer l (padded)
inline int in_width(const sedsurr_handle *h, int l) { return h->fip[l]; }

inline int tiles(int n, int t) { return (n + t - 1) / t; }

// blocks of the output layer's product for b rows, each with a partial loss
inline int loss_parts(const sedsurr_handle *h, int b) { return tiles(b, ss::BM) * tiles(h->nout_p, ss::BN); }

// forward pass of b rows from h->xb; the n_out real columns, compact, to out,
// or, without out, the loss against h->yb: squared errors per block to h->part
// and dZ of the output layer to h->dz0
void forward(sedsurr_handle *h, int b, int *launches, float *out = nullptr)
{
  const int L = h->nl;
  for (int l = 0; l < L; ++l) {
    const bf16 *A = l == 0 ? h->xb : h->hs[l - 1];
    const int lda = in_width(h, l);
    ss::Epi e{};
    e.bias = h->w + h->boff[l];
    if (l < L - 1) {
      e.out_f = h->zs[l];
      e.ldo = h->fop[l];
      e.out_h = h->hs[l];
      e.ldh = h->fop[l];
      gemm<ss::EPI_BIAS_GELU>(h, b, h->fop[l], h->fip[l], A, lda, h->wb + h->woff[l], h->fop[l], e,
                                            launches);
    } else if (out) {
      e.out_f = out;
      e.ldo = h->s.n_out;
      gemm<ss::EPI_BIAS>(h, b, h->s.n_out, h->fip[l], A, lda, h->wb + h->woff[l], h->fop[l], e, launches);
    } else {
      e.out_f = h->part;
      e.out_h = h->dz0;
      e.ldh = h->nout_p;
      e.zin = h->yb;
      e.ldz = h->nout_p;
      e.scale = 2.0f / ((float)b * (float)h->s.n_out);
      e.n_out = h->s.n_out;
      gemm<ss::EPI_LOSS>(h, b, h->nout_p, h->fip[l], A, lda, h->wb + h->woff[l], h->fop[l], e, launches);
    }
  }
}

// gradient of the loss of forward(): into h->g, or as slices in h->kpart_all
// for the layers whose product over the batch is split (h->slices)
void backward(sedsurr_handle *h, int b, int *launches)
{
  bf16 *dz = h->dz0, *dzn = h->dz1;
  for (int l = h->nl - 1; l >= 0; --l) {
    const int win = in_width(h, l), wout = h->fop[l];
    // [dW_l; db_l] = [H_in, 1]^T dZ_l in one product: the bias gradient
    // (the column sums of dZ_l) is the row of a ones column appended to
    // H_in, and b_l follows W_l in the parameter vector, so that row lands
    // on it; split over the batch into slices summed in order
    const int split = split_for(win + 1, wout, b);
    const long long welems = (long long)(win + 1) * wout;
    const int kc = ((b + split - 1) / split + ss::BK - 1) / ss::BK * ss::BK;
    const int nz = (b + kc - 1) / kc;
    ss::Bwd p{};
    p.dz = dz;
    p.w = h->wb + h->woff[l];
    p.hin = l == 0 ? h->xb : h->hs[l - 1];
    p.b = b;
    p.win = win;
    p.wout = wout;
    p.kchunk = kc;
    p.ndx = tiles(win, ss::BN);
    p.nd = l > 0 ? p.ndx * tiles(b, ss::BM) : 0;  // the input needs no gradient
    p.nwx = tiles(wout, ss::BN);
    p.nwy = tiles(win + 1, ss::BM);
    p.ng = p.nwx * p.nwy * nz;
    // dZ_{l-1} = GELU'(Z_{l-1}) * (dZ_l W_l^T)
    p.d.out_h = dzn;
    p.d.ldh = win;
    p.d.zin = l > 0 ? h->zs[l - 1] : nullptr;
    p.d.ldz = win;
    p.g.out_f = nz > 1 ? h->kpart_all + h->kpofs[l] : h->g + h->woff[l];
    p.g.ldo = wout;
    p.g.zstride = welems;
    hipLaunchKernelGGL(ss::k_bwd, dim3(p.nd + p.ng), dim3(256), 0, h->st, p);
    ++*launches;
    h->slices.woff[l] = h->woff[l];
    h->slices.welems[l] = welems;
    h->slices.pofs[l] = h->kpofs[l];
    h->slices.nz[l] = nz;
    std::swap(dz, dzn);
  }
}

ss::Gather gather_of(const sedsurr_handle *h, const float *X, const float *Y, const int *rows, int b)
{
  return ss::Gather{X, Y, rows, h->s.n_in, h->s.n_out, b, h->kin, h->nout_p, h->xb, Y ? h->yb : nullptr};
}

void gather(sedsurr_handle *h, const ss::Gather &q, int *launches)
{
  hipLaunchKernelGGL(ss::k_gather, dim3((q.b + 3) / 4), dim3(256), 0, h->st, q);
  ++*launches;
}

}  // namespace

extern "C" {

const char *sedsurr_last_error(void) { return g_err.c_str(); }

int sedsurr_create(const sedsurr_shape *shape, sedsurr_handle **out)
{
  if (!shape || !out) return fail(SEDCOL_EINVAL, "null argument");
  *out = nullptr;
  const sedsurr_shape s = *shape;
  if (s.n_in < 1 || s.n_in > 64) return fail(SEDCOL_EINVAL, "n_in outside 1..64");
  if (s.n_hidden < 64 || s.n_hidden % 64 || s.n_hidden > 4096)
    return fail(SEDCOL_EINVAL, "n_hidden must be a multiple of 64 in 64..4096");
  if (s.n_layers < 1 || s.n_layers > 16) return fail(SEDCOL_EINVAL, "n_layers outside 1..16");
  if (s.n_out < 1 || s.n_out > 4096) return fail(SEDCOL_EINVAL, "n_out outside 1..4096");
  if (s.max_batch < 64 || s.max_batch % 64 || s.max_batch > 65536)
    return fail(SEDCOL_EINVAL, "max_batch must be a multiple of 64 in 64..65536");
  if (s.reserved != 0) return fail(SEDCOL_EINVAL, "reserved must be 0");
  sedsurr_handle *h = new sedsurr_handle();
  h->s = s;
  h->kin = round_up(s.n_in, 32);
  h->nout_p = round_up(s.n_out, 64);
  h->nl = s.n_layers + 1;
  long long off = 0;
  for (int l = 0; l < h->nl; ++l) {
    const int fi = l == 0 ? s.n_in : s.n_hidden, fo = l == h->nl - 1 ? s.n_out : s.n_hidden;
    const int fip = l == 0 ? h->kin : s.n_hidden, fop = l == h->nl - 1 ? h->nout_p : s.n_hidden;
    h->fi.push_back(fi);
    h->fo.push_back(fo);
    h->fip.push_back(fip);
    h->fop.push_back(fop);
    h->woff.push_back(off);
    off += (long long)fip * fop;
    h->boff.push_back(off);
    off += fop;
    h->np += (long long)fi * fo + fo;
  }
  h->np_pad = off;
  auto cleanup = [&](int code) {
    sedsurr_destroy(h);
    return code;
  };
#define HIPOK_C(call)                                                                       \
  do {                                                                                      \
    hipError_t e_ = (call);                                                                 \
    if (e_ != hipSuccess)                                                                   \
      return cleanup(fail(SEDCOL_EHIP, std::string(#call) + ": " + hipGetErrorString(e_))); \
  } while (0)
  HIPOK_C(hipGetDevice(&h->device));
  HIPOK_C(hipStreamCreateWithFlags(&h->st, hipStreamNonBlocking));
  HIPOK_C(hipEventCreate(&h->e0));
  HIPOK_C(hipEventCreate(&h->e1));
  const size_t P = (size_t)h->np_pad, B = (size_t)s.max_batch;
  for (float **q : {&h->w, &h->g, &h->m, &h->v}) {
    HIPOK_C(hipMalloc(q, sizeof(float) * P));
    HIPOK_C(hipMemset(*q, 0, sizeof(float) * P));
  }
  HIPOK_C(hipMalloc(&h->wb, sizeof(bf16) * P));
  HIPOK_C(hipMemset(h->wb, 0, sizeof(bf16) * P));
  HIPOK_C(hipMalloc(&h->xb, sizeof(bf16) * B * h->kin));
  for (int l = 0; l < s.n_layers; ++l) {
    bf16 *hb = nullptr;
    float *zb = nullptr;
    HIPOK_C(hipMalloc(&hb, sizeof(bf16) * B * s.n_hidden));
    h->hs.push_back(hb);
    HIPOK_C(hipMalloc(&zb, sizeof(float) * B * s.n_hidden));
    h->zs.push_back(zb);
  }
  const size_t wmax = (size_t)std::max(s.n_hidden, h->nout_p);
  HIPOK_C(hipMalloc(&h->yb, sizeof(float) * B * h->nout_p));
  HIPOK_C(hipMalloc(&h->dz0, sizeof(bf16) * B * wmax));
  HIPOK_C(hipMalloc(&h->dz1, sizeof(bf16) * B * wmax));
  HIPOK_C(hipMalloc(&h->part, sizeof(float) * (loss_parts(h, s.max_batch) + 1)));  // + the loss of sedsurr_loss_grad
  HIPOK_C(hipMalloc(&h->flat, sizeof(float) * (size_t)h->np));
  HIPOK_C(hipHostMalloc((void **)&h->h_loss, sizeof(float), hipHostMallocDefault));
  if (h->nl > ss::kMaxLayers) return cleanup(fail(SEDCOL_EINVAL, "too many layers"));
  long long kall = 0;
  for (int l = 0; l < h->nl; ++l) {
    h->kpofs.push_back(kall);
    kall += (long long)kMaxSplit * (h->fip[l] + 1) * h->fop[l];
  }
  HIPOK_C(hipMalloc(&h->kpart_all, sizeof(float) * kall));
  h->slices.nl = h->nl;
  h->layers.nl = h->nl;
  long long fofs = 0;
  for (int l = 0; l < h->nl; ++l) {
    h->layers.fi[l] = h->fi[l];
    h->layers.fo[l] = h->fo[l];
    h->layers.fip[l] = h->fip[l];
    h->layers.fop[l] = h->fop[l];
    h->layers.woff[l] = h->woff[l];
    h->layers.fofs[l] = fofs;
    fofs += (long long)(h->fi[l] + 1) * h->fo[l];
  }
  HIPOK_C(hipMalloc(&h->xin, sizeof(float) * B * s.n_in));
  HIPOK_C(hipMalloc(&h->yin, sizeof(float) * B * s.n_out));
#undef HIPOK_C
  *out = h;
  return SEDCOL_OK;
}

int sedsurr_destroy(sedsurr_handle *h)
{
  if (!h) return SEDCOL_OK;
  const DeviceScope dscope(h->device);
  if (h->st) (void)hipStreamSynchronize(h->st);
  std::vector<void *> ptrs = {h->w, h->g, h->m, h->v, h->wb, h->xb, h->yb, h->dz0, h->dz1,
                              h->part, h->loss, h->X, h->Y, h->rows, h->xin, h->yin, h->kpart_all,
                              h->ydev, h->flat};
  for (auto *q : h->hs) ptrs.push_back(q);
  for (auto *q : h->zs) ptrs.push_back(q);
  for (void *q : ptrs)
    if (q) (void)hipFree(q);
  if (h->h_loss) (void)hipHostFree(h->h_loss);
  if (h->e0) (void)hipEventDestroy(h->e0);
  if (h->e1) (void)hipEventDestroy(h->e1);
  if (h->st) (void)hipStreamDestroy(h->st);
  delete h;
  return SEDCOL_OK;
}

int sedsurr_num_params(sedsurr_handle *h, int64_t *n)
{
  if (!h || !n) return fail(SEDCOL_EINVAL, "null argument");
  const DeviceScope dscope(h->device);
  *n = h->np;
  return SEDCOL_OK;
}

int sedsurr_set_params(sedsurr_handle *h, const float *params)
{
  if (!h || !params) return fail(SEDCOL_EINVAL, "null argument");
  const DeviceScope dscope(h->device);
  for (long long i = 0; i < h->np; ++i)
    if (!std::isfinite(params[i])) return fail(SEDCOL_EDOMAIN, "non-finite parameter");
  HIPOK(hipMemcpyAsync(h->flat, params, sizeof(float) * (size_t)h->np, hipMemcpyHostToDevice, h->st));
  hipLaunchKernelGGL(ss::k_set_params, dim3(kParamBlocks, h->nl), dim3(256), 0, h->st, h->layers, h->flat, h->w, h->wb,
                     h->m, h->v);
  HIPOK(hipGetLastError());
  HIPOK(hipStreamSynchronize(h->st));
  h->step = 0;
  return SEDCOL_OK;
}

int sedsurr_get_params(sedsurr_handle *h, float *params)
{
  if (!h || !params) return fail(SEDCOL_EINVAL, "null argument");
  const DeviceScope dscope(h->device);
  hipLaunchKernelGGL(ss::k_get_params, dim3(kParamBlocks, h->nl), dim3(256), 0, h->st, h->layers, h->w, h->flat, 0,
                     h->slices, (const float *)nullptr, (const float *)nullptr, 0, 0.0f, (float *)nullptr);
  HIPOK(hipGetLastError());
  HIPOK(hipMemcpyAsync(params, h->flat, sizeof(float) * (size_t)h->np, hipMemcpyDeviceToHost, h->st));
  HIPOK(hipStreamSynchronize(h->st));
  return SEDCOL_OK;
}

int sedsurr_set_data(sedsurr_handle *h, const float *X, const float *Y, int64_t n)
{
  if (!h || !X || !Y) return fail(SEDCOL_EINVAL, "null argument");
  const DeviceScope dscope(h->device);
  if (n < 1) return fail(SEDCOL_EINVAL, "need n >= 1");
  if (h->X) (void)hipFree(h->X);
  if (h->Y) (void)hipFree(h->Y);
  h->X = h->Y = nullptr;
  h->ndata = 0;
  HIPOK(hipMalloc(&h->X, sizeof(float) * (size_t)n * h->s.n_in));
  HIPOK(hipMalloc(&h->Y, sizeof(float) * (size_t)n * h->s.n_out));
  HIPOK(hipMemcpyAsync(h->X, X, sizeof(float) * (size_t)n * h->s.n_in, hipMemcpyHostToDevice, h->st));
  HIPOK(hipMemcpyAsync(h->Y, Y, sizeof(float) * (size_t)n * h->s.n_out, hipMemcpyHostToDevice, h->st));
  HIPOK(hipStreamSynchronize(h->st));
  h->ndata = n;
  return SEDCOL_OK;
}

int sedsurr_train(sedsurr_handle *h, int32_t steps, int32_t batch, const int32_t *rows, const sedsurr_adam *adam,
                  float *loss)
{
  if (!h || !rows || !adam) return fail(SEDCOL_EINVAL, "null argument");
  const DeviceScope dscope(h->device);
  if (!h->X) return fail(SEDCOL_EINVAL, "no training set (sedsurr_set_data)");
  if (steps < 1) return fail(SEDCOL_EINVAL, "need steps >= 1");
  if (batch < 1 || batch > h->s.max_batch) return fail(SEDCOL_EINVAL, "batch outside 1..max_batch");
  if (!(adam->lr > 0.0f) || !(adam->beta1 >= 0.0f && adam->beta1 < 1.0f) ||
      !(adam->beta2 >= 0.0f && adam->beta2 < 1.0f) || !(adam->eps > 0.0f))
    return fail(SEDCOL_EINVAL, "Adam settings out of range");
  const long long nr = (long long)steps * batch;
  for (long long i = 0; i < nr; ++i)
    if (rows[i] < 0 || rows[i] >= h->ndata) return fail(SEDCOL_EINVAL, "row index outside the training set");
  if (nr > h->rows_cap) {
    if (h->rows) (void)hipFree(h->rows);
    h->rows = nullptr;
    h->rows_cap = 0;
    HIPOK(hipMalloc(&h->rows, sizeof(int) * nr));
    h->rows_cap = nr;
  }
  if (steps > h->loss_cap) {
    if (h->loss) (void)hipFree(h->loss);
    h->loss = nullptr;
    h->loss_cap = 0;
    HIPOK(hipMalloc(&h->loss, sizeof(float) * steps));
    h->loss_cap = steps;
  }
  HIPOK(hipMemcpyAsync(h->rows, rows, sizeof(int) * nr, hipMemcpyHostToDevice, h->st));
  int launches = 0;
  HIPOK(hipEventRecord(h->e0, h->st));
  gather(h, gather_of(h, h->X, h->Y, h->rows, batch), &launches);
  for (int s = 0; s < steps; ++s) {
    forward(h, batch, &launches);
    backward(h, batch, &launches);
    ++h->step;
    ss::Step p{};
    p.w = h->w;
    p.g = h->g;
    p.m = h->m;
    p.v = h->v;
    p.wb = h->wb;
    p.n = h->np_pad;
    p.lr = adam->lr;
    p.b1 = adam->beta1;
    p.b2 = adam->beta2;
    p.eps = adam->eps;
    p.bc1 = 1.0f - std::pow(adam->beta1, (float)h->step);
    p.bc2 = 1.0f - std::pow(adam->beta2, (float)h->step);
    p.part = h->kpart_all;
    p.na = (int)((h->np_pad / 4 + 255) / 256);
    p.ng = s + 1 < steps ? (batch + 3) / 4 : 0;
    p.lpart = h->part;
    p.nlpart = loss_parts(h, batch);
    p.lscale = 1.0f / ((float)batch * (float)h->s.n_out);
    p.loss = h->loss + s;
    if (p.ng) p.next = gather_of(h, h->X, h->Y, h->rows + (long long)(s + 1) * batch, batch);
    hipLaunchKernelGGL(ss::k_adam, dim3(p.na + p.ng + 1), dim3(256), 0, h->st, p, h->slices);
    ++launches;
  }
  HIPOK(hipGetLastError());
  HIPOK(hipEventRecord(h->e1, h->st));
  HIPOK(hipEventSynchronize(h->e1));
  float ms = 0.f;
  HIPOK(hipEventElapsedTime(&ms, h->e0, h->e1));
  h->last_ms = ms;
  h->last_launches = launches;
  if (loss) {
    HIPOK(hipMemcpyAsync(loss, h->loss, sizeof(float) * steps, hipMemcpyDeviceToHost, h->st));
    HIPOK(hipStreamSynchronize(h->st));
  }
  return SEDCOL_OK;
}

int sedsurr_loss_grad(sedsurr_handle *h, const float *X, const float *Y, int32_t n, float *loss, float *grad)
{
  if (!h || !X || !Y || !loss || !grad) return fail(SEDCOL_EINVAL, "null argument");
  const DeviceScope dscope(h->device);
  if (n < 1 || n > h->s.max_batch) return fail(SEDCOL_EINVAL, "n outside 1..max_batch");
  HIPOK(hipMemcpyAsync(h->xin, X, sizeof(float) * (size_t)n * h->s.n_in, hipMemcpyHostToDevice, h->st));
  HIPOK(hipMemcpyAsync(h->yin, Y, sizeof(float) * (size_t)n * h->s.n_out, hipMemcpyHostToDevice, h->st));
  int launches = 0;
  gather(h, gather_of(h, h->xin, h->yin, nullptr, n), &launches);
  forward(h, n, &launches);
  backward(h, n, &launches);
  const int np = loss_parts(h, n);
  float *loss_dev = h->part + np;
  // the gradient straight into the caller's layout, slices summed on the way
  hipLaunchKernelGGL(ss::k_get_params, dim3(kParamBlocks, h->nl + 1), dim3(256), 0, h->st, h->layers, h->g, h->flat, 1,
                     h->slices, h->kpart_all, h->part, np, 1.0f / ((float)n * (float)h->s.n_out), loss_dev);
  HIPOK(hipGetLastError());
  HIPOK(hipMemcpyAsync(h->h_loss, loss_dev, sizeof(float), hipMemcpyDeviceToHost, h->st));
  HIPOK(hipMemcpyAsync(grad, h->flat, sizeof(float) * (size_t)h->np, hipMemcpyDeviceToHost, h->st));
  HIPOK(hipStreamSynchronize(h->st));
  *loss = *h->h_loss;
  return SEDCOL_OK;
}

// prediction passes of max_batch rows; Y on the device (written by the last
// layer's product directly) or in host memory (copied per pass)
static int predict_rows(sedsurr_handle *h, const float *X, int64_t n, float *Y, bool y_on_device)
{
  int launches = 0;
  HIPOK(hipEventRecord(h->e0, h->st));
  const int B = h->s.max_batch, no = h->s.n_out;
  for (int64_t r0 = 0; r0 < n; r0 += B) {
    const int b = (int)std::min<int64_t>(B, n - r0);
    HIPOK(hipMemcpyAsync(h->xin, X + r0 * h->s.n_in, sizeof(float) * (size_t)b * h->s.n_in, hipMemcpyHostToDevice,
                         h->st));
    gather(h, gather_of(h, h->xin, nullptr, nullptr, b), &launches);
    // compact b x n_out output, in place on the device or staged for the host
    forward(h, b, &launches, y_on_device ? Y + r0 * no : h->yb);
    HIPOK(hipGetLastError());
    if (!y_on_device)
      HIPOK(hipMemcpyAsync(Y + r0 * no, h->yb, sizeof(float) * (size_t)b * no, hipMemcpyDeviceToHost, h->st));
  }
  HIPOK(hipEventRecord(h->e1, h->st));
  HIPOK(hipEventSynchronize(h->e1));
  float ms = 0.f;
  HIPOK(hipEventElapsedTime(&ms, h->e0, h->e1));
  h->last_ms = ms;
  h->last_launches = launches;
  return SEDCOL_OK;
}

int sedsurr_predict(sedsurr_handle *h, const float *X, int64_t n, float *Y)
{
  if (!h || !X || !Y) return fail(SEDCOL_EINVAL, "null argument");
  const DeviceScope dscope(h->device);
  if (n < 0) return fail(SEDCOL_EINVAL, "need n >= 0");
  return predict_rows(h, X, n, Y, false);
}

int sedsurr_predict_device(sedsurr_handle *h, const float *X, int64_t n, const float **Y_device)
{
  if (!h || !X || !Y_device) return fail(SEDCOL_EINVAL, "null argument");
  const DeviceScope dscope(h->device);
  if (n < 1) return fail(SEDCOL_EINVAL, "need n >= 1");
  if (n > h->ydev_rows) {
    HIPOK(hipStreamSynchronize(h->st));
    if (h->ydev) HIPOK(hipFree(h->ydev));
    h->ydev = nullptr;
    h->ydev_rows = 0;
    HIPOK(hipMalloc(&h->ydev, sizeof(float) * (size_t)n * h->s.n_out));
    h->ydev_rows = n;
  }
  const int rc = predict_rows(h, X, n, h->ydev, true);
  *Y_device = rc == SEDCOL_OK ? h->ydev : nullptr;
  return rc;
}

int sedsurr_last_timing(sedsurr_handle *h, double *ms, int32_t *launches)
{
  if (!h || !ms || !launches) return fail(SEDCOL_EINVAL, "null argument");
  const DeviceScope dscope(h->device);
  *ms = h->last_ms;
  *launches = h->last_launches;
  return SEDCOL_OK;
}

}  // extern "C"
