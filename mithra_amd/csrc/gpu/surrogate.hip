// Learned surrogate of a scan point: an ensemble of multilayer perceptrons (SiLU hidden layers,
// linear output) trained and evaluated on the GPU.  Weights are kept in FP32 (the Adam master
// copy) and in BF16 (what the products read); every product is a BF16 x BF16 -> FP32 MFMA GEMM
// (v_mfma_f32_32x32x16_bf16) with FP32 accumulation.  Activations enter the products as BF16;
// pre-activations, losses and gradients stay FP32 until they feed the next product.
//
// The members of the ensemble are marched together: every kernel takes the member from
// blockIdx.z (GEMMs) or blockIdx.y (elementwise), so one launch per layer and pass serves the
// whole ensemble.  Training on a resident data set (mithra_mlp_set_data / _train_epochs) runs
// whole epochs as one captured HIP graph: the mini-batch gather, the forward and backward
// passes, the loss and the Adam update of every member, with the epoch number, learning rate
// and Adam bias corrections read on the device.
//
// GEMM: C[M x N] (FP32, row-major, ldc) = op(A)[M x K] * op(B)[K x N], where op(A)(m, k) is read
// at A[m * sam + k * sak] and op(B)(k, n) at B[k * sbk + n * sbn] (BF16): one kernel serves the
// forward product and both backward products (transposed operands) without copies.  Four
// wavefronts of (32 WM) x (32 WN) make a (64 WM) x (64 WN) workgroup tile; K is staged through
// LDS 32 or 64 at a time, double-buffered: the next stage's 16-byte global loads are in flight
// while the current stage feeds the matrix cores.  Operands contiguous along k are written to
// LDS as they come; operands contiguous along m (or n) are transposed on the way in.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <new>
#include <random>
#include <vector>

#include "common.h"

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float floatx16;

namespace {

inline int status(hipError_t e) { return e == hipSuccess ? MITHRA_OK : MITHRA_E_HIP - (int)e; }

#define SG_TRY(expr)                          \
  do {                                        \
    hipError_t _e = (expr);                   \
    if (_e != hipSuccess) return status(_e);  \
  } while (0)

constexpr int kPadK = 8;  // LDS row padding (bf16): rows stay 16-byte aligned

struct GemmArgs {
  const __bf16* A;
  long sam, sak, sae;  // op(A)(m, k) of member e at A[e sae + m sam + k sak]
  const __bf16* B;
  long sbk, sbn, sbe;  // op(B)(k, n) of member e at B[e sbe + k sbk + n sbn]
  float* C;
  long ldc, sce;       // C(m, n) of member e at C[e sce + m ldc + n]
  int M, N, K;
  int veca, vecb;      // 16-byte loads allowed (aligned bases and strides along the vector)
};

// One 8-element vector of an operand tile: elements (r0 + i dr, c0 + i dc), i < 8, of a matrix
// whose element (r, c) is at P[r sr + c sc]; rows < R and columns < Cn are in range.  `vec`:
// the 8 elements are contiguous and 16-byte aligned whenever they are all in range.
__device__ inline bf16x8 load8(const __bf16* __restrict__ P, long sr, long sc, int r0, int c0, int dr, int dc, int R,
                               int Cn, bool vec) {
  const bool full = r0 + 7 * dr < R && c0 + 7 * dc < Cn && r0 < R && c0 < Cn;
  if (vec && full) return *reinterpret_cast<const bf16x8*>(P + r0 * sr + c0 * sc);
  bf16x8 v;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int r = r0 + i * dr, c = c0 + i * dc;
    v[i] = (r < R && c < Cn) ? P[r * sr + c * sc] : (__bf16)0.0f;
  }
  return v;
}

// Staging of one operand tile of ROWS x TK (rows m of op(A), or n of op(B); k contiguous in LDS)
// by 256 threads.  KC: the operand is contiguous along k, each thread moves 8-element vectors
// straight into LDS rows.  Otherwise it is contiguous along the rows: a thread loads the same 8
// rows at two neighbouring k and writes each row's pair as one 32-bit LDS word (the transpose).
template <int ROWS, int TK, bool KC>
struct Stage {
  static constexpr int kChunks = KC ? ROWS * TK / 8 : (TK / 2) * (ROWS / 8);
  static constexpr int kPasses = kChunks / 256;
  static_assert(kPasses >= 1 && kChunks % 256 == 0, "tile not covered by whole passes");
  bf16x8 r[kPasses][KC ? 1 : 2];
  // P[row sr + k sc] with sr/sc the strides of (row, k); R rows, K columns in range
  __device__ inline void load(const __bf16* __restrict__ P, long sr, long sk, int row0, int k0, int R, int K, bool vec) {
#pragma unroll
    for (int p = 0; p < kPasses; ++p) {
      const int c = threadIdx.x + 256 * p;
      if (KC) {
        r[p][0] = load8(P, sr, sk, row0 + c / (TK / 8), k0 + (c % (TK / 8)) * 8, 0, 1, R, K, vec);
      } else {
        const int row = row0 + (c % (ROWS / 8)) * 8, k = k0 + 2 * (c / (ROWS / 8));
        r[p][0] = load8(P, sr, sk, row, k, 1, 0, R, K, vec);
        r[p][1] = load8(P, sr, sk, row, k + 1, 1, 0, R, K, vec);
      }
    }
  }
  __device__ inline void store(__bf16 (*T)[TK + kPadK]) const {
#pragma unroll
    for (int p = 0; p < kPasses; ++p) {
      const int c = threadIdx.x + 256 * p;
      if (KC) {
        *reinterpret_cast<bf16x8*>(&T[c / (TK / 8)][(c % (TK / 8)) * 8]) = r[p][0];
      } else {
        const int row = (c % (ROWS / 8)) * 8, k = 2 * (c / (ROWS / 8));
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          typedef __attribute__((__vector_size__(2 * sizeof(__bf16)))) __bf16 bf16x2;
          const bf16x2 w = {r[p][0][i], r[p][1][i]};
          *reinterpret_cast<bf16x2*>(&T[row + i][k]) = w;
        }
      }
    }
  }
};

__device__ inline float silu(float z) { return z / (1.0f + expf(-z)); }
__device__ inline float silu_grad(float z) {
  const float s = 1.0f / (1.0f + expf(-z));
  return s * (1.0f + z * (1.0f - s));
}

// What a product's workgroup does with its tile (member e's slab at e times the stride):
//   kPlain  C = acc
//   kHidden z = acc + bias; Z = z (when kept for the backward pass), act = bf16(silu(z))
//   kOutput z = acc + bias; Z = z
//   kLoss   y = acc + bias against the targets: dZ = bf16(2 (y - t) scale), the tile's column sums of
//           2 (y - t) scale (FP32) and its sum of (y - t)^2 (FP64: a tile has up to 16384 terms)
//   kBack   g = acc silu'(Z): dZ = bf16(g), the tile's column sums of g (FP32)
// so that biases, activations, losses and bias gradients cost no launches and no passes of their own.
// A training step of 256 rows (five members, 264-512-512-512-256) is a chain of short launches: 30 of
// them and 280 us with bias, activation, loss and column sums apart (the column sums 17 us a layer), 11
// and 165 us so.  A prediction of 4096 rows: four products of 42 us and four passes of 22 us each, 58 to 70
// us and 34 us (the output) so.
enum Epilogue { kPlain, kHidden, kOutput, kLoss, kBack };

struct Epi {
  const float* bias;   // of the layer, FP32
  long sbias;
  float* Z;            // pre-activations, rows of N (nullptr: not kept)
  long sz;
  __bf16* act;         // kHidden: the next layer's inputs; kLoss, kBack: dZ; rows of N
  long sact;
  const float* tgt;    // kLoss: targets, rows of N, shared
  float scale;
  float* colsum;       // kLoss, kBack: [row tile][N] column sums
  long scol;
  double* loss;        // kLoss: [tile] sums of squares
  long sloss;
};

// Lane layout of v_mfma_f32_32x32x16_bf16 (64 lanes, l = lane): A supplies row l % 32 and
// k = 8 (l / 32) .. +7, B column l % 32 and the same k; accumulator i of lane l is row
// 8 (i / 4) + 4 (l / 32) + i % 4, column l % 32.
// AK: op(A) contiguous along k (sak = 1), else along m (sam = 1); BK: op(B) along k (sbk = 1),
// else along n (sbn = 1).  With general strides the vector flags are off and any form is exact.
// lds: gemm_lds<WM, WN, TK>() bytes; tile (bx, by) of member e.
template <int WM, int WN, int TK>
constexpr int gemm_lds() {
  return 2 * (64 * WM + 64 * WN) * (TK + kPadK) * (int)sizeof(__bf16);
}

template <int WM, int WN, int TK, bool AK, bool BK, Epilogue EPI>
__device__ inline void gemm_tile(const GemmArgs& g, const Epi& q, char* lds, int bx, int by, int nbx, int e) {
  constexpr int BM = 64 * WM, BN = 64 * WN, LD = TK + kPadK;
  auto As = reinterpret_cast<__bf16(*)[BM][LD]>(lds);                                   // rows m, k contiguous
  auto Bs = reinterpret_cast<__bf16(*)[BN][LD]>(lds + 2 * BM * LD * sizeof(__bf16));  // rows n, k contiguous
  const __bf16* __restrict__ A = g.A + e * g.sae;
  const __bf16* __restrict__ B = g.B + e * g.sbe;
  const int m0 = by * BM, n0 = bx * BN;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int wm = (w >> 1) * 32 * WM, wn = (w & 1) * 32 * WN;
  const bool va = g.veca, vb = g.vecb;
  Stage<BM, TK, AK> sa;
  Stage<BN, TK, BK> sb;
  // op(B)(k, n) = B[k sbk + n sbn] is staged as rows n: the matrix (n, k) with strides (sbn, sbk)
  auto load = [&](int k0) {
    sa.load(A, g.sam, g.sak, m0, k0, g.M, g.K, va);
    sb.load(B, g.sbn, g.sbk, n0, k0, g.N, g.K, vb);
  };
  floatx16 acc[WM][WN];
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j) acc[i][j] = floatx16{};
  load(0);
  sa.store(As[0]);
  sb.store(Bs[0]);
  __syncthreads();
  int buf = 0;
  for (int k0 = 0; k0 < g.K; k0 += TK) {
    const bool next = k0 + TK < g.K;
    if (next) load(k0 + TK);  // in flight while this stage computes
#pragma unroll
    for (int kk = 0; kk < TK; kk += 16) {
      bf16x8 a[WM], b[WN];
#pragma unroll
      for (int i = 0; i < WM; ++i)
        a[i] = *reinterpret_cast<const bf16x8*>(&As[buf][wm + 32 * i + (lane & 31)][kk + 8 * (lane >> 5)]);
#pragma unroll
      for (int j = 0; j < WN; ++j)
        b[j] = *reinterpret_cast<const bf16x8*>(&Bs[buf][wn + 32 * j + (lane & 31)][kk + 8 * (lane >> 5)]);
#pragma unroll
      for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int j = 0; j < WN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
    }
    // the other buffer was last read in the previous stage, which the barrier below it closed
    if (next) {
      sa.store(As[buf ^ 1]);
      sb.store(Bs[buf ^ 1]);
    }
    __syncthreads();
    buf ^= 1;
  }
  // the epilogue reuses the staging memory: every wavefront is past its last read of it
  float* const sums = reinterpret_cast<float*>(lds);  // [2][BN] column sums
  double* const losses = reinterpret_cast<double*>(sums + 2 * BN);  // [4]
  constexpr bool kSums = EPI == kLoss || EPI == kBack;
  double sq = 0.0;
#pragma unroll
  for (int j = 0; j < WN; ++j) {
    const int c = n0 + wn + 32 * j + (lane & 31);
    const bool cok = c < g.N;
    const float bias = (EPI == kHidden || EPI == kOutput || EPI == kLoss) && cok ? q.bias[e * q.sbias + c] : 0.0f;
    float col = 0.0f;
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int r = m0 + wm + 32 * i + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
        if (r >= g.M || !cok) continue;
        const float x = acc[i][j][v];
        const long at = (long)r * g.N + c;
        if (EPI == kPlain) {
          g.C[e * g.sce + (long)r * g.ldc + c] = x;
        } else if (EPI == kHidden) {
          const float z = x + bias;
          if (q.Z) q.Z[e * q.sz + at] = z;
          q.act[e * q.sact + at] = (__bf16)silu(z);
        } else if (EPI == kOutput) {
          q.Z[e * q.sz + at] = x + bias;
        } else if (EPI == kLoss) {
          const float d = (x + bias) - q.tgt[at];
          const float gr = 2.0f * d * q.scale;
          q.act[e * q.sact + at] = (__bf16)gr;
          col += gr;
          sq += (double)d * (double)d;
        } else {
          const float gr = x * silu_grad(q.Z[e * q.sz + at]);
          q.act[e * q.sact + at] = (__bf16)gr;
          col += gr;
        }
      }
    if (kSums) {
      col += __shfl_xor(col, 32);
      if (lane < 32) sums[(w >> 1) * BN + wn + 32 * j + lane] = col;
    }
  }
  if (EPI == kLoss) {
#pragma unroll
    for (int h = 32; h > 0; h >>= 1) sq += __shfl_xor(sq, h);
    if (lane == 0) losses[w] = sq;
  }
  if (kSums) {
    __syncthreads();
    if ((int)threadIdx.x < BN && n0 + (int)threadIdx.x < g.N)
      q.colsum[e * q.scol + (long)by * g.N + n0 + threadIdx.x] = sums[threadIdx.x] + sums[BN + threadIdx.x];
    if (EPI == kLoss && threadIdx.x == 0)
      q.loss[e * q.sloss + (long)by * nbx + bx] = (losses[0] + losses[1]) + (losses[2] + losses[3]);
  }
}

template <int WM, int WN, int TK, bool AK, bool BK, Epilogue EPI>
__global__ __launch_bounds__(256) void k_gemm(GemmArgs g, Epi q) {
  __shared__ __attribute__((aligned(16))) char lds[gemm_lds<WM, WN, TK>()];
  gemm_tile<WM, WN, TK, AK, BK, EPI>(g, q, lds, blockIdx.x, blockIdx.y, gridDim.x, blockIdx.z);
}

// The two products that read dZ of a layer, in one launch: dW = X^T dZ (plain) in the first `nw`
// workgroups, dZ of the layer below (kBack) in the rest; both 64 x 64 tiles.
__global__ __launch_bounds__(256) void k_gemm_back(GemmArgs gw, GemmArgs ga, Epi q, int nw) {
  __shared__ __attribute__((aligned(16))) char lds[gemm_lds<1, 1, 64>()];
  const int e = blockIdx.z;
  if ((int)blockIdx.x < nw) {
    const int nx = (gw.N + 63) / 64;
    gemm_tile<1, 1, 64, false, false, kPlain>(gw, q, lds, blockIdx.x % nx, blockIdx.x / nx, nx, e);
  } else {
    const int nx = (ga.N + 63) / 64, b = blockIdx.x - nw;
    gemm_tile<1, 1, 64, true, true, kBack>(ga, q, lds, b % nx, b / nx, nx, e);
  }
}

__global__ void k_to_bf16(const float* __restrict__ x, __bf16* __restrict__ y, long n) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) y[t] = (__bf16)x[t];
}

// Bias gradients of every layer: member blockIdx.y, layer blockIdx.z, the row tiles' column sums in
// order.  The last workgroup column of layer 0 adds the mini-batch's loss to the epoch's entry (out set).
struct BiasLayer {
  const float* col;    // [tiles][d] per member
  long scol;
  int d, tiles;
  long off;            // of the biases in a member's parameters
};
constexpr int kBiasLayers = 16;  // layers per launch
struct BiasLayers {
  BiasLayer l[kBiasLayers];
};

__global__ __launch_bounds__(64) void k_bias_grad(BiasLayers t, float* __restrict__ g, long pm,
                                                  const double* __restrict__ loss, int nb,
                                                  const int* __restrict__ epoch, float* __restrict__ out, int members,
                                                  float scale) {
  if (out && blockIdx.x == gridDim.x - 1) {  // one more column of workgroups than the biases take
    const int e = threadIdx.x;
    if (blockIdx.y == 0 && blockIdx.z == 0 && e < members) {
      double s = 0.0;
      for (int i = 0; i < nb; ++i) s += loss[(long)e * nb + i];
      out[(long)*epoch * members + e] += (float)(s * (double)scale);
    }
    return;
  }
  const BiasLayer L = t.l[blockIdx.z];
  const int j = blockIdx.x * 64 + threadIdx.x, e = blockIdx.y;
  if (j >= L.d) return;
  float s = 0.0f;
  for (int b = 0; b < L.tiles; ++b) s += L.col[e * L.scol + (long)b * L.d + j];
  g[e * pm + L.off + j] = s;
}

// The schedule of a captured epoch: the epoch number lives on the device (*epoch), so one graph
// serves every epoch.  Step t = step0 + epoch steps + b + 1 (Adam's count, from 1); learning rate
// max(lr_max (1 + cos(pi epoch / epochs)) / 2, lr_min).
struct EpochSched {
  const int* epoch;
  long step0;
  int steps, b, epochs;
  float lr_max, lr_min;
};

constexpr float kB1 = 0.9f, kB2 = 0.999f, kEps = 1e-8f;

// Adam on the FP32 master weights (all members); the BF16 copy follows.  With s.epoch set, the
// rate and bias corrections come from the schedule, else from lr, c1, c2.  HBM and the schedule's
// powers bound it: four parameters a thread (16-byte accesses; the arrays are padded to four) 36 ->
// 19.4 us for the surrogate's five members of 793k parameters.
__global__ __launch_bounds__(256) void k_adam(float* __restrict__ w, __bf16* __restrict__ wb,
                                              const float* __restrict__ g, float* __restrict__ m,
                                              float* __restrict__ v, long n, float lr, float c1, float c2,
                                              EpochSched s) {
  const long t = 4 * ((long)blockIdx.x * blockDim.x + threadIdx.x);
  if (t >= n) return;
  if (s.epoch) {
    const int ep = *s.epoch;
    const float step = (float)(s.step0 + (long)ep * s.steps + s.b + 1);
    c1 = 1.0f - powf(kB1, step);
    c2 = 1.0f - powf(kB2, step);
    lr = fmaxf(s.lr_max * 0.5f * (1.0f + cosf(3.14159265358979f * (float)ep / (float)s.epochs)), s.lr_min);
  }
  typedef float floatx4 __attribute__((ext_vector_type(4)));
  typedef __attribute__((__vector_size__(4 * sizeof(__bf16)))) __bf16 bf16x4;
  const floatx4 gv = *reinterpret_cast<const floatx4*>(g + t);
  floatx4 mv = *reinterpret_cast<const floatx4*>(m + t), vv = *reinterpret_cast<const floatx4*>(v + t),
          wv = *reinterpret_cast<const floatx4*>(w + t);
  bf16x4 wq;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const float gi = gv[q];
    const float mi = kB1 * mv[q] + (1.0f - kB1) * gi;
    const float vi = kB2 * vv[q] + (1.0f - kB2) * gi * gi;
    mv[q] = mi;
    vv[q] = vi;
    wv[q] = wv[q] - lr * (mi / c1) / (sqrtf(vi / c2) + kEps);
    wq[q] = (__bf16)wv[q];
  }
  *reinterpret_cast<floatx4*>(m + t) = mv;
  *reinterpret_cast<floatx4*>(v + t) = vv;
  *reinterpret_cast<floatx4*>(w + t) = wv;
  *reinterpret_cast<bf16x4*>(wb + t) = wq;
}

// Mini-batch b of the epoch *epoch: rows perm[epoch n_data + b batch + r] of the resident data
// set, inputs (BF16) and targets (FP32).
__global__ void k_gather(const __bf16* __restrict__ dx, const float* __restrict__ dt, const int* __restrict__ perm,
                         const int* __restrict__ epoch, long n_data, int b, int batch, int d0, int dL,
                         __bf16* __restrict__ xb, float* __restrict__ tb) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const int r = blockIdx.y;
  if (r >= batch) return;
  const long src = perm[(long)*epoch * n_data + (long)b * batch + r];
  if (t < d0) xb[(long)r * d0 + t] = dx[src * d0 + t];
  if (t < dL) tb[(long)r * dL + t] = dt[src * dL + t];
}

__global__ void k_next_epoch(int* epoch) {
  if (threadIdx.x == 0) *epoch += 1;
}

// A chunk of the outputs into pinned memory.
__global__ __launch_bounds__(256) void k_copy_out(const float* __restrict__ y, float* __restrict__ out, long n) {
  const long t = (long)blockIdx.x * 256 + threadIdx.x;
  if (t < n) out[t] = y[t];
}

__global__ void k_fill(float* __restrict__ p, long n, float v) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) p[t] = v;
}

unsigned blocks(long n, int per = 256) { return (unsigned)((n + per - 1) / per); }
long tiles64(long n) { return (n + 63) / 64; }

}  // namespace

struct mithra_mlp {
  int members = 0, layers = 0;
  std::vector<int> dims;            // layers + 1 widths
  std::vector<long> woff, boff;     // offsets of W_l (d_l x d_{l+1}, row-major) and b_l in one member
  long per_member = 0;              // parameters per member
  hipStream_t stream = nullptr;
  float* w = nullptr;               // FP32 master parameters, members x per_member
  __bf16* wb = nullptr;             // BF16 copy (the biases' entries unused)
  float* g = nullptr;               // gradients, members x per_member
  float* m = nullptr;               // Adam moments
  float* v = nullptr;
  long step = 0;                    // Adam steps taken
  // activations for a batch of up to cap rows; every buffer but X[0] holds one slab per member
  long cap = 0;
  std::vector<__bf16*> X;           // layer inputs (BF16): X[0] n x d_0 (shared), X[l] members x n x d_l
  std::vector<float*> Z;            // pre-activations (FP32), members x n x d_{l+1}
  __bf16* dZ[2] = {nullptr, nullptr};  // gradients of the pre-activations, members x n x max width
  std::vector<float*> col;          // per layer: dZ's column sums per row tile, members x tiles x d_{l+1}
  mithra::HostStage stage = {};     // pinned slots of transfers to the host
  float* xin = nullptr;             // FP32 staging of the inputs, n x d_0
  float* tgt = nullptr;             // targets, n x d_L (shared)
  double* partial = nullptr;        // the loss's sums per tile, members x tiles
  int maxw = 0;
  // resident training data
  long n_data = 0;
  __bf16* data_x = nullptr;         // n_data x d_0
  float* data_t = nullptr;          // n_data x d_L
};

namespace {

void free_acts(mithra_mlp* p) {
  for (auto* x : p->X) (void)hipFree(x);
  for (auto* z : p->Z) (void)hipFree(z);
  for (auto* c : p->col) (void)hipFree(c);
  p->X.clear();
  p->Z.clear();
  p->col.clear();
  (void)hipFree(p->dZ[0]); (void)hipFree(p->dZ[1]);
  (void)hipFree(p->xin); (void)hipFree(p->tgt); (void)hipFree(p->partial);
  p->dZ[0] = p->dZ[1] = nullptr;
  p->xin = p->tgt = nullptr;
  p->partial = nullptr;
  p->cap = 0;
}

int ensure_acts(mithra_mlp* p, long n) {
  if (n <= p->cap) return MITHRA_OK;
  SG_TRY(hipStreamSynchronize(p->stream));
  free_acts(p);
  const int L = p->layers;
  const long E = p->members;
  p->X.assign(L, nullptr);
  p->Z.assign(L, nullptr);
  p->col.assign(L, nullptr);
  bool ok = true;
  for (int l = 0; l < L && ok; ++l) {
    ok = hipMalloc(&p->X[l], sizeof(__bf16) * (l ? E : 1) * n * p->dims[l]) == hipSuccess &&
         hipMalloc(&p->Z[l], sizeof(float) * E * n * p->dims[l + 1]) == hipSuccess &&
         hipMalloc(&p->col[l], sizeof(float) * E * tiles64(n) * p->dims[l + 1]) == hipSuccess;
  }
  ok = ok && hipMalloc(&p->dZ[0], sizeof(__bf16) * E * n * p->maxw) == hipSuccess &&
       hipMalloc(&p->dZ[1], sizeof(__bf16) * E * n * p->maxw) == hipSuccess &&
       hipMalloc(&p->xin, sizeof(float) * n * p->dims[0]) == hipSuccess &&
       hipMalloc(&p->tgt, sizeof(float) * n * p->dims[L]) == hipSuccess &&
       hipMalloc(&p->partial, sizeof(double) * E * tiles64(n) * tiles64(p->dims[L])) == hipSuccess;
  if (!ok) {
    free_acts(p);
    return MITHRA_E_NOMEM;
  }
  p->cap = n;
  return MITHRA_OK;
}

bool aligned16(const void* q) { return ((uintptr_t)q & 15) == 0; }

// The workgroup tile of a product: 128 x 128 where that still makes a workgroup per compute unit
// (half the operand traffic), else 64 x 64.
int gemm_tile_size(long M, long N, int members) {
  return ((M + 127) / 128) * ((N + 127) / 128) * members >= 256 ? 128 : 64;
}

// The vector flags: each 8-element run along the operand's contiguous direction (k with AK/BK, else
// m or n) must start 16-byte aligned.
template <bool AK, bool BK>
void vector_flags(GemmArgs& g) {
  g.veca = aligned16(g.A) && g.sae % 8 == 0 && (AK ? g.sak == 1 && g.sam % 8 == 0 : g.sam == 1 && g.sak % 8 == 0);
  g.vecb = aligned16(g.B) && g.sbe % 8 == 0 && (BK ? g.sbk == 1 && g.sbn % 8 == 0 : g.sbn == 1 && g.sbk % 8 == 0);
}

// T: 128 (k staged 32 at a time) or 64 (k staged 64 at a time: half the barriers on short products)
template <bool AK, bool BK, Epilogue EPI>
hipError_t gemm(hipStream_t s, GemmArgs g, const Epi& q, int members, int T) {
  vector_flags<AK, BK>(g);
  const dim3 grid((unsigned)((g.N + T - 1) / T), (unsigned)((g.M + T - 1) / T), (unsigned)members);
  if (T == 128)
    hipLaunchKernelGGL((k_gemm<2, 2, 32, AK, BK, EPI>), grid, dim3(256), 0, s, g, q);
  else
    hipLaunchKernelGGL((k_gemm<1, 1, 64, AK, BK, EPI>), grid, dim3(256), 0, s, g, q);
  return hipGetLastError();
}

// Forward pass of members e0 .. e0 + ne - 1 on X[0] (already BF16, n rows): X[l + 1] in the members'
// slabs.  Without targets the outputs go to Z[L - 1]; with them (train) the hidden layers' Z are kept,
// dZ of the last layer goes to dZ[0], with its column sums and the loss's sums.
int forward(mithra_mlp* p, int e0, int ne, long n, bool train) {
  hipStream_t s = p->stream;
  const int L = p->layers;
  const long pm = p->per_member;
  for (int l = 0; l < L; ++l) {
    const int di = p->dims[l], dout = p->dims[l + 1];
    const int T = gemm_tile_size(n, dout, ne);
    GemmArgs g{};
    g.A = p->X[l]; g.sam = di; g.sak = 1; g.sae = l ? n * di : 0;
    g.B = p->wb + e0 * pm + p->woff[l]; g.sbk = dout; g.sbn = 1; g.sbe = pm;
    g.M = (int)n; g.N = dout; g.K = di;
    Epi q{};
    q.bias = p->w + e0 * pm + p->boff[l]; q.sbias = pm;
    q.Z = p->Z[l]; q.sz = n * dout; q.sact = n * dout;
    if (l + 1 < L) {
      if (!train) q.Z = nullptr;
      q.act = p->X[l + 1];
      SG_TRY((gemm<true, false, kHidden>(s, g, q, ne, T)));
    } else if (!train) {
      SG_TRY((gemm<true, false, kOutput>(s, g, q, ne, T)));
    } else {
      const long rows = (n + T - 1) / T, cols = (dout + T - 1) / T;
      q.act = p->dZ[0];
      q.tgt = p->tgt;
      q.scale = 1.0f / (float)(n * dout);
      q.colsum = p->col[l]; q.scol = rows * dout;
      q.loss = p->partial; q.sloss = rows * cols;
      SG_TRY((gemm<true, false, kLoss>(s, g, q, ne, T)));
    }
  }
  return MITHRA_OK;
}

// The loss's sums per member that forward(..., train) leaves in p->partial
long loss_tiles(const mithra_mlp* p, int ne, long n) {
  const int dL = p->dims[p->layers], T = gemm_tile_size(n, dL, ne);
  return ((n + T - 1) / T) * ((dL + T - 1) / T);
}

// Gradients of members e0 .. e0 + ne - 1 into their slots of p->g (the training forward pass must
// have run on the batch).  epoch_loss: the mini-batch's loss, times loss_scale, is added to the
// entries of *epoch there; `loss`: the per-member loss to the host.
int backward(mithra_mlp* p, int e0, int ne, long n, float* loss, const int* epoch = nullptr, float* epoch_loss = nullptr,
             float loss_scale = 0.0f) {
  hipStream_t s = p->stream;
  const int L = p->layers;
  const long pm = p->per_member, nb = loss_tiles(p, ne, n);
  std::vector<long> tiles(L);  // row tiles of each layer's column sums
  tiles[L - 1] = (n + gemm_tile_size(n, p->dims[L], ne) - 1) / gemm_tile_size(n, p->dims[L], ne);
  for (int l = L - 1; l >= 0; --l) {
    const int di = p->dims[l], dout = p->dims[l + 1];
    const __bf16* dz = p->dZ[(L - 1 - l) & 1];
    // dW_l = X_l^T dZ_l  (di x dout)
    GemmArgs g{};
    g.A = p->X[l]; g.sam = 1; g.sak = di; g.sae = l ? n * di : 0;
    g.B = dz; g.sbk = dout; g.sbn = 1; g.sbe = n * dout;
    g.C = p->g + e0 * pm + p->woff[l]; g.ldc = dout; g.sce = pm;
    g.M = di; g.N = dout; g.K = (int)n;
    const int Tw = gemm_tile_size(di, dout, ne);
    if (l == 0) {
      SG_TRY((gemm<false, false, kPlain>(s, g, Epi{}, ne, Tw)));
      break;
    }
    // dA_{l-1} = dZ_l W_l^T  (n x di), dZ_{l-1} = dA_{l-1} silu'(Z_{l-1})
    GemmArgs h{};
    h.A = dz; h.sam = dout; h.sak = 1; h.sae = n * dout;
    h.B = p->wb + e0 * pm + p->woff[l]; h.sbk = 1; h.sbn = dout; h.sbe = pm;
    h.M = (int)n; h.N = di; h.K = dout;
    const int T = gemm_tile_size(n, di, ne);
    tiles[l - 1] = (n + T - 1) / T;
    Epi q{};
    q.Z = p->Z[l - 1]; q.sz = n * di;
    q.act = p->dZ[(L - l) & 1]; q.sact = n * di;
    q.colsum = p->col[l - 1]; q.scol = tiles[l - 1] * di;
    if (T == 64 && Tw == 64) {  // neither fills the chip by itself
      vector_flags<false, false>(g);
      vector_flags<true, true>(h);
      const long nw = tiles64(g.M) * tiles64(g.N), nh = tiles64(h.M) * tiles64(h.N);
      hipLaunchKernelGGL(k_gemm_back, dim3((unsigned)(nw + nh), 1, ne), dim3(256), 0, s, g, h, q, (int)nw);
      SG_TRY(hipGetLastError());
    } else {
      SG_TRY((gemm<false, false, kPlain>(s, g, Epi{}, ne, Tw)));
      SG_TRY((gemm<true, true, kBack>(s, h, q, ne, T)));
    }
  }
  for (int l0 = 0; l0 < L; l0 += kBiasLayers) {
    BiasLayers t{};
    const int nl = std::min(kBiasLayers, L - l0);
    int dmax = 1;
    for (int i = 0; i < nl; ++i) {
      const int d = p->dims[l0 + i + 1];
      t.l[i] = BiasLayer{p->col[l0 + i], tiles[l0 + i] * d, d, (int)tiles[l0 + i], p->boff[l0 + i]};
      dmax = std::max(dmax, d);
    }
    float* out = l0 == 0 ? epoch_loss : nullptr;
    hipLaunchKernelGGL(k_bias_grad, dim3((unsigned)tiles64(dmax) + (out ? 1 : 0), ne, nl), dim3(64), 0, s, t,
                       p->g + e0 * pm, pm, p->partial, (int)nb, epoch, out, ne, loss_scale);
    SG_TRY(hipGetLastError());
  }
  if (loss) {
    std::vector<double> part((size_t)ne * nb);
    SG_TRY(hipMemcpyAsync(part.data(), p->partial, sizeof(double) * part.size(), hipMemcpyDeviceToHost, s));
    SG_TRY(hipStreamSynchronize(s));
    for (int e = 0; e < ne; ++e) {
      double sum = 0.0;
      for (long i = 0; i < nb; ++i) sum += part[(size_t)e * nb + i];
      loss[e] = (float)(sum / ((double)n * p->dims[L]));
    }
  }
  return MITHRA_OK;
}

int load_inputs(mithra_mlp* p, const float* x, const float* t, long n) {
  if (int rc = ensure_acts(p, n)) return rc;
  hipStream_t s = p->stream;
  const long nx = n * p->dims[0];
  SG_TRY(hipMemcpyAsync(p->xin, x, sizeof(float) * nx, hipMemcpyHostToDevice, s));
  hipLaunchKernelGGL(k_to_bf16, dim3(blocks(nx)), dim3(256), 0, s, p->xin, p->X[0], nx);
  SG_TRY(hipGetLastError());
  if (t) SG_TRY(hipMemcpyAsync(p->tgt, t, sizeof(float) * n * p->dims[p->layers], hipMemcpyHostToDevice, s));
  SG_TRY(hipStreamSynchronize(s));  // the host arrays may go away on return
  return MITHRA_OK;
}

hipError_t adam(mithra_mlp* p, float lr, float c1, float c2, EpochSched sched) {
  const long n = (long)p->members * p->per_member;
  hipLaunchKernelGGL(k_adam, dim3(blocks(n, 1024)), dim3(256), 0, p->stream, p->w, p->wb, p->g, p->m, p->v, n, lr, c1, c2,
                     sched);
  return hipGetLastError();
}

// One epoch of `steps` mini-batches of the resident data, every member, as stream work (for
// capture): gather, forward, backward, loss, Adam; then the epoch counter advances.
int enqueue_epoch(mithra_mlp* p, const int* perm, int* epoch, float* epoch_loss, int steps, int batch, int epochs,
                  float lr_max, float lr_min) {
  hipStream_t s = p->stream;
  const int d0 = p->dims[0], dL = p->dims[p->layers];
  for (int b = 0; b < steps; ++b) {
    hipLaunchKernelGGL(k_gather, dim3(blocks(std::max(d0, dL)), batch), dim3(256), 0, s, p->data_x, p->data_t, perm,
                       epoch, p->n_data, b, batch, d0, dL, p->X[0], p->tgt);
    SG_TRY(hipGetLastError());
    if (int rc = forward(p, 0, p->members, batch, true)) return rc;
    if (int rc = backward(p, 0, p->members, batch, nullptr, epoch, epoch_loss,
                          1.0f / ((float)batch * dL * steps * p->members)))
      return rc;
    EpochSched sched{epoch, p->step, steps, b, epochs, lr_max, lr_min};
    SG_TRY(adam(p, 0.0f, 1.0f, 1.0f, sched));
  }
  hipLaunchKernelGGL(k_next_epoch, dim3(1), dim3(64), 0, s, epoch);
  SG_TRY(hipGetLastError());
  return MITHRA_OK;
}

}  // namespace

extern "C" {

int mithra_mlp_create(int members, int layers, const int* dims, unsigned long long seed, mithra_mlp** out) {
  if (!out || members < 1 || members > 64 || layers < 1 || !dims) return MITHRA_E_ARG;
  for (int l = 0; l <= layers; ++l)
    if (dims[l] < 1) return MITHRA_E_ARG;
  *out = nullptr;
  mithra_mlp* p = new (std::nothrow) mithra_mlp();
  if (!p) return MITHRA_E_NOMEM;
  p->members = members;
  p->layers = layers;
  p->dims.assign(dims, dims + layers + 1);
  long off = 0;
  for (int l = 0; l < layers; ++l) {
    p->woff.push_back(off);
    off += (long)dims[l] * dims[l + 1];
    p->boff.push_back(off);
    off += dims[l + 1];
    p->maxw = std::max(p->maxw, std::max(dims[l], dims[l + 1]));
  }
  p->per_member = off;
  const size_t total = ((size_t)members * off + 3) / 4 * 4;  // whole vectors of the Adam update
  int rc = status(hipStreamCreateWithFlags(&p->stream, hipStreamNonBlocking));
  if (!rc && (hipMalloc(&p->w, sizeof(float) * total) != hipSuccess ||
              hipMalloc(&p->wb, sizeof(__bf16) * total) != hipSuccess ||
              hipMalloc(&p->g, sizeof(float) * total) != hipSuccess ||
              hipMalloc(&p->m, sizeof(float) * total) != hipSuccess ||
              hipMalloc(&p->v, sizeof(float) * total) != hipSuccess))
    rc = MITHRA_E_NOMEM;
  if (rc) {
    mithra_mlp_destroy(p);
    return rc;
  }
  // He-normal weights, zero biases; each member from its own stream of the seed
  std::vector<float> h(total, 0.0f);
  for (int e = 0; e < members; ++e) {
    std::mt19937_64 gen(seed * 1000003ull + (unsigned long long)e);
    for (int l = 0; l < layers; ++l) {
      std::normal_distribution<float> nd(0.0f, std::sqrt(2.0f / (float)dims[l]));
      float* W = h.data() + (size_t)e * off + p->woff[l];
      for (long i = 0; i < (long)dims[l] * dims[l + 1]; ++i) W[i] = nd(gen);
    }
  }
  rc = mithra_mlp_set_params(p, -1, h.data());
  if (!rc) {
    std::fill(h.begin(), h.end(), 0.0f);
    rc = status(hipMemcpy(p->m, h.data(), sizeof(float) * total, hipMemcpyHostToDevice));
    if (!rc) rc = status(hipMemcpy(p->v, h.data(), sizeof(float) * total, hipMemcpyHostToDevice));
  }
  if (rc) {
    mithra_mlp_destroy(p);
    return rc;
  }
  *out = p;
  return MITHRA_OK;
}

int mithra_mlp_destroy(mithra_mlp* p) {
  if (!p) return MITHRA_E_ARG;
  if (p->stream) (void)hipStreamSynchronize(p->stream);
  free_acts(p);
  mithra::stage_free(&p->stage);
  (void)hipFree(p->w); (void)hipFree(p->wb); (void)hipFree(p->g); (void)hipFree(p->m); (void)hipFree(p->v);
  (void)hipFree(p->data_x); (void)hipFree(p->data_t);
  if (p->stream) (void)hipStreamDestroy(p->stream);
  delete p;
  return MITHRA_OK;
}

long mithra_mlp_param_count(const mithra_mlp* p) { return p ? p->per_member : -1; }

// member = -1: all members from params (members x per-member); else one member.
int mithra_mlp_set_params(mithra_mlp* p, int member, const float* params) {
  if (!p || !params || member < -1 || member >= p->members) return MITHRA_E_ARG;
  const size_t n = (size_t)(member < 0 ? p->members : 1) * p->per_member;
  float* w = p->w + (member < 0 ? 0 : (size_t)member * p->per_member);
  __bf16* wb = p->wb + (member < 0 ? 0 : (size_t)member * p->per_member);
  SG_TRY(hipMemcpyAsync(w, params, sizeof(float) * n, hipMemcpyHostToDevice, p->stream));
  hipLaunchKernelGGL(k_to_bf16, dim3(blocks((long)n)), dim3(256), 0, p->stream, w, wb, (long)n);
  SG_TRY(hipGetLastError());
  SG_TRY(hipStreamSynchronize(p->stream));
  return MITHRA_OK;
}

int mithra_mlp_get_params(mithra_mlp* p, int member, float* params) {
  if (!p || !params || member < -1 || member >= p->members) return MITHRA_E_ARG;
  const size_t n = (size_t)(member < 0 ? p->members : 1) * p->per_member;
  SG_TRY(hipStreamSynchronize(p->stream));
  SG_TRY(hipMemcpy(params, p->w + (member < 0 ? 0 : (size_t)member * p->per_member), sizeof(float) * n,
                   hipMemcpyDeviceToHost));
  return MITHRA_OK;
}

// y: members x n x d_out, each member's prediction for the n rows of x (n x d_in).
int mithra_mlp_forward(mithra_mlp* p, const float* x, long n, float* y) {
  if (!p || !x || !y || n < 1) return MITHRA_E_ARG;
  if (int rc = load_inputs(p, x, nullptr, n)) return rc;
  const int dL = p->dims[p->layers];
  if (int rc = forward(p, 0, p->members, n, false)) return rc;
  const float* out = p->Z[p->layers - 1];
  const long values = (long)p->members * n * dL;
  // the layout is the caller's: a network's only prediction, when small, is a plain copy (see kOnce)
  if (mithra::stage_first(&p->stage, sizeof(float) * values, 3 << 19)) {
    SG_TRY(hipMemcpyAsync(y, out, sizeof(float) * values, hipMemcpyDeviceToHost, p->stream));
    SG_TRY(hipStreamSynchronize(p->stream));
    return MITHRA_OK;
  }
  auto put = [&](long i, long m, char* slot) {
    hipLaunchKernelGGL(k_copy_out, dim3(blocks(m)), dim3(256), 0, p->stream, out + i, (float*)slot, m);
    return hipGetLastError();
  };
  auto take = [&](long i, long m, const char* slot) { std::memcpy(y + i, slot, sizeof(float) * m); };
  return mithra::stage_chunks(&p->stage, p->stream, values, sizeof(float), put, take);
}

// Loss (mean squared error over the n x d_out targets) and its gradient for one member, in the
// parameter layout of mithra_mlp_get_params.
int mithra_mlp_gradients(mithra_mlp* p, int member, const float* x, const float* t, long n, float* grads,
                         float* loss) {
  if (!p || !x || !t || n < 1 || member < 0 || member >= p->members) return MITHRA_E_ARG;
  if (int rc = load_inputs(p, x, t, n)) return rc;
  if (int rc = forward(p, member, 1, n, true)) return rc;
  if (int rc = backward(p, member, 1, n, loss)) return rc;
  if (grads) {
    SG_TRY(hipMemcpyAsync(grads, p->g + (size_t)member * p->per_member, sizeof(float) * p->per_member,
                          hipMemcpyDeviceToHost, p->stream));
    SG_TRY(hipStreamSynchronize(p->stream));
  }
  return MITHRA_OK;
}

// One Adam step of every member on the same mini-batch; loss[e] (optional) before the step.
int mithra_mlp_train_step(mithra_mlp* p, const float* x, const float* t, long n, float lr, float* loss) {
  if (!p || !x || !t || n < 1 || !(lr > 0.0f)) return MITHRA_E_ARG;
  if (int rc = load_inputs(p, x, t, n)) return rc;
  ++p->step;
  const float c1 = 1.0f - std::pow(kB1, (float)p->step), c2 = 1.0f - std::pow(kB2, (float)p->step);
  if (int rc = forward(p, 0, p->members, n, true)) return rc;
  if (int rc = backward(p, 0, p->members, n, loss)) return rc;
  SG_TRY(adam(p, lr, c1, c2, EpochSched{}));
  SG_TRY(hipStreamSynchronize(p->stream));
  return MITHRA_OK;
}

// The training set, resident on the device: n rows of inputs x (n x d_0, rounded to BF16) and
// targets t (n x d_out), replacing any set before.
int mithra_mlp_set_data(mithra_mlp* p, const float* x, const float* t, long n) {
  if (!p || !x || !t || n < 1) return MITHRA_E_ARG;
  SG_TRY(hipStreamSynchronize(p->stream));
  (void)hipFree(p->data_x);
  (void)hipFree(p->data_t);
  p->data_x = nullptr;
  p->data_t = nullptr;
  p->n_data = 0;
  const long nx = n * p->dims[0], nt = n * p->dims[p->layers];
  float* stage = nullptr;
  if (hipMalloc(&p->data_x, sizeof(__bf16) * nx) != hipSuccess ||
      hipMalloc(&p->data_t, sizeof(float) * nt) != hipSuccess || hipMalloc(&stage, sizeof(float) * nx) != hipSuccess) {
    (void)hipFree(stage);
    (void)hipFree(p->data_x);
    (void)hipFree(p->data_t);
    p->data_x = nullptr;
    p->data_t = nullptr;
    return MITHRA_E_NOMEM;
  }
  hipError_t e = hipMemcpyAsync(stage, x, sizeof(float) * nx, hipMemcpyHostToDevice, p->stream);
  if (e == hipSuccess) {
    hipLaunchKernelGGL(k_to_bf16, dim3(blocks(nx)), dim3(256), 0, p->stream, stage, p->data_x, nx);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipMemcpyAsync(p->data_t, t, sizeof(float) * nt, hipMemcpyHostToDevice, p->stream);
  if (e == hipSuccess) e = hipStreamSynchronize(p->stream);
  (void)hipFree(stage);
  SG_TRY(e);
  p->n_data = n;
  return MITHRA_OK;
}

// `epochs` epochs of Adam on the resident training set, every member on the same mini-batches of
// `batch` rows (n / batch per epoch, each epoch a fresh permutation drawn from `seed`), learning
// rate max(lr_max (1 + cos(pi epoch / epochs)) / 2, lr_min).  One epoch is one captured HIP graph,
// replayed `epochs` times without the host.  loss (optional, epochs entries): each epoch's mean
// training loss over the members and mini-batches, before each step.
int mithra_mlp_train_epochs(mithra_mlp* p, int epochs, int batch, float lr_max, float lr_min,
                            unsigned long long seed, float* loss) {
  if (!p || epochs < 1 || batch < 1 || !(lr_max > 0.0f) || !(lr_min >= 0.0f)) return MITHRA_E_ARG;
  if (!p->data_x || batch > p->n_data) return MITHRA_E_STATE;
  const int steps = (int)(p->n_data / batch);
  const long nperm = (long)epochs * p->n_data;
  if (int rc = ensure_acts(p, batch)) return rc;
  // the permutations of every epoch (Fisher-Yates on one generator)
  std::vector<int> perm((size_t)nperm);
  std::mt19937_64 gen(seed);
  for (int ep = 0; ep < epochs; ++ep) {
    int* q = perm.data() + (size_t)ep * p->n_data;
    for (long i = 0; i < p->n_data; ++i) q[i] = (int)i;
    for (long i = p->n_data - 1; i > 0; --i) {
      std::uniform_int_distribution<long> u(0, i);
      std::swap(q[i], q[u(gen)]);
    }
  }
  int* dperm = nullptr;
  int* depoch = nullptr;
  float* dloss = nullptr;
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  int rc = MITHRA_OK;
  if (hipMalloc(&dperm, sizeof(int) * nperm) != hipSuccess || hipMalloc(&depoch, sizeof(int)) != hipSuccess ||
      hipMalloc(&dloss, sizeof(float) * (size_t)epochs * p->members) != hipSuccess)
    rc = MITHRA_E_NOMEM;
  const int zero = 0;
  hipStream_t s = p->stream;
  if (!rc) rc = status(hipMemcpyAsync(dperm, perm.data(), sizeof(int) * nperm, hipMemcpyHostToDevice, s));
  if (!rc) rc = status(hipMemcpyAsync(depoch, &zero, sizeof(int), hipMemcpyHostToDevice, s));
  if (!rc) {
    hipLaunchKernelGGL(k_fill, dim3(blocks((long)epochs * p->members)), dim3(256), 0, s, dloss,
                       (long)epochs * p->members, 0.0f);
    rc = status(hipGetLastError());
  }
  if (!rc) rc = status(hipStreamSynchronize(s));  // `zero` and `perm` are host locals
  if (!rc) {
    rc = status(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
    if (!rc) {
      const int erc = enqueue_epoch(p, dperm, depoch, dloss, steps, batch, epochs, lr_max, lr_min);
      const hipError_t ec = hipStreamEndCapture(s, &graph);
      rc = erc ? erc : status(ec);
    }
  }
  if (!rc) rc = status(hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0));
  for (int ep = 0; ep < epochs && !rc; ++ep) rc = status(hipGraphLaunch(exec, s));
  if (!rc) rc = status(hipStreamSynchronize(s));
  if (!rc) p->step += (long)epochs * steps;
  if (!rc && loss) {
    std::vector<float> l((size_t)epochs * p->members);
    rc = status(hipMemcpy(l.data(), dloss, sizeof(float) * l.size(), hipMemcpyDeviceToHost));
    for (int ep = 0; ep < epochs && !rc; ++ep) {
      double sum = 0.0;
      for (int e = 0; e < p->members; ++e) sum += l[(size_t)ep * p->members + e];
      loss[ep] = (float)sum;
    }
  }
  (void)hipStreamSynchronize(s);
  if (exec) (void)hipGraphExecDestroy(exec);
  if (graph) (void)hipGraphDestroy(graph);
  (void)hipFree(dperm);
  (void)hipFree(depoch);
  (void)hipFree(dloss);
  return rc;
}

// One product of the surrogate's GEMM on host arrays (BF16 given as raw 16-bit patterns), for
// tests and timing: C = op(A) op(B) with the strides of k_gemm; tile 0 (by size), 1 (64 x 64)
// or 2 (128 x 128).
int mithra_mlp_gemm(const unsigned short* A, long sam, long sak, long a_len, const unsigned short* B, long sbk,
                    long sbn, long b_len, float* C, int M, int N, int K, int tile, int reps, float* ms) {
  if (!A || !B || !C || M < 1 || N < 1 || K < 1 || reps < 1 || tile < 0 || tile > 2) return MITHRA_E_ARG;
  // every element op(A) and op(B) reach must lie inside the arrays given
  if ((M - 1) * sam + (K - 1) * sak >= a_len || (K - 1) * sbk + (N - 1) * sbn >= b_len || sam < 0 || sak < 0 ||
      sbk < 0 || sbn < 0)
    return MITHRA_E_ARG;
  __bf16 *dA = nullptr, *dB = nullptr;
  float* dC = nullptr;
  int rc = MITHRA_OK;
  if (hipMalloc(&dA, 2 * a_len) != hipSuccess || hipMalloc(&dB, 2 * b_len) != hipSuccess ||
      hipMalloc(&dC, sizeof(float) * (size_t)M * N) != hipSuccess)
    rc = MITHRA_E_NOMEM;
  if (!rc) rc = status(hipMemcpy(dA, A, 2 * a_len, hipMemcpyHostToDevice));
  if (!rc) rc = status(hipMemcpy(dB, B, 2 * b_len, hipMemcpyHostToDevice));
  GemmArgs g{};
  g.A = dA; g.sam = sam; g.sak = sak; g.sae = 0;
  g.B = dB; g.sbk = sbk; g.sbn = sbn; g.sbe = 0;
  g.C = dC; g.ldc = N; g.sce = 0;
  g.M = M; g.N = N; g.K = K;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  if (!rc) rc = status(hipEventCreate(&e0));
  if (!rc) rc = status(hipEventCreate(&e1));
  const int T = tile == 2 ? 128 : tile == 1 ? 64 : gemm_tile_size(M, N, 1);
  const bool ak = sak == 1 || sam != 1, bk = sbk == 1 || sbn != 1;
  auto product = [&]() {
    if (ak) return bk ? gemm<true, true, kPlain>(0, g, Epi{}, 1, T) : gemm<true, false, kPlain>(0, g, Epi{}, 1, T);
    return bk ? gemm<false, true, kPlain>(0, g, Epi{}, 1, T) : gemm<false, false, kPlain>(0, g, Epi{}, 1, T);
  };
  if (!rc) rc = status(product());  // warm-up
  if (!rc) rc = status(hipEventRecord(e0, 0));
  for (int r = 0; r < reps && !rc; ++r) rc = status(product());
  if (!rc) rc = status(hipEventRecord(e1, 0));
  if (!rc) rc = status(hipEventSynchronize(e1));
  float t = 0.0f;
  if (!rc) rc = status(hipEventElapsedTime(&t, e0, e1));
  if (!rc && ms) *ms = t / reps;
  if (!rc) rc = status(hipMemcpy(C, dC, sizeof(float) * (size_t)M * N, hipMemcpyDeviceToHost));
  if (e0) (void)hipEventDestroy(e0);
  if (e1) (void)hipEventDestroy(e1);
  (void)hipFree(dA);
  (void)hipFree(dB);
  (void)hipFree(dC);
  return rc;
}

}  // extern "C"
