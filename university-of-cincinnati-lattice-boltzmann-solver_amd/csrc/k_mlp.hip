// Learned initial guess of the D3Q27 entropic alpha: feature logging,
// hand-written training kernels (FP32 forward / backward / Adam) and the
// inference kernel on BF16 MFMA with FP32 accumulation.
//
// The network (12 -> 64 -> 64 -> 64 -> 1, GELU, 9,217 parameters) maps 12
// scale-free invariants of a node's non-equilibrium part to
// y = (alpha - 2) / m, m = max_i |D_i / f_i|; the Newton root-find of
// H(f + alpha D) = H(f) then starts from alpha0 = 2 + m (y_mean + y_std * net)
// and falls back to the plain start alpha = 2 when that start does not
// converge.  The reference has no learned component (its closest precedent,
// the fitted multiplier guesses of amr_processes.f95:1871-2039, is disabled at
// calculate_lagrangian_mults.f95:729-741).
//
// Parameter layout (FP32 master copy): W1 (12 x 64, row-major in x out), b1,
// W2 (64 x 64), b2, W3 (64 x 64), b3, W4 (64), b4.
#include "d3q27.h"
#include "kernels.h"
#include "philox.h"

#include <hip/hip_bf16.h>

#include <algorithm>

namespace uclbs {

namespace {

constexpr int kIn = 12, kH = 64;
constexpr int oW1 = 0, oB1 = oW1 + kIn * kH, oW2 = oB1 + kH, oB2 = oW2 + kH * kH,
              oW3 = oB2 + kH, oB3 = oW3 + kH * kH, oW4 = oB3 + kH, oB4 = oW4 + kH;
static_assert(oB4 + 1 == kMlpParams, "parameter count");

// The 12 features of a node from its pre-collision shifted populations, in
// FP32 (they feed a BF16 network; the moments and equilibrium behind D are the
// streaming kernel's FP64-summed ones).  Returns m = max|x| (0 for a node at
// equilibrium or with f <= 0).
//
// The ratio features are formed over the scaled deviations xh = x / m, which
// lie in [-1, 1]: with R_k = sum_i D_i xh_i^k,
//   (S_n / S_2) / m^(n-2) = R_(n-1) / R_1,   S_2 = m R_1,
// so no intermediate leaves the range of its result.  (Forming
// S_n * (1 / S_2) * (1 / m)^(n-2) instead overflows FP32 near equilibrium:
// at m = 1e-7, S_2 = 1e-14 the factor (1 / S_2) m^-4 is 1e42.)
__device__ __forceinline__ float features27(const float (&f)[27], float (&phi)[kIn]) {
  float D[27], x[27];
  double rho, u[3];
  prep27_shifted(f, D, rho, u);
  float m = 0.0f, xmin = 0.0f;
  bool nonpos = false;
#pragma unroll
  for (int i = 0; i < 27; ++i) {
    const float fi = (float)W27[i] + f[i];
    nonpos |= !(fi > 0.0f);
    x[i] = D[i] * __builtin_amdgcn_rcpf(fi);
    m = fmaxf(m, fabsf(x[i]));
    xmin = fminf(xmin, x[i]);
  }
  const bool ok = !nonpos && m > 1e-30f && m < 1e30f;
  const float mi = ok ? __builtin_amdgcn_rcpf(m) : 0.0f;
  float R[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < 27; ++i) {
    const float xh = x[i] * mi;
    float t = D[i];
#pragma unroll
    for (int k = 1; k <= 5; ++k) {
      t *= xh;
      R[k] += t;
    }
  }
  if (!ok || !(R[1] > 0.0f)) {
#pragma unroll
    for (int j = 0; j < kIn; ++j) phi[j] = 0.0f;
    return 0.0f;
  }
  constexpr float kLog10_2 = 0.30102999566398120f;
  const float r1 = __builtin_amdgcn_rcpf(R[1]);
  phi[0] = __builtin_amdgcn_logf(m) * (kLog10_2 * 0.25f) + 1.0f;  // log10(m) / 4 + 1
#pragma unroll
  for (int n = 3; n <= 6; ++n) phi[n - 2] = R[n - 1] * r1;  // (S_n / S_2) / m^(n-2)
  phi[5] = xmin * mi;
  phi[6] = R[1] * mi * __builtin_amdgcn_rcpf((float)rho);  // S_2 / (rho m^2)
  const float S2 = m * R[1];
  phi[7] = (float)(5.0 * u[0]);
  phi[8] = (float)(5.0 * u[1]);
  phi[9] = (float)(5.0 * u[2]);
  phi[10] = (float)(25.0 * (u[0] * u[0] + u[1] * u[1] + u[2] * u[2]));
  phi[11] = __builtin_amdgcn_logf(S2) * (kLog10_2 * 0.125f) + 1.0f;  // log10(S2) / 8 + 1
  return m;
}

// pull of an interior node of a periodic box or of a level whose flag is
// kFlagInterior (no boundary link): f~_i(x) = f~_i(x - c_i) with wrap
__device__ __forceinline__ void pull27(const float* __restrict__ fin, unsigned node, const Box& b,
                                       float (&f)[27]) {
  const unsigned nx = (unsigned)b.nx, ny = (unsigned)b.ny, nz = (unsigned)b.nz, nn = (unsigned)b.n;
  const unsigned x = node % nx, yz = node / nx, y = yz % ny, z = yz / ny;
  unsigned ox[3], oy[3], oz[3];
  ox[0] = x + 1 == nx ? 0u : x + 1;
  ox[1] = x;
  ox[2] = x == 0 ? nx - 1 : x - 1;
  oy[0] = (y + 1 == ny ? 0u : y + 1) * nx;
  oy[1] = y * nx;
  oy[2] = (y == 0 ? ny - 1 : y - 1) * nx;
  oz[0] = (z + 1 == nz ? 0u : z + 1) * nx * ny;
  oz[1] = z * nx * ny;
  oz[2] = (z == 0 ? nz - 1 : z - 1) * nx * ny;
#pragma unroll
  for (int i = 0; i < 27; ++i)
    f[i] = (fin + (size_t)i * nn)[ox[CX27[i] + 1] + oy[CY27[i] + 1] + oz[CZ27[i] + 1]];
}

// Sample logging: every stride-th interior node with m above 1e-8 and finite
// features is a pair (features, node, m); the target is filled after the plain
// step has produced alpha (k_collect_targets).  The pairs of one collection
// land in node order: a counting pass records each wavefront's ballot of taken
// nodes and each block's count, one block turns the counts into slot offsets
// after the pairs already held, and a writing pass places each taken node at
// its block's offset plus its rank in the block.
__device__ __forceinline__ bool collect_take(const float* __restrict__ fin, const Box& b,
                                             const uint8_t* __restrict__ flags, int stride,
                                             int phase, unsigned gid, float (&phi)[kIn],
                                             float& m) {
  float f[27];
  bool take = gid < (unsigned)b.n && (int)(gid % (unsigned)stride) == phase;
  if (take && flags) take = flags[gid] == kFlagInterior;
  m = 0.0f;
  if (take) {
    pull27(fin, gid, b, f);
    m = features27(f, phi);
    take = m > 1e-8f;
    // a pair with a non-finite feature never enters the training set
#pragma unroll
    for (int j = 0; j < kIn; ++j) take = take && __builtin_isfinite(phi[j]);
  }
  return take;
}

__global__ __launch_bounds__(256) void k27_collect_count(const float* __restrict__ fin, Box b,
                                                         const uint8_t* __restrict__ flags,
                                                         int stride, int phase,
                                                         unsigned long long* __restrict__ ballots,
                                                         unsigned long long* __restrict__ blk) {
  const unsigned gid = blockIdx.x * blockDim.x + threadIdx.x;
  float phi[kIn], m;
  const bool take = collect_take(fin, b, flags, stride, phase, gid, phi, m);
  const unsigned long long bm = __ballot(take);
  __shared__ unsigned wc[4];
  const int w = threadIdx.x / 64;
  if (__lane_id() == 0) {
    ballots[gid / 64] = bm;
    wc[w] = (unsigned)__popcll(bm);
  }
  __syncthreads();
  if (threadIdx.x == 0) blk[blockIdx.x] = (unsigned long long)(wc[0] + wc[1] + wc[2] + wc[3]);
}

// blk[i] <- count + sum of blk[0..i) (one block of 1024 threads); count <- the new total
__global__ __launch_bounds__(1024) void k_scan_counts(unsigned long long* __restrict__ blk,
                                                      unsigned nb,
                                                      unsigned long long* __restrict__ count) {
  __shared__ unsigned long long part[1024];
  const unsigned t = threadIdx.x;
  const unsigned chunk = (nb + 1023u) / 1024u;
  const unsigned lo = min(nb, t * chunk), hi = min(nb, lo + chunk);
  const unsigned long long base = *count;
  unsigned long long own = 0;
  for (unsigned i = lo; i < hi; ++i) own += blk[i];
  part[t] = own;
  __syncthreads();
  for (unsigned off = 1; off < 1024u; off <<= 1) {
    const unsigned long long v = t >= off ? part[t - off] : 0ull;
    __syncthreads();
    part[t] += v;
    __syncthreads();
  }
  unsigned long long run = base + part[t] - own;
  for (unsigned i = lo; i < hi; ++i) {
    const unsigned long long c = blk[i];
    blk[i] = run;
    run += c;
  }
  __syncthreads();
  if (t == 0) *count = base + part[1023];
}

__global__ __launch_bounds__(256) void k27_collect(const float* __restrict__ fin, Box b,
                                                   const uint8_t* __restrict__ flags, int stride,
                                                   int phase,
                                                   const unsigned long long* __restrict__ ballots,
                                                   const unsigned long long* __restrict__ blk,
                                                   float* __restrict__ X,
                                                   unsigned* __restrict__ node_of,
                                                   float* __restrict__ m_of,
                                                   unsigned long long cap) {
  const unsigned gid = blockIdx.x * blockDim.x + threadIdx.x;
  // the counting pass's decision, so the slots match its counts exactly
  const unsigned long long bm = ballots[gid / 64];
  const bool take = (bm >> __lane_id()) & 1ull;
  __shared__ unsigned wc[4];
  const int w = threadIdx.x / 64;
  if (__lane_id() == 0) wc[w] = (unsigned)__popcll(bm);
  __syncthreads();
  if (!take) return;
  unsigned before = 0;
  for (int q = 0; q < w; ++q) before += wc[q];
  const unsigned long long slot =
      blk[blockIdx.x] + before + __popcll(bm & ((1ull << __lane_id()) - 1ull));
  if (slot >= cap) return;
  float phi[kIn], m;
  (void)collect_take(fin, b, flags, stride, phase, gid, phi, m);
#pragma unroll
  for (int j = 0; j < kIn; ++j) X[slot * kIn + j] = phi[j];
  node_of[slot] = gid;
  m_of[slot] = (float)m;
}

__global__ void k_collect_targets(const double* __restrict__ alpha, const unsigned* __restrict__ node_of,
                                  const float* __restrict__ m_of, float* __restrict__ y,
                                  unsigned long long first, unsigned long long last) {
  const unsigned long long k = first + blockIdx.x * (unsigned long long)blockDim.x + threadIdx.x;
  if (k >= last) return;
  y[k] = (float)((alpha[node_of[k]] - 2.0) / (double)m_of[k]);
}

// ---- training (FP32) -------------------------------------------------------
// One launch takes a batch through the network and back, a second adds the
// weight gradients up (and, in training, applies Adam); activations stay in
// registers and LDS.  Launch per layer and direction, the same step took 18
// launches whose threads each ran a serial loop over a row or a chunk of rows.
//
// A block of four wavefronts holds 32 rows; wavefront w computes 16 of them
// (w & 1) and 32 of a layer's 64 outputs (w >> 1), so that a batch of 8,192
// gives each of the 256 CUs one block.  All products run on
// v_mfma_f32_16x16x4_f32 (FP32 in, FP32 accumulation): A lane l = row l % 16,
// k = l / 16; B lane l = column l % 16, the same k; D lane l = column l % 16,
// rows 4 (l / 16) + 0..3.  Layers are computed transposed, O^T = W^T X^T, and
// MFMA step s of a 16-wide chunk takes k = 4 (l / 16) + s for both operands, so
// that a D tile's rows are the next product's k.  Every tile lives in LDS as
// [feature][row] (pitch kTp): the forward and backward products read it by
// column, the weight gradients, which contract over the rows, by float4.  Each
// wavefront reads its half of a weight matrix once, into registers.
// Bound by the FP32 matrix rate and the chain of seven layer products with a
// barrier after each: 206 MFMA a wavefront (2.8 us at 32 cycles each) of the
// 17 us that the launch takes at 8,192 rows; the rest is the draw of the rows,
// two dependent reads and the barriers.  Before: 490 us a step in 18 launches.
constexpr int kTrainRows = 32;
constexpr int kMaxRowBlocks = 256;
constexpr int kTp = kTrainRows + 4;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;

__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// h = gelu(z), gp = gelu'(z): (1 + tanh u) / 2 = s = 1 / (1 + exp(-2 u)), so that
// h = z s and gp = s + 2 z u' s (1 - s), over one exponential and one quotient
__device__ __forceinline__ float gelu_both(float x, float& gp) {
  const float c = 0.7978845608028654f;
  const float s = 1.0f / (1.0f + expf(-2.0f * c * (x + 0.044715f * x * x * x)));
  gp = fmaf(2.0f * c * x * s * (1.0f - s), 1.0f + 3.0f * 0.044715f * x * x, s);
  return x * s;
}

// A operand of a forward product: W^T[o = 16 ot + l % 16][k], 16 k-steps
__device__ __forceinline__ void load_fwd(const float* __restrict__ W, int ot, int c16, int g,
                                         float (&a)[16]) {
#pragma unroll
  for (int t = 0; t < 16; ++t) a[t] = W[(16 * (t / 4) + 4 * g + t % 4) * kH + 16 * ot + c16];
}
// A operand of a backward product: W[k = 16 kt + l % 16][o], 16 o-steps
__device__ __forceinline__ void load_bwd(const float* __restrict__ W, int kt, int c16, int g,
                                         f32x4 (&a)[4]) {
#pragma unroll
  for (int q = 0; q < 4; ++q)
    a[q] = *reinterpret_cast<const f32x4*>(W + (16 * kt + c16) * kH + 16 * q + 4 * g);
}

enum { kRowsForward = 0, kRowsGrad = 1, kRowsGather = 2 };

// kRowsForward: yhat of rows 0..B-1 of X.  kRowsGrad: the block's sums of the
// weight gradients over its rows into part[block][kMlpParams] and of the loss
// into lpart[block].  kRowsGather: the same over rows drawn from n samples
// (Philox4x32-10 indices, with replacement).
template <int kMode>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 2))) void k_mlp_rows(const float* __restrict__ P,
                                                  const float* __restrict__ X,
                                                  const float* __restrict__ y, int B,
                                                  unsigned long long n, uint64_t seed,
                                                  uint64_t step, float* __restrict__ part,
                                                  double* __restrict__ lpart,
                                                  float* __restrict__ yhat) {
  constexpr bool kBack = kMode != kRowsForward;
  __shared__ __attribute__((aligned(16))) float Xs[16][kTp];
  __shared__ __attribute__((aligned(16))) float H[3][kH][kTp];
  __shared__ __attribute__((aligned(16))) float D[kBack ? 3 : 1][kBack ? kH : 1][kTp];
  __shared__ float ysum[2][kTrainRows];
  __shared__ __attribute__((aligned(16))) float dz[kTrainRows];
  __shared__ unsigned sidx[kTrainRows];
  const int tid = (int)threadIdx.x, l = tid % 64, w = tid / 64;
  const int c16 = l % 16, g = l / 16;
  const int nt = w & 1, hf = w >> 1;  // rows 16 nt .., output tiles 2 hf, 2 hf + 1
  const int col = 16 * nt + c16;      // this lane's row of the tile
  const float *W1 = P + oW1, *W2 = P + oW2, *W3 = P + oW3;

  float a1[2][3], a2[2][16], a3[2][16];
  f32x4 b1[2], b2[2], b3[2], w4[2];
#pragma unroll
  for (int o = 0; o < 2; ++o) {
    const int ot = 2 * hf + o;
#pragma unroll
    for (int s = 0; s < 3; ++s) a1[o][s] = W1[(4 * s + g) * kH + 16 * ot + c16];
    load_fwd(W2, ot, c16, g, a2[o]);
    load_fwd(W3, ot, c16, g, a3[o]);
    const int r = 16 * ot + 4 * g;
    b1[o] = *reinterpret_cast<const f32x4*>(P + oB1 + r);
    b2[o] = *reinterpret_cast<const f32x4*>(P + oB2 + r);
    b3[o] = *reinterpret_cast<const f32x4*>(P + oB3 + r);
    w4[o] = *reinterpret_cast<const f32x4*>(P + oW4 + r);
  }
  const float b4 = P[oB4];

  // sums over this block's tiles: gW3, gW2 (k-tile w, the four o-tiles), gW1
  // (o-tile w), one entry of gW4 / gb3 / gb2 / gb1 a thread, gb4 and the loss
  f32x4 s3[4], s2[4], s1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int o = 0; o < 4; ++o) s3[o] = s2[o] = f32x4{0.f, 0.f, 0.f, 0.f};
  float sv = 0.0f, sb4 = 0.0f;
  double sl = 0.0;

  const int ntiles = (B + kTrainRows - 1) / kTrainRows;
  for (int tile = (int)blockIdx.x; tile < ntiles; tile += (int)gridDim.x) {
    const int r0 = tile * kTrainRows;
    float yt = 0.0f;
    if (tid < kTrainRows) {
      const int r = r0 + tid;
      unsigned k = (unsigned)(r < B ? r : 0);
      if constexpr (kMode == kRowsGather) {
        uint32_t c[4] = {(uint32_t)r, (uint32_t)step, (uint32_t)(step >> 32), 0x6d6c70u};
        philox4x32_10(c, (uint32_t)seed, (uint32_t)(seed >> 32));
        k = (unsigned)((((unsigned long long)c[0] << 32) | c[1]) % n);
      }
      sidx[tid] = k;
      if constexpr (kBack) yt = y[k];
    }
    __syncthreads();
    if (tid < 4 * kTrainRows) {
      const int r = tid / 4, q = tid % 4;
      f32x4 v = {0.f, 0.f, 0.f, 0.f};
      if (q < 3 && r0 + r < B)
        v = *reinterpret_cast<const f32x4*>(X + (size_t)sidx[r] * kIn + 4 * q);
#pragma unroll
      for (int j = 0; j < 4; ++j) Xs[4 * q + j][r] = v[j];
    }
    __syncthreads();

    f32x4 p1[2], p2[2], p3[2];  // gelu' of the three layers at (16 ot + 4 g + j, col)
    auto act = [&](float (*Hl)[kTp], const f32x4 (&z)[2], f32x4 (&p)[2]) __attribute__((always_inline)) {
#pragma unroll
      for (int o = 0; o < 2; ++o)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          float gp;
          Hl[16 * (2 * hf + o) + 4 * g + j][col] = gelu_both(z[o][j], gp);
          p[o][j] = gp;
        }
    };
    f32x4 z[2] = {b1[0], b1[1]};
#pragma unroll
    for (int s = 0; s < 3; ++s) {
      const float b = Xs[4 * s + g][col];
#pragma unroll
      for (int o = 0; o < 2; ++o) z[o] = mfma4(a1[o][s], b, z[o]);
    }
    act(H[0], z, p1);
    __syncthreads();
    auto layer = [&](const float (*Hl)[kTp], const float (&a)[2][16], const f32x4 (&b)[2]) __attribute__((always_inline)) {
      z[0] = b[0];
      z[1] = b[1];
#pragma unroll
      for (int t = 0; t < 16; ++t) {
        const float h = Hl[16 * (t / 4) + 4 * g + t % 4][col];
#pragma unroll
        for (int o = 0; o < 2; ++o) z[o] = mfma4(a[o][t], h, z[o]);
      }
    };
    layer(H[0], a2, b2);
    act(H[1], z, p2);
    __syncthreads();
    layer(H[1], a3, b3);
    float yp = 0.0f;
#pragma unroll
    for (int o = 0; o < 2; ++o)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float gp;
        const float h = gelu_both(z[o][j], gp);
        p3[o][j] = gp;
        if constexpr (kBack) H[2][16 * (2 * hf + o) + 4 * g + j][col] = h;
        yp = fmaf(h, w4[o][j], yp);
      }
    yp += __shfl_xor(yp, 16);
    yp += __shfl_xor(yp, 32);
    if (g == 0) ysum[hf][col] = yp;
    __syncthreads();
    if (tid < kTrainRows) {
      const float yh = (ysum[0][tid] + ysum[1][tid]) + b4;
      const bool in = r0 + tid < B;
      if constexpr (kBack) {
        const float d = in ? yh - yt : 0.0f;
        const float v = d / (float)B;
        dz[tid] = v;
        sb4 += v;
        sl += 0.5 * (double)d * d;
      } else if (in) {
        yhat[r0 + tid] = yh;
      }
    }
    __syncthreads();
    if constexpr (kBack) {
      f32x4 w3[2][4], w2[2][4];
#pragma unroll
      for (int o = 0; o < 2; ++o) {
        load_bwd(W3, 2 * hf + o, c16, g, w3[o]);
        load_bwd(W2, 2 * hf + o, c16, g, w2[o]);
      }
      {
        const float d4 = dz[col];
#pragma unroll
        for (int o = 0; o < 2; ++o)
#pragma unroll
          for (int j = 0; j < 4; ++j)
            D[2][16 * (2 * hf + o) + 4 * g + j][col] = (d4 * w4[o][j]) * p3[o][j];
      }
      __syncthreads();
      auto back = [&](const float (*Dl)[kTp], const f32x4 (&a)[2][4], const f32x4 (&p)[2],
                      float (*Dp)[kTp]) __attribute__((always_inline)) {
        z[0] = z[1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
          for (int s = 0; s < 4; ++s) {
            const float d = Dl[16 * q + 4 * g + s][col];
#pragma unroll
            for (int o = 0; o < 2; ++o) z[o] = mfma4(a[o][q][s], d, z[o]);
          }
#pragma unroll
        for (int o = 0; o < 2; ++o)
#pragma unroll
          for (int j = 0; j < 4; ++j) Dp[16 * (2 * hf + o) + 4 * g + j][col] = z[o][j] * p[o][j];
      };
      back(D[2], w3, p2, D[1]);
      __syncthreads();
      back(D[1], w2, p1, D[0]);
      __syncthreads();
      // weight gradients, contracted over the 32 rows
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int rr = 16 * q + 4 * g;
        const f32x4 h2 = *reinterpret_cast<const f32x4*>(&H[1][16 * w + c16][rr]);
        const f32x4 h1 = *reinterpret_cast<const f32x4*>(&H[0][16 * w + c16][rr]);
        const f32x4 x = *reinterpret_cast<const f32x4*>(&Xs[c16][rr]);
        const f32x4 d1 = *reinterpret_cast<const f32x4*>(&D[0][16 * w + c16][rr]);
#pragma unroll
        for (int s = 0; s < 4; ++s) s1 = mfma4(x[s], d1[s], s1);
#pragma unroll
        for (int o = 0; o < 4; ++o) {
          const f32x4 d3 = *reinterpret_cast<const f32x4*>(&D[2][16 * o + c16][rr]);
          const f32x4 d2 = *reinterpret_cast<const f32x4*>(&D[1][16 * o + c16][rr]);
#pragma unroll
          for (int s = 0; s < 4; ++s) {
            s3[o] = mfma4(h2[s], d3[s], s3[o]);
            s2[o] = mfma4(h1[s], d2[s], s2[o]);
          }
        }
      }
      // wavefront 0: gW4, 1: gb3, 2: gb2, 3: gb1, one feature a lane
      const float* src = w == 0 ? &H[2][l][0] : &D[3 - w][l][0];
#pragma unroll
      for (int r = 0; r < kTrainRows; r += 4) {
        const f32x4 v = *reinterpret_cast<const f32x4*>(src + r);
        const f32x4 m = *reinterpret_cast<const f32x4*>(&dz[r]);
#pragma unroll
        for (int j = 0; j < 4; ++j) sv = w == 0 ? fmaf(v[j], m[j], sv) : sv + v[j];
      }
      __syncthreads();
    }
  }
  if constexpr (kBack) {
    float* o = part + (size_t)blockIdx.x * kMlpParams;
#pragma unroll
    for (int ot = 0; ot < 4; ++ot)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        o[oW3 + (16 * w + 4 * g + j) * kH + 16 * ot + c16] = s3[ot][j];
        o[oW2 + (16 * w + 4 * g + j) * kH + 16 * ot + c16] = s2[ot][j];
      }
    if (g < 3) {
#pragma unroll
      for (int j = 0; j < 4; ++j) o[oW1 + (4 * g + j) * kH + 16 * w + c16] = s1[j];
    }
    o[(w == 0 ? oW4 : w == 1 ? oB3 : w == 2 ? oB2 : oB1) + l] = sv;
    if (w == 0) {
      // lanes 0..31 hold the rows' sums, the others zero
#pragma unroll
      for (int d = 16; d > 0; d >>= 1) {
        sb4 += __shfl_xor(sb4, d);
        sl += __shfl_xor(sl, d);
      }
      if (l == 0) {
        o[oB4] = sb4;
        lpart[blockIdx.x] = sl;
      }
    }
  }
}

// The gradient as the sum of nb blocks' parts, 32 slices of the blocks a
// weight (a fixed order, so the result is the same from run to run), and the
// mean loss.  kAdam: applied to the parameters at once; else stored in g.
// 32 weights a block: a slice's loads are 128 B rows of part.  Bound by the
// latency of a thread's loads, so that all of them (8 at 256 blocks) are in
// flight; with 8 slices of up to 32 loads the launch took 11 us.
constexpr int kSlices = 32;
template <bool kAdam>
__global__ __launch_bounds__(32 * kSlices) void k_mlp_reduce(
    const float* __restrict__ part, const double* __restrict__ lpart, int nb, int B,
    float* __restrict__ gout, double* __restrict__ loss, float* __restrict__ p,
    float* __restrict__ m, float* __restrict__ v, float lr, float c1, float c2) {
  __shared__ float red[kSlices][33];
  __shared__ double lred[256];
  const int t = (int)threadIdx.x, c = t % 32, sl = t / 32;
  const int k = (int)blockIdx.x * 32 + c;
  float s = 0.0f;
  if (k < kMlpParams) {
    // blocks sl, sl + 32, ..: at most eight
    static_assert(kMaxRowBlocks == 8 * kSlices && kMaxRowBlocks == 256, "slices, loss sums");
    float q[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int b = sl + kSlices * j;
      q[j] = b < nb ? part[(size_t)b * kMlpParams + k] : 0.0f;
    }
    s = ((q[0] + q[1]) + (q[2] + q[3])) + ((q[4] + q[5]) + (q[6] + q[7]));
  }
  red[sl][c] = s;
  if (blockIdx.x == 0) {
    if (t < 256) lred[t] = t < nb ? lpart[t] : 0.0;
    __syncthreads();
    for (int d = 128; d > 0; d >>= 1) {
      if (t < d) lred[t] += lred[t + d];
      __syncthreads();
    }
    if (t == 0) *loss = lred[0] / B;
  }
  __syncthreads();
  // a half-wavefront a weight adds its 32 slices
  float gk = red[t % 32][t / 32];
#pragma unroll
  for (int d = 16; d > 0; d >>= 1) gk += __shfl_xor(gk, d);
  const int kw = (int)blockIdx.x * 32 + t / 32;
  if (t % 32 != 0 || kw >= kMlpParams) return;
  if constexpr (kAdam) {
    const float mk = 0.9f * m[kw] + 0.1f * gk;
    const float vk = 0.999f * v[kw] + 0.001f * gk * gk;
    m[kw] = mk;
    v[kw] = vk;
    p[kw] -= lr * (mk / c1) / (sqrtf(vk / c2) + 1e-8f);
  } else {
    gout[kw] = gk;
  }
}

// mean and standard deviation of the targets in FP64: a block's sums, then
// one block over the blocks (with one block over all of 786k targets the first
// training on them took 2 ms longer than the next)
constexpr int kMomentBlocks = 256;
__device__ __forceinline__ void sum2_256(double& a, double& b) {
  __shared__ double s1[256], s2[256];
  const int t = (int)threadIdx.x;
  s1[t] = a;
  s2[t] = b;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (t < s) {
      s1[t] += s1[t + s];
      s2[t] += s2[t + s];
    }
    __syncthreads();
  }
  a = s1[0];
  b = s2[0];
}
__global__ __launch_bounds__(256) void k_moments_part(const float* __restrict__ y,
                                                      unsigned long long n,
                                                      double* __restrict__ sums) {
  double a = 0.0, b = 0.0;
  for (unsigned long long k = blockIdx.x * 256ull + threadIdx.x; k < n; k += gridDim.x * 256ull) {
    a += y[k];
    b += (double)y[k] * y[k];
  }
  sum2_256(a, b);
  if (threadIdx.x == 0) {
    sums[2 * blockIdx.x] = a;
    sums[2 * blockIdx.x + 1] = b;
  }
}
__global__ __launch_bounds__(256) void k_moments(const double* __restrict__ sums,
                                                 unsigned long long n, double* __restrict__ out) {
  double a = sums[2 * threadIdx.x], b = sums[2 * threadIdx.x + 1];
  sum2_256(a, b);
  if (threadIdx.x == 0) {
    const double mean = a / (double)n;
    out[0] = mean;
    out[1] = sqrt(fmax(b / (double)n - mean * mean, 1e-30));
  }
}

// y <- (y - mean) / std on the device copy the trainer uses
__global__ void k_normalise(float* __restrict__ y, unsigned long long n, const double* __restrict__ ms) {
  const unsigned long long k = blockIdx.x * (unsigned long long)blockDim.x + threadIdx.x;
  if (k < n) y[k] = (float)(((double)y[k] - ms[0]) / ms[1]);
}

// ---- inference on BF16 MFMA -----------------------------------------------
// One wavefront evaluates 64 nodes.  v_mfma_f32_16x16x16_bf16 layouts (wave64):
// A (16x16): lane l holds row l%16, k = 4(l/16)..4(l/16)+3; B (16x16): lane l
// holds column l%16, the same k; D (16x16 FP32): lane l holds column l%16,
// rows 4(l/16)..4(l/16)+3.
typedef __attribute__((__vector_size__(4 * sizeof(short)))) short bf16x4;
typedef __attribute__((__vector_size__(8 * sizeof(short)))) short bf16x8;
typedef __bf16 bf16v8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ bf16x8 cat8(bf16x4 a, bf16x4 b) {
  return bf16x8{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
}
// D += A B on v_mfma_f32_16x16x32_bf16 (two K-slots of eight per lane group)
__device__ __forceinline__ f32x4 mfma32(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16v8, a),
                                                 __builtin_bit_cast(bf16v8, b), c, 0, 0, 0);
}

__device__ __forceinline__ short bf16_bits(float x) {
  return (short)__bfloat16_as_ushort(__float2bfloat16(x));
}

// GELU for the BF16 inference path: x sigmoid(2 sqrt(2/pi)(x + 0.044715 x^3)),
// the tanh form rewritten as x / (1 + 2^(x (a + b x^2))) with
// a = -2 sqrt(2/pi) log2(e), b = 0.044715 a, on the hardware exp2 and
// reciprocal (its ~1e-6 relative error is far below the BF16 rounding of the
// activations)
__device__ __forceinline__ float gelu_fast(float x) {
  const float e = __builtin_amdgcn_exp2f(x * fmaf(-0.10294324f, x * x, -2.3022082f));
  return x * __builtin_amdgcn_rcpf(1.0f + e);
}

// Inference on v_mfma_f32_16x16x16_bf16, one wavefront per 64 nodes.  Each
// layer is computed transposed, O^T = W^T X^T: the weights are the A operand
// (lane l: W^T[row l%16][k 4(l/16)..+3]), the activations the B operand
// (lane l: X^T[k 4(l/16)..+3][node l%16]), and the result tile D holds
// O^T[out 4(l/16)..+3][node l%16] -- exactly the B operand of the next layer
// for the same lane.  So for each group of 16 nodes the three hidden layers
// chain in registers; only the input features pass through LDS (one transpose)
// and the 64 -> 1 output layer is a dot product reduced across the four lane
// groups.  LDS weight layout (bf16 bits, row = output, pitch kWp):
// W1t 64 x 16 (K padded), W2t and W3t 64 x 64.
constexpr int kWp1 = 24, kWp = 72;
constexpr int kWsmem = 64 * kWp1 + 2 * 64 * kWp;  // shorts
struct MlpSmem {
  short w[kWsmem];
  float bias[3][64];
  float w4[64];
};

// stage the bf16 weights (global layout of k_pack_bf16: W1t 64 x 16, W2t, W3t
// 64 x 64, rows = outputs) and the FP32 biases / output weights in LDS
__device__ __forceinline__ void mlp_stage(MlpSmem& sm, const short* __restrict__ Wbf,
                                          const float* __restrict__ P) {
  for (int t = threadIdx.x; t < 64 * 16; t += blockDim.x) sm.w[(t / 16) * kWp1 + t % 16] = Wbf[t];
  for (int t = threadIdx.x; t < 2 * 64 * 64; t += blockDim.x) {
    const int layer = t / 4096, v = t % 4096;
    sm.w[64 * kWp1 + layer * 64 * kWp + (v / 64) * kWp + v % 64] = Wbf[64 * 16 + t];
  }
  for (int t = threadIdx.x; t < 64; t += blockDim.x) {
    sm.bias[0][t] = P[oB1 + t];
    sm.bias[1][t] = P[oB2 + t];
    sm.bias[2][t] = P[oB3 + t];
    sm.w4[t] = P[oW4 + t];
  }
}

__device__ __forceinline__ bf16x4 pack_gelu(const f32x4& z) {
  bf16x4 r;
#pragma unroll
  for (int j = 0; j < 4; ++j) r[j] = bf16_bits(gelu_fast(z[j]));
  return r;
}

// Network output y (normalised) for the wavefront's 64 nodes; lane l passes
// the features of node l and receives y of node l.  feat: this wavefront's
// 64 x 16 bf16 transpose buffer (pitch kWp1).
__device__ __forceinline__ float mlp_wave(const float (&phi)[kIn], const MlpSmem& sm,
                                          short* __restrict__ feat, float b4) {
  const int l = __lane_id();
  const int r16 = l % 16, g4 = 4 * (l / 16);
#pragma unroll
  for (int j = 0; j < 16; ++j) feat[l * kWp1 + j] = bf16_bits(j < kIn ? phi[j] : 0.0f);
  __builtin_amdgcn_wave_barrier();
  // A operands for this lane (same for every node group).  Layers 2 and 3 run
  // on the K = 32 instruction: K-chunk c takes the previous layer's output
  // tiles 2c and 2c + 1, whose rows this lane holds as 32c + g4 + (0..3) and
  // 32c + 16 + g4 + (0..3); the weights take the same eight K indices, so the
  // pairs line up whatever the instruction's K-slot order.
  bf16x4 A1[4];
  bf16x8 A2[4][2], A3[4][2];
  const short* w2 = sm.w + 64 * kWp1;
  const short* w3 = w2 + 64 * kWp;
#pragma unroll
  for (int ot = 0; ot < 4; ++ot) {
    A1[ot] = *reinterpret_cast<const bf16x4*>(sm.w + (ot * 16 + r16) * kWp1 + g4);
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const int row = (ot * 16 + r16) * kWp + 32 * c + g4;
      A2[ot][c] = cat8(*reinterpret_cast<const bf16x4*>(w2 + row),
                       *reinterpret_cast<const bf16x4*>(w2 + row + 16));
      A3[ot][c] = cat8(*reinterpret_cast<const bf16x4*>(w3 + row),
                       *reinterpret_cast<const bf16x4*>(w3 + row + 16));
    }
  }
  // biases and output weights of this lane's rows 4(l/16)..+3 of each output tile
  auto bias = [&](int layer, int ot) __attribute__((always_inline)) {
    return *reinterpret_cast<const f32x4*>(&sm.bias[layer][ot * 16 + g4]);
  };
  float mine = 0.0f;
#pragma unroll 1
  for (int ct = 0; ct < 4; ++ct) {
    // features 4(l/16)..+3 of node ct*16 + l%16
    const bf16x4 x = *reinterpret_cast<const bf16x4*>(feat + (ct * 16 + r16) * kWp1 + g4);
    bf16x4 h1[4], h2[4];
#pragma unroll
    for (int ot = 0; ot < 4; ++ot)
      h1[ot] = pack_gelu(__builtin_amdgcn_mfma_f32_16x16x16bf16_1k(A1[ot], x, bias(0, ot), 0, 0, 0));
    const bf16x8 b1[2] = {cat8(h1[0], h1[1]), cat8(h1[2], h1[3])};
#pragma unroll
    for (int ot = 0; ot < 4; ++ot) {
      f32x4 acc = bias(1, ot);
#pragma unroll
      for (int c = 0; c < 2; ++c) acc = mfma32(A2[ot][c], b1[c], acc);
      h2[ot] = pack_gelu(acc);
    }
    const bf16x8 b2[2] = {cat8(h2[0], h2[1]), cat8(h2[2], h2[3])};
    float y = 0.0f;
#pragma unroll
    for (int ot = 0; ot < 4; ++ot) {
      f32x4 acc = bias(2, ot);
#pragma unroll
      for (int c = 0; c < 2; ++c) acc = mfma32(A3[ot][c], b2[c], acc);
      const f32x4 w4 = *reinterpret_cast<const f32x4*>(&sm.w4[ot * 16 + g4]);
#pragma unroll
      for (int j = 0; j < 4; ++j) y = fmaf(gelu_fast(acc[j]), w4[j], y);
    }
    // sum over the four output groups held by lanes l%16 + 16q
    y += __shfl_xor(y, 16);
    y += __shfl_xor(y, 32);
    if (l / 16 == ct) mine = y;
  }
  __builtin_amdgcn_wave_barrier();
  return mine + b4;
}

// forward of a host-given batch through the MFMA path (checks of the layout)
__global__ __launch_bounds__(256) void k_mlp_infer(const float* __restrict__ X, int B,
                                                   const short* __restrict__ Wbf,
                                                   const float* __restrict__ P,
                                                   float* __restrict__ yhat) {
  __shared__ MlpSmem sm;
  __shared__ short feat[4][64 * kWp1];
  mlp_stage(sm, Wbf, P);
  __syncthreads();
  const int r = blockIdx.x * 256 + threadIdx.x;
  float phi[kIn];
#pragma unroll
  for (int j = 0; j < kIn; ++j) phi[j] = r < B ? X[r * kIn + j] : 0.0f;
  const float y = mlp_wave(phi, sm, feat[threadIdx.x / 64], P[oB4]);
  if (r < B) yhat[r] = y;
}

// Initial guesses for the step: interior nodes get alpha0 = 2 + m (mean +
// std * net(phi)); every other node 2.  Written to alpha[].  Blocks of four
// wavefronts stage the weights once and stride over 64-node tiles.
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k27_alpha_guess(const float* __restrict__ fin, Box b,
                                                       const uint8_t* __restrict__ flags,
                                                       const short* __restrict__ Wbf,
                                                       const float* __restrict__ P, float ymean,
                                                       float ystd, double* __restrict__ alpha) {
  __shared__ MlpSmem sm;
  __shared__ short feat[4][64 * kWp1];
  mlp_stage(sm, Wbf, P);
  __syncthreads();
  const float b4 = P[oB4];
  const unsigned nn = (unsigned)b.n;
  const unsigned ntiles = (nn + 63u) / 64u;
  short* fw = feat[threadIdx.x / 64];
  for (unsigned tile = blockIdx.x * 4u + threadIdx.x / 64u; tile < ntiles; tile += gridDim.x * 4u) {
    const unsigned gid = tile * 64u + __lane_id();
    bool ok = gid < nn;
    if (ok && flags) ok = flags[gid] == kFlagInterior;
    float f[27], phi[kIn];
    float m = 0.0f;
    if (ok) {
      pull27(fin, gid, b, f);
      m = features27(f, phi);
    } else {
#pragma unroll
      for (int j = 0; j < kIn; ++j) phi[j] = 0.0f;
    }
    // the whole wave evaluates the network (MFMA needs all lanes)
    const float y = mlp_wave(phi, sm, fw, b4);
    if (gid < nn)
      alpha[gid] = m > 1e-12f ? 2.0 + (double)m * ((double)ymean + (double)ystd * (double)y) : 2.0;
  }
}

// bf16 transposed copies of W1 (padded to K = 16), W2, W3 for the MFMA path
__global__ void k_pack_bf16(const float* __restrict__ P, short* __restrict__ Wbf) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t < 64 * 16) {
    const int o = t / 16, k = t % 16;
    Wbf[t] = bf16_bits(k < kIn ? P[oW1 + k * kH + o] : 0.0f);
  } else if (t < 64 * 16 + 2 * 64 * 64) {
    const int u = t - 64 * 16;
    const int layer = u / 4096, v = u % 4096;
    const int o = v / 64, k = v % 64;
    Wbf[t] = bf16_bits(P[(layer == 0 ? oW2 : oW3) + k * kH + o]);
  }
}

}  // namespace

hipError_t launch_mlp_collect(const Box& b, const float* fin, const uint8_t* flags, int stride,
                              int phase, MlpSamples& s, hipStream_t st) {
  const unsigned blocks = (unsigned)((b.n + 255) / 256);
  if ((size_t)blocks > s.blk_n) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k27_collect_count, dim3(blocks), dim3(256), 0, st, fin, b, flags, stride,
                     phase, s.ballots, s.blk);
  hipLaunchKernelGGL(k_scan_counts, dim3(1), dim3(1024), 0, st, s.blk, blocks, s.count);
  hipLaunchKernelGGL(k27_collect, dim3(blocks), dim3(256), 0, st, fin, b, flags, stride, phase,
                     s.ballots, s.blk, s.X, s.node_of, s.m_of, (unsigned long long)s.cap);
  return hipGetLastError();
}

hipError_t launch_mlp_targets(const double* alpha, MlpSamples& s, unsigned long long first,
                              unsigned long long last, hipStream_t st) {
  if (last <= first) return hipSuccess;
  const unsigned blocks = (unsigned)((last - first + 255) / 256);
  hipLaunchKernelGGL(k_collect_targets, dim3(blocks), dim3(256), 0, st, alpha, s.node_of, s.m_of,
                     s.y, first, last);
  return hipGetLastError();
}

int mlp_blocks(int B) {
  // one block a CU (its weights and sums take 363 VGPRs, one wavefront a SIMD);
  // a block strides over the tiles beyond and keeps its weights and sums
  return std::min((B + kTrainRows - 1) / kTrainRows, kMaxRowBlocks);
}

// forward + backward of one batch (X: B x 12, y: B targets); gradients into g
// (kMlpParams), loss into *loss
hipError_t launch_mlp_loss_grad(const float* P, const float* X, const float* y, int B,
                                const MlpWork& w, float* g, double* loss, hipStream_t st) {
  const int nb = mlp_blocks(B);
  hipLaunchKernelGGL(k_mlp_rows<kRowsGrad>, dim3(nb), dim3(256), 0, st, P, X, y, B, 0ull,
                     (uint64_t)0, (uint64_t)0, w.part, w.loss, (float*)nullptr);
  hipLaunchKernelGGL(k_mlp_reduce<false>, dim3((kMlpParams + 31) / 32), dim3(32 * kSlices), 0, st, w.part,
                     w.loss, nb, B, g, loss, (float*)nullptr, (float*)nullptr, (float*)nullptr,
                     0.0f, 0.0f, 0.0f);
  return hipGetLastError();
}

// training step t of Adam on a batch of B drawn from the n samples (X, y);
// the batch's loss before the step into *loss
hipError_t launch_mlp_train_step(float* P, float* m, float* v, const float* X, const float* y,
                                 unsigned long long n, uint64_t seed, uint64_t step, int B, int t,
                                 float lr, const MlpWork& w, double* loss, hipStream_t st) {
  const int nb = mlp_blocks(B);
  const float c1 = 1.0f - powf(0.9f, (float)t), c2 = 1.0f - powf(0.999f, (float)t);
  hipLaunchKernelGGL(k_mlp_rows<kRowsGather>, dim3(nb), dim3(256), 0, st, P, X, y, B, n, seed, step,
                     w.part, w.loss, (float*)nullptr);
  hipLaunchKernelGGL(k_mlp_reduce<true>, dim3((kMlpParams + 31) / 32), dim3(32 * kSlices), 0, st, w.part,
                     w.loss, nb, B, (float*)nullptr, loss, P, m, v, lr, c1, c2);
  return hipGetLastError();
}

hipError_t launch_mlp_forward_fp32(const float* P, const float* X, int B, float* yhat,
                                   hipStream_t st) {
  hipLaunchKernelGGL(k_mlp_rows<kRowsForward>, dim3(mlp_blocks(B)), dim3(256), 0, st, P, X,
                     (const float*)nullptr, B, 0ull, (uint64_t)0, (uint64_t)0, (float*)nullptr,
                     (double*)nullptr, yhat);
  return hipGetLastError();
}

// sums: scratch of 2 kMomentBlocks doubles
hipError_t launch_mlp_normalise(float* y, unsigned long long n, double* sums, double* ms,
                                hipStream_t st) {
  hipLaunchKernelGGL(k_moments_part, dim3(kMomentBlocks), dim3(256), 0, st, y, n, sums);
  hipLaunchKernelGGL(k_moments, dim3(1), dim3(256), 0, st, sums, n, ms);
  hipLaunchKernelGGL(k_normalise, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, y, n, ms);
  return hipGetLastError();
}

hipError_t launch_mlp_pack(const float* P, short* Wbf, hipStream_t st) {
  hipLaunchKernelGGL(k_pack_bf16, dim3((64 * 16 + 2 * 4096 + 255) / 256), dim3(256), 0, st, P, Wbf);
  return hipGetLastError();
}

hipError_t launch_mlp_infer(const float* X, int B, const short* Wbf, const float* P, float* yhat,
                            hipStream_t st) {
  hipLaunchKernelGGL(k_mlp_infer, dim3((B + 255) / 256), dim3(256), 0, st, X, B, Wbf, P, yhat);
  return hipGetLastError();
}

hipError_t launch_alpha_guess27(const Box& b, const float* fin, const uint8_t* flags,
                                const short* Wbf, const float* P, float ymean, float ystd,
                                double* alpha, hipStream_t st) {
  // persistent-style grid: 8 blocks of four wavefronts per CU of a 256-CU device
  const unsigned tiles = (unsigned)((b.n + 63) / 64);
  const unsigned blocks = std::min<unsigned>((tiles + 3) / 4, 2048u);
  hipLaunchKernelGGL(k27_alpha_guess, dim3(blocks), dim3(256), 0, st, fin, b, flags, Wbf, P, ymean,
                     ystd, alpha);
  return hipGetLastError();
}

}  // namespace uclbs
