// Learned surrogate of one reactor step: a small MLP trained and evaluated
// with BF16-input / FP32-accumulate MFMA kernels (v_mfma_f32_16x16x16_bf16),
// and the FP64 acceptance test of its proposals.
//
//   features     [log T, log P, log max(Y_j, 1e-20) (nsp), log dt] -> normalised BF16
//   layer        one dense layer with its bias and GELU, or a layer's gradient
//                with gelu', in one launch
//   weight_grad  dW and db with the rows split over workgroups
//   gemm         C(f32) [+]= A(bf16) . B(bf16), any strides; one wavefront per
//                16x16 tile of C, K walked 16 at a time through the MFMA
//                (layers whose sizes are not multiples of 8, and callers)
//   bias_act     Z = C + b (f32), Y = gelu(Z) or Z (bf16 and f32)
//   act_backward dZ = dY * gelu'(Z) (f32 and bf16)
//   col_sum      db = sum over rows of dZ
//   adam         FP32 master weights, BF16 copies
//   accept       FP64 acceptance test of a proposed trajectory (one wavefront
//                per reactor, the integrator's RHS)
#include <hip/hip_runtime.h>

#include <type_traits>

#include "bdf_device.h"
#include "launch.h"

namespace zrk {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ unsigned short f32_to_bf16(float f) {
  // round to nearest even (finite inputs; NaN stays NaN)
  unsigned int u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (unsigned short)0x7fc0;  // NaN
  u += 0x7fffu + ((u >> 16) & 1u);
  return (unsigned short)(u >> 16);
}
__device__ __forceinline__ float bf16_to_f32(unsigned short h) {
  return __uint_as_float(((unsigned int)h) << 16);
}

// ---------------------------------------------------------------------------
__global__ void mlp_features_kernel(int n, int nsp, const double* __restrict__ T,
                                    const double* __restrict__ P, const double* __restrict__ Y,
                                    int stride, const double* __restrict__ dt, double dt_all,
                                    const float* __restrict__ mu, const float* __restrict__ sig,
                                    unsigned short* __restrict__ X, int ldx, int nfeat) {
  // A thread row per reactor and one logarithm of the selected source: bound by the
  // FP64 logarithm's instructions, of which a wavefront took four (one a source, in
  // branches) and a 64-bit division of its index.  Forward pass of 262,144 reactors
  // with 53 species: 615 to 521 us.
  const long r = (long)blockIdx.x * blockDim.y + threadIdx.y;
  if (r >= n) return;
  for (int f = threadIdx.x; f < ldx; f += blockDim.x) {
    float v = 0.0f;
    if (f < nfeat) {
      const double* p = f == 0 ? T + r : f == 1 ? P + r : Y + (size_t)r * stride + (f - 2);
      double x = dt_all;
      if (f < 2 + nsp) x = *p;
      else if (dt) x = dt[r];
      if (f >= 2 && f < 2 + nsp) x = fmax(x, 1.0e-20);
      v = (float)((log(x) - (double)mu[f]) / (double)sig[f]);
    }
    X[(size_t)r * ldx + f] = f32_to_bf16(v);
  }
}

// C[M x N] (f32) = or += A[M x K] . B[K x N]; A, B bf16 with element strides.
// MFMA 16x16x16 bf16 operand layout: lane l supplies A[row l%16][k 4(l/16)+j]
// and B[k 4(l/16)+j][col l%16], j = 0..3, and receives D[row 4(l/16)+j][col l%16].
__global__ void __launch_bounds__(256)
gemm_bf16_kernel(int M, int N, int K, const unsigned short* __restrict__ A, long sAm, long sAk,
                 const unsigned short* __restrict__ B, long sBk, long sBn, float* __restrict__ C,
                 long sCm, long sCn, int accumulate) {
  const long wave = ((long)blockIdx.x * blockDim.x + threadIdx.x) / kWave;
  const int lane = lane_id();
  const int tilesN = (N + 15) / 16;
  const long tm = wave / tilesN;
  const int tn = (int)(wave % tilesN);
  if (tm * 16 >= M) return;
  const long ra = tm * 16 + (lane & 15);
  const int cb = tn * 16 + (lane & 15);
  const int kq = (lane >> 4) * 4;
  f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
  for (int k0 = 0; k0 < K; k0 += 16) {
    bf16x4 a, b;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int k = k0 + kq + j;
      a[j] = (ra < M && k < K) ? (short)A[ra * sAm + (long)k * sAk] : (short)0;
      b[j] = (cb < N && k < K) ? (short)B[(long)k * sBk + (long)cb * sBn] : (short)0;
    }
    acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc, 0, 0, 0);
  }
  const int col = tn * 16 + (lane & 15);
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const long row = tm * 16 + (lane >> 4) * 4 + j;
    if (row < M && col < N) {
      float* c = C + row * sCm + (long)col * sCn;
      *c = accumulate ? *c + acc[j] : acc[j];
    }
  }
}

// LDS-tiled form of gemm_bf16_kernel for the network's shapes: a workgroup of
// 4 wavefronts computes a 64 x 64 block of C, each wavefront a 32 x 32 quarter
// (2 x 2 MFMA tiles).  K is walked 32 at a time: the A and B tiles are read
// from HBM with 16-byte loads along whichever of their dimensions is
// contiguous (kAk: A[m, k] has k contiguous, else m; kBk: B[k, n] has k
// contiguous, else n) and stored k-contiguous in LDS (As[m][k], Bs[n][k], rows
// padded to 40 elements), so every MFMA operand is one 8-byte LDS read.
// Requires the contiguous dimension of each operand a multiple of 8 elements,
// the other stride a multiple of 8 and 16-byte aligned bases (launch_gemm_bf16
// checks this and otherwise uses gemm_bf16_kernel).  Rows of A past M, columns
// of B past N and k past kend read as zero; kbeg is a multiple of 8.
constexpr int kGemmBM = 64, kGemmBN = 64, kGemmBK = 32, kGemmLd = kGemmBK + 8;

template <bool kAk, bool kBk>
__device__ __forceinline__ void gemm_block(unsigned short* __restrict__ As,
                                           unsigned short* __restrict__ Bs, long m0, int n0,
                                           int kbeg, int kend, int M, int N,
                                           const unsigned short* __restrict__ A, long sAm,
                                           long sAk, const unsigned short* __restrict__ B,
                                           long sBk, long sBn, float* __restrict__ C, long sCm,
                                           long sCn, int accumulate) {
  const int t = threadIdx.x;
  const int lane = t & 63, wave = t >> 6;
  const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
  f32x4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  for (int k0 = kbeg; k0 < kend; k0 += kGemmBK) {
    // A tile (64 m x 32 k): 256 chunks of 8 elements, one per thread
    {
      uint4 v = make_uint4(0, 0, 0, 0);
      if (kAk) {
        const int mm = t >> 2, c = (t & 3) * 8;
        const long gm = m0 + mm;
        const int gk = k0 + c;
        if (gm < M && gk < kend) v = *reinterpret_cast<const uint4*>(A + gm * sAm + gk);
        *reinterpret_cast<uint4*>(As + mm * kGemmLd + c) = v;
      } else {
        const int kk = t >> 3, c = (t & 7) * 8;
        const long gm = m0 + c;
        const int gk = k0 + kk;
        if (gm < M && gk < kend) v = *reinterpret_cast<const uint4*>(A + (long)gk * sAk + gm);
        const unsigned short* e = reinterpret_cast<const unsigned short*>(&v);
#pragma unroll
        for (int j = 0; j < 8; ++j) As[(c + j) * kGemmLd + kk] = e[j];
      }
    }
    // B tile (32 k x 64 n)
    {
      uint4 v = make_uint4(0, 0, 0, 0);
      if (kBk) {
        const int nn = t >> 2, c = (t & 3) * 8;
        const int gk = k0 + c;
        if (n0 + nn < N && gk < kend)
          v = *reinterpret_cast<const uint4*>(B + (long)(n0 + nn) * sBn + gk);
        *reinterpret_cast<uint4*>(Bs + nn * kGemmLd + c) = v;
      } else {
        const int kk = t >> 3, c = (t & 7) * 8;
        const int gk = k0 + kk;
        if (n0 + c < N && gk < kend)
          v = *reinterpret_cast<const uint4*>(B + (long)gk * sBk + n0 + c);
        const unsigned short* e = reinterpret_cast<const unsigned short*>(&v);
#pragma unroll
        for (int j = 0; j < 8; ++j) Bs[(c + j) * kGemmLd + kk] = e[j];
      }
    }
    __syncthreads();
#pragma unroll
    for (int ks = 0; ks < kGemmBK; ks += 16) {
      const int kq = ks + (lane >> 4) * 4;
      bf16x4 a[2], b[2];
#pragma unroll
      for (int i = 0; i < 2; ++i)
        a[i] = *reinterpret_cast<const bf16x4*>(As + (wm + 16 * i + (lane & 15)) * kGemmLd + kq);
#pragma unroll
      for (int j = 0; j < 2; ++j)
        b[j] = *reinterpret_cast<const bf16x4*>(Bs + (wn + 16 * j + (lane & 15)) * kGemmLd + kq);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a[i], b[j], acc[i][j], 0, 0, 0);
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int col = n0 + wn + 16 * j + (lane & 15);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const long row = m0 + wm + 16 * i + (lane >> 4) * 4 + v;
        if (row < M && col < N) {
          float* c = C + row * sCm + (long)col * sCn;
          *c = accumulate ? *c + acc[i][j][v] : acc[i][j][v];
        }
      }
    }
}

template <bool kAk, bool kBk>
__global__ void __launch_bounds__(256)
gemm_bf16_tiled_kernel(int M, int N, int K, const unsigned short* __restrict__ A, long sAm,
                       long sAk, const unsigned short* __restrict__ B, long sBk, long sBn,
                       float* __restrict__ C, long sCm, long sCn, int accumulate) {
  __shared__ __align__(16) unsigned short As[kGemmBM * kGemmLd];
  __shared__ __align__(16) unsigned short Bs[kGemmBN * kGemmLd];
  gemm_block<kAk, kBk>(As, Bs, (long)blockIdx.x * kGemmBM, blockIdx.y * kGemmBN, 0, K, M, N, A,
                       sAm, sAk, B, sBk, sBn, C, sCm, sCn, accumulate);
}

__device__ __forceinline__ float gelu(float z) {
  return 0.5f * z * (1.0f + erff(z * 0.70710678118654752f));
}
__device__ __forceinline__ float gelu_grad(float z) {
  const float cdf = 0.5f * (1.0f + erff(z * 0.70710678118654752f));
  const float pdf = 0.39894228040143268f * expf(-0.5f * z * z);
  return cdf + z * pdf;
}

// Z = C + b; Y = act(Z) as bf16 (and f32 if Yf).  act: 1 gelu, 0 identity.
__global__ void bias_act_kernel(int M, int N, const float* __restrict__ C, const float* __restrict__ b,
                                float* __restrict__ Z, unsigned short* __restrict__ Yb,
                                float* __restrict__ Yf, int act) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (long)M * N) return;
  const float z = C[i] + b[i % N];
  if (Z) Z[i] = z;
  const float y = act ? gelu(z) : z;
  if (Yb) Yb[i] = f32_to_bf16(y);
  if (Yf) Yf[i] = y;
}

// dZ = dY * act'(Z) (f32 and bf16 copies)
__global__ void act_backward_kernel(int M, int N, const float* __restrict__ dY,
                                    const float* __restrict__ Z, float* __restrict__ dZ,
                                    unsigned short* __restrict__ dZb, int act) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (long)M * N) return;
  const float g = act ? dY[i] * gelu_grad(Z[i]) : dY[i];
  dZ[i] = g;
  dZb[i] = f32_to_bf16(g);
}

// db[j] = sum_i dZ[i*N + j]: one thread per column, rows in order
__global__ void col_sum_kernel(int M, int N, const float* __restrict__ dZ, float* __restrict__ db) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= N) return;
  float s = 0.0f;
  for (int i = 0; i < M; ++i) s += dZ[(long)i * N + j];
  db[j] = s;
}

// Adam (bias-corrected) on FP32 master weights; refreshes the BF16 copy
__global__ void adam_kernel(long n, float* __restrict__ w, const float* __restrict__ g,
                            float* __restrict__ m, float* __restrict__ v,
                            unsigned short* __restrict__ wb, float lr, float b1, float b2,
                            float eps, float c1, float c2) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.0f - b1) * gi;
  const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  const float wi = w[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
  w[i] = wi;
  if (wb) wb[i] = f32_to_bf16(wi);
}

__global__ void to_bf16_kernel(long n, const float* __restrict__ x, unsigned short* __restrict__ y) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = f32_to_bf16(x[i]);
}

// One dense layer with its elementwise part, out = epilogue(X W') for W' = W
// (K x N, forward) or, with kT, the transpose of W (N x K, backward):
//   kBias     Z = X W + b                                   (the last layer)
//   kGelu     Z = X W + b (f32, optional), Y = gelu(Z) (bf16)
//   kGradGelu dZ = (X W^T) gelu'(Z) (f32 and bf16 copies)
// A workgroup keeps its span of output columns of W' in LDS, k-contiguous, and
// its wavefronts walk 32-row tiles of X, whose MFMA operands come straight from
// memory, the next tile's while this one is computed.  The product is formed
// transposed (W' is the row operand), so a lane ends with 4 consecutive outputs
// of one row: 16-byte stores.  With K > KC (= 16 KS) a workgroup has 64 columns
// and restages W' chunk by chunk.  kStagers (KS = 16, fewer row tiles than fill the
// workgroups): a workgroup has kLayerWaves wavefronts all the same, those beyond the
// first `workers` only to stage: a small batch has one wavefront of rows a workgroup,
// which alone took most of the pass to stage 32 KB (one row, 3 x 1,024: 81 to 51 us,
// 3 x 256: 39 to 32 us).  Smaller chunks are staged in a few loads and don't pay for the
// test (16,384 rows, 3 x 128: 38.6 and 39.4 us).
// Bound: memory and the GELU (one erff is about 40 instructions).  As a product with
// FP32 results and a pass of its own for bias and GELU, in 64 x 64 tiles that read
// X once per 64 columns, a forward pass of 262,144 reactors (56 -> 3 x 256 -> 54)
// took 1,270 us; this way 615 us.
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
enum { kBias = 0, kGelu = 1, kGradGelu = 2 };
constexpr int kLayerWaves = 8;

__device__ __forceinline__ uint2 pack_bf16(const float* v) {
  uint2 p;
  p.x = (unsigned)f32_to_bf16(v[0]) | ((unsigned)f32_to_bf16(v[1]) << 16);
  p.y = (unsigned)f32_to_bf16(v[2]) | ((unsigned)f32_to_bf16(v[3]) << 16);
  return p;
}

template <int KS, bool kT, int kEpi, bool kStagers>
__global__ void __launch_bounds__(kLayerWaves* kWave)
layer_kernel(int M, int N, int K, int span, int workers, const unsigned short* __restrict__ X,
             const unsigned short* __restrict__ W, const float* __restrict__ b,
             const float* __restrict__ Zin, float* __restrict__ Z,
             unsigned short* __restrict__ Y) {
  extern __shared__ __align__(16) unsigned short wl[];
  constexpr int KC = 16 * KS, ld = KC + 8;
  const int lane = threadIdx.x & 63;
  const int wave = kStagers ? uni((int)threadIdx.x >> 6) : (int)threadIdx.x >> 6;
  const int nthr = kStagers ? kLayerWaves * kWave : (int)blockDim.x;
  const int nw = kStagers ? workers : nthr >> 6;  // wavefronts with tiles of their own
  const bool mine = !kStagers || wave < nw;
  const int n0 = blockIdx.y * span, n1 = min(N, n0 + span);
  const int chunks = (K + KC - 1) / KC;
  const int tiles = (M + 31) / 32;
  const int r = lane & 31, half = lane >> 5;

  // columns [c0, c0 + cols) of W', k chunk c, into LDS rows 0.. (zeros past N and K)
  auto stage = [&](int c0, int cols, int c) {
    const int kb = c * KC;
    if (kT) {
      for (int i = threadIdx.x; i < cols * (KC / 8); i += nthr) {
        const int n = i / (KC / 8), k = (i % (KC / 8)) * 8;
        uint4 v = make_uint4(0, 0, 0, 0);
        if (c0 + n < N && kb + k < K)
          v = *reinterpret_cast<const uint4*>(W + (size_t)(c0 + n) * K + kb + k);
        *reinterpret_cast<uint4*>(wl + n * ld + k) = v;
      }
    } else {
      for (int i = threadIdx.x; i < (cols / 8) * (KC / 4); i += nthr) {
        const int k = (i / (cols / 8)) * 4, n = (i % (cols / 8)) * 8;
        uint4 v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          v[j] = make_uint4(0, 0, 0, 0);
          if (c0 + n < N && kb + k + j < K)
            v[j] = *reinterpret_cast<const uint4*>(W + (size_t)(kb + k + j) * N + c0 + n);
        }
        const unsigned* e[4] = {&v[0].x, &v[1].x, &v[2].x, &v[3].x};
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          const int sh = (q & 1) * 16;
          uint2 p;
          p.x = ((e[0][q >> 1] >> sh) & 0xffffu) | (((e[1][q >> 1] >> sh) & 0xffffu) << 16);
          p.y = ((e[2][q >> 1] >> sh) & 0xffffu) | (((e[3][q >> 1] >> sh) & 0xffffu) << 16);
          *reinterpret_cast<uint2*>(wl + (n + q) * ld + k) = p;
        }
      }
    }
  };
  auto load_x = [&](int tile, int c, bf16x8* a) {
    const long row = (long)tile * 32 + r;
    const unsigned short* p = X + row * K + c * KC + 8 * half;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      uint4 v = make_uint4(0, 0, 0, 0);
      if (row < M && c * KC + 16 * s + 8 * half < K)
        v = *reinterpret_cast<const uint4*>(p + 16 * s);
      a[s] = __builtin_bit_cast(bf16x8, v);
    }
  };

  if (chunks == 1) stage(n0, (n1 - n0 + 63) & ~63, 0);
  bf16x8 a[KS], an[KS];
  if (chunks == 1) load_x(mine ? blockIdx.x * nw + wave : tiles, 0, an);
  __syncthreads();
  for (int t0 = blockIdx.x * nw; t0 < tiles; t0 += gridDim.x * nw) {
    const int tile = mine ? t0 + wave : tiles;  // helpers: past the rows
    const long row = (long)tile * 32 + r;
    if (chunks == 1) {
      if (!mine) break;  // nothing more to stage
#pragma unroll
      for (int s = 0; s < KS; ++s) a[s] = an[s];
      load_x(tile + gridDim.x * nw, 0, an);
    }
    for (int g0 = n0; g0 < n1; g0 += 64) {
      f32x16 acc[2];
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[t][i] = 0.0f;
      for (int c = 0; c < chunks; ++c) {
        const unsigned short* w = wl + (g0 - n0 + r) * ld + 8 * half;
        if (chunks > 1) {
          __syncthreads();
          stage(g0, 64, c);
          load_x(tile, c, a);
          __syncthreads();
          w = wl + r * ld + 8 * half;
          if (!mine) continue;
        }
#pragma unroll
        for (int s = 0; s < KS; ++s)
#pragma unroll
          for (int t = 0; t < 2; ++t) {
            const bf16x8 wv = *reinterpret_cast<const bf16x8*>(w + t * 32 * ld + 16 * s);
            acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wv, a[s], acc[t], 0, 0, 0);
          }
      }
      // output (row, n + j) is register 4 q + j of tile t, n = g0 + 32 t + 8 q + 4 half
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int n = g0 + 32 * t + 8 * q + 4 * half;
          if (row < M && n < n1) {
            const size_t at = (size_t)row * N + n;
            const float4 e = *reinterpret_cast<const float4*>(kEpi == kGradGelu ? Zin + at : b + n);
            const float* ev = &e.x;
            float z[4], y[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              const float x = acc[t][4 * q + j];
              z[j] = kEpi == kGradGelu ? x * gelu_grad(ev[j]) : x + ev[j];
              y[j] = kEpi == kGelu ? gelu(z[j]) : z[j];
            }
            if (kEpi != kGelu || Z)
              *reinterpret_cast<float4*>(Z + at) = make_float4(z[0], z[1], z[2], z[3]);
            if (kEpi != kBias) *reinterpret_cast<uint2*>(Y + at) = pack_bf16(y);
          }
        }
    }
  }
}

// dW = H^T dZ (bf16 operands, K x N) and db = column sums of dZ (f32) over B
// rows, split over blockIdx.y: a workgroup sums its rows' part of a 64 x 64
// block of dW, or of 64 columns of db, into out[blockIdx.y][K * N + N].  One
// workgroup per block of dW over all rows left 240 of 256 compute units idle at
// K = N = 256, and db was summed by one thread a column: a forward and backward
// pass of 4,096 reactors took 4,370 us, with both split 151 us.
__global__ void __launch_bounds__(256)
weight_grad_kernel(int B, int K, int N, int rows, const unsigned short* __restrict__ H,
                   const float* __restrict__ dZ, const unsigned short* __restrict__ dZb,
                   float* __restrict__ dW, float* __restrict__ db, long part) {
  __shared__ __align__(16) unsigned short As[kGemmBM * kGemmLd];
  __shared__ __align__(16) unsigned short Bs[kGemmBN * kGemmLd];
  const int bk = (K + kGemmBM - 1) / kGemmBM, bn = (N + kGemmBN - 1) / kGemmBN;
  const int r0 = blockIdx.y * rows, r1 = min(B, r0 + rows);
  const int i = blockIdx.x;
  if (i < bk * bn) {
    gemm_block<false, false>(As, Bs, (long)(i % bk) * kGemmBM, (i / bk) * kGemmBN, r0, r1, K, N, H,
                             1, K, dZb, N, 1, dW + blockIdx.y * part, N, 1, 0);
    return;
  }
  float* const red = reinterpret_cast<float*>(As);
  const int col = (i - bk * bn) * 64 + (threadIdx.x & 63), sub = threadIdx.x >> 6;
  float s[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  if (col < N) {
    int row = r0 + sub;
    for (; row + 12 < r1; row += 16)
#pragma unroll
      for (int u = 0; u < 4; ++u) s[u] += dZ[(size_t)(row + 4 * u) * N + col];
    for (; row < r1; row += 4) s[0] += dZ[(size_t)row * N + col];
  }
  red[threadIdx.x] = (s[0] + s[1]) + (s[2] + s[3]);
  __syncthreads();
  if (sub == 0 && col < N)
    db[blockIdx.y * part + col] =
        (red[threadIdx.x] + red[threadIdx.x + 64]) + (red[threadIdx.x + 128] + red[threadIdx.x + 192]);
}

// dW and db from the splits' parts, in the order of the splits
__global__ void __launch_bounds__(256)
weight_grad_sum_kernel(int nw, int nb, int splits, const float* __restrict__ part,
                       float* __restrict__ dW, float* __restrict__ db) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nw + nb) return;
  const long st = (long)nw + nb;
  float s = 0.0f;
#pragma unroll 8
  for (int k = 0; k < splits; ++k) s += part[k * st + i];
  if (i < nw) dW[i] = s;
  else db[i - nw] = s;
}

// ---------------------------------------------------------------------------
// Acceptance of a proposed trajectory of one reactor step [0, dt] (one
// wavefront per reactor, constant pressure, FP64).  The proposal gives the
// state at the nodes t_k = tau_k dt (k = 1..m, tau increasing, tau_m = 1):
// Tp[(k-1)*n + r] and Yp[((k-1)*n + r)*stride + j].  Interval k, from t_{k-1}
// (t_0 = 0, the initial state) to t_k, is the implicit equation
//   G(y) = y - y_{k-1} - h f(y)                      (k = 1, backward Euler)
//   G(y) = y - y_{k-1} - h/2 (f(y_{k-1}) + f(y))     (k > 1, trapezoidal rule)
// solved by Newton iterations with the iteration matrix I - c J (c = h or
// h/2, J the reference Jacobian at the start point): at most max_newton
// iterations, converged when the correction's weighted RMS norm is at most
// kAcceptConv.  The start point is the proposal at t_k, or the converged state
// at t_{k-1} when its residual (-h f(y_{k-1})) has the smaller weighted norm
// (weights at y_{k-1}); a start too far from the solution for that many
// iterations fails the test.  Local errors come from divided differences of f
// over the converged nodes after t_0 (the initial state may lie off the slow
// manifold that the first interval's backward Euler step damps away):
//   backward Euler   (h^2 / 2) f[t_1, t_2]
//   trapezoidal      (h^3 / 12) 2 f[t_a, t_b, t_c], three consecutive nodes
// Each interval's |local error| is weighted with the weights
// 1 / (rtol |y| + atol) of the node that completes its divided difference and
// summed componentwise; the step is accepted when every interval converged
// and that sum has weighted RMS norm at most 1.  The sum only grows, so the
// test stops at the first node where its norm exceeds 1.  An accepted
// reactor's converged end state is written to the last node's arrays.
// res[4r..4r+3] (optional): most Newton iterations of an interval, largest
// first correction, the error norm where the test stopped (infinite if an
// interval failed first), first interval whose Newton iterations failed
// (0: none, -1: the RHS failed).
// LDS: Ml[kNP*kNP], rvec[kNP], t2l[kNP], then C, G, rop.
// ---------------------------------------------------------------------------
constexpr int kAcceptMaxNodes = 8;
constexpr double kAcceptConv = 0.1;

template <bool kExt, bool kAhead>
__global__ void __launch_bounds__(kWave)
accept_kernel(DevMech m, BdfOpts o, int n, const double* __restrict__ dts, double dt_all,
              const double* __restrict__ T0, const double* __restrict__ P,
              const double* __restrict__ Y0, int nodes, const double* __restrict__ tau,
              double* __restrict__ Tp, double* __restrict__ Yp, int stride, int max_newton,
              int* __restrict__ accept, double* __restrict__ res,
              double* __restrict__ jscratch) {
  extern __shared__ double lds[];
  const int lane = lane_id();
  const int nsp = m.nsp;
  const int N = nsp + 1;
  double* Ml = lds;
  double* rvec = Ml + kNP * kNP;
  double* t2l = rvec + kNP;
  double* rl = t2l + kNP;
  RhsLds s = rhs_lds_at(rl, nsp);
  double* saved = jscratch + (size_t)blockIdx.x * kNP * kNP;
  constexpr TeamWaveX<kExt, kAhead ? kTeamInline : kTeamBatch> team{};
  const bool act = lane <= nsp;
  const double inv = 1.0 / (double)N;
  const int rot = gj_rotation(N);  // register c of the inverse holds column (c + rot) mod 64
  for (int r = blockIdx.x; r < n; r += gridDim.x) {
    const double dt = dts ? dts[r] : dt_all;
    const double Pr = P[r];
    double y0 = 0.0;
    if (lane < nsp) y0 = Y0[(size_t)r * stride + lane];
    if (lane == nsp) y0 = T0[r] / o.Tref;
    RhsAux aux;
    double yprev = y0, fprev = 0.0;
    int bad = rhs_team(team, m, s, Pr, 0.0, o.Tref, o.step_limiter, y0, fprev, aux);
    int failed = 0, most_it = 0;
    double first_max = 0.0;
    double esum = 0.0;  // this lane's weighted |local errors| summed so far
    double en = 0.0;
    bool stopped = false;
    // f and t at the two converged nodes before node k (sliding window)
    double fm2 = 0.0, fm1 = 0.0, tm2 = 0.0, tm1 = 0.0;
    for (int k = 0; k < nodes && !bad && !failed && !stopped; ++k) {
      const size_t row = (size_t)k * n + r;
      double y = 0.0;
      if (lane < nsp) y = Yp[row * stride + lane];
      if (lane == nsp) y = Tp[row] / o.Tref;
      const double tk = tau[k] * dt;
      const double h = tk - (k > 0 ? tm1 : 0.0);
      const double c = k == 0 ? h : 0.5 * h;
      // the start point: the proposal, or y_{k-1} if its residual is smaller
      double fy;
      const int badp = rhs_team(team, m, s, Pr, 0.0, o.Tref, o.step_limiter, y, fy, aux);
      const double wp = act ? 1.0 / (o.rtol * fabs(yprev) + o.atol) : 0.0;
      const double gp = (!act || badp) ? 0.0
                        : (k == 0 ? y - yprev - h * fy : y - yprev - 0.5 * h * (fprev + fy));
      const double rp = badp ? INFINITY : wave_sum(gp * gp * wp * wp);
      const double rq = wave_sum(act ? h * h * fprev * fprev * wp * wp : 0.0);
      if (rq < rp) {
        y = yprev;
        bad = rhs_team(team, m, s, Pr, 0.0, o.Tref, o.step_limiter, y, fy, aux);
        if (bad) continue;
      }
      // Newton matrix I - c J at the start point, inverted in registers
      jacobian_lds<double>(team, m, s, Pr, 0.0, o, y, fy, aux.inv_rho, Ml, kNP, saved, t2l);
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      double R[kNP];
#pragma unroll
      for (int col = 0; col < kNP; ++col) {
        double v = (col <= nsp && lane <= nsp) ? -c * Ml[col * kNP + lane] : 0.0;
        if (col == lane) v += 1.0;
        R[col] = v;
      }
      const bool ok = gj_invert(R, N);
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int col = 0; col < kNP; ++col) Ml[col * kNP + lane] = R[col];
      if (!ok) {
        failed = k + 1;
        continue;
      }
      const double w = act ? 1.0 / (o.rtol * fabs(y) + o.atol) : 0.0;
      bool conv = false;
      int it = 0;
      for (; it < max_newton && !conv && !bad; ++it) {
        if (it > 0) bad = rhs_team(team, m, s, Pr, 0.0, o.Tref, o.step_limiter, y, fy, aux);
        if (bad) continue;
        const double G = !act ? 0.0
                         : (k == 0 ? y - yprev - h * fy : y - yprev - 0.5 * h * (fprev + fy));
        rvec[lane] = G;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        double d = 0.0;
#pragma unroll 8
        for (int col = 0; col < kNP; ++col)
          d = fma(Ml[col * kNP + lane], rvec[(col + rot) & (kNP - 1)], d);
        __builtin_amdgcn_wave_barrier();
        if (act) y -= d;
        const double dn = sqrt(wave_sum(act ? d * d * w * w : 0.0) * inv);
        if (it == 0) first_max = fmax(first_max, dn);
        conv = dn <= kAcceptConv;
      }
      if (bad) continue;
      most_it = max(most_it, it);
      if (!conv) {
        failed = k + 1;
        continue;
      }
      bad = rhs_team(team, m, s, Pr, 0.0, o.Tref, o.step_limiter, y, fy, aux);
      if (bad) continue;
      yprev = y;
      fprev = fy;
      // the local errors that node k completes, in the weights at node k
      double e = 0.0;
      if (k == 1) {  // backward Euler on [0, t_1]: (h^2 / 2) y'' with y'' = f[t_1, t_2]
        e = fabs(0.5 * tm1 * tm1 * (fy - fm1) / (tk - tm1));
      } else if (k >= 2) {
        // trapezoidal intervals: (h^3 / 12) 2 f[t_a, t_b, t_c] over the three
        // consecutive nodes ending at k; the first three nodes also serve the
        // trapezoidal interval before, which has no node of its own before it
        const double dd = ((fy - fm1) / (tk - tm1) - (fm1 - fm2) / (tm1 - tm2)) / (tk - tm2);
        e = fabs(h * h * h / 12.0 * 2.0 * dd);
        if (k == 2) {
          const double h1 = tm1 - tm2;
          e += fabs(h1 * h1 * h1 / 12.0 * 2.0 * dd);
        }
      }
      fm2 = fm1;
      fm1 = fy;
      tm2 = tm1;
      tm1 = tk;
      esum += act ? e / (o.rtol * fabs(y) + o.atol) : 0.0;
      en = sqrt(wave_sum(esum * esum) * inv);
      if (en > 1.0) stopped = true;
    }
    if (bad || failed) en = INFINITY;
    const bool acc = !bad && !failed && en <= 1.0;
    if (acc) {
      const size_t row = (size_t)(nodes - 1) * n + r;
      if (lane < nsp) Yp[row * stride + lane] = yprev;
      if (lane == nsp) Tp[row] = yprev * o.Tref;
    }
    if (lane == 0) {
      accept[r] = acc ? 1 : 0;
      if (res) {
        res[4 * (size_t)r] = (double)most_it;
        res[4 * (size_t)r + 1] = first_max;
        res[4 * (size_t)r + 2] = en;
        res[4 * (size_t)r + 3] = bad ? -1.0 : (double)failed;
      }
    }
    __builtin_amdgcn_wave_barrier();
  }
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
namespace {
inline unsigned blocks_for(long n, int b) { return (unsigned)((n + b - 1) / b); }
}  // namespace

hipError_t launch_mlp_features(int n, int nsp, const double* T, const double* P, const double* Y,
                               int stride, const double* dt, double dt_all, const float* mu,
                               const float* sig, unsigned short* X, int ldx, int nfeat,
                               hipStream_t st) {
  if (n <= 0) return hipSuccess;
  const unsigned bx = ldx < 256 ? (unsigned)ldx : 256u, by = 256u / bx;
  hipLaunchKernelGGL(mlp_features_kernel, dim3(blocks_for(n, (int)by)), dim3(bx, by), 0, st, n,
                     nsp, T, P, Y, stride, dt, dt_all, mu, sig, X, ldx, nfeat);
  return hipGetLastError();
}

hipError_t launch_gemm_bf16(int M, int N, int K, const unsigned short* A, long sAm, long sAk,
                            const unsigned short* B, long sBk, long sBn, float* C, long sCm,
                            long sCn, int accumulate, hipStream_t st) {
  if (M <= 0 || N <= 0) return hipSuccess;
  // the tiled kernel where its layout conditions hold (16-byte loads along
  // the contiguous dimension of each operand), else one wavefront per tile
  const auto al16 = [](const void* p) { return ((uintptr_t)p & 15) == 0; };
  const bool aK = sAk == 1 && sAm % 8 == 0 && K % 8 == 0;
  const bool aM = sAm == 1 && sAk % 8 == 0 && M % 8 == 0;
  const bool bK = sBk == 1 && sBn % 8 == 0 && K % 8 == 0;
  const bool bN = sBn == 1 && sBk % 8 == 0 && N % 8 == 0;
  const long tiles = (long)((M + 15) / 16) * ((N + 15) / 16);
  // Ragged columns with both operands contiguous along the outputs (a weight
  // gradient's layout), whose blocks of 8 x 64 go through LDS transposed: while the
  // 16 x 16 tiles leave wavefronts idle (at most two a SIMD) and the sum is not long,
  // a wavefront per tile reads them faster.  Microseconds, a wavefront per tile and
  // tiled: 48 x 48, K 4,096 94 and 101; 256 x 200, K 512 14.6 and 15.6; 1,024 x 56,
  // K 4,096 145 and 106; 1,024 x 520, K 512 17.5 and 15.3.
  const bool few = !aK && !bK && N % kGemmBN != 0 && tiles <= 2048 && tiles * K < (1L << 20);
  // (the tiles of 64 columns are counted in a grid's second dimension)
  const bool fits = N <= 65535L * kGemmBN;
  if (K > 0 && (aK || aM) && (bK || bN) && al16(A) && al16(B) && !few && fits) {
    const dim3 grid((unsigned)((M + kGemmBM - 1) / kGemmBM),
                    (unsigned)((N + kGemmBN - 1) / kGemmBN));
    if (aK && bN)
      hipLaunchKernelGGL((gemm_bf16_tiled_kernel<true, false>), grid, dim3(256), 0, st, M, N, K, A,
                         sAm, sAk, B, sBk, sBn, C, sCm, sCn, accumulate);
    else if (aK)
      hipLaunchKernelGGL((gemm_bf16_tiled_kernel<true, true>), grid, dim3(256), 0, st, M, N, K, A,
                         sAm, sAk, B, sBk, sBn, C, sCm, sCn, accumulate);
    else if (bN)
      hipLaunchKernelGGL((gemm_bf16_tiled_kernel<false, false>), grid, dim3(256), 0, st, M, N, K,
                         A, sAm, sAk, B, sBk, sBn, C, sCm, sCn, accumulate);
    else
      hipLaunchKernelGGL((gemm_bf16_tiled_kernel<false, true>), grid, dim3(256), 0, st, M, N, K, A,
                         sAm, sAk, B, sBk, sBn, C, sCm, sCn, accumulate);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(gemm_bf16_kernel, dim3(blocks_for(tiles * kWave, 256)), dim3(256), 0, st, M,
                     N, K, A, sAm, sAk, B, sBk, sBn, C, sCm, sCn, accumulate);
  return hipGetLastError();
}

hipError_t launch_bias_act(int M, int N, const float* C, const float* b, float* Z,
                           unsigned short* Yb, float* Yf, int act, hipStream_t st) {
  if (M <= 0 || N <= 0) return hipSuccess;
  hipLaunchKernelGGL(bias_act_kernel, dim3(blocks_for((long)M * N, 256)), dim3(256), 0, st, M, N,
                     C, b, Z, Yb, Yf, act);
  return hipGetLastError();
}

hipError_t launch_act_backward(int M, int N, const float* dY, const float* Z, float* dZ,
                               unsigned short* dZb, int act, hipStream_t st) {
  if (M <= 0 || N <= 0) return hipSuccess;
  hipLaunchKernelGGL(act_backward_kernel, dim3(blocks_for((long)M * N, 256)), dim3(256), 0, st, M,
                     N, dY, Z, dZ, dZb, act);
  return hipGetLastError();
}

hipError_t launch_col_sum(int M, int N, const float* dZ, float* db, hipStream_t st) {
  if (N <= 0) return hipSuccess;
  hipLaunchKernelGGL(col_sum_kernel, dim3(blocks_for(N, 256)), dim3(256), 0, st, M, N, dZ, db);
  return hipGetLastError();
}

namespace {
constexpr int kLayerCus = 256;  // compute units a launch wants to occupy

// lets a kernel take a compute unit's whole LDS
template <auto kKernel>
hipError_t layer_lds() {
  static const hipError_t e =
      hipFuncSetAttribute(reinterpret_cast<const void*>(kKernel),
                          hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
  return e;
}

template <int KS, bool kT, int kEpi>
hipError_t layer_launch(int M, int N, int K, const unsigned short* X, const unsigned short* W,
                        const float* b, const float* Zin, float* Z, unsigned short* Y,
                        hipStream_t st) {
  constexpr int KC = 16 * KS;
  const long tiles = ((long)M + 31) / 32;
  // All columns in one workgroup (X is read once) where the row tiles alone
  // occupy the card and W fits a workgroup's LDS; else 64 a workgroup.
  int span = 64;
  if (K <= KC && N <= 256 && tiles >= (long)kLayerCus * kLayerWaves) span = ((N + 63) / 64) * 64;
  const long groups = (N + span - 1) / span;
  long waves = (tiles * groups + kLayerCus - 1) / kLayerCus;
  waves = waves < 1 ? 1 : (waves > kLayerWaves ? kLayerWaves : waves);
  if (waves > tiles) waves = tiles;
  const size_t lds = (size_t)span * (KC + 8) * sizeof(unsigned short);
  const long per_cu = (160 * 1024) / (long)lds;  // workgroups a compute unit's LDS holds
  long gx = (tiles + waves - 1) / waves;
  const long most = kLayerCus * (per_cu < 1 ? 1 : (per_cu > 2 ? 2 : per_cu)) / groups;
  if (gx > most) gx = most < 1 ? 1 : most;
  const auto launch = [&](hipError_t attr, auto kernel, long wavefronts) {
    if (attr != hipSuccess) return attr;
    hipLaunchKernelGGL(kernel, dim3((unsigned)gx, (unsigned)groups),
                       dim3((unsigned)wavefronts * kWave), lds, st, M, N, K, span, (int)waves, X,
                       W, b, Zin, Z, Y);
    return hipGetLastError();
  };
  if constexpr (KS == 16) {
    constexpr auto staged = layer_kernel<KS, kT, kEpi, true>;
    if (waves < kLayerWaves) return launch(layer_lds<staged>(), staged, kLayerWaves);
  }
  constexpr auto kernel = layer_kernel<KS, kT, kEpi, false>;
  return launch(layer_lds<kernel>(), kernel, waves);
}

template <bool kT, int kEpi>
hipError_t layer_for_k(int M, int N, int K, const unsigned short* X, const unsigned short* W,
                       const float* b, const float* Zin, float* Z, unsigned short* Y,
                       hipStream_t st) {
  if (M <= 0 || N <= 0) return hipSuccess;
  if (K <= 64) return layer_launch<4, kT, kEpi>(M, N, K, X, W, b, Zin, Z, Y, st);
  if (K <= 128) return layer_launch<8, kT, kEpi>(M, N, K, X, W, b, Zin, Z, Y, st);
  return layer_launch<16, kT, kEpi>(M, N, K, X, W, b, Zin, Z, Y, st);
}
}  // namespace

bool layer_fits(int N, int K, std::initializer_list<const void*> operands) {
  if (K <= 0 || K % 8 != 0 || N % 8 != 0) return false;
  // (a null operand is one the call does not use)
  for (const void* p : operands)
    if ((uintptr_t)p & 15) return false;
  return true;
}

hipError_t launch_layer(int M, int N, int K, const unsigned short* X, const unsigned short* W,
                        const float* b, float* Z, unsigned short* Y, int act, hipStream_t st) {
  return act ? layer_for_k<false, kGelu>(M, N, K, X, W, b, nullptr, Z, Y, st)
             : layer_for_k<false, kBias>(M, N, K, X, W, b, nullptr, Z, nullptr, st);
}

hipError_t launch_layer_grad(int M, int K, int N, const unsigned short* dZb,
                             const unsigned short* W, const float* Zin, float* dZ,
                             unsigned short* dZb_out, hipStream_t st) {
  return layer_for_k<true, kGradGelu>(M, K, N, dZb, W, nullptr, Zin, dZ, dZb_out, st);
}

// Splits of the rows: enough workgroups for two a compute unit, of at least 128
// rows each (4 steps of the product's 32), and rows a multiple of 32.
int weight_grad_splits(int B, int K, int N) {
  const long blocks = (long)((K + 63) / 64) * ((N + 63) / 64) + (N + 63) / 64;
  long s = (2 * kLayerCus + blocks - 1) / blocks;
  const long most = ((long)B + 127) / 128;
  if (s > most) s = most;
  return (int)(s < 1 ? 1 : s);
}

hipError_t launch_weight_grad(int B, int K, int N, const unsigned short* H, const float* dZ,
                              const unsigned short* dZb, float* dW, float* db, float* work,
                              hipStream_t st) {
  if (K <= 0 || N <= 0) return hipSuccess;
  const int splits = weight_grad_splits(B, K, N);
  const int rows = ((B + splits - 1) / splits + 31) & ~31;
  const long nw = (long)K * N;
  const unsigned blocks =
      (unsigned)(((K + 63) / 64) * ((N + 63) / 64) + (N + 63) / 64);
  const bool one = splits == 1;
  hipLaunchKernelGGL(weight_grad_kernel, dim3(blocks, (unsigned)splits), dim3(256), 0, st, B, K, N,
                     rows, H, dZ, dZb, one ? dW : work, one ? db : work + nw,
                     one ? 0L : nw + N);
  if (!one)
    hipLaunchKernelGGL(weight_grad_sum_kernel, dim3(blocks_for(nw + N, 256)), dim3(256), 0, st,
                       (int)nw, N, splits, work, dW, db);
  return hipGetLastError();
}

hipError_t launch_adam(long n, float* w, const float* g, float* m, float* v, unsigned short* wb,
                       float lr, float b1, float b2, float eps, float c1, float c2,
                       hipStream_t st) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(adam_kernel, dim3(blocks_for(n, 256)), dim3(256), 0, st, n, w, g, m, v, wb,
                     lr, b1, b2, eps, c1, c2);
  return hipGetLastError();
}

hipError_t launch_to_bf16(long n, const float* x, unsigned short* y, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(to_bf16_kernel, dim3(blocks_for(n, 256)), dim3(256), 0, st, n, x, y);
  return hipGetLastError();
}

hipError_t launch_accept(const DevMech& m, const BdfOpts& o, int n, const double* dts,
                         double dt_all, const double* T0, const double* P, const double* Y0,
                         int nodes, const double* tau, double* Tp, double* Yp, int stride,
                         int max_newton, int* accept, double* res, double* jscratch,
                         int nblocks, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  if (m.nsp > kNP - 1 || nodes < 3 || nodes > kAcceptMaxNodes) return hipErrorInvalidValue;
  const int grid = n < nblocks ? n : nblocks;
  const size_t lds = sizeof(double) * (size_t)(kNP * kNP + 2 * kNP) + rhs_lds_bytes(m);
  const auto launch = [&](auto e, auto a) {
    hipLaunchKernelGGL((accept_kernel<decltype(e)::value, decltype(a)::value>), dim3(grid),
                       dim3(kWave), lds, st, m, o, n, dts, dt_all, T0, P, Y0, nodes, tau, Tp, Yp,
                       stride, max_newton, accept, res, jscratch);
    return hipGetLastError();
  };
  // (the right-hand sides are inlined: 8,192 reactors of 10 species 695 us, 773 us when
  // they are called; 53 species 9.5 and 10.1 ms)
  const bool ahead = records_ahead(m, kWave);
  if (m.n_ext > 0)
    return ahead ? launch(std::true_type{}, std::true_type{})
                 : launch(std::true_type{}, std::false_type{});
  return ahead ? launch(std::false_type{}, std::true_type{})
               : launch(std::false_type{}, std::false_type{});
}

}  // namespace zrk
