// Host interface of the integrator kernels (bdf_kernels.h): one launch
// description and the per-family launch / occupancy entry points, whose
// explicit instantiations live in bdf_{wave,team}_{direct,krylov}.hip.
#pragma once

#include <hip/hip_runtime.h>

#include "dev_mech.h"

namespace zrk {

// Variants of the one-wavefront integrator by mechanism size (bdf_size).
enum BdfSize : int {
  kBdfAny,
  kBdfSmall,  // FP32 matrix of two tiles a side at most, records of one iteration
  kBdfTile,   // the Newton matrix is one tile
};

// doubles of the Krylov solver's uniform block (Givens rotations, triangular
// factor, least-squares right side) after the RHS arrays of a team's LDS
constexpr size_t kKryDoubles = 46;

// Column stride of a Newton matrix of N rows: odd, so that neither a column read
// by consecutive lanes nor a row's elements share an LDS bank.
__host__ __device__ constexpr int gj_stride(int N) { return N | 1; }

// Buffers of the published row and column in gj_invert_tiles, by team size.
constexpr int gj_buffers(int W) { return W == 3 ? 2 : 1; }

// Elements of one 16 x 16 operand tile in LDS (gj_place).
constexpr int kGjTile = 4 * 68;

// LDS elements of gj_invert_tiles for an N x N matrix: the published columns
// and rows, D^-1 as a left and as a right operand, and the diagonal tile on its
// way to gj_invert16.
__host__ __device__ constexpr int gj_lds_elems(int N, int W) {
  return (2 * gj_buffers(W) * ((N + 15) >> 4) + 2) * kGjTile + 16 * 20;
}

// LDS bytes of a team's matrix region: the (nsp+1) x (nsp+1) FP32 matrix (column stride
// gj_stride) or what the blocked inverse publishes while the matrix is in registers,
// padded to 16 bytes; FP64 teams keep theirs in device memory.
__host__ __device__ constexpr size_t team_matrix_lds_bytes(int nsp, size_t mt, int W) {
  const int N = nsp + 1;
  if (mt != sizeof(float)) return 0;
  const size_t gj = (size_t)gj_lds_elems(N, W) * mt, mat = (size_t)N * gj_stride(N) * mt;
  return ((gj > mat ? gj : mat) + 15) & ~(size_t)15;
}

// Doubles of the RHS arrays C[nsp+1], G[nsp+1], rop[nstep+1].
__host__ __device__ constexpr size_t rhs_doubles(int nsp, int nstep) {
  return (size_t)(2 * (nsp + 1) + nstep + 1);
}

// LDS of a one-wavefront reactor after its CvUni, in bytes from there: the matrix of
// element size mt (FP32: column stride gj_stride; FP64: nsp + 1), the Jacobian's column
// factors (kNP doubles), the RHS arrays (rhs bytes) and, for kIter, the Krylov block.
// The FP32 matrix's blocked inverse publishes from the matrix's place on, over the
// column factors and the RHS arrays, none of which outlive a Jacobian or a right-hand
// side; its zero-pivot flag lies behind both.  (With a region of its own a reactor of 40
// species and 600 reactions took 21,192 bytes of LDS instead of 17,952, and 1,792
// instead of 2,048 reactors were in flight.)
struct WaveLds {
  size_t t2l, rhs, flag, kry, end;
};
__host__ __device__ constexpr WaveLds wave_lds(int nsp, size_t mt, size_t rhs) {
  const int N = nsp + 1;
  const bool f32 = mt == sizeof(float);
  WaveLds l{};
  l.t2l = ((size_t)N * (f32 ? gj_stride(N) : N) * mt + 15) & ~(size_t)15;
  l.rhs = l.t2l + sizeof(double) * kNP;
  l.flag = l.rhs + rhs;
  if (f32 && (size_t)gj_lds_elems(N, 1) * mt > l.flag) l.flag = (size_t)gj_lds_elems(N, 1) * mt;
  l.flag = (l.flag + 7) & ~(size_t)7;
  l.kry = l.flag + (f32 ? sizeof(double) : 0);
  l.end = l.kry;
  return l;
}

struct BdfLaunch {
  const DevMech& m;
  const BdfOpts& o;
  int n;
  double dt;
  const double* dts;
  double *T, *P, *Y;
  int stride;
  int *nsteps, *stats;
  const int* order;
  unsigned int* counter;
  double* jscratch;
  int grid;
  size_t lds;
  hipStream_t st;
};

template <bool kIter>
hipError_t launch_bdf_wave(const BdfLaunch& a, bool ext, bool f32, BdfSize size);
template <bool kIter>
hipError_t launch_bdf_team(const BdfLaunch& a, bool ext, int W, size_t slot, bool f32);
template <bool kIter>
int resident_bdf_wave(bool ext, bool f32, BdfSize size, size_t lds);
template <bool kIter>
int resident_bdf_team(bool ext, int W, size_t lds, bool f32);

inline size_t max_lds_per_block() {
  int dev = 0, v = 0;
  if (hipGetDevice(&dev) != hipSuccess) return 0;
  if (hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess)
    return 0;
  return (size_t)v;
}

template <class K>
inline int resident_blocks(K kernel, int threads, size_t lds) {
  int dev = 0, ncu = 0, per_cu = 0;
  if (lds > max_lds_per_block()) return 0;
  if (hipGetDevice(&dev) != hipSuccess) return 0;
  if (hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
    return 0;
  (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, threads, lds) != hipSuccess)
    return 0;
  return ncu * (per_cu > 0 ? per_cu : 1);
}


}  // namespace zrk
