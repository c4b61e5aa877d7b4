// One block step of a Householder update on a panel's targets (gfx950),
//   C <- (I - V T V^T)^T C = C - V (T^T (V^T C))
// with V rows x w unit lower trapezoidal (w <= 32) and T w x w upper
// triangular: the larfb of util.cpp:421-443 (side 'L', trans 'T', forward,
// columnwise), one launch for all targets of a batch of panels.
//
// Bound by C's traffic: 4 w flops a value where 16 bytes move at least once.  So C
// is read once and written once: a workgroup holds all rows of 16 columns in
// registers, the 16-row tiles dealt to its waves, as the right operand of V^T C
// and as the accumulators of the update alike.  (As two GEMMs C was read twice,
// Y made a round through memory, and long sums over few tiles had to be split:
// 64^3, 640 steps of 106 GB of C in all: 98.8 -> 50.3 ms; 33^3 16.4 -> 5.5 ms;
// 2-D 128^2 2.57 -> 0.79 ms.)  Forms of 128 rows and more move 2.1-2.4 TB/s of
// C: a workgroup waits for memory twice and at three barriers, with 3-7 of
// them on a CU.  32 columns a workgroup, which halve V's reads, took as long.
//
// A lane (k4 = lane / 16, c16 = lane % 16) holds rows 4 k4 .. 4 k4 + 3 of a tile
// in column c16, which are 16-byte loads along the column.  The contraction over
// rows may take them in any order that V follows; the result rows of the matrix
// instruction (k4 + 4 c in accumulator c for FP64, 4 k4 + c for FP32) are made to
// be these by the order in which V's rows enter the second product.
#include <algorithm>

#include "kcommon.hpp"
#include "descs.hpp"
#include "launch.hpp"

namespace spq {

constexpr int kLB = 32, kLC = 16;  // reflectors of a block, columns of a workgroup

// four consecutive entries (the entries' own alignment)
template <typename T>
__device__ __forceinline__ void load4(gptr<T> p, T (&v)[4]) {
  typedef T V4 __attribute__((ext_vector_type(4), aligned(sizeof(T))));
  const V4 x = *(const __attribute__((address_space(1))) V4*)p;
#pragma unroll
  for (int q = 0; q < 4; ++q) v[q] = x[q];
}
template <typename T>
__device__ __forceinline__ void store4(gmut<T> p, const T (&v)[4]) {
  typedef T V4 __attribute__((ext_vector_type(4), aligned(sizeof(T))));
  *(__attribute__((address_space(1))) V4*)p = V4{v[0], v[1], v[2], v[3]};
}

template <typename T, int NW, int RT>  // waves, row tiles per wave
__global__ __launch_bounds__(NW * kWave) void k_larfb(const LarfbDesc<T>* __restrict__ descs,
                                                      const int* __restrict__ tstart, int nd) {
  using M = Mfma<T>;
  using V4 = typename M::v4;
  constexpr int LD = kLC + 1;
  __shared__ T Ys[NW][kLB][LD];
  __shared__ T Zs[kLB][LD];
  const int p = find_owner(tstart, nd, blockIdx.x);
  const LarfbDesc<T> d = descs[p];
  const int tid = threadIdx.x, lane = tid & (kWave - 1), c16 = lane & 15, k4 = lane >> 4;
  const int wv = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int j = (blockIdx.x - tstart[p]) * kLC + c16, rows = d.rows, w = d.w;
  const bool in = j < d.cols;
  const gmut<T> C = to_global_mut(d.C) + (int64_t)min(j, d.cols - 1) * d.ldc + 4 * k4;
  T c[RT][4];
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    const int rb = (t * NW + wv) * 16;
    if (rb + 16 <= rows) {
      load4<T>(C + rb, c[t]);
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q) c[t][q] = rb + 4 * k4 + q < rows ? C[rb + q] : T(0);
    }
  }
  // ---- Y = V^T C, this wave's rows
  const gptr<T> V = to_global(d.V);
  V4 y[2] = {V4{0, 0, 0, 0}, V4{0, 0, 0, 0}};
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    const int rb = (t * NW + wv) * 16;
    if (rb < rows) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int i = 16 * h + c16;
        if (16 * h < w) {
          const gptr<T> v = V + (int64_t)min(i, w - 1) * d.ldv + rb + 4 * k4;
          T a[4];
          if (rb + 16 <= rows) {
            load4<T>(v, a);
          } else {
#pragma unroll
            for (int q = 0; q < 4; ++q) a[q] = rb + 4 * k4 + q < rows ? v[q] : T(0);
          }
          if (rb < kLB || w < kLB) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              const int r = rb + 4 * k4 + q;
              a[q] = i < w ? (r > i ? a[q] : (r == i ? T(1) : T(0))) : T(0);
            }
          }
#pragma unroll
          for (int q = 0; q < 4; ++q) y[h] = M::mac(a[q], c[t][q], y[h]);
        }
      }
    }
  }
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int q = 0; q < 4; ++q) Ys[wv][16 * h + M::row(k4, q)][c16] = y[h][q];
  __syncthreads();
  // ---- Z = -T^T Y, 16 rows by each of two waves
  if (NW > 4) {
    for (int e = tid; e < kLB * kLC; e += NW * kWave) {
      const int l = e / kLC, cc = e % kLC;
      T s = Ys[0][l][cc];
#pragma unroll
      for (int q = 1; q < NW; ++q) s += Ys[q][l][cc];
      Ys[0][l][cc] = s;
    }
    __syncthreads();
  }
  if (wv < 2) {
    V4 z = V4{0, 0, 0, 0};
    const int i = 16 * wv + c16;
#pragma unroll
    for (int kk = 0; kk < kLB / 4; ++kk) {
      if ((kk < 4 || wv == 1) && 4 * kk < w) {
        const int l = 4 * kk + k4;
        T s = Ys[0][l][c16];
        if (NW <= 4) {
#pragma unroll
          for (int q = 1; q < NW; ++q) s += Ys[q][l][c16];
        }
        const T tt = to_global(d.Tb)[i * kLB + l];
        z = M::mac(l <= i && i < w ? tt : T(0), s, z);
      }
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) Zs[16 * wv + M::row(k4, q)][c16] = -z[q];
  }
  __syncthreads();
  // ---- C += V Z
  // row i of the instruction's result is row `pi` of the tile
  const int pi = sizeof(T) == 8 ? 4 * (c16 & 3) + (c16 >> 2) : c16;
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    const int rb = (t * NW + wv) * 16;
    if (rb < rows) {
      V4 acc = V4{c[t][0], c[t][1], c[t][2], c[t][3]};
      const int r = rb + pi;
      const gptr<T> v = V + min(r, rows - 1);
#pragma unroll
      for (int h = 0; h < 2; ++h)
        if (16 * h < w) {
#pragma unroll
          for (int kk = 0; kk < 4; ++kk) {
            const int i = 16 * h + 4 * k4 + kk;
            T a = v[(int64_t)min(i, w - 1) * d.ldv];
            if (rb < kLB || w < kLB) a = i < w ? (r > i ? a : (r == i ? T(1) : T(0))) : T(0);
            acc = M::mac(a, Zs[i][c16], acc);
          }
        }
      if (in) {
        if (rb + 16 <= rows) {
          const T o[4] = {acc[0], acc[1], acc[2], acc[3]};
          store4<T>(C + rb, o);
        } else {
#pragma unroll
          for (int q = 0; q < 4; ++q)
            if (rb + 4 * k4 + q < rows) C[rb + q] = acc[q];
        }
      }
    }
  }
}

namespace {
struct LarfbForm { int nw, rt; };
constexpr LarfbForm kLarfbForms[] = {{4, 1}, {4, 2}, {4, 4}, {4, 6}, {4, 8}, {8, 6}, {8, 8}, {16, 6}, {16, 8}};
constexpr int kNumLarfb = sizeof(kLarfbForms) / sizeof(kLarfbForms[0]);
}  // namespace
int larfb_forms() { return kNumLarfb; }
int larfb_form_rows(int f) { return 16 * kLarfbForms[f].nw * kLarfbForms[f].rt; }
int larfb_tiles(int cols) { return (cols + kLC - 1) / kLC; }
template <typename T>
void launch_larfb(hipStream_t s, const LarfbDesc<T>* d, const int* tstart, int nd, int ntiles, int form) {
  if (nd <= 0 || ntiles <= 0) return;
  auto go = [&](auto nw, auto rt) {
    constexpr int NW = decltype(nw)::value, RT = decltype(rt)::value;
    hipLaunchKernelGGL((k_larfb<T, NW, RT>), dim3(ntiles), dim3(NW * kWave), 0, s, d, tstart, nd);
  };
#define SPQ_FORM(f)                                                                                             \
  case f:                                                                                                       \
    go(std::integral_constant<int, kLarfbForms[f].nw>{}, std::integral_constant<int, kLarfbForms[f].rt>{});     \
    break;
  switch (form) {
    SPQ_FORM(0) SPQ_FORM(1) SPQ_FORM(2) SPQ_FORM(3) SPQ_FORM(4) SPQ_FORM(5) SPQ_FORM(6) SPQ_FORM(7) SPQ_FORM(8)
  }
#undef SPQ_FORM
}
template void launch_larfb<double>(hipStream_t, const LarfbDesc<double>*, const int*, int, int, int);
template void launch_larfb<float>(hipStream_t, const LarfbDesc<float>*, const int*, int, int, int);

}  // namespace spq
