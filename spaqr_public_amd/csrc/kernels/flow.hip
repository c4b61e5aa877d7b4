// The preconditioner apply of a tree as one dataflow kernel (gfx950).
//
// The tape is a chain of 50-250 dependent steps, most of a few small ops (the
// elimination waves of a level: 1-24 ops of 250-500 rows), so an apply is bound
// by what lies between two dependent ops, not by the factors' bytes: cold
// instructions and descriptors, first touches of the factors (2-4 us from HBM),
// and the hand-over of x.  Here workgroups draw (op, part) pairs from a ticket
// counter in tape order and fetch descriptors, row lists and the first tile of
// both factors while the op's inputs are still being made.
//
// x is in single-assignment form: every op writes its rows to places of their
// own, so an input is a list of segments of earlier outputs and nothing is
// overwritten, merged or split.  A place holds the value's complement and is
// zero until then: consumers poll the values themselves, which costs one trip
// through memory per link where store, counter and load cost three.
//
// Reflector products are applied whole: with W = V T^T (T the k x k compact-WY
// factor, formed once per factorization) H^T x = x - W (V^T x) and H x = x - V
// (W^T x), two matrix-vector products and one exchange whatever k is, where
// 32-column blocks with their 32 x 32 T factors need an exchange per block.
//
// One link of the chain (an op of one part) takes 3-4 us: 0.6-1 us from the
// last store to the polled value, 0.6 us for y, 0.7 us for x, the rest fetching
// what could not be fetched ahead; a part that exchanges sums 1.2 us more; a
// triangular block of 32 rows 0.9 us (3.3 us as k_bwdr's block step).  Whole
// applies, against one kernel per stage with a graph around them: 2-D 64^2 472
// -> 146 us, 3-D 40^3 2.9 -> 0.8 ms, 52^3 5.3 -> 1.6 ms (the first with the launches
// of launch_flow_begin; 165 us inside a graph of seven nodes).
//
// Progress: a workgroup waits only for ops with earlier tickets and for the
// other parts of its own op.  Tickets are drawn when a workgroup is running
// and past its last wait, so the unfinished op with the earliest tickets always
// has all its parts running (an op has at most kFlowMaxParts parts, fewer than
// the resident workgroups of the grid).  Every wait is bounded all the same:
// one that gives up sets the error flag and the kernel ends.
#include <limits.h>

#include <algorithm>
#include <type_traits>

#include "kcommon.hpp"
#include "descs.hpp"
#include "launch.hpp"

namespace spq {

constexpr int kFT = 256, kFW = kFT / kWave;
constexpr int kFNB = 32;
constexpr int kFlowTouch = 8;

// *p through the scalar cache (p uniform, *p constant during the kernel)
template <typename S>
__device__ __forceinline__ S scalar_get(const S* p) {
  static_assert(sizeof(S) % 4 == 0, "");
  const auto q = (const __attribute__((address_space(4))) int*)p;
  int w[sizeof(S) / 4];
#pragma unroll
  for (size_t i = 0; i < sizeof(S) / 4; ++i) w[i] = q[i];
  S s;
  __builtin_memcpy(&s, w, sizeof(S));
  return s;
}

// Buffer view of a column-major matrix of `cols` columns of `rows` rows: reads
// past its last entry give zero.
template <typename T>
struct Tiles {
  __amdgpu_buffer_rsrc_t rsrc;
  unsigned step;
  __device__ __forceinline__ Tiles(const T* M, int ld, int rows, int cols)
      : rsrc(__builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(M), 0,
                                               ((unsigned)(cols - 1) * (unsigned)ld + (unsigned)rows) * sizeof(T),
                                               0x00027000u)),
        step((unsigned)ld * (unsigned)sizeof(T)) {}
  // 32 columns from c0 on, one row in each lane: the row's offset stays in one
  // register, the columns follow as scalar offsets (columns past k repeat the
  // last one)
  __device__ __forceinline__ void rows32(int row, int c0, int k, T (&v)[kFNB]) const {
    const unsigned off = (unsigned)row * (unsigned)sizeof(T);
    int w = __builtin_amdgcn_readfirstlane(k - c0);
    unsigned so = __builtin_amdgcn_readfirstlane((int)((unsigned)c0 * step));
#pragma unroll
    for (int u = 0; u < kFNB; ++u) {
      if constexpr (sizeof(T) == 8) {
        const auto b = __builtin_amdgcn_raw_buffer_load_b64(rsrc, off, so, 0);
        __builtin_memcpy(&v[u], &b, sizeof(T));
      } else {
        const auto b = __builtin_amdgcn_raw_buffer_load_b32(rsrc, off, so, 0);
        __builtin_memcpy(&v[u], &b, sizeof(T));
      }
      so += u + 1 < w ? step : 0u;
      asm volatile("" : "+s"(so), "+s"(w));  // one offset at a time, not 32 kept in registers
    }
  }
  // 32 consecutive entries of one column in each lane, from row r0 on (16-byte
  // loads, which need the entries' own alignment only)
  __device__ __forceinline__ void col32(int col, int r0, T (&v)[kFNB]) const {
    const unsigned off = (unsigned)col * step + (unsigned)r0 * (unsigned)sizeof(T);
    constexpr int per = 16 / sizeof(T);
#pragma unroll
    for (int u = 0; u < kFNB; u += per) {
      const auto b = __builtin_amdgcn_raw_buffer_load_b128(rsrc, off + u * (unsigned)sizeof(T), 0, 0);
      __builtin_memcpy(&v[u], &b, 16);
    }
  }
};

// Entries of a tile outside a trapezoid become zero, one after the other (32
// lane masks at once do not fit the SGPRs).  row_edge: a row whose diagonal
// lies in column e of its tile, V unit lower trapezoidal, W lower trapezoidal.
// col_edge: 32 entries of a column whose diagonal is entry e, with n rows left.
template <typename T>
__device__ __forceinline__ void row_edge(T (&v)[kFNB], int unit, int e) {
#pragma unroll
  for (int u = 0; u < kFNB; ++u) {
    const T dg = unit ? T(1) : v[u];
    v[u] = e > u ? v[u] : (e == u ? dg : T(0));
    asm volatile("" : "+v"(v[u]), "+v"(e));
  }
}
template <typename T>
__device__ __forceinline__ void col_edge(T (&v)[kFNB], int unit, int e, int n) {
#pragma unroll
  for (int u = 0; u < kFNB; ++u) {
    const T dg = unit ? T(1) : v[u];
    v[u] = u < n ? (u > e ? v[u] : (u == e ? dg : T(0))) : T(0);
    asm volatile("" : "+v"(v[u]), "+v"(e), "+v"(n));
  }
}
// sum of v[u] x[u], x in LDS (32 values, 16-byte aligned)
template <typename T>
__device__ __forceinline__ T dot32(const T (&v)[kFNB], const T* x) {
  T s4[4] = {T(0), T(0), T(0), T(0)};
#pragma unroll
  for (int u = 0; u < kFNB; ++u) s4[u & 3] = fma(v[u], x[u], s4[u & 3]);
  return (s4[0] + s4[1]) + (s4[2] + s4[3]);
}

// row l of diagonal block b, as k_flow_diag leaves it
template <typename T>
__device__ __forceinline__ void diag_load(const T* D, int b, int l, T (&v)[kFNB]) {
  constexpr int per = 16 / sizeof(T);
  const auto p = (const __attribute__((address_space(1))) char*)(D + (int64_t)b * kFNB * kFNB) + l * 16;
  typedef float f4 __attribute__((ext_vector_type(4)));
#pragma unroll
  for (int u = 0; u < kFNB; u += per) {
    const f4 q = *(const __attribute__((address_space(1))) f4*)(p + u / per * (kFNB * 16));
    __builtin_memcpy(&v[u], &q, 16);
  }
}
template <typename T>
__device__ __forceinline__ void zero32(T (&v)[kFNB]) {
#pragma unroll
  for (int u = 0; u < kFNB; ++u) v[u] = T(0);
}

// the value in place `at` of x, once it is there
template <typename T>
__device__ __forceinline__ T flow_poll(const T* X, int at, int* err) {
  using B = typename Bits<sizeof(T)>::type;
  const gmut<B> p = to_global_mut((B*)const_cast<T*>(X)) + at;
  unsigned int spins = 0;
  B b;
  while ((b = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) == 0) {
    __builtin_amdgcn_s_sleep(2);
    if ((++spins & 255u) == 0 &&
        __hip_atomic_load(to_global_mut(err), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0)
      break;
    if (spins > (1u << 20)) {
      __hip_atomic_fetch_or(to_global_mut(err), 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      break;
    }
  }
  b = ~b;
  T v;
  __builtin_memcpy(&v, &b, sizeof(T));
  return v;
}

// A column half of 32 entries in each lane (col32) makes y a sum along the
// lane's registers and one exchange between the half waves, where a row in each
// lane needs a 32-way reduction over the wave (2.4 -> 0.6 us an op, masks at the
// trapezoids' edges included: they are applied while x is still awaited).
// Two workgroups a CU: bounded to three, FP64 spills 109 registers, and with as
// many more parts to fill them an apply is 1.3-1.5x slower (2D n = 64: 147 -> 189
// us, 3D n = 52: 1575 -> 2222 us; bound and part count were changed together).
template <typename T>
__global__ __launch_bounds__(kFT, 2) void k_flow(const FlowArgs<T> P) {
  constexpr int KM = kFlowMaxK;
  __shared__ __align__(16) T xs[KM + kWave], ys[KM + kFNB], ps[4 * 128];  // a tile reads on past the rows or k
  __shared__ __align__(16) T xw[kFW][kWave];
  __shared__ int sbase[kFlowMaxSegs + 1], soff[kFlowMaxSegs + 1];
  __shared__ int s_next;
  T* const X = P.x;
  if (threadIdx.x == 0)
    s_next = (int)__hip_atomic_fetch_add(to_global_mut(P.ctl), 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  for (;;) {
    const int ticket = __builtin_amdgcn_readfirstlane(s_next);
    if (ticket >= P.nparts) break;  // every later ticket is past the end too
    // the lane's constants are formed anew for each op: kept over the loop,
    // its masks and addresses do not fit the registers
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int lane = tid & (kWave - 1);
    const int w = __builtin_amdgcn_readfirstlane(tid / kWave);
    const FlowOp<T> d = scalar_get(P.parts + ticket);
    const int g = d.g, nwg = d.nwg;
    const int k = d.k, nb = (k + kFNB - 1) / kFNB;
    // draws the next ticket (after the last wait for the op's other parts)
    auto draw = [&] {
      if (tid == 0)
        s_next = (int)__hip_atomic_fetch_add(to_global_mut(P.ctl), 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    // table of the op's input segments, in LDS
    auto seg_table_begin = [&] {
      if (w == 0) {
        int carry = 0;
        for (int s0 = 0; s0 < d.nseg; s0 += kWave) {
          const int s = s0 + lane;
          int len = 0;
          if (s < d.nseg) {
            const FlowSeg sg = P.segs[d.seg0 + s];
            len = sg.len;
            soff[s] = sg.off;
          }
          int v = len;
#pragma unroll
          for (int o = 1; o < kWave; o <<= 1) {
            const int u = __shfl_up(v, o, kWave);
            if (lane >= o) v += u;
          }
          if (s < d.nseg) sbase[s] = carry + v - len;
          carry += __shfl(v, kWave - 1, kWave);
        }
      }
    };
    // place of input row i
    auto place = [&](int i) {
      int lo = 0, hi = d.nseg - 1;
      while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (sbase[mid] <= i) lo = mid;
        else hi = mid - 1;
      }
      return soff[lo] + i - sbase[lo];
    };

    if (d.type == kFlowWY) {
      T va[kFNB], vb[kFNB];
      const Tiles<T> A(d.A, d.lda, d.m, k), B(d.B, d.ldb, d.m, k);
      const int rp = d.rows_per;  // rows per part
      const int r0 = g * rp, rows = min(d.m - r0, rp), nc = (rows + kWave - 1) / kWave;
      // y = A^T x: waves over column blocks, over row chunks where there are
      // few blocks; (b, c) is block b of row chunk c, of which a lane holds
      // half a column
      const bool bycol = nb >= 3;
      const int ba = bycol ? w : 0, bs = bycol ? kFW : 1, ca = bycol ? 0 : w, cs = bycol ? 1 : kFW;
      const int half = (lane >> 5) * kFNB;
      auto load_a = [&](int b, int c) {
        const int i = r0 + c * kWave + half, j = b * kFNB + (lane & (kFNB - 1));
        A.col32(min(j, k - 1), i, va);
        if (r0 + c * kWave < (b + 1) * kFNB || r0 + (c + 1) * kWave > d.m) col_edge(va, d.unit_a, j - i, d.m - i);
      };
      // first chunk of this wave that reaches into block b
      auto chunk0 = [&](int b) {
        const int lo = (b * kFNB - r0) >> 6;
        return lo <= ca ? ca : (bycol ? lo : ca + ((lo - ca + kFW - 1) & ~(kFW - 1)));
      };
      // x -= B y: waves over row chunks, over column blocks too where there
      // are few chunks
      const int cw = nc >= 3 ? kFW : (nc == 2 ? 2 : 1);  // waves side by side over the chunks
      const int cfirst = w % cw, bfirst = w / cw, bstep = kFW / cw;
      auto blocks = [&](int c) { return min(nb, (r0 + c * kWave + kWave - 1) / kFNB + 1); };
      auto load_b = [&](int b, int c) {
        const int i = r0 + c * kWave + lane;
        B.rows32(min(i, d.m - 1), b * kFNB, k, vb);
        if (r0 + c * kWave < (b + 1) * kFNB) row_edge(vb, d.unit_b, i - b * kFNB);
      };
      seg_table_begin();
      // the first tiles of both, on their way while x is made (some tile in
      // any case: a tile not loaded would stay live around the loop)
      load_b(min(bfirst, nb - 1), min(cfirst, nc - 1));
      load_a(min(ba, nb - 1), min(chunk0(min(ba, nb - 1)), nc - 1));
      if (tid < kFNB) ys[k + tid] = T(0);
      __syncthreads();
      for (int r = tid; r < nc * kWave; r += kFT) xs[r] = r < rows ? flow_poll(X, place(r0 + r), P.err) : T(0);
      __syncthreads();
      if (nwg == 1) draw();
      // ---- y = A^T x, the next tile on its way after each
      {
        int b = ba, c = ba < nb ? chunk0(ba) : nc;
        auto put = [&](T y) {
          if (lane < kFNB) {
            if (!bycol) ps[(w * 2 + b) * kFNB + lane] = y;
            else if (b * kFNB + lane < k) ys[b * kFNB + lane] = y;
          }
        };
        if (c < nc) {
          T acc = T(0);
          for (;;) {
            acc += dot32(va, xs + c * kWave + half);
            c += cs;
            if (c >= nc) {
              put(acc + lane_xor<32>(acc));
              b += bs;
              if (b >= nb) break;
              c = chunk0(b);
              if (c >= nc) break;
              acc = T(0);
            }
            load_a(b, c);
          }
        }
        for (; b < nb; b += bs) put(T(0));  // blocks below these rows
      }
      __syncthreads();
      if (!bycol) {
        if (tid < k) {
          T y = T(0);
#pragma unroll
          for (int q = 0; q < kFW; ++q) y += ps[(q * 2 + tid / kFNB) * kFNB + (tid & (kFNB - 1))];
          ys[tid] = y;
        }
        if (nwg == 1) __syncthreads();
      }
      if (nwg > 1) {
        // the sum over the op's parts, in part order, in every part (each
        // thread its own columns)
        T* const sl = d.slots;
        for (int c = tid; c < k; c += kFT) slot_put(sl, (int64_t)g * k + c, true, ys[c]);
        for (int c = tid; c < k; c += kFT) ys[c] = slot_sum<T, 8>(sl + c, k, nwg, nwg, P.err);
        __syncthreads();
        draw();
      }
      // ---- x - B y
      if (cfirst < nc) {
        int c = cfirst, b = bfirst, nbc = blocks(c);
        T s = T(0);
        for (;;) {
          if (b < nbc) s += dot32(vb, ys + b * kFNB);
          b += bstep;
          if (b >= nbc) {
            const int r = c * kWave + lane;
            if (bstep > 1) ps[bfirst * 128 + r] = s;
            else slot_put(X, d.out + r0 + r, r < rows, xs[r] - s);
            c += cw;
            if (c >= nc) break;
            b = bfirst;
            nbc = blocks(c);
            s = T(0);
          }
          load_b(b, c);
        }
      }
      if (bstep > 1) {
        __syncthreads();
        if (tid < rows) {
          T s = T(0);
          for (int q = 0; q < bstep; ++q) s += ps[q * 128 + tid];
          slot_put(X, d.out + r0 + tid, true, xs[tid] - s);
        }
      }
    } else if (d.type == kFlowPull) {
      // ---- x_n - sum over blocks A_c^T x_c: this part's 32 rows of n are
      // columns of the blocks, whose tiles of 64 rows are dealt to the waves
      const int j0 = g * kFNB, nt = d.nblk, half = (lane >> 5) * kFNB;
      T va[kFNB], acc = T(0);
      FlowBlk<T> q;
      auto load = [&](int t) {
        q = scalar_get(P.blks + d.blk0 + t);
        Tiles<T>(q.A, q.ld, q.n, d.m).col32(min(j0 + (lane & (kFNB - 1)), d.m - 1), half, va);
        if (q.n < kWave) col_edge(va, 0, -1, q.n - half);
      };
      load(min(w, nt - 1));
      seg_table_begin();
      __syncthreads();
      for (int t = w; t < nt;) {
        xw[w][lane] = lane < q.n ? flow_poll(X, q.off + lane, P.err) : T(0);
        wave_sync();
        acc += dot32(va, xw[w] + half);
        wave_sync();
        t += kFW;
        if (t >= nt) break;
        load(t);
      }
      acc += lane_xor<32>(acc);
      if (lane < kFNB) ps[w * kFNB + lane] = acc;
      const int j = j0 + tid;
      T xj = T(0);
      if (tid < kFNB && j < d.m) xj = flow_poll(X, place(j), P.err);
      draw();
      __syncthreads();
      if (tid < kFNB && j < d.m) {
        T s = T(0);
#pragma unroll
        for (int v = 0; v < kFW; ++v) s += ps[v * kFNB + tid];
        slot_put(X, d.out + j, true, xj - s);
      }
    } else {
      // ---- triangular ops: x_c <- R^{-1} (x_c - sum_n A_n x_n), or transposed
      // x_c <- R^{-T} x_c.  The blocks' tiles of 32 columns are dealt to the
      // parts; part 0 holds x_c and solves.
      const bool tr = d.type == kFlowSolveT;
      const Tiles<T> R(d.A, d.lda, k, k);
      const int nc = (k + kWave - 1) / kWave;
      const int t0 = (int)((int64_t)g * d.nblk / nwg), t1 = (int)((int64_t)(g + 1) * d.nblk / nwg);
      const int cw = nc >= 3 ? kFW : (nc == 2 ? 2 : 1), cfirst = w % cw, jfirst = w / cw, jstep = kFW / cw;
      // the first tile, on its way while x is made
      T va[kFNB];
      FlowBlk<T> q{};
      auto load = [&](int t, int c) {
        q = scalar_get(P.blks + d.blk0 + t);
        Tiles<T>(q.A, q.ld, k, q.n).rows32(min(c * kWave + lane, k - 1), 0, q.n, va);
      };
      if (t0 + jfirst < t1 && cfirst < nc) {
        load(t0 + jfirst, cfirst);
      } else {
        zero32(va);
      }
      // and, in the part that solves, R's lines into this die's cache
      T touch[kFlowTouch];
      const int lines = (k * (int)sizeof(T) + 127) / 128;
#pragma unroll
      for (int u = 0; u < kFlowTouch; ++u) {
        const int q2 = tid + u * kFT, c = q2 / lines, l = q2 - c * lines;
        touch[u] = T(0);
        if (g == 0 && c < k && l * 128 <= c * (int)sizeof(T))
          touch[u] = to_global(d.A)[(int64_t)c * d.lda + l * (128 / (int)sizeof(T))];
      }
      if (tid < kFNB) xs[k + tid] = T(0);
      seg_table_begin();
      __syncthreads();
      if (t0 + jfirst < t1 && cfirst < nc) {
        int t = t0 + jfirst, c = cfirst;
        T s = T(0);
        for (;;) {
          if (lane < kFNB) xw[w][lane] = lane < q.n ? flow_poll(X, q.off + lane, P.err) : T(0);
          wave_sync();
          s += dot32(va, xw[w]);
          wave_sync();
          t += jstep;
          if (t >= t1) {
            const int r = c * kWave + lane;
            if (jstep == 1) ys[r] = s;
            else ps[jfirst * 128 + r] = s;
            s = T(0);
            t = t0 + jfirst;
            c += cw;
            if (c >= nc) break;
          }
          load(t, c);
        }
      }
#pragma unroll
      for (int u = 0; u < kFlowTouch; ++u) asm volatile("" ::"v"(touch[u]));
      if (g == 0)
        for (int r = tid; r < k; r += kFT) xs[r] = flow_poll(X, place(r), P.err);
      __syncthreads();
      if (jstep > 1) {
        if (tid < k) {
          T s = T(0);
          for (int v = 0; v < jstep; ++v)
            if (t0 + v < t1) s += ps[v * 128 + tid];
          ys[tid] = s;
        }
        __syncthreads();
      } else if (t0 == t1) {
        for (int r = tid; r < k; r += kFT) ys[r] = T(0);
      }
      if (g != 0) {
        for (int r = tid; r < k; r += kFT) slot_put(d.slots, (int64_t)g * k + r, true, ys[r]);
        draw();
      } else {
        for (int r = tid; r < k; r += kFT) {
          T s = ys[r];
          if (nwg > 1) s += slot_sum<T, 8>(d.slots + k + r, k, nwg - 1, nwg - 1, P.err);
          xs[r] -= s;
        }
        draw();
        __syncthreads();
        // Blocks of 32 rows from the last (or, transposed, the first).  Wave 0
        // goes from diagonal block to diagonal block, with the update of the
        // next block's rows between; the other waves update the rows after
        // those, a block behind.
        auto solve = [&](auto trans) {
          constexpr bool TR = decltype(trans)::value;
          auto load_rows = [&](int r, int jb, T(&v)[kFNB]) {
            if constexpr (TR) R.col32(max(min(r, k - 1), 0), jb, v);
            else R.rows32(max(min(r, k - 1), 0), jb, k, v);
          };
          const int l = lane & (kFNB - 1), dirn = TR ? kFNB : -kFNB;
          const int first = TR ? 0 : (nb - 1) * kFNB;
          if (w == 0) {
            T dd[kFNB], v[kFNB];
            diag_load(d.B, first / kFNB, l, dd);
            load_rows(first + dirn + l, first, v);  // (clamped when there is one block)
            for (int s = 0; s < nb; ++s) {
              const int jb = first + s * dirn;
              T z = jb + l < k ? xs[jb + l] : T(0);
              if (s > 0) {
                z -= dot32(v, xs + (jb - dirn));
                load_rows(jb + dirn + l, jb, v);
              }
              z *= d.B[(int64_t)nb * kFNB * kFNB + jb + l];
              if constexpr (TR) {
#pragma unroll
                for (int u = 0; u < kFNB; ++u) z = fma(-dd[u], lane_bcast(z, u), z);
              } else {
#pragma unroll
                for (int u = kFNB - 1; u >= 0; --u) z = fma(-dd[u], lane_bcast(z, u), z);
              }
              if (s + 1 < nb) diag_load(d.B, (jb + dirn) / kFNB, l, dd);
              if (lane < min(kFNB, k - jb)) {
                xs[jb + lane] = z;
                slot_put(X, d.out + jb + lane, true, z);
              }
              __syncthreads();
            }
          } else {
            for (int s = 0; s < nb; ++s) {
              const int jb = first + s * dirn;
              // rows past the next block
              const int rl = TR ? jb + 2 * kFNB : 0, rh = TR ? k : jb - kFNB, r0 = rl + tid - kWave;
              T v[kFNB];
              if (rl < rh) load_rows(r0, jb, v);
              else zero32(v);
              __syncthreads();
              if (r0 < rh) xs[r0] -= dot32(v, xs + jb);
#pragma unroll 1
              for (int r = r0 + kFT - kWave; r < rh; r += kFT - kWave) {
                T v2[kFNB];
                load_rows(r, jb, v2);
                xs[r] -= dot32(v2, xs + jb);
              }
            }
          }
        };
        if (tr) solve(std::true_type{});
        else solve(std::false_type{});
      }
    }
    __syncthreads();
  }
}

// Diagonal blocks of R (k x k upper) for the solves of k_flow: row l of block b
// divided by its diagonal, entries the solve does not use (u <= l, or with R^T
// u >= l; rows past k) zero, in 16-byte pieces [u][l]; the reciprocals of the
// diagonal follow the last block.  With z = x / diag a step is z_l -= D[l][u]
// z_u, one multiply-add after a broadcast.
template <typename T>
__global__ __launch_bounds__(kFNB * 8) void k_flow_diag(const FlowDiag<T>* ds, const int* start, int nd) {
  const int i = find_owner(start, nd, blockIdx.x);
  const FlowDiag<T> d = ds[i];
  const int b = blockIdx.x - start[i], nb = (d.k + kFNB - 1) / kFNB;
  constexpr int per = 16 / sizeof(T);
  T* const D = d.D + (int64_t)b * kFNB * kFNB;
  for (int e = threadIdx.x; e < kFNB * kFNB; e += kFNB * 8) {
    const int l = e % kFNB, u = e / kFNB, r = b * kFNB + l, c = b * kFNB + u;
    T v = T(0);
    if (r < d.k && c < d.k && (d.tr ? u < l : u > l))
      v = (d.tr ? d.R[c + (int64_t)r * d.ld] : d.R[r + (int64_t)c * d.ld]) * (T(1) / d.R[r + (int64_t)r * d.ld]);
    D[u / per * (kFNB * per) + l * per + u % per] = v;
  }
  if (threadIdx.x < kFNB) {
    const int r = b * kFNB + threadIdx.x;
    d.D[(int64_t)nb * kFNB * kFNB + r] = r < d.k ? T(1) / d.R[r + (int64_t)r * d.ld] : T(0);
  }
}
size_t flow_diag_elems(int k) { return (size_t)((k + kFNB - 1) / kFNB) * kFNB * (kFNB + 1); }
template <typename T>
void launch_flow_diag(hipStream_t s, const FlowDiag<T>* d, const int* start, int nd, int nblocks) {
  if (nblocks > 0) hipLaunchKernelGGL((k_flow_diag<T>), dim3(nblocks), dim3(kFNB * 8), 0, s, d, start, nd);
}
template void launch_flow_diag<double>(hipStream_t, const FlowDiag<double>*, const int*, int, int);
template void launch_flow_diag<float>(hipStream_t, const FlowDiag<float>*, const int*, int, int);

template <typename T>
int flow_capacity() {
  int per_cu = 0, dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess) return 0;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, (const void*)k_flow<T>, kFT, 0) != hipSuccess) return 0;
  return per_cu * cus;
}
template <typename T>
void launch_flow(hipStream_t s, const FlowArgs<T>& a, int grid) {
  if (a.nparts <= 0 || grid <= 0) return;
  hipLaunchKernelGGL((k_flow<T>), dim3(std::min(grid, a.nparts)), dim3(kFT), 0, s, a);
}
template int flow_capacity<double>();
template int flow_capacity<float>();
template void launch_flow<double>(hipStream_t, const FlowArgs<double>&, int);
template void launch_flow<float>(hipStream_t, const FlowArgs<float>&, int);

template <typename T>
__global__ __launch_bounds__(256) void k_flow_begin(const int* __restrict__ src, int n, const double* __restrict__ b,
                                                    T* x, int nz, FlowClear c) {
  const int64_t i0 = (int64_t)blockIdx.x * 256 + threadIdx.x, step = (int64_t)gridDim.x * 256;
  for (int64_t i = i0; i < n + nz; i += step) slot_put(x, i, true, i < n ? (T)b[src ? src[i] : i] : T(0));
#pragma unroll
  for (int q = 0; q < 5; ++q)
    for (int64_t i = i0; i < c.n[q]; i += step) c.p[q][i] = 0;
}
template <typename T, typename D>
__global__ __launch_bounds__(256) void k_flow_out(const int* __restrict__ loc, int n, const T* __restrict__ x,
                                                  const int* __restrict__ dst, D* __restrict__ y) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  using B = typename Bits<sizeof(T)>::type;
  const B b = ~((const B*)x)[loc[i]];
  T v;
  __builtin_memcpy(&v, &b, sizeof(T));
  y[dst ? dst[i] : i] = (D)v;
}
// values of places of one x in places of another
template <typename T, typename D>
__global__ __launch_bounds__(256) void k_flow_cvt(const int* __restrict__ loc, int n, const T* __restrict__ x, D* y,
                                                  int at) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  using B = typename Bits<sizeof(T)>::type;
  const B b = ~((const B*)x)[loc[i]];
  T v;
  __builtin_memcpy(&v, &b, sizeof(T));
  slot_put(y, (int64_t)at + i, true, (D)v);
}
template <typename T>
void launch_flow_begin(hipStream_t s, const int* src, int n, const double* b, T* x, int nz, const FlowClear& c) {
  int64_t most = n + nz;
  for (int64_t w : c.n) most = std::max(most, w);
  if (most <= 0) return;
  hipLaunchKernelGGL((k_flow_begin<T>), dim3(std::min<int64_t>((most + 255) / 256, 2048)), dim3(256), 0, s, src, n, b, x,
                     nz, c);
}
template <typename T>
void launch_flow_out(hipStream_t s, const int* loc, int n, const T* x, const int* dst, double* y) {
  if (n > 0) hipLaunchKernelGGL((k_flow_out<T, double>), dim3((n + 255) / 256), dim3(256), 0, s, loc, n, x, dst, y);
}
template <typename T, typename D>
void launch_flow_cvt(hipStream_t s, const int* loc, int n, const T* x, D* y, int at) {
  if (n > 0) hipLaunchKernelGGL((k_flow_cvt<T, D>), dim3((n + 255) / 256), dim3(256), 0, s, loc, n, x, y, at);
}
template void launch_flow_begin<double>(hipStream_t, const int*, int, const double*, double*, int, const FlowClear&);
template void launch_flow_begin<float>(hipStream_t, const int*, int, const double*, float*, int, const FlowClear&);
template void launch_flow_out<double>(hipStream_t, const int*, int, const double*, const int*, double*);
template void launch_flow_out<float>(hipStream_t, const int*, int, const float*, const int*, double*);
template void launch_flow_cvt<float, double>(hipStream_t, const int*, int, const float*, double*, int);
template void launch_flow_cvt<double, float>(hipStream_t, const int*, int, const double*, float*, int);
template void launch_flow_cvt<double, double>(hipStream_t, const int*, int, const double*, double*, int);

}  // namespace spq
