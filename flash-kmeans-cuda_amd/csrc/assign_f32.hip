// fp32 assignment on the matrix cores, and row squared norms.
//
// The labels are those of the reference's tensor-core-free kernel
// (flash_kmeans_cuda/csrc/assign/assign_safe.cu:38-81): for each point,
//     dist_k = max(0, x_sq + c_sq[k] - 2 * <x, c_k>)      (assign_common.cuh:33-36)
// with the dot product accumulated in fp32 as one fused multiply-add chain in
// feature order, and the strict-< running minimum that keeps the lowest k on
// ties (assign_common.cuh:23-28).  It serves fp32 inputs, fp16/bf16 with
// D % 8 != 0 or D > 512, and FKC_ASSIGN_FORCE_SAFE (api.cpp:12-25).
//
// v_mfma_f32_16x16x4_f32 and v_mfma_f32_32x32x2_f32 add their products to
// the accumulator as a chain of fused multiply-adds in k order (the tests of
// this route compare its labels bit for bit with that chain, with subnormal,
// overflowing, infinite and NaN rows among them), so a sequence of them over the
// features gives the chain's bits at the matrix cores' fp32 rate (133 and 149
// TFLOP/s measured in registers alone; 78 is the vector peak without packed
// instructions).  Norms that the caller leaves out are the same chain: the
// points scored against themselves, read from the diagonal.
//
// Operands: A = M centroids x 64 / M features, B = as many features x M
// points, so lane l holds centroid (A) or point (B) l % M.  Both are loaded
// as quads of four consecutive features, lane group l / M the (l / M)-th
// quad of a group of 4 * 64 / M features, and transposed over the lane groups
// (v_permlane16_swap, v_permlane32_swap) into the operands of the group's
// four steps.  The points' operands stay in registers for the whole scan
// over K; the centroids' quads stream from the caches straight into
// registers up to eight groups ahead, with neither LDS nor barriers.  One
// quad feeds 4 * PT MFMAs, so a CU asks its L1 for at most 32 bytes a cycle.
//
// Bound by the matrix pipe and, on top of it, the vector instructions: fp32
// MFMAs and vector work hardly overlap here (at (131072, 1024, 128), timing
// copies without fold, loads and transposes ran 145 TFLOP/s, with them 110
// to 115), so the fold is five instructions per score.  Measured against the
// vector kernel this replaced, same labels: (1, 131072, 1024, 128) fp32 897
// -> 300 us, (1, 8192, 256, 128) 45 -> 13, (1, 1000, 1000, 512) 614 -> 78,
// (1, 100000, 300, 37) fp16 81 -> 39.  Staging the centroids through LDS in
// operand order (no transposes) gained at most 5% at large N and lost at
// small; folding a tile under the next one's MFMAs gained nothing.
#include "device_util.hpp"
#include "fkc_internal.hpp"

#include <algorithm>

#include <float.h>

namespace fkc {

int launch_assign_mfma(const void* x, const void* c, const float* c_sq,
                       int32_t* ids, int64_t B, int64_t N, int64_t K,
                       int64_t D, int dtype, const int32_t* ctrl,
                       hipStream_t s, hipEvent_t ev0, hipEvent_t ev1,
                       void* ws, size_t ws_bytes);

namespace {

constexpr int FT = 256;  // threads: four waves
// assign_rows_kernel: widest rows, most centroids, floats per row in LDS.
constexpr int kRowsMaxD = 32, kRowsMaxK = 8;
__host__ __device__ constexpr int rows_ld(int D) { return 4 * (D / 4 | 1); }

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));

// Four consecutive elements of a row.  Rows start wherever the caller's
// tensor and D put them, so the loads ask for element alignment only.
template <int DT>
struct Quad {
  typedef uint16_t Raw __attribute__((ext_vector_type(4), aligned(2)));
  __device__ static f32x4 cvt(Raw r) {
    typename Elem<DT>::T e[4];
    const uint16_t h[4] = {r[0], r[1], r[2], r[3]};
    __builtin_memcpy(e, h, 8);
    return f32x4{Elem<DT>::load(e[0]), Elem<DT>::load(e[1]),
                 Elem<DT>::load(e[2]), Elem<DT>::load(e[3])};
  }
};
template <>
struct Quad<FKC_F32> {
  typedef float Raw __attribute__((ext_vector_type(4), aligned(4)));
  __device__ static f32x4 cvt(Raw r) { return f32x4{r[0], r[1], r[2], r[3]}; }
};

// Features d .. d + 3 of a row of D.  whole: all four exist (d + 3 < D);
// else those at D and after read as zero, which adds nothing to a chain.
// Such a quad is the row's last whole one, moved down by the features it
// starts early: four clamped loads of one feature each took twice the time of
// whole quads at few features ((1, 400000, 8, D) fp32, us: D = 8 14.5, D = 12
// 11.4, against 8.1 at D = 16).  Only rows of less than a quad are loaded so.
template <int DT>
__device__ inline typename Quad<DT>::Raw load_quad(
    const typename Elem<DT>::T* row, int d, int D, bool whole, bool tiny) {
  using Raw = typename Quad<DT>::Raw;
  if (whole) return *reinterpret_cast<const Raw*>(row + d);
  Raw r = {};
  if (tiny) {
#pragma unroll
    for (int e = 0; e < 3; ++e) {
      const typename Elem<DT>::T v = row[min(d + e, D - 1)];
      if constexpr (DT == FKC_F32) {
        r[e] = d + e < D ? v : 0.f;
      } else {
        uint16_t h;
        __builtin_memcpy(&h, &v, 2);
        r[e] = d + e < D ? h : (uint16_t)0;
      }
    }
    return r;
  }
  const int d0 = min(d, D - 4), early = d - d0;
  r = *reinterpret_cast<const Raw*>(row + d0);
  if (D % 4 != 0) {
    if (early & 1) r = Raw{r[1], r[2], r[3], 0};
    if (early & 2) r = Raw{r[2], r[3], 0, 0};
  }
  if (early > 3) r = Raw{0, 0, 0, 0};
  return r;
}

// The two instruction shapes: M x M scores, FG features per group of quads
// (64 / M lane groups of four), four steps per group.
template <int M>
struct Shape;

template <>
struct Shape<16> {
  static constexpr int FG = 16, R = 4;
  typedef float Acc __attribute__((ext_vector_type(4)));
  __device__ static Acc mfma(float a, float b, Acc c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  // 4 x 4 transpose over the lane groups of 16: in, lane group q holds
  // features 4 q + e of the group in register e; out, it holds feature
  // 4 s + q in register s, the operand of step s.
  __device__ static void steps(f32x4 v, float (&o)[4]) {
    const u32x2 a = __builtin_amdgcn_permlane16_swap(
        __float_as_uint(v[0]), __float_as_uint(v[1]), false, false);
    const u32x2 b = __builtin_amdgcn_permlane16_swap(
        __float_as_uint(v[2]), __float_as_uint(v[3]), false, false);
    const u32x2 lo = __builtin_amdgcn_permlane32_swap(a[0], b[0], false, false);
    const u32x2 hi = __builtin_amdgcn_permlane32_swap(a[1], b[1], false, false);
    o[0] = __uint_as_float(lo[0]);
    o[1] = __uint_as_float(hi[0]);
    o[2] = __uint_as_float(lo[1]);
    o[3] = __uint_as_float(hi[1]);
  }
  // Accumulator register r of lane group q holds centroid row(r) + 4 q.
  __device__ static constexpr int row(int r) { return r; }
  // Register and lane of the diagonal's entry col.
  __device__ static int diag_reg(int col) { return col & 3; }
  __device__ static int diag_lane(int col) { return 16 * (col >> 2) + col; }
};

template <>
struct Shape<32> {
  static constexpr int FG = 8, R = 16;
  typedef float Acc __attribute__((ext_vector_type(16)));
  __device__ static Acc mfma(float a, float b, Acc c) {
    return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
  }
  // In, half q of the wave holds features 4 q + e in register e; out, it
  // holds feature 2 s + q in register s.
  __device__ static void steps(f32x4 v, float (&o)[4]) {
    const u32x2 a = __builtin_amdgcn_permlane32_swap(
        __float_as_uint(v[0]), __float_as_uint(v[1]), false, false);
    const u32x2 b = __builtin_amdgcn_permlane32_swap(
        __float_as_uint(v[2]), __float_as_uint(v[3]), false, false);
    o[0] = __uint_as_float(a[0]);
    o[1] = __uint_as_float(b[0]);
    o[2] = __uint_as_float(a[1]);
    o[3] = __uint_as_float(b[1]);
  }
  __device__ static constexpr int row(int r) { return 8 * (r / 4) + r % 4; }
  __device__ static int diag_reg(int col) { return 4 * (col >> 3) + (col & 3); }
  __device__ static int diag_lane(int col) { return 32 * (col >> 2 & 1) + col; }
};

// Where a wave's work lies: ks (1, 2 or 4) waves of the workgroup share one
// group of points and take every ks-th tile of 16 centroids.
struct WaveWork {
  int wave, kpart, n0;
  __device__ WaveWork(int ks, int pts) {
    wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    kpart = wave & (ks - 1);
    const int per = 4 / ks;  // point groups of the workgroup
    n0 = (blockIdx.x * per + wave / ks) * pts;
  }
};

// c_sq of the centroids whose scores a lane holds of the block at k0 (row
// K - 1 again past K).  Row by row, clamped, this costs four vector
// instructions a value, a quarter of the vector work of a 32 x 32 block at
// D = 37; QUADS loads four consecutive rows at a time and clamps only in the
// last, partial block.  That branch costs the four-tile 16 x 16 loop more
// than it saves ((1, 131072, 1024, 128) fp32 +1%), so it stays with the others
// ((8, 34594, 1712, 19) bf16 334 -> 257 us, (1, 3000, 4000, 96) fp32 63 -> 49).
template <int M, bool QUADS>
__device__ inline void load_csq(const float* qb, int k0, int q, int K,
                                float (&cq)[Shape<M>::R]) {
  if (QUADS && k0 + M <= K) {
    const float* p = qb + k0 + 4 * q;
#pragma unroll
    for (int r = 0; r < Shape<M>::R; r += 4) {
      const Quad<FKC_F32>::Raw v =
          *reinterpret_cast<const Quad<FKC_F32>::Raw*>(p + Shape<M>::row(r));
#pragma unroll
      for (int j = 0; j < 4; ++j) cq[r + j] = v[j];
    }
  } else {
#pragma unroll
    for (int r = 0; r < Shape<M>::R; ++r)
      cq[r] = qb[min(k0 + Shape<M>::row(r) + 4 * q, K - 1)];
  }
}

// The scores a lane holds of one block (one point, centroid rows rising with
// r) folded into its running minimum; strict < keeps the first.  best starts
// at FLT_MAX and stays >= 0, so the median of dist, 0 and best is
// min(max(dist, 0), best), and a NaN distance counts as 0 as the chain's
// clamp has it.  bidx lacks the lane group's 4 q until the end: the index is
// then wave-uniform and costs no vector instruction.
template <int M, bool WHOLE>
__device__ inline void fold_dist(const typename Shape<M>::Acc& acc, float xs,
                                 const float (&cq)[Shape<M>::R], int k0, int q,
                                 int K, float& best, int& bidx) {
#pragma unroll
  for (int r = 0; r < Shape<M>::R; ++r) {
    const int k = k0 + Shape<M>::row(r);
    const float dist = fmaf(-2.0f, acc[r], xs + cq[r]);
    float nb = __builtin_amdgcn_fmed3f(dist, 0.f, best);
    if constexpr (!WHOLE) nb = k + 4 * q < K ? nb : best;
    bidx = nb < best ? k : bidx;
    best = nb;
  }
}

// fold_dist over a wave's PT point tiles.
template <int M, int PT>
__device__ inline void fold_tile(const typename Shape<M>::Acc (&acc)[PT],
                                 const float (&xs)[PT],
                                 const float (&cq)[Shape<M>::R], int k0, int q,
                                 int K, float (&best)[PT], int (&bidx)[PT]) {
  if (k0 + M <= K) {
#pragma unroll
    for (int p = 0; p < PT; ++p)
      fold_dist<M, true>(acc[p], xs[p], cq, k0, q, K, best[p], bidx[p]);
  } else {
#pragma unroll
    for (int p = 0; p < PT; ++p)
      fold_dist<M, false>(acc[p], xs[p], cq, k0, q, K, best[p], bidx[p]);
  }
}

// Merge the lane groups of each point, then the ks waves that share them
// (smaller distance, then smaller index), and store the labels.
template <int M, int PT>
__device__ inline void merge_store(float (&best)[PT], int (&bidx)[PT], int ks,
                                   const WaveWork& w, int32_t* ids, int N) {
  static_assert(M * PT <= 64, "one point per lane");
  __shared__ float s_best[4][M * PT];
  __shared__ int s_idx[4][M * PT];
  const int lane = threadIdx.x & 63, q = lane / M;
#pragma unroll
  for (int p = 0; p < PT; ++p) {
    // No score below FLT_MAX: index 0, as the scan starts.
    bidx[p] = best[p] < FLT_MAX ? bidx[p] + 4 * q : 0;
#pragma unroll
    for (int off = M; off < 64; off <<= 1) {
      const float ob = __shfl_xor(best[p], off, 64);
      const int oi = __shfl_xor(bidx[p], off, 64);
      if (ob < best[p] || (ob == best[p] && oi < bidx[p])) {
        best[p] = ob;
        bidx[p] = oi;
      }
    }
  }
  // Lane group q keeps point tile q: lane l then holds point n0 + l.
  float b = best[0];
  int i = bidx[0];
#pragma unroll
  for (int p = 1; p < PT; ++p) {
    b = q == p ? best[p] : b;
    i = q == p ? bidx[p] : i;
  }
  if (ks > 1) {
    if (lane < M * PT) {
      s_best[w.wave][lane] = b;
      s_idx[w.wave][lane] = i;
    }
    __syncthreads();
    if (w.kpart != 0) return;
    if (lane < M * PT) {
      for (int j = 1; j < ks; ++j) {
        const float ob = s_best[w.wave + j][lane];
        const int oi = s_idx[w.wave + j][lane];
        if (ob < b || (ob == b && oi < i)) {
          b = ob;
          i = oi;
        }
      }
    }
  }
  if (lane < M * PT && w.n0 + lane < N) ids[w.n0 + lane] = i;
}

// ||x_n||^2 of the points of tile p, given.
template <int M, int PT>
__device__ inline void given_norms(const float* x_sq, int n0, int N,
                                   float (&xs)[PT]) {
#pragma unroll
  for (int p = 0; p < PT; ++p)
    xs[p] = x_sq[min(n0 + M * p + (int)threadIdx.x % M, N - 1)];
}

// ||x_n||^2 computed: points scored against themselves give the chain of
// v * v on the block's diagonal; every lane takes its own point's entry.  (A
// loop over the features in the vector unit waits for a round trip each: (1,
// 35, 5, 768) fp32 283 us of 300.)
template <int M>
__device__ inline float diagonal(const typename Shape<M>::Acc& acc) {
  using S = Shape<M>;
  const int col = threadIdx.x % M;
  float v = acc[0];
#pragma unroll
  for (int r = 1; r < S::R; ++r) v = S::diag_reg(col) == r ? acc[r] : v;
  return __shfl(v, S::diag_lane(col), 64);
}

// D <= 512.  M: instruction shape; G: feature groups a row takes (D <= FG G),
// the first NF of them certainly whole; PT: M-point tiles per wave.
template <int DT, int M, int G, int NF, int PT>
__global__ void __launch_bounds__(FT, 2)
assign_f32_kernel(const typename Elem<DT>::T* __restrict__ x,
                  const typename Elem<DT>::T* __restrict__ c,
                  const float* __restrict__ x_sq,
                  const float* __restrict__ c_sq, int32_t* __restrict__ ids,
                  int N, int K, int D, int ks,
                  const int32_t* __restrict__ ctrl) {
  using T = typename Elem<DT>::T;
  using Raw = typename Quad<DT>::Raw;
  using S = Shape<M>;
  // Quads in flight: eight against two gained 15% at (131072, 1024, 128).
  constexpr int PD = G < 8 ? G : 8;
  if (loop_done(ctrl)) return;
  const int lane = threadIdx.x & 63, col = lane % M, q = lane / M;
  const int b = blockIdx.y;
  const WaveWork w(ks, M * PT);
  const T* xb = x + (size_t)b * N * D;
  const T* cb = c + (size_t)b * K * D;
  const float* qb = c_sq + (size_t)b * K;

  const int nt = (K + M - 1) / M;
  const bool tiny = G == 1 && D < 4;
  // Quad g of this lane's row of tile t (row K - 1 past K: such rows are
  // loaded but never win).
  auto load_c = [&](int t, int g) -> Raw {
    const T* row = cb + (size_t)min(M * t + col, K - 1) * D;
    return load_quad<DT>(row, S::FG * g + 4 * q, D, g < NF, tiny);
  };
  Raw ring[PD];
#pragma unroll
  for (int i = 0; i < PD; ++i) ring[i] = load_c(w.kpart, i);

  float bx[PT][G][4];
#pragma unroll
  for (int p = 0; p < PT; ++p) {
    const T* row = xb + (size_t)min(w.n0 + M * p + col, N - 1) * D;
    Raw raw[G];
#pragma unroll
    for (int g = 0; g < G; ++g)
      raw[g] = load_quad<DT>(row, S::FG * g + 4 * q, D, g < NF, tiny);
#pragma unroll
    for (int g = 0; g < G; ++g) S::steps(Quad<DT>::cvt(raw[g]), bx[p][g]);
  }
  float xs[PT], best[PT];
  int bidx[PT];
  if (x_sq != nullptr) {
    given_norms<M, PT>(x_sq + (size_t)b * N, w.n0, N, xs);
  } else {
#pragma unroll
    for (int p = 0; p < PT; ++p) {
      typename S::Acc acc = {};
#pragma unroll
      for (int g = 0; g < G; ++g)
#pragma unroll
        for (int s = 0; s < 4; ++s) acc = S::mfma(bx[p][g][s], bx[p][g][s], acc);
      xs[p] = diagonal<M>(acc);
    }
  }
#pragma unroll
  for (int p = 0; p < PT; ++p) {
    best[p] = FLT_MAX;
    bidx[p] = 0;
  }

  for (int t = w.kpart; t < nt; t += ks) {
    float cq[S::R];
    load_csq<M, M == 32 || PT == 1>(qb, M * t, q, K, cq);
    typename S::Acc acc[PT];
#pragma unroll
    for (int p = 0; p < PT; ++p)
#pragma unroll
      for (int r = 0; r < S::R; ++r) acc[p][r] = 0.f;
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const Raw cur = ring[0];
#pragma unroll
      for (int i = 0; i + 1 < PD; ++i) ring[i] = ring[i + 1];
      ring[PD - 1] = g + PD < G ? load_c(t, g + PD) : load_c(t + ks, g + PD - G);
      float a[4];
      S::steps(Quad<DT>::cvt(cur), a);
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int p = 0; p < PT; ++p) acc[p] = S::mfma(a[s], bx[p][g][s], acc[p]);
    }
    fold_tile<M, PT>(acc, xs, cq, M * t, q, K, best, bidx);
  }
  merge_store<M, PT>(best, bidx, ks, w, ids + (size_t)b * N, N);
}

// Any D (used above 512, where a point tile's operands no longer fit the
// registers): both operands stream, and CT x PT blocks of 16 x 16 scores per
// wave give each quad CT or PT uses.  4 x 4 blocks where N and K fill them:
// (1, 20000, 500, 768) fp32 974 us with the vector kernel, 289 with this one;
// fp16 2362 and 284.  Smaller blocks (plan_wide) for few points or few
// centroids, with PD groups of quads in flight: with one in flight a wave
// waits for a round trip per group.
template <int DT, int PT, int CT, int PD>
__global__ void __launch_bounds__(FT, 2)
assign_f32_wide_kernel(const typename Elem<DT>::T* __restrict__ x,
                       const typename Elem<DT>::T* __restrict__ c,
                       const float* __restrict__ x_sq,
                       const float* __restrict__ c_sq,
                       int32_t* __restrict__ ids, int N, int K, int D, int ks,
                       const int32_t* __restrict__ ctrl) {
  using T = typename Elem<DT>::T;
  using Raw = typename Quad<DT>::Raw;
  using S = Shape<16>;
  constexpr int M = 16;
  if (loop_done(ctrl)) return;
  const int lane = threadIdx.x & 63, col = lane % M, q = lane / M;
  const int b = blockIdx.y;
  const WaveWork w(ks, M * PT);
  const T* xb = x + (size_t)b * N * D;
  const T* cb = c + (size_t)b * K * D;
  const float* qb = c_sq + (size_t)b * K;
  float xs[PT], best[PT];
  int bidx[PT];
  const T* xrow[PT];
#pragma unroll
  for (int p = 0; p < PT; ++p) {
    best[p] = FLT_MAX;
    bidx[p] = 0;
    xrow[p] = xb + (size_t)min(w.n0 + M * p + col, N - 1) * D;
  }
  const int nfull = D / S::FG;  // > PD
  const bool rest = D % S::FG != 0;

  // The groups of a row in order: load(i, g, whole) fills slot i of PD with
  // group g's quads, use(i) scores a slot.  (Past the last whole group a slot
  // is filled with that again.)
  auto stream = [&](auto load, auto use) {
#pragma unroll
    for (int i = 0; i < PD; ++i) load(i, i, true);
    int g = 0;
    for (; g + PD <= nfull; g += PD) {
#pragma unroll
      for (int i = 0; i < PD; ++i) use(i, min(g + i + PD, nfull - 1));
    }
#pragma unroll
    for (int i = 0; i < PD - 1; ++i)
      if (g + i < nfull) use(i, nfull - 1);
    if (rest) {
      load(0, nfull, false);
      use(0, nfull - 1);
    }
  };

  Raw rx[PD][PT], rc[PD][CT];
  auto load_x = [&](int i, int g, bool whole) {
#pragma unroll
    for (int p = 0; p < PT; ++p)
      rx[i][p] = load_quad<DT>(xrow[p], S::FG * g + 4 * q, D, whole, false);
  };
  if (x_sq != nullptr) {
    given_norms<M, PT>(x_sq + (size_t)b * N, w.n0, N, xs);
  } else {
    S::Acc acc[PT];
#pragma unroll
    for (int p = 0; p < PT; ++p) acc[p] = S::Acc{0.f, 0.f, 0.f, 0.f};
    stream(load_x, [&](int i, int next) {
      Raw u[PT];
#pragma unroll
      for (int p = 0; p < PT; ++p) u[p] = rx[i][p];
      load_x(i, next, true);
#pragma unroll
      for (int p = 0; p < PT; ++p) {
        float v[4];
        S::steps(Quad<DT>::cvt(u[p]), v);
#pragma unroll
        for (int s = 0; s < 4; ++s) acc[p] = S::mfma(v[s], v[s], acc[p]);
      }
    });
#pragma unroll
    for (int p = 0; p < PT; ++p) xs[p] = diagonal<M>(acc[p]);
  }

  const int nt = (K + M * CT - 1) / (M * CT);
  for (int t = w.kpart; t < nt; t += ks) {
    const int k0 = M * CT * t;
    const T* crow[CT];
#pragma unroll
    for (int j = 0; j < CT; ++j)
      crow[j] = cb + (size_t)min(k0 + M * j + col, K - 1) * D;
    S::Acc acc[CT][PT];
#pragma unroll
    for (int j = 0; j < CT; ++j)
#pragma unroll
      for (int p = 0; p < PT; ++p) acc[j][p] = S::Acc{0.f, 0.f, 0.f, 0.f};
    auto load = [&](int i, int g, bool whole) {
      load_x(i, g, whole);
#pragma unroll
      for (int j = 0; j < CT; ++j)
        rc[i][j] = load_quad<DT>(crow[j], S::FG * g + 4 * q, D, whole, false);
    };
    stream(load, [&](int i, int next) {
      Raw ux[PT], uc[CT];
#pragma unroll
      for (int p = 0; p < PT; ++p) ux[p] = rx[i][p];
#pragma unroll
      for (int j = 0; j < CT; ++j) uc[j] = rc[i][j];
      load(i, next, true);
      float a[CT][4], bx[PT][4];
#pragma unroll
      for (int p = 0; p < PT; ++p) S::steps(Quad<DT>::cvt(ux[p]), bx[p]);
#pragma unroll
      for (int j = 0; j < CT; ++j) S::steps(Quad<DT>::cvt(uc[j]), a[j]);
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int j = 0; j < CT; ++j)
#pragma unroll
          for (int p = 0; p < PT; ++p)
            acc[j][p] = S::mfma(a[j][s], bx[p][s], acc[j][p]);
    });
#pragma unroll
    for (int j = 0; j < CT; ++j) {
      float cq[S::R];
      load_csq<M, false>(qb, k0 + M * j, q, K, cq);
      fold_tile<M, PT>(acc[j], xs, cq, k0 + M * j, q, K, best, bidx);
    }
  }
  merge_store<M, PT>(best, bidx, ks, w, ids + (size_t)b * N, N);
}

// The better of two candidates: smaller distance, then smaller index.
__device__ inline void take_better(float& b, int& i, float ob, int oi) {
  const bool other = ob < b || (ob == b && oi < i);
  b = other ? ob : b;
  i = other ? oi : i;
}

// Few centroids of few features (K <= 16 KT, D <= 16 G) and many points: the
// centroids' operands and c_sq stay in registers and a wave walks groups of 64
// points, the next group's loads in flight.  What bounds it is the vector
// work per group, so a tile's centroids are laid out with lane group q's
// register r holding centroid 4 r + q (registers past K are skipped whole),
// and the four lane groups' winners of four point tiles are merged with lane
// swaps, each group ending with one tile.  At (1, 3000000, 8, D) fp32, us, the
// vector kernel (one lane per point), the kernel above, this one: D = 1 28 /
// 44 / 24, D = 8 33 / 50 / 29, D = 16 40 / 41 / 39 (216 MB: 5.5 TB/s, partly
// from the cache); D = 24 57 / 70 / 66.  (Those of whole quads take
// assign_rows_kernel since.)
template <int DT, int G, int KT>
__global__ void __launch_bounds__(FT, G == 1 ? 4 : 2)
assign_few_kernel(const typename Elem<DT>::T* __restrict__ x,
                  const typename Elem<DT>::T* __restrict__ c,
                  const float* __restrict__ x_sq,
                  const float* __restrict__ c_sq, int32_t* __restrict__ ids,
                  int N, int K, int D, const int32_t* __restrict__ ctrl) {
  using T = typename Elem<DT>::T;
  using Raw = typename Quad<DT>::Raw;
  using S = Shape<16>;
  constexpr int M = 16, PT = 4;
  if (loop_done(ctrl)) return;
  const int lane = threadIdx.x & 63, col = lane % M, q = lane / M;
  const int b = blockIdx.y;
  const T* xb = x + (size_t)b * N * D;
  const T* cb = c + (size_t)b * K * D;
  const float* qb = c_sq + (size_t)b * K;
  const float* xq = x_sq != nullptr ? x_sq + (size_t)b * N : nullptr;
  int32_t* ib = ids + (size_t)b * N;
  const bool tiny = D < 4;

  int n0 = WaveWork(1, M * PT).n0;
  const int stride = (int)gridDim.x * 4 * M * PT;
  Raw rx[PT][G];
  float rq[PT];
  auto load_x = [&](int at) {
#pragma unroll
    for (int p = 0; p < PT; ++p) {
      const int n = min(at + M * p + col, N - 1);
      const T* row = xb + (size_t)n * D;
#pragma unroll
      for (int g = 0; g < G; ++g)
        rx[p][g] = load_quad<DT>(row, S::FG * g + 4 * q, D, g < G - 1, tiny);
      rq[p] = xq != nullptr ? xq[n] : 0.f;
    }
  };
  load_x(n0);

  float a[KT][G][4], cq[KT][S::R];
#pragma unroll
  for (int t = 0; t < KT; ++t) {
    const T* row = cb + (size_t)min(M * t + 4 * (col & 3) + col / 4, K - 1) * D;
#pragma unroll
    for (int g = 0; g < G; ++g)
      S::steps(Quad<DT>::cvt(load_quad<DT>(row, S::FG * g + 4 * q, D,
                                           g < G - 1, tiny)),
               a[t][g]);
#pragma unroll
    for (int r = 0; r < S::R; ++r) cq[t][r] = qb[min(M * t + 4 * r + q, K - 1)];
  }

  for (bool more = n0 < N; more; n0 += stride) {
    more = stride < N - n0;
    float bx[PT][G][4], xs[PT], best[PT];
    int bidx[PT];
#pragma unroll
    for (int p = 0; p < PT; ++p) {
#pragma unroll
      for (int g = 0; g < G; ++g) S::steps(Quad<DT>::cvt(rx[p][g]), bx[p][g]);
      xs[p] = rq[p];
    }
    if (more) load_x(n0 + stride);
    if (xq == nullptr) {
#pragma unroll
      for (int p = 0; p < PT; ++p) {
        S::Acc acc = {};
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
          for (int s = 0; s < 4; ++s)
            if (S::FG * g + 4 * s < D)
              acc = S::mfma(bx[p][g][s], bx[p][g][s], acc);
        xs[p] = diagonal<M>(acc);
      }
    }
#pragma unroll
    for (int p = 0; p < PT; ++p) {
      best[p] = FLT_MAX;
      bidx[p] = 0;
    }
#pragma unroll
    for (int t = 0; t < KT; ++t) {
      S::Acc acc[PT];
#pragma unroll
      for (int p = 0; p < PT; ++p) acc[p] = S::Acc{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int g = 0; g < G; ++g)
#pragma unroll
        for (int s = 0; s < 4; ++s)
          if (S::FG * g + 4 * s < D) {
#pragma unroll
            for (int p = 0; p < PT; ++p)
              acc[p] = S::mfma(a[t][g][s], bx[p][g][s], acc[p]);
          }
      // As fold_dist; centroid k0 + q, the last register's past K masked.
      auto fold = [&](int r, bool whole) {
        const int k0 = M * t + 4 * r;
#pragma unroll
        for (int p = 0; p < PT; ++p) {
          const float dist = fmaf(-2.0f, acc[p][r], xs[p] + cq[t][r]);
          float nb = __builtin_amdgcn_fmed3f(dist, 0.f, best[p]);
          if (!whole) nb = k0 + q < K ? nb : best[p];
          bidx[p] = nb < best[p] ? k0 : bidx[p];
          best[p] = nb;
        }
      };
#pragma unroll
      for (int r = 0; r < S::R; ++r) {
        if (M * t + 4 * r + 4 <= K)
          fold(r, true);
        else if (M * t + 4 * r < K)
          fold(r, false);
      }
    }
    // No score below FLT_MAX: index 0, as the scan starts.
#pragma unroll
    for (int p = 0; p < PT; ++p) bidx[p] = best[p] < FLT_MAX ? bidx[p] + q : 0;
    // Tiles 0 | 2 and 1 | 3 over the halves of the wave, then even | odd tiles
    // over the halves' halves: lane group q keeps tile q.
    float bv[2];
    int bi[2];
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      const u32x2 v = __builtin_amdgcn_permlane32_swap(
          __float_as_uint(best[p]), __float_as_uint(best[p + 2]), false, false);
      const u32x2 i = __builtin_amdgcn_permlane32_swap(
          (unsigned)bidx[p], (unsigned)bidx[p + 2], false, false);
      bv[p] = __uint_as_float(v[0]);
      bi[p] = (int)i[0];
      take_better(bv[p], bi[p], __uint_as_float(v[1]), (int)i[1]);
    }
    const u32x2 v = __builtin_amdgcn_permlane16_swap(
        __float_as_uint(bv[0]), __float_as_uint(bv[1]), false, false);
    const u32x2 i = __builtin_amdgcn_permlane16_swap((unsigned)bi[0],
                                                     (unsigned)bi[1], false, false);
    float win = __uint_as_float(v[0]);
    int id = (int)i[0];
    take_better(win, id, __uint_as_float(v[1]), (int)i[1]);
    if (lane < N - n0) ib[n0 + lane] = id;
  }
}

// KM centroids at most, rows of whole quads and many points: one lane per
// point.  A workgroup's rows pass through LDS so that they are loaded as one
// contiguous block; every lane reads the same centroids from LDS.  Bound by
// the loads: at (1, 3000000, 4, D) fp32, us, the vector kernel that passed
// everything through LDS, assign_few_kernel, this one: D = 8 29 / 29 / 22,
// D = 16 34 / 39 / 33, D = 24 52 / 65 / 53 (312 MB: 5.9 TB/s, partly from the
// cache); norms left out cost it nothing.
template <int DT, int KM>
__global__ void __launch_bounds__(FT, 5)
assign_rows_kernel(const typename Elem<DT>::T* __restrict__ x,
                   const typename Elem<DT>::T* __restrict__ c,
                   const float* __restrict__ x_sq,
                   const float* __restrict__ c_sq, int32_t* __restrict__ ids,
                   int N, int K, int D, const int32_t* __restrict__ ctrl) {
  using T = typename Elem<DT>::T;
  using Raw = typename Quad<DT>::Raw;
  constexpr int QM = kRowsMaxD / 4;  // quads of a row, at most
  if (loop_done(ctrl)) return;
  // Rows of an odd number of quads: lanes that read their own rows spread
  // over the banks.
  extern __shared__ __attribute__((aligned(16))) float s_x[];
  __shared__ __attribute__((aligned(16))) float s_c[KM][kRowsMaxD];
  __shared__ float s_q[KM];
  static_assert(KM * kRowsMaxD <= FT, "one centroid value per thread");
  const int tid = threadIdx.x, b = blockIdx.y;
  const int n0 = blockIdx.x * FT, n = n0 + tid;
  const int qd = D / 4, nq = min(FT, N - n0) * qd, ld = rows_ld(D);
  const T* xb = x + ((size_t)b * N + n0) * D;
  const T* cb = c + (size_t)b * K * D;
  float xs = 0.f;
  Raw v[QM];
#pragma unroll
  for (int i = 0; i < QM; ++i)
    if (i < qd)
      v[i] = *reinterpret_cast<const Raw*>(xb + 4 * min(i * FT + tid, nq - 1));
  if (x_sq != nullptr) xs = x_sq[(size_t)b * N + min(n, N - 1)];
  if (tid < KM * kRowsMaxD) {
    const int k = tid / kRowsMaxD, d = tid % kRowsMaxD;
    s_c[k][d] = k < K && d < D ? Elem<DT>::load(cb[k * D + d]) : 0.f;
  }
  if (tid < KM) s_q[tid] = c_sq[(size_t)b * K + min(tid, K - 1)];
  int r = tid / qd, q = tid - r * qd;
  const int dr = FT / qd, dq = FT - dr * qd;
#pragma unroll
  for (int i = 0; i < QM; ++i)
    if (i < qd) {
      *reinterpret_cast<f32x4*>(s_x + r * ld + 4 * q) = Quad<DT>::cvt(v[i]);
      r += dr;
      q += dq;
      if (q >= qd) {
        q -= qd;
        ++r;
      }
    }
  __syncthreads();
  const f32x4* row = reinterpret_cast<const f32x4*>(s_x + tid * ld);
  float acc[KM], own = 0.f;
#pragma unroll
  for (int k = 0; k < KM; ++k) acc[k] = 0.f;
  for (int i = 0; i < qd; ++i) {
    const f32x4 xv = row[i];
    if (x_sq == nullptr) {
#pragma unroll
      for (int e = 0; e < 4; ++e) own = fmaf(xv[e], xv[e], own);
    }
#pragma unroll
    for (int k = 0; k < KM; ++k) {
      const f32x4 cv = *reinterpret_cast<const f32x4*>(&s_c[k][4 * i]);
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[k] = fmaf(xv[e], cv[e], acc[k]);
    }
  }
  if (x_sq == nullptr) xs = own;
  float best = FLT_MAX;
  int bidx = 0;
#pragma unroll
  for (int k = 0; k < KM; ++k)
    if (k < K) {
      const float dist = fmaf(-2.0f, acc[k], xs + s_q[k]);
      const float nb = __builtin_amdgcn_fmed3f(dist, 0.f, best);
      bidx = nb < best ? k : bidx;
      best = nb;
    }
  if (n < N) ids[(size_t)b * N + n] = bidx;
}

// Bound by HBM at many rows.  R rows per wave, their loads in flight together:
// one row per wave waits for a round trip with 2 to 8 bytes per lane
// outstanding.  One and four rows, us: 65536 x 128 fp16 11.3 / 6.2, 100000 x
// 37 fp16 11.0 / 6.1, 131072 x 128 fp32 20.6 / 10.7 (6.3 TB/s, partly from the
// cache).  Every row is summed in the same order for any R.
template <int DT, int R>
__global__ void __launch_bounds__(256)
row_sqnorm_kernel(const typename Elem<DT>::T* __restrict__ src,
                  float* __restrict__ out, int64_t rows, int D,
                  const int32_t* __restrict__ ctrl) {
  using E = Elem<DT>;
  if (loop_done(ctrl)) return;
  const int lane = threadIdx.x & 63;
  const int64_t row = ((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * R;
  if (row >= rows) return;
  const typename E::T* r[R];
#pragma unroll
  for (int i = 0; i < R; ++i) r[i] = src + min(row + i, rows - 1) * D;
  // Column order and reduction shared with the finalize kernels.
  float acc[R] = {};
  if (row_vec(D) == 2) {
    for (int c = 2 * lane; c < D; c += 128) {
      float f[R][2];
#pragma unroll
      for (int i = 0; i < R; ++i) {
        f[i][0] = E::load(r[i][c]);
        f[i][1] = E::load(r[i][c + 1]);
      }
#pragma unroll
      for (int i = 0; i < R; ++i) {
        acc[i] = fmaf(f[i][0], f[i][0], acc[i]);
        acc[i] = fmaf(f[i][1], f[i][1], acc[i]);
      }
    }
  } else {
    for (int c = lane; c < D; c += 64) {
      float f[R];
#pragma unroll
      for (int i = 0; i < R; ++i) f[i] = E::load(r[i][c]);
#pragma unroll
      for (int i = 0; i < R; ++i) acc[i] = fmaf(f[i], f[i], acc[i]);
    }
  }
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const float v = row_sum(acc[i]);
    if (lane == i && row + i < rows) out[row + i] = v;
  }
}

// The launch of a shape: instruction shape m (64: one lane per point), m-point
// tiles per wave (pt), 16-centroid tiles at a time (ct: rows above D = 512, and
// the few-centroid kernel's KT; one lane per point: KM), waves of a workgroup that share their points and split K (ks).
struct F32Plan {
  int m, pt, ct, ks;
};

// 32 x 32 blocks step eight features at a time, 16 x 16 blocks sixteen: where
// D's last sixteen are at most half used, 32 x 32 saves the padding
// ((131072, 1000, D) fp32, 16 x 16 against 32 x 32: D = 24 103 / 79 us, 40
// 132 / 110, 72 203 / 177, 104 261 / 246, 200 536 / 497); elsewhere 16 x 16
// is as fast or faster (64 159 / 160, 96 223 / 228, 128 292 / 302, 160 413 /
// 426) and wastes less of a small K.
bool f32_has_m32(int64_t D) { return D <= 248 && (D + 7) / 8 % 2 == 1; }

// 32 x 32 blocks need more than 16 centroids: (1, 1500000, 16, 24) fp32 67 us,
// with 16 x 16 blocks 33.
//
// The candidate with the least modelled time: waves per SIMD, rounded up,
// times a wave's work in 16 x 16 blocks.  A wave's own start costs about two
// 16-centroid tiles; fewer points per wave mean more centroid loads per MFMA
// (factors measured at (131072, 1024, 128): four tiles 1, two 1.05, one 1.5);
// one wave alone on a SIMD reaches 0.77 of what two do.
F32Plan plan_f32(int64_t B, int64_t N, int64_t K, int64_t D) {
  const int64_t simds = 4 * (int64_t)device_shape().cus;
  F32Plan best{16, 1, 1, 1};
  double least = 0;
  for (int m = 16; m <= 32; m *= 2) {
    if (m == 32 && (!f32_has_m32(D) || K <= 16)) break;
    const int u = m / 16;
    const int64_t nt = (K + m - 1) / m;
    const double groups = m == 16 ? 2 * ((D + 15) / 16) : (D + 7) / 8;
    const int pt_max = (D <= 128 ? 4 : D <= 256 ? 2 : 1) / u;
    for (int pt = pt_max; pt >= 1; pt >>= 1) {
      const double reuse = pt * u >= 4 ? 1.0 : pt * u == 2 ? 1.05 : 1.5;
      for (int ks = 1; ks <= 4 && ks <= nt; ks *= 2) {
        const int64_t waves = B * ((N + m * pt - 1) / (m * pt)) * ks;
        const double t = (double)((waves + simds - 1) / simds) *
                         (waves <= simds ? 1.3 : 1.0) * pt * u * reuse *
                         groups * ((double)((nt + ks - 1) / ks) * u + 2);
        if (least == 0 || t < least) {
          least = t;
          best = {m, pt, 1, ks};
        }
      }
    }
  }
  return best;
}

// Where assign_few_kernel is taken: its registers hold the centroids, and
// there are enough points for its waves to walk.  At (1, N, K, D) fp32, us,
// assign_f32_kernel / this: N = 500000: (16, 16) 10 / 10, (48, 16) 16 / 16,
// (16, 24) 15 / 14, (48, 8) 14 / 12; N = 3000000: (16, 16) 41 / 40, (48, 16)
// 73 / 73, (16, 24) 70 / 67, (16, 28) 75 / 77, (32, 20) 68 / 78, (32, 8) 46 /
// 45, (17, 1) 47 / 36; below 131072 points both end before the next launch.
bool f32_few(int64_t B, int64_t N, int64_t K, int64_t D) {
  return ((D <= 16 && K <= 48) || (D <= 24 && K <= 16)) && N >= 1024 &&
         B * N >= 131072;
}

// The launch of rows above D = 512: point (1 or 4) and centroid (1, 2 or 4)
// tiles per wave, waves that split K.  The candidate with the least modelled
// time: waves per SIMD times a wave's blocks; waves of fewer blocks load more
// per MFMA (factors that fit the best of all forms at 100 .. 100000 points and
// 1 .. 1000 centroids; 4 x 1 blocks never were).  Against 4 x 4
// blocks alone, fp32 us: (1, 1000, 4, 768) 76 -> 11, (1, 20000, 32, 1024) 116
// -> 47, (1, 100000, 16, 513) 121 -> 65; the vector kernel before them took
// 18, 86 and 86.
F32Plan plan_wide(int64_t B, int64_t N, int64_t K) {
  const int64_t simds = 4 * (int64_t)device_shape().cus;
  F32Plan best{16, 1, 1, 1};
  double least = 0;
  for (int pt = 4; pt >= 1; pt /= 4) {
    for (int ct = 4; ct >= (pt == 4 ? 2 : 1); ct /= 2) {
      const int64_t nt = (K + 16 * ct - 1) / (16 * ct);
      const double reuse = pt == 4 ? (ct == 4 ? 1.0 : 1.2)
                                   : (ct == 4 ? 1.3 : ct == 2 ? 1.6 : 2.0);
      for (int ks = 1; ks <= 4 && ks <= nt; ks *= 2) {
        const int64_t waves = B * ((N + 16 * pt - 1) / (16 * pt)) * ks;
        const double t = std::max(1.3, (double)waves / (double)simds) * pt *
                         ct * reuse * (double)((nt + ks - 1) / ks);
        if (least == 0 || t < least) {
          least = t;
          best = {16, pt, ct, ks};
        }
      }
    }
  }
  return best;
}

// Where assign_rows_kernel is taken, against the better of the two above, at
// (1, N, K, D) fp32, us: N = 400000: (8, 24) 11 / 11, (4, 20) 10 / 7, (8, 32)
// 15 / 14; N = 3000000: (8, 8) 29 / 23, (8, 16) 39 / 34, (8, 24) 65 / 55, (8, 32)
// 82 / 76.
bool f32_rows(int64_t B, int64_t N, int64_t K, int64_t D) {
  return K <= kRowsMaxK && D <= kRowsMaxD && D % 4 == 0 && N >= 1024 &&
         B * N >= 131072;
}

enum F32Kind { kChain, kWide, kFew, kRows = 8 };  // as in fkc_assign_plan

F32Kind f32_kind(int64_t B, int64_t N, int64_t K, int64_t D) {
  return D > 512                 ? kWide
         : f32_rows(B, N, K, D) ? kRows
         : f32_few(B, N, K, D)  ? kFew
                                : kChain;
}

F32Plan f32_plan(F32Kind kind, int64_t B, int64_t N, int64_t K, int64_t D) {
  if (kind == kWide) return plan_wide(B, N, K);
  if (kind == kRows) return {64, 1, K <= 4 ? 4 : 8, 1};
  if (kind == kFew) return {16, 4, D > 16 || K <= 16 ? 1 : K <= 32 ? 2 : 3, 1};
  return plan_f32(B, N, K, D);
}

template <int DT>
int launch_f32_t(const void* x, const void* c, const float* x_sq,
                 const float* c_sq, int32_t* ids, int64_t B, int64_t N,
                 int64_t K, int64_t D, const int32_t* ctrl, hipStream_t s) {
  using T = typename Elem<DT>::T;
  const F32Kind kind = f32_kind(B, N, K, D);
  const F32Plan p = f32_plan(kind, B, N, K, D);
  const int64_t per = p.m * p.pt * (4 / p.ks);  // points per workgroup
  dim3 grid((unsigned)((N + per - 1) / per), (unsigned)B);
  if (kind == kRows) {
    auto rows = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, grid, dim3(FT),
                         (size_t)FT * rows_ld((int)D) * sizeof(float), s,
                         static_cast<const T*>(x), static_cast<const T*>(c),
                         x_sq, c_sq, ids, (int)N, (int)K, (int)D, ctrl);
      return check_launch("assign_rows");
    };
    return p.ct == 4 ? rows(assign_rows_kernel<DT, 4>)
                     : rows(assign_rows_kernel<DT, 8>);
  }
  if (kind == kFew) {
    // One round of resident workgroups (4 per CU), or two of 6 for the
    // smallest: us at 3, 4, 6, 8, 12 per CU, (1, 3000000, 8, 8) 41 / 34 / 28 /
    // 34 / 29, (1, 3000000, 24, 8) 51 / 44 / 53 / 45 / 46.
    const int64_t most = (D <= 16 && K <= 16 ? 12 : 4) * device_shape().cus;
    grid.x = (unsigned)std::min<int64_t>(grid.x, std::max<int64_t>(most / B, 1));
    auto few = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, grid, dim3(FT), 0, s,
                         static_cast<const T*>(x), static_cast<const T*>(c),
                         x_sq, c_sq, ids, (int)N, (int)K, (int)D, ctrl);
      return check_launch("assign_few");
    };
    return D > 16      ? few(assign_few_kernel<DT, 2, 1>)
           : p.ct == 1 ? few(assign_few_kernel<DT, 1, 1>)
           : p.ct == 2 ? few(assign_few_kernel<DT, 1, 2>)
                       : few(assign_few_kernel<DT, 1, 3>);
  }
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(FT), 0, s, static_cast<const T*>(x),
                       static_cast<const T*>(c), x_sq, c_sq, ids, (int)N,
                       (int)K, (int)D, p.ks, ctrl);
    return check_launch("assign_f32");
  };
  if (kind == kWide) {
    if (p.pt == 1)
      return p.ct == 1   ? go(assign_f32_wide_kernel<DT, 1, 1, 8>)
             : p.ct == 2 ? go(assign_f32_wide_kernel<DT, 1, 2, 6>)
                         : go(assign_f32_wide_kernel<DT, 1, 4, 4>);
    return p.ct == 2 ? go(assign_f32_wide_kernel<DT, 4, 2, 3>)
                     : go(assign_f32_wide_kernel<DT, 4, 4, 1>);
  }
  // G feature groups cover D; the NF groups of the next smaller variant are
  // certainly whole (all G where fp32 fills them exactly).  The points'
  // operands take 128 registers at most, which leaves two waves per SIMD.
#define FKC_F32_G(M, G, NF, PTMAX)                                           \
  if (p.m == M && D <= Shape<M>::FG * G) {                                   \
    if constexpr (DT == FKC_F32 && M == 16) {                                \
      if (D == Shape<M>::FG * G) {                                           \
        if (p.pt == 1) return go(assign_f32_kernel<DT, M, G, G, 1>);         \
        if constexpr (PTMAX >= 2)                                            \
          if (p.pt == 2) return go(assign_f32_kernel<DT, M, G, G, 2>);       \
        if constexpr (PTMAX >= 4)                                            \
          if (p.pt == 4) return go(assign_f32_kernel<DT, M, G, G, 4>);       \
      }                                                                      \
    }                                                                        \
    if (p.pt == 1) return go(assign_f32_kernel<DT, M, G, NF, 1>);            \
    if constexpr (PTMAX >= 2)                                                \
      if (p.pt == 2) return go(assign_f32_kernel<DT, M, G, NF, 2>);          \
    if constexpr (PTMAX >= 4)                                                \
      if (p.pt == 4) return go(assign_f32_kernel<DT, M, G, NF, 4>);          \
  }
  FKC_F32_G(16, 1, 0, 4)
  FKC_F32_G(16, 2, 1, 4)
  FKC_F32_G(16, 3, 2, 4)
  FKC_F32_G(16, 4, 3, 4)
  FKC_F32_G(16, 5, 4, 4)
  FKC_F32_G(16, 6, 5, 4)
  FKC_F32_G(16, 7, 6, 4)
  FKC_F32_G(16, 8, 7, 4)
  FKC_F32_G(16, 10, 8, 2)
  FKC_F32_G(16, 12, 10, 2)
  FKC_F32_G(16, 14, 12, 2)
  FKC_F32_G(16, 16, 14, 2)
  FKC_F32_G(16, 20, 16, 1)
  FKC_F32_G(16, 24, 20, 1)
  FKC_F32_G(16, 28, 24, 1)
  FKC_F32_G(16, 32, 28, 1)
  FKC_F32_G(32, 1, 0, 2)
  FKC_F32_G(32, 3, 2, 2)
  FKC_F32_G(32, 5, 4, 2)
  FKC_F32_G(32, 7, 6, 2)
  FKC_F32_G(32, 9, 8, 2)
  FKC_F32_G(32, 11, 10, 2)
  FKC_F32_G(32, 13, 12, 2)
  FKC_F32_G(32, 15, 14, 2)
  FKC_F32_G(32, 17, 16, 1)
  FKC_F32_G(32, 19, 18, 1)
  FKC_F32_G(32, 21, 20, 1)
  FKC_F32_G(32, 23, 22, 1)
  FKC_F32_G(32, 25, 24, 1)
  FKC_F32_G(32, 27, 26, 1)
  FKC_F32_G(32, 29, 28, 1)
  FKC_F32_G(32, 31, 30, 1)
#undef FKC_F32_G
  return fail(FKC_ERR_UNSUPPORTED, "assign_f32: no kernel for D = %lld",
              (long long)D);
}

template <int DT>
int launch_rowsq_t(const void* src, float* out, int64_t rows, int64_t D,
                   const int32_t* ctrl, hipStream_t s) {
  using T = typename Elem<DT>::T;
  // Four rows per wave while the grid still has 8 workgroups (32 waves) per CU.
  const bool many = rows >= 32768;
  const int64_t per = many ? 16 : 4;
  dim3 grid((unsigned)((rows + per - 1) / per));
  auto fn = many ? &row_sqnorm_kernel<DT, 4> : &row_sqnorm_kernel<DT, 1>;
  hipLaunchKernelGGL(fn, grid, dim3(256), 0, s, static_cast<const T*>(src), out,
                     rows, (int)D, ctrl);
  return check_launch("row_sqnorm");
}

}  // namespace

int launch_assign(const void* x, const void* c, const float* x_sq,
                  const float* c_sq, int32_t* ids, int64_t B, int64_t N,
                  int64_t K, int64_t D, int dtype, const int32_t* ctrl,
                  hipStream_t s, hipEvent_t ev0, hipEvent_t ev1, void* ws,
                  size_t ws_bytes) {
  if (B == 0 || N == 0) return FKC_OK;
  if (assign_uses_mfma(dtype, D))
    return launch_assign_mfma(x, c, c_sq, ids, B, N, K, D, dtype, ctrl, s,
                              ev0, ev1, ws, ws_bytes);
  // The fp32 route marks its span with event records on the stream.
  if (ev0 != nullptr) (void)hipEventRecord(ev0, s);
  int rc = FKC_OK;
  switch (dtype) {
    case FKC_F32:
      rc = launch_f32_t<FKC_F32>(x, c, x_sq, c_sq, ids, B, N, K, D, ctrl, s);
      break;
    case FKC_F16:
      rc = launch_f32_t<FKC_F16>(x, c, x_sq, c_sq, ids, B, N, K, D, ctrl, s);
      break;
    case FKC_BF16:
      rc = launch_f32_t<FKC_BF16>(x, c, x_sq, c_sq, ids, B, N, K, D, ctrl, s);
      break;
    default:
      return fail(FKC_ERR_INVALID, "assign: unknown dtype %d", dtype);
  }
  if (ev1 != nullptr) (void)hipEventRecord(ev1, s);
  return rc;
}

void assign_plan(int64_t B, int64_t N, int64_t K, int64_t D, int dtype,
                 bool slices, int32_t out[6]) {
  if (assign_uses_mfma(dtype, D)) {
    assign_mfma_plan(B, N, K, D, slices, out);
    return;
  }
  const F32Kind kind = f32_kind(B, N, K, D);
  const F32Plan p = f32_plan(kind, B, N, K, D);
  const int32_t v[6] = {(int32_t)kind, p.m, p.pt, p.ct, p.ks, (int32_t)K};
  std::copy(v, v + 6, out);
}

int launch_row_sqnorm(const void* src, float* out, int64_t rows, int64_t D,
                      int dtype, const int32_t* ctrl, hipStream_t s) {
  if (rows == 0) return FKC_OK;
  switch (dtype) {
    case FKC_F32: return launch_rowsq_t<FKC_F32>(src, out, rows, D, ctrl, s);
    case FKC_F16: return launch_rowsq_t<FKC_F16>(src, out, rows, D, ctrl, s);
    case FKC_BF16: return launch_rowsq_t<FKC_BF16>(src, out, rows, D, ctrl, s);
  }
  return fail(FKC_ERR_INVALID, "row_sqnorm: unknown dtype %d", dtype);
}

}  // namespace fkc
