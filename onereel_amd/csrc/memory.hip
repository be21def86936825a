// Bounded cross-scene memory on the GPU: the per-head choice of representatives among the boundary-frame keys
// (k-means over L2-normalised keys, one medoid per non-empty cluster) and the per-(head, piece) key lists of the
// head-major attention that reads them.
//
// Reference: BoundaryMemory.select (src/onereel/memory.py:58-93) and the index building of MemoryAttention.__call__
// (memory.py:152-168). The reference runs torch ops: batched fp32 matmuls for the distances, one-hot matmuls for the
// cluster sums, a host read per iteration for the convergence test, stable sorts for the tie-break.
//
// Here, per call:
//   prep     one wavefront per (candidate, 16 heads): inv = 1 / max(|row|, 1e-12) and |x|^2 of x = row * inv in fp32. bf16
//            keys are left where they are and x is formed again from row and inv wherever it is used (the same fp32
//            product; half the bytes of a stored x); fp32 keys are stored as x [H, B, D].
//   start    |c|^2 of the centroids; a cold start first copies the evenly spaced candidates into them.
//   assign   dot products x . c by fp32 MFMA (v_mfma_f32_16x16x4_f32), d = |x|^2 - 2 x . c + |c|^2, the nearest centroid
//            (the lowest index on equal distances).
//   update   per cluster: the mean of its members in ascending order (fp32, four partial sums), or the old centroid when
//            the cluster is empty; a flag per head records whether any of its centroids moved.
//   medoid   one workgroup per head: per non-empty cluster, in cluster order, the member nearest its centroid (the
//            lowest candidate on equal distances) -> rep[h, r] (int64) and valid[h, r] = 1, then zeros.
// assign / update of iteration it > 0 return at once for the heads whose centroids iteration it - 1 did not move (a
// fixed point: every later iteration would give the same assignment), so the host launches all passes without reading
// anything back, and the result equals a loop that stops at convergence. A pass that finds nothing to do costs its
// launch, so the grids are about two blocks per CU whatever the sizes.
// Measured, 12 720 candidates x 16 heads x 128, M = 128: prep 49 -> 12.5 us, an assign 97 -> 79, an update 37 -> 25 (and a
// counting sort of the candidates ahead of it 25 -> 0: every update block finds its clusters' members itself), medoids
// 22 -> 12. 2340 candidates, first pass of a request: assign 23.5 -> 18, sort and update 17 to 35 -> 9 to 13.
#include <math.h>

#include <algorithm>

#include "common.h"

namespace onereel {

namespace {

constexpr int kMaxClusters = 1024;  // M of one call (one thread of the medoid kernel each)
constexpr int kAssignThreads = 256;  // 4 wavefronts
constexpr int kAssignTiles = 32;     // 16-candidate tiles per assign block at most (their results wait in LDS)
constexpr int kPassBlocks = 512;     // blocks of an assign pass: two per CU
constexpr int kUpdThreads = 512;
constexpr int kUpdClusters = kUpdThreads / 128;   // clusters per update block
constexpr int kUpdPer = 8;           // assignments per thread and chunk of an update block
constexpr int kUpdChunk = kUpdThreads * kUpdPer;  // candidates looked at at once
constexpr int kUpdFly = 16;          // member rows in flight per thread

typedef float f32x4v __attribute__((ext_vector_type(4)));

struct SelArgs {
  const void* keys;         // candidate key rows: bf16 or fp32
  const int32_t* rows;      // [B] row of each candidate in keys (NULL: candidate b is row b)
  int64_t stride;           // elements between consecutive rows of keys
  int B, H, D, M, fp32_in, iters;
  float* X;                 // [H, B, D] normalised keys (fp32 keys only: bf16 keys have no room for it)
  float* inv;               // [H, B] 1 / max(|key|, 1e-12)
  float* xx;                // [H, B] |x|^2
  float* C;                 // [H, M, D] centroids (in / out)
  float* cc;                // [H, M] |c|^2 of the current centroids
  int32_t* z;               // [H, B] cluster of each candidate
  float* dist;              // [H, B] its squared distance to that centroid
  int32_t* moved;           // [iters + 1, H] moved[it, h] != 0: iteration it changed a centroid of head h
  int64_t* rep;             // [H, M]
  uint8_t* valid;           // [H, M]
};

// ------------------------------------------------------------------------------------------------------------------
// prep: one wavefront per (candidate b, group of 64 / LPH heads); LPH = D / 32 lanes per head, 32 consecutive elements
// per lane (4 x 16-byte loads of bf16, or 8 of fp32), the head's |row|^2 summed over its lanes by shuffles
template <int D>
__global__ __launch_bounds__(256) void mem_prep_kernel(SelArgs g, int n_moved) {
  constexpr int LPH = D / 32, HPW = 64 / LPH;   // lanes per head, heads per wavefront
  const int lane = threadIdx.x & 63;
  const int b = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int h = blockIdx.y * HPW + lane / LPH, part = lane % LPH;
  if (blockIdx.x == 0 && blockIdx.y == 0)
    for (int i = threadIdx.x; i < n_moved; i += 256) g.moved[i] = 0;   // until an update says otherwise
  if (b >= g.B) return;
  const bool live = h < g.H;
  const int64_t row = g.rows ? g.rows[b] : b;
  float v[32];
  const int64_t off = row * g.stride + (int64_t)min(h, g.H - 1) * D + 32 * part;
  if (g.fp32_in) {
    const f32x4v* p = (const f32x4v*)((const float*)g.keys + off);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const f32x4v t = p[k];
#pragma unroll
      for (int j = 0; j < 4; ++j) v[4 * k + j] = t[j];
    }
  } else {
    const u32x4* p = (const u32x4*)((const uint16_t*)g.keys + off);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const u32x4 t = p[k];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        v[8 * k + 2 * j] = bf2f((uint16_t)(t[j] & 0xffffu));
        v[8 * k + 2 * j + 1] = bf2f((uint16_t)(t[j] >> 16));
      }
    }
  }
  float ss = 0.0f;
#pragma unroll
  for (int e = 0; e < 32; ++e) ss += v[e] * v[e];
#pragma unroll
  for (int o = 1; o < LPH; o <<= 1) ss += __shfl_xor(ss, o, 64);
  const float inv = 1.0f / fmaxf(sqrtf(ss), 1e-12f);
  float q = 0.0f;
#pragma unroll
  for (int e = 0; e < 32; ++e) {
    v[e] *= inv;
    q += v[e] * v[e];
  }
#pragma unroll
  for (int o = 1; o < LPH; o <<= 1) q += __shfl_xor(q, o, 64);
  if (!live) return;
  if (g.fp32_in) {
    f32x4v* x = (f32x4v*)(g.X + ((int64_t)h * g.B + b) * D + 32 * part);
#pragma unroll
    for (int k = 0; k < 8; ++k) x[k] = f32x4v{v[4 * k], v[4 * k + 1], v[4 * k + 2], v[4 * k + 3]};
  }
  if (part == 0) {
    g.inv[(int64_t)h * g.B + b] = inv;
    g.xx[(int64_t)h * g.B + b] = q;
  }
}

// |c|^2 of a centroid held one element per thread (threads 0..D-1 of a 128-thread group), summed by a fixed tree in
// LDS: the same bits wherever it is computed
__device__ __forceinline__ float centroid_norm2(float c, int d, int D, float* red) {
  if (d < 128) red[d] = d < D ? c * c : 0.0f;   // threads with d >= 128 only take part in the barriers
  __syncthreads();
  for (int o = 64; o >= 1; o >>= 1) {
    if (d < o) red[d] += red[d + o];
    __syncthreads();
  }
  const float r = red[0];
  __syncthreads();
  return r;
}

// start of a call: a cold start copies x of candidate init[i] into centroid i; every start computes |c|^2
__global__ __launch_bounds__(128) void mem_start_kernel(SelArgs g, const int32_t* init) {
  __shared__ float red[128];
  const int i = blockIdx.x, h = blockIdx.y, d = threadIdx.x;
  float* dst = g.C + ((int64_t)h * g.M + i) * g.D;
  float c = 0.0f;
  if (d < g.D) {
    if (!init) {
      c = dst[d];
    } else if (g.fp32_in) {
      c = g.X[((int64_t)h * g.B + init[i]) * g.D + d];
    } else {
      const int64_t row = g.rows ? g.rows[init[i]] : init[i];
      c = bf2f(((const uint16_t*)g.keys)[row * g.stride + (int64_t)h * g.D + d]) * g.inv[(int64_t)h * g.B + init[i]];
    }
    if (init) dst[d] = c;
  }
  const float n2 = centroid_norm2(c, d, g.D, red);
  if (d == 0) g.cc[(int64_t)h * g.M + i] = n2;
}

// ------------------------------------------------------------------------------------------------------------------
// assign: bound by the fp32 matrix rate (B x M x D x 2 FLOP; 135 TFLOP/s in a bare loop: 49 us at 12 720 candidates x 16
// heads x 128 clusters x 128). A wavefront keeps 32 centroids in registers for the whole pass and streams 16-candidate
// tiles past them; the wavefronts of a block split the centroids (WR = 1: four groups of 32) or, with few of them, the
// tiles (up to 64 clusters: WR = 2, up to 32: WR = 4). The block reads WR tiles a stage ahead in whole rows, forms x and
// leaves it in LDS, where every wavefront finds its operands: gathered by each wavefront from memory in operand order
// (16 bytes here and there of 32 lines per load) a pass took 85 to 97 us, and so it did with the centroids in LDS and
// the candidates in registers.
// MFMA 16x16x4 f32: lane l supplies A[l % 16][l / 16] (a centroid) and B[l / 16][l % 16] (a candidate) and holds
// D[4 (l / 16) + r][l % 16]: four centroids of one candidate, so that the nearest is found in the lane but for two
// exchanges. The reduction dimension is visited in the order d = (l / 16) * (D / 4) + s at step s (any order of the same
// products is the same dot product), so that every lane reads D / 4 consecutive elements of its row and centroid.
template <int D, bool BF, int WR>
struct StageIn {
  static constexpr int ROWS = 16 * WR;
  static constexpr int PER = ROWS * (D / 8) / kAssignThreads > 0 ? ROWS * (D / 8) / kAssignThreads : 1;
  u32x4 raw[PER][BF ? 1 : 2];   // 8 elements of a row per thread and step
  float inv[PER], xx[PER];
};

__device__ __forceinline__ bool nearer(float d, int i, float od, int oi) { return d < od || (d == od && i < oi); }

template <int D, bool BF, int WR>
__global__ __launch_bounds__(kAssignThreads) __attribute__((amdgpu_waves_per_eu(2, 2)))
void mem_assign_kernel(SelArgs g, int it) {
  const int h = blockIdx.y;
  if (it > 0 && g.moved[(int64_t)(it - 1) * g.H + h] == 0) return;
  typedef StageIn<D, BF, WR> Stage;
  constexpr int KS = D / 4;          // MFMA steps per dot product
  constexpr int WC = 4 / WR;         // centroid groups
  constexpr int PITCH = D + 4;       // floats per row in LDS (16 rows of one 16-byte column on different banks)
  constexpr int CPR = D / 8;         // 8-element chunks per row
  __shared__ __attribute__((aligned(16))) float xs[2][Stage::ROWS > 32 ? Stage::ROWS : 32][PITCH];   // centroids first
  __shared__ float xxs[2][Stage::ROWS];
  __shared__ float bestv[WC][16 * kAssignTiles];
  __shared__ int besti[WC][16 * kAssignTiles];
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kq = lane >> 4, c16 = lane & 15;
  const int cw = w % WC, rw = w / WC;   // this wavefront's centroid group and tile of a stage
  const int tiles = (g.B + 15) / 16, nb = gridDim.x;
  const int mine = ((int)blockIdx.x < tiles ? (tiles - 1 - (int)blockIdx.x) / nb : -1) + 1;   // this block's tiles
  const int stages = (mine + WR - 1) / WR;
  // candidate of row r of a stage (past the last: the last one again, not stored)
  auto cand_of = [&](int stage, int r) {
    return min(16 * ((int)blockIdx.x + nb * (WR * stage + (r >> 4))) + (r & 15), g.B - 1);
  };
  const bool loads = Stage::ROWS * CPR >= kAssignThreads || tid < Stage::ROWS * CPR;
  auto load_rows = [&](int stage, int (&row)[Stage::PER]) {
#pragma unroll
    for (int p = 0; p < Stage::PER; ++p) {
      const int b = cand_of(stage, (tid + p * kAssignThreads) / CPR % Stage::ROWS);
      row[p] = BF && g.rows ? g.rows[b] : b;
    }
  };
  auto load_stage = [&](int stage, const int (&row)[Stage::PER], Stage& in) {
#pragma unroll
    for (int p = 0; p < Stage::PER; ++p) {
      const int e = tid + p * kAssignThreads, c = e % CPR;
      const int64_t hb = (int64_t)h * g.B + cand_of(stage, e / CPR % Stage::ROWS);
      if constexpr (BF) {
        in.raw[p][0] = *(const u32x4*)((const uint16_t*)g.keys + row[p] * g.stride + (int64_t)h * D + 8 * c);
        in.inv[p] = g.inv[hb];
      } else {
        const u32x4* x = (const u32x4*)(g.X + hb * D + 8 * c);
        in.raw[p][0] = x[0];
        in.raw[p][1] = x[1];
      }
      in.xx[p] = g.xx[hb];
    }
  };
  auto store_stage = [&](int buf, const Stage& in) {
    if (loads)
#pragma unroll
      for (int p = 0; p < Stage::PER; ++p) {
        const int e = tid + p * kAssignThreads, r = e / CPR, c = e % CPR;
        f32x4v* o = (f32x4v*)&xs[buf][r][8 * c];
        if constexpr (BF) {
          float x[8];
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            x[2 * j] = bf2f((uint16_t)(in.raw[p][0][j] & 0xffffu)) * in.inv[p];
            x[2 * j + 1] = bf2f((uint16_t)(in.raw[p][0][j] >> 16)) * in.inv[p];
          }
          o[0] = f32x4v{x[0], x[1], x[2], x[3]};
          o[1] = f32x4v{x[4], x[5], x[6], x[7]};
        } else {
          o[0] = __builtin_bit_cast(f32x4v, in.raw[p][0]);
          o[1] = __builtin_bit_cast(f32x4v, in.raw[p][1]);
        }
        if (c == 0) xxs[buf][r] = in.xx[p];
      }
  };
  const float* Ch = g.C + (int64_t)h * g.M * D;
  for (int c0 = 0; c0 < g.M; c0 += 32 * WC) {
    const int ci = c0 + 32 * cw;    // this wavefront's first centroid (past the last: its results stay infinite)
    int row[Stage::PER];
    Stage in;
    load_rows(0, row);
    // the centroids by whole rows through LDS, 16 of every group at a time (group k in rows 16 k ..)
    f32x4v cen[2][KS / 4];
    float cc[2][4];
    float* cs = &xs[0][0][0];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      constexpr int N = 16 * WC * (D / 4) / kAssignThreads;   // 16-byte chunks per thread
      f32x4v v[N];
#pragma unroll
      for (int n = 0; n < N; ++n) {
        const int e = tid + n * kAssignThreads, r = e / (D / 4), i = c0 + 32 * (r >> 4) + 16 * t + (r & 15);
        v[n] = *(const f32x4v*)(Ch + (int64_t)min(i, g.M - 1) * D + 4 * (e % (D / 4)));
      }
      __syncthreads();   // what the buffer held is no longer read
#pragma unroll
      for (int n = 0; n < N; ++n) {
        const int e = tid + n * kAssignThreads;
        *(f32x4v*)(cs + e / (D / 4) * PITCH + 4 * (e % (D / 4))) = v[n];
      }
      __syncthreads();
#pragma unroll
      for (int s = 0; s < KS / 4; ++s) cen[t][s] = *(const f32x4v*)(cs + (16 * cw + c16) * PITCH + kq * KS + 4 * s);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = ci + 16 * t + 4 * kq + r;
        const float v1 = g.cc[(int64_t)h * g.M + min(i, g.M - 1)];
        cc[t][r] = i < g.M ? v1 : __builtin_inff();
      }
    }
    load_stage(0, row, in);
    load_rows(1, row);
    __syncthreads();     // the centroids are in registers
    store_stage(0, in);
    load_stage(1, row, in);
    load_rows(2, row);
    for (int st = 0; st < stages; ++st) {
      __syncthreads();   // stage st is in its buffer, and stage st - 1 no longer read
      store_stage((st + 1) & 1, in);
      load_stage(st + 2, row, in);
      load_rows(st + 3, row);
      const int n = WR * st + rw;
      f32x4v x[KS / 4];
#pragma unroll
      for (int s = 0; s < KS / 4; ++s) x[s] = *(const f32x4v*)&xs[st & 1][16 * rw + c16][kq * KS + 4 * s];
      const float xx = xxs[st & 1][16 * rw + c16];
      f32x4v acc[2] = {f32x4v{0.0f, 0.0f, 0.0f, 0.0f}, f32x4v{0.0f, 0.0f, 0.0f, 0.0f}};
#pragma unroll
      for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int t = 0; t < 2; ++t)
          acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(cen[t][s / 4][s % 4], x[s / 4][s % 4], acc[t], 0, 0, 0);
      float best = __builtin_inff();
      int bi = 0;   // stays 0 only if no distance is finite (non-finite keys): still a valid cluster
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float dd = (xx - 2.0f * acc[t][r]) + cc[t][r];
          if (dd < best) {    // centroids visited in ascending order: the first minimum stays
            best = dd;
            bi = ci + 16 * t + 4 * kq + r;
          }
        }
#pragma unroll
      for (int o = 16; o <= 32; o <<= 1) {
        const float od = __shfl_xor(best, o, 64);
        const int oi = __shfl_xor(bi, o, 64);
        const bool nr = nearer(od, oi, best, bi);
        best = nr ? od : best;
        bi = nr ? oi : bi;
      }
      if (kq == 0 && n < mine) {   // this wavefront's own entries
        const int e = 16 * n + c16;
        if (c0 == 0 || nearer(best, bi, bestv[cw][e], besti[cw][e])) {
          bestv[cw][e] = best;
          besti[cw][e] = bi;
        }
      }
    }
  }
  __syncthreads();
  for (int e = tid; e < 16 * mine; e += kAssignThreads) {
    const int b = 16 * ((int)blockIdx.x + nb * (e >> 4)) + (e & 15);
    float best = bestv[0][e];
    int bi = besti[0][e];
#pragma unroll
    for (int k = 1; k < WC; ++k)
      if (nearer(bestv[k][e], besti[k][e], best, bi)) {
        best = bestv[k][e];
        bi = besti[k][e];
      }
    if (b < g.B) {
      g.z[(int64_t)h * g.B + b] = bi;
      g.dist[(int64_t)h * g.B + b] = best;
    }
  }
}

// ------------------------------------------------------------------------------------------------------------------
// update: a block averages kUpdClusters clusters of one head, 128 threads each: four groups of 32 take the members j = q,
// q + 4, ... (group q) in ascending order, four elements of D per thread, and the four partial sums are added in group
// order. The block finds the members itself: it reads the head's assignments (from the L2: a few tens of KB) a chunk at a
// time, wavefront w the w-th part of a chunk; one ballot per 64 assignments gathers the members of any of its clusters,
// and a wavefront per cluster then picks its own from those few.
// Bound by latency for small clusters (assignments, member rows) and by the read of the keys for many: one cluster per
// block with four rows of 4-byte loads in flight took 28 us where the first passes put hundreds of keys into one cluster.
template <int D, bool BF>
__global__ __launch_bounds__(kUpdThreads) void mem_update_kernel(SelArgs g, int it) {
  const int h = blockIdx.y;
  if (it > 0 && g.moved[(int64_t)(it - 1) * g.H + h] == 0) return;
  constexpr int W = kUpdThreads / 64, K = kUpdClusters;
  __shared__ int found[kUpdChunk];      // the chunk's members of any of the clusters, cluster << 16 | place in the chunk
  __shared__ int mrow[kUpdChunk];       // cluster after cluster, ascending: the members' key rows (fp32: candidates)
  __shared__ float minv[kUpdChunk];
  __shared__ int wcnt[W], beg[K], len[K];
  __shared__ float part[K][4][128];
  __shared__ float norm[K][128];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int i0 = blockIdx.x * K;
  const int k = tid >> 7, q = (tid >> 5) & 3, d4 = 4 * (tid & 31);   // this thread's cluster, member group and elements
  const int32_t* zh = g.z + (int64_t)h * g.B;
  const uint64_t below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
  f32x4v sum = {0.0f, 0.0f, 0.0f, 0.0f};
  int seen = 0;     // members of cluster k in the chunks before
  for (int c0 = 0; c0 < g.B; c0 += kUpdChunk) {
    int zi[kUpdPer];
#pragma unroll
    for (int u = 0; u < kUpdPer; ++u) {
      const int b = c0 + w * (64 * kUpdPer) + 64 * u + lane;
      const int z = zh[min(b, g.B - 1)];
      zi[u] = b < g.B ? z - i0 : -1;
    }
    int cnt = 0;
    uint64_t bal[kUpdPer];
#pragma unroll
    for (int u = 0; u < kUpdPer; ++u) {
      bal[u] = __ballot(zi[u] >= 0 && zi[u] < K);
      cnt += __popcll(bal[u]);
    }
    if (lane == 0) wcnt[w] = cnt;
    __syncthreads();   // the lists of the chunk before are no longer read either
    int at = 0, all = 0;
#pragma unroll
    for (int x = 0; x < W; ++x) {
      if (x < w) at += wcnt[x];
      all += wcnt[x];
    }
#pragma unroll
    for (int u = 0; u < kUpdPer; ++u) {
      if (zi[u] >= 0 && zi[u] < K) found[at + __popcll(bal[u] & below)] = zi[u] << 16 | (w * (64 * kUpdPer) + 64 * u + lane);
      at += __popcll(bal[u]);
    }
    __syncthreads();
    if ((w & 1) == 0) {   // the first wavefront of each cluster picks its own
      int before = 0, n = 0;
      for (int x = 0; x < all; x += 64) before += __popcll(__ballot(x + lane < all && found[x + lane] >> 16 < k));
      for (int x = 0; x < all; x += 64) {
        const int f = x + lane < all ? found[x + lane] : -1;
        const uint64_t own = __ballot(f >> 16 == k);
        if (f >> 16 == k) {
          const int place = before + n + __popcll(own & below), b = c0 + (f & 0xffff);
          mrow[place] = BF && g.rows ? g.rows[b] : b;
          if constexpr (BF) minv[place] = g.inv[(int64_t)h * g.B + b];
        }
        n += __popcll(own);
      }
      if (lane == 0) {
        beg[k] = before;
        len[k] = n;
      }
    }
    __syncthreads();
    const int n = len[k], mine = beg[k];
    if (d4 < D) {
      for (int m = (q - seen) & 3; m < n; m += 4 * kUpdFly) {
        f32x4v x[kUpdFly];
#pragma unroll
        for (int u = 0; u < kUpdFly; ++u) {
          const int j = mine + min(m + 4 * u, n - 1);
          if constexpr (BF) {
#pragma clang fp contract(off)
            const uint2 v = *(const uint2*)((const uint16_t*)g.keys + mrow[j] * g.stride + (int64_t)h * D + d4);
            const float inv = minv[j];
            x[u] = f32x4v{bf2f((uint16_t)(v.x & 0xffffu)) * inv, bf2f((uint16_t)(v.x >> 16)) * inv,
                          bf2f((uint16_t)(v.y & 0xffffu)) * inv, bf2f((uint16_t)(v.y >> 16)) * inv};
          } else {
            x[u] = *(const f32x4v*)(g.X + ((int64_t)h * g.B + mrow[j]) * D + d4);
          }
        }
#pragma unroll
        for (int u = 0; u < kUpdFly; ++u)
          if (m + 4 * u < n)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
#pragma clang fp contract(off)
              sum[e] = sum[e] + x[u][e];
            }
      }
    }
    seen += n;
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) part[k][q][d4 + e] = sum[e];
  __syncthreads();
  const int d = tid & 127, i = i0 + k;
  const bool live = i < g.M && seen > 0;   // empty: the centroid (and its |c|^2) stays
  float c = 0.0f;
  bool change = false;
  if (live && d < D) {
    c = ((part[k][0][d] + part[k][1][d]) + part[k][2][d]) + part[k][3][d];
    c = c / (float)seen;
    float* cp = g.C + ((int64_t)h * g.M + i) * D + d;
    change = *cp != c;
    *cp = c;
  }
  // |c|^2 by the tree of centroid_norm2: the halves of the row first, then within a wavefront
  norm[k][d] = c * c;
  const bool any = __syncthreads_or(change);
  if (d < 64) {
    float n2 = norm[k][d] + norm[k][d + 64];
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) n2 += __shfl_down(n2, o, 64);
    if (d == 0 && live) g.cc[(int64_t)h * g.M + i] = n2;
  }
  if (any && tid == 0) atomicOr(&g.moved[(int64_t)it * g.H + h], 1);
}

// ------------------------------------------------------------------------------------------------------------------
// medoid: one workgroup per head. The smallest (distance, candidate) of every cluster by 64-bit minima in LDS (the
// distance's bits mapped so that their order is that of the values); rep / valid compacted in cluster order.
__global__ __launch_bounds__(1024) void mem_medoid_kernel(SelArgs g) {
  __shared__ unsigned long long pick[kMaxClusters];
  __shared__ int wsum[16];
  const int h = blockIdx.x, tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int32_t* zh = g.z + (int64_t)h * g.B;
  const float* dh = g.dist + (int64_t)h * g.B;
  pick[tid] = ~0ull;
  __syncthreads();
  for (int b0 = tid; b0 < g.B; b0 += 4 * 1024) {
    int z[4];
    float d[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int b = min(b0 + 1024 * u, g.B - 1);   // the last candidate again: no change
      z[u] = zh[b];
      d[u] = dh[b];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const uint32_t x = __float_as_uint(d[u] + 0.0f);   // -0 equals +0
      const uint32_t ord = x & 0x80000000u ? ~x : x | 0x80000000u;
      const unsigned long long key = (unsigned long long)ord << 32 | (uint32_t)min(b0 + 1024 * u, g.B - 1);
      if (key < pick[z[u]]) atomicMin(&pick[z[u]], key);
    }
  }
  __syncthreads();
  const bool has = tid < g.M && pick[tid] != ~0ull;
  const uint64_t bal = __ballot(has);
  if (lane == 0) wsum[w] = __popcll(bal);
  __syncthreads();
  int before = 0, total = 0;
#pragma unroll
  for (int x = 0; x < 16; ++x) {
    if (x < w) before += wsum[x];
    total += wsum[x];
  }
  int64_t* rp = g.rep + (int64_t)h * g.M;
  uint8_t* vp = g.valid + (int64_t)h * g.M;
  if (has) {
    const int r = before + __popcll(bal & (lane == 0 ? 0ull : (~0ull >> (64 - lane))));
    rp[r] = (int64_t)(pick[tid] & 0xffffffffull);
    vp[r] = 1;
  }
  if (tid >= total && tid < g.M) {
    rp[tid] = 0;
    vp[tid] = 0;
  }
}

// ------------------------------------------------------------------------------------------------------------------
// foreign keys of the head-major attention: block (piece i, head h) appends, after piece i's local keys, the rows of
// head h's valid representatives that belong to another scene (when the piece reads the memory), in rep order
__global__ __launch_bounds__(256) void mem_index_kernel(const int64_t* rep, const uint8_t* valid, const int64_t* cand_row,
                                                        const int64_t* cand_scene, const int64_t* piece_scene,
                                                        const uint8_t* piece_mem, const int32_t* piece_len,
                                                        const int32_t* k_off, int32_t* kidx, int32_t* k_len, int n,
                                                        int H, int M) {
  __shared__ int wave_cnt[4];
  const int i = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int seg = h * n + i;
  const int base = k_off[seg] + piece_len[i];
  const int64_t scene = piece_scene[i];
  const bool reads = piece_mem[i] != 0;
  int total = 0;
  for (int r0 = 0; r0 < M; r0 += 256) {
    const int r = r0 + tid;
    bool f = false;
    int64_t row = 0;
    if (reads && r < M && valid[(int64_t)h * M + r]) {
      const int64_t c = rep[(int64_t)h * M + r];
      f = cand_scene[c] != scene;
      row = cand_row[c];
    }
    const uint64_t bal = __ballot(f);
    if (lane == 0) wave_cnt[w] = __popcll(bal);
    __syncthreads();
    int before = total;
    for (int x = 0; x < w; ++x) before += wave_cnt[x];
    const uint64_t below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    if (f) kidx[base + before + __popcll(bal & below)] = (int32_t)(row * H + h);
    total += wave_cnt[0] + wave_cnt[1] + wave_cnt[2] + wave_cnt[3];
    __syncthreads();
  }
  if (tid == 0) k_len[seg] = piece_len[i] + total;
}

// The multi-head form of the per-call key lists (the packed K / V hold every head of a row, and each head's
// representatives sit in its own head slot after the piece's local keys): block (i, h) writes, for slot r < M of piece
// i and head h, src = cand_row[c] * H + h (the representative's row in the [rows * H, 1, D] view of the key buffer, or
// -1 for an unused slot) and dst = (k_off[i] + piece_len[i] + r) * H + h (its row in that view of the packed buffer),
// in the representatives' order, and k_len_head[i * H + h] = piece_len[i] + the count. Pieces that do not read the
// memory get no representatives.
__global__ __launch_bounds__(256) void mem_foreign_kernel(const int64_t* rep, const uint8_t* valid,
                                                          const int64_t* cand_row, const int64_t* cand_scene,
                                                          const int64_t* piece_scene, const uint8_t* piece_mem,
                                                          const int32_t* piece_len, const int32_t* k_off,
                                                          int32_t* fsrc, int32_t* fdst, int32_t* k_len_head, int n,
                                                          int H, int M) {
  __shared__ int wave_cnt[4];
  const int i = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int64_t slot0 = ((int64_t)i * H + h) * M;
  const int64_t dst0 = (int64_t)k_off[i] + piece_len[i];
  const int64_t scene = piece_scene[i];
  const bool reads = piece_mem[i] != 0;
  for (int r = tid; r < M; r += 256) {
    fsrc[slot0 + r] = -1;
    fdst[slot0 + r] = (int32_t)((dst0 + r) * H + h);
  }
  __syncthreads();
  int total = 0;
  for (int r0 = 0; r0 < M; r0 += 256) {
    const int r = r0 + tid;
    bool f = false;
    int64_t row = 0;
    if (reads && r < M && valid[(int64_t)h * M + r]) {
      const int64_t c = rep[(int64_t)h * M + r];
      f = cand_scene[c] != scene;
      row = cand_row[c];
    }
    const uint64_t bal = __ballot(f);
    if (lane == 0) wave_cnt[w] = __popcll(bal);
    __syncthreads();
    int before = total;
    for (int x = 0; x < w; ++x) before += wave_cnt[x];
    const uint64_t below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    if (f) fsrc[slot0 + before + __popcll(bal & below)] = (int32_t)(row * H + h);
    total += wave_cnt[0] + wave_cnt[1] + wave_cnt[2] + wave_cnt[3];
    __syncthreads();
  }
  if (tid == 0) k_len_head[(int64_t)i * H + h] = piece_len[i] + total;
}

template <int D, bool BF>
auto assign_fn(int share) {
  return share == 4 ? mem_assign_kernel<D, BF, 4> : share == 2 ? mem_assign_kernel<D, BF, 2> : mem_assign_kernel<D, BF, 1>;
}

struct WsParts {
  int64_t X, inv, xx, cc, z, dist, moved, total;
};

// (bf16 keys need no X)
WsParts ws_parts(int B, int H, int D, int M, int iters, bool fp32_keys) {
  WsParts p;
  int64_t o = 0;
  auto take = [&](int64_t bytes) {
    const int64_t at = o;
    o += (bytes + 255) / 256 * 256;
    return at;
  };
  p.X = take(fp32_keys ? (int64_t)H * B * D * 4 : 0);
  p.inv = take((int64_t)H * B * 4);
  p.xx = take((int64_t)H * B * 4);
  p.cc = take((int64_t)H * M * 4);
  p.z = take((int64_t)H * B * 4);
  p.dist = take((int64_t)H * B * 4);
  p.moved = take((int64_t)(iters + 1) * H * 4);
  p.total = o;
  return p;
}

}  // namespace
}  // namespace onereel

using namespace onereel;

extern "C" int64_t or_memory_select_workspace_bytes(int32_t B, int32_t H, int32_t D, int32_t M, int32_t iters,
                                                    int32_t fp32_keys) {
  if (B < 1 || H < 1 || M < 1 || iters < 0 || (D != 64 && D != 128)) return -1;
  return ws_parts(B, H, D, M, iters, fp32_keys != 0).total;
}

extern "C" int64_t or_memory_select_workspace_size(int32_t B, int32_t H, int32_t D, int32_t M, int32_t iters) {
  return or_memory_select_workspace_bytes(B, H, D, M, iters, 1);
}

extern "C" int or_memory_select(const void* keys, int32_t fp32_keys, const int32_t* rows, int64_t key_row_stride,
                                int32_t B, int32_t H, int32_t D, int32_t M, float* centroids, const int32_t* init,
                                int32_t iters, int64_t* rep, uint8_t* valid, void* workspace, int64_t workspace_bytes,
                                void* stream) {
  if (B < 1 || H < 1 || (D != 64 && D != 128))
    return fail_arg("or_memory_select: need B >= 1, H >= 1 and D 64 or 128 (B=%d H=%d D=%d)", B, H, D);
  if (M < 1 || M > B || M > kMaxClusters)
    return fail_arg("or_memory_select: M=%d outside [1, min(B=%d, %d)]", M, B, kMaxClusters);
  if (iters < 0 || iters > 1000) return fail_arg("or_memory_select: iters=%d outside [0, 1000]", iters);
  if (!keys || !centroids || !rep || !valid || key_row_stride < (int64_t)H * D)
    return fail_arg("or_memory_select: keys, centroids, rep and valid are required, rows of at least H*D elements");
  const WsParts wp = ws_parts(B, H, D, M, iters, fp32_keys != 0);
  if (!workspace || workspace_bytes < wp.total || ((uintptr_t)workspace & 255u))
    return fail_arg("or_memory_select: a 256-byte aligned workspace of %lld bytes is needed", (long long)wp.total);
  if (((uintptr_t)centroids & 15u) || ((uintptr_t)keys & 15u) || key_row_stride % (fp32_keys ? 4 : 8))
    return fail_arg("or_memory_select: centroids and keys must be 16-byte aligned and the key row stride a multiple "
                    "of 16 bytes");
  char* w = (char*)workspace;
  SelArgs g;
  g.keys = keys;
  g.rows = rows;
  g.stride = key_row_stride;
  g.B = B;
  g.H = H;
  g.D = D;
  g.M = M;
  g.fp32_in = fp32_keys ? 1 : 0;
  g.iters = iters;
  g.X = (float*)(w + wp.X);
  g.inv = (float*)(w + wp.inv);
  g.xx = (float*)(w + wp.xx);
  g.cc = (float*)(w + wp.cc);
  g.C = centroids;
  g.z = (int32_t*)(w + wp.z);
  g.dist = (float*)(w + wp.dist);
  g.moved = (int32_t*)(w + wp.moved);
  g.rep = rep;
  g.valid = valid;
  hipStream_t st = (hipStream_t)stream;
  const int n_moved = (iters + 1) * H;
  if (D == 128) hipLaunchKernelGGL(mem_prep_kernel<128>, dim3((B + 3) / 4, (H + 15) / 16), dim3(256), 0, st, g, n_moved);
  else hipLaunchKernelGGL(mem_prep_kernel<64>, dim3((B + 3) / 4, (H + 31) / 32), dim3(256), 0, st, g, n_moved);
  if (int rc = check_hip(hipGetLastError(), "mem_prep_kernel launch")) return rc;
  hipLaunchKernelGGL(mem_start_kernel, dim3(M, H), dim3(128), 0, st, g, init);
  if (int rc = check_hip(hipGetLastError(), "mem_start_kernel launch")) return rc;
  // the tiles of a head over enough blocks to fill the chip twice
  const int share = M <= 32 ? 4 : M <= 64 ? 2 : 1, tiles = (B + 15) / 16;
  const int nb = std::max(std::min((tiles + share - 1) / share, std::max(1, kPassBlocks / H)),
                          (tiles + kAssignTiles - 1) / kAssignTiles);
  const dim3 agrid(nb, H), ugrid((M + kUpdClusters - 1) / kUpdClusters, H);
  const auto assign = D == 128 ? (fp32_keys ? assign_fn<128, false>(share) : assign_fn<128, true>(share))
                               : (fp32_keys ? assign_fn<64, false>(share) : assign_fn<64, true>(share));
  const auto update = D == 128 ? (fp32_keys ? mem_update_kernel<128, false> : mem_update_kernel<128, true>)
                               : (fp32_keys ? mem_update_kernel<64, false> : mem_update_kernel<64, true>);
  for (int it = 0; it <= iters; ++it) {
    hipLaunchKernelGGL(assign, agrid, dim3(kAssignThreads), 0, st, g, it);
    if (it < iters) hipLaunchKernelGGL(update, ugrid, dim3(kUpdThreads), 0, st, g, it);
    if (int rc = check_hip(hipGetLastError(), "k-means launch")) return rc;
  }
  hipLaunchKernelGGL(mem_medoid_kernel, dim3(H), dim3(1024), 0, st, g);
  return check_hip(hipGetLastError(), "mem_medoid_kernel launch");
}

extern "C" int or_memory_index(const int64_t* rep, const uint8_t* valid, const int64_t* cand_row,
                               const int64_t* cand_scene, const int64_t* piece_scene, const uint8_t* piece_mem,
                               const int32_t* piece_len, const int32_t* k_off, int32_t n_pieces, int32_t H, int32_t M,
                               int32_t* kidx, int32_t* k_len, void* stream) {
  if (n_pieces < 1 || H < 1 || M < 1 || n_pieces > 65535 || H > 65535)
    return fail_arg("or_memory_index: need 1 <= pieces, heads <= 65535 and M >= 1 (n=%d H=%d M=%d)", n_pieces, H, M);
  if (!rep || !valid || !cand_row || !cand_scene || !piece_scene || !piece_mem || !piece_len || !k_off || !kidx || !k_len)
    return fail_arg("or_memory_index: every array is required");
  hipLaunchKernelGGL(mem_index_kernel, dim3(n_pieces, H), dim3(256), 0, (hipStream_t)stream, rep, valid, cand_row,
                     cand_scene, piece_scene, piece_mem, piece_len, k_off, kidx, k_len, n_pieces, H, M);
  return check_hip(hipGetLastError(), "mem_index_kernel launch");
}

extern "C" int or_memory_foreign(const int64_t* rep, const uint8_t* valid, const int64_t* cand_row,
                                 const int64_t* cand_scene, const int64_t* piece_scene, const uint8_t* piece_mem,
                                 const int32_t* piece_len, const int32_t* k_off, int32_t n_pieces, int32_t H,
                                 int32_t M, int32_t* fsrc, int32_t* fdst, int32_t* k_len_head, void* stream) {
  if (n_pieces < 1 || H < 1 || M < 1 || n_pieces > 65535 || H > 65535)
    return fail_arg("or_memory_foreign: need 1 <= pieces, heads <= 65535 and M >= 1 (n=%d H=%d M=%d)", n_pieces, H, M);
  if (!rep || !valid || !cand_row || !cand_scene || !piece_scene || !piece_mem || !piece_len || !k_off || !fsrc ||
      !fdst || !k_len_head)
    return fail_arg("or_memory_foreign: every array is required");
  hipLaunchKernelGGL(mem_foreign_kernel, dim3(n_pieces, H), dim3(256), 0, (hipStream_t)stream, rep, valid, cand_row,
                     cand_scene, piece_scene, piece_mem, piece_len, k_off, fsrc, fdst, k_len_head, n_pieces, H, M);
  return check_hip(hipGetLastError(), "mem_foreign_kernel launch");
}
