// Frame memory on the device: per-frame pooling of hidden states, and the k-means (cosine) choice of representative
// frames with their medoids.
//
// Reference: FrameMemory.collect (src/onereel/frame_memory.py:76-85): the per-frame sums and counts of one layer's
// video rows (index_add_), and FrameMemory.select (frame_memory.py:114-132): farthest-point initialisation, k-means
// on L2-normalised features with the dot product as similarity, then per cluster the member most similar to its
// centre (the first on ties). Here:
//
// - frame_pool_kernel: rows are frame-major (frame of row r = (row0 + r) / T, as the one-GPU processors build
//   them), so a frame's rows are contiguous. A block per (frame, 128 columns) adds them in row order:
//   deterministic, unlike an atomic index_add_. Per lane, 2 consecutive columns in fp32. With many short frames
//   frame_pool_wave_kernel, a wavefront per (frame, 512 columns), in the same order: the same bits.
// - frame_select_kernel: the whole selection in one workgroup of 1024 threads, centres in LDS (k * C floats); no
//   host round trip per iteration. Ties are broken towards the lower index, as torch.argmax does. A pass stops when
//   the new centres equal the old ones exactly (torch.equal).
#include <math.h>

#include <algorithm>

#include "common.h"

namespace onereel {

namespace {

constexpr int kPoolThreads = 256;
constexpr int kPoolRows = 64;    // rows per stage of the pooling
constexpr int kSelThreads = 1024;
constexpr int kSelWaves = kSelThreads / 64;
constexpr int kSelRows = 16;      // rows of a column in flight in the member sums
constexpr int kMaxCand = 1024;
constexpr int kMaxCentreFloats = 32768;   // k * C: the centres, 128 KiB of LDS
constexpr int kMaxK = 64;

struct PoolArgs {
  const uint16_t* hs;
  int64_t n_rows, row_stride, row0;
  int C, T, n_frames;
  float* sums;       // [n_frames, C]
  float* counts;     // [n_frames]
};

// A block per (frame, 128 columns): its wavefronts load the frame's rows in whole 256-byte pieces, kPoolRows at a time and
// the next ones in flight, through LDS, and the lanes of the first wavefront, two columns each, add them in row order:
// the sums have the same bits whatever the launch, and the chain of dependent additions is short (1590 rows: 3 us).
// HBM-bound, so what counts is the bytes in flight: 32 frames x 1590 rows x 2048 columns took 168 us with eight columns
// per lane and four rows in flight (128 wavefronts, 1.2 TB/s), 65 with a wavefront per 128 columns that loaded what it
// added in batches of 32 (of 64: 69), now 33 (6.3 TB/s).
__global__ __launch_bounds__(kPoolThreads) void frame_pool_kernel(PoolArgs g) {
  constexpr int PER = kPoolRows * 16 / kPoolThreads;   // 16-byte chunks per thread and stage (16 per row)
  __shared__ __attribute__((aligned(16))) u32x4 buf[2][kPoolRows][16];
  const int f = blockIdx.y, col0 = blockIdx.x * 128, tid = threadIdx.x;
  int64_t r0 = (int64_t)f * g.T - g.row0, r1 = r0 + g.T;
  r0 = r0 < 0 ? 0 : r0;
  r1 = r1 > g.n_rows ? g.n_rows : r1;
  if (r1 <= r0) return;
  const int n = (int)(r1 - r0);
  // this thread's chunk of a row (a chunk past the last column repeats the row's last one; its sums are not stored)
  const uint16_t* p = g.hs + r0 * g.row_stride + min(col0 + 8 * (tid & 15), g.C - 8);
  u32x4 v[PER];
  auto load = [&](int s) {   // stage s, rows past the last repeat it
#pragma unroll
    for (int u = 0; u < PER; ++u)
      v[u] = *(const u32x4*)(p + (int64_t)min(s * kPoolRows + u * (kPoolThreads / 16) + (tid >> 4), n - 1) * g.row_stride);
  };
  float a0 = 0.0f, a1 = 0.0f;
  const int stages = (n + kPoolRows - 1) / kPoolRows;
  load(0);
  for (int s = 0; s < stages; ++s) {
#pragma unroll
    for (int u = 0; u < PER; ++u) buf[s & 1][u * (kPoolThreads / 16) + (tid >> 4)][tid & 15] = v[u];
    if (s + 1 < stages) load(s + 1);
    __syncthreads();   // stage s is there; the sums of stage s - 2 in this half are long done (the barrier before)
    if (tid < 64) {
      const uint32_t* x = (const uint32_t*)&buf[s & 1][0][0] + tid;
      const int rows = min(kPoolRows, n - s * kPoolRows);
      if (rows == kPoolRows) {
#pragma unroll
        for (int r = 0; r < kPoolRows; ++r) {
          a0 += bf2f((uint16_t)(x[64 * r] & 0xffffu));
          a1 += bf2f((uint16_t)(x[64 * r] >> 16));
        }
      } else {
        for (int r = 0; r < rows; ++r) {
          a0 += bf2f((uint16_t)(x[64 * r] & 0xffffu));
          a1 += bf2f((uint16_t)(x[64 * r] >> 16));
        }
      }
    }
  }
  const int col = col0 + 2 * tid;
  if (tid < 64 && col < g.C) {
    float* sp = g.sums + (int64_t)f * g.C + col;
    sp[0] += a0;
    sp[1] += a1;
    if (col == 0) g.counts[f] += (float)n;
  }
}

// The same sums, a wavefront per (frame, 512 columns): eight columns per lane, four rows in flight, no LDS and no barrier.
// Where its wavefronts fill the chip by themselves, what a block of frame_pool_kernel costs beside the rows (a stage of 64
// rows however few there are, the barriers) is what counts: 5000 frames of one row of 1024 columns 46 -> 7 us, 240 frames
// of 48 rows x 3072 columns 16.6 -> 12.5.
__global__ __launch_bounds__(kPoolThreads) void frame_pool_wave_kernel(PoolArgs g) {
  const int lane = threadIdx.x & 63;
  const int cb = blockIdx.x * (kPoolThreads / 64) + (threadIdx.x >> 6);   // 512-column block
  const int f = blockIdx.y, col = cb * 512 + 8 * lane;
  int64_t r0 = (int64_t)f * g.T - g.row0, r1 = r0 + g.T;
  r0 = r0 < 0 ? 0 : r0;
  r1 = r1 > g.n_rows ? g.n_rows : r1;
  if (r1 <= r0 || col >= g.C) return;
  float acc[8] = {};
  auto add = [&](const u32x4& v) {
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      acc[2 * p] += bf2f((uint16_t)(v[p] & 0xffffu));
      acc[2 * p + 1] += bf2f((uint16_t)(v[p] >> 16));
    }
  };
  const uint16_t* p = g.hs + r0 * g.row_stride + col;
  int n = (int)(r1 - r0);
  for (; n >= 4; n -= 4, p += 4 * g.row_stride) {
    u32x4 v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) v[u] = *(const u32x4*)(p + u * g.row_stride);
#pragma unroll
    for (int u = 0; u < 4; ++u) add(v[u]);
  }
  for (; n > 0; --n, p += g.row_stride) add(*(const u32x4*)p);
  float* sp = g.sums + (int64_t)f * g.C + col;
#pragma unroll
  for (int e = 0; e < 8; ++e) sp[e] += acc[e];
  if (col == 0) g.counts[f] += (float)(r1 - r0);
}

// Which of the two pools a call: w wavefronts of 512 columns. Staged / direct, us: up to 32 rows a frame the direct kernel
// from 400 wavefronts on (20 000 frames x 16 rows x 64 columns 36 / 19, 100 x 24 x 3072 5.7 / 4.4; 1000 x 24 x 64, 125
// wavefronts, 3.7 / 5.8), up to 48 from 1500 on (20 000 x 48 x 64 46 / 39; 5000 x 48 x 128, 1250, 12.7 / 16). Past that only
// with whole wavefronts of columns (5000 x 64 x 128: 16.5 / 19.4) and from 700 on, where a stage or two are less than full
// (200 x 64 x 2048 12.0 / 11.0, 240 x 192 x 2048 29.6 / 27.4; 150 x 64 x 2048, 600 wavefronts, 9.7 / 10.1; 400 x 128 x 3072,
// 2400 wavefronts, 51 / 59), or while eight wavefronts per CU hold the whole call (240 x 1590 x 3072 404 / 384, 400 x 1590 x
// 2048 446 / 422; 240 x 1590 x 2048, 960 wavefronts, 269 / 302; 400 x 1590 x 3072, 2400 wavefronts, 670 / 761).
static bool pool_by_wave(int64_t frames, int C, int T) {
  const int64_t w = frames * C / 512;
  if (T <= 32) return w >= 400;
  if (T <= 48 && w >= 1500) return true;
  if (C < 512 || w < 700) return false;
  return T <= 96 || (w <= 2048 && (T < 200 || w >= 1200));
}

// sum over the 64 lanes, the same in every lane: the tree of a butterfly with partners 32, 16, 8, 4, 2 and 1 lanes away,
// on the vector unit (after the first steps the lanes of a row of 16 repeat every 8, 4, .. lanes, so that a rotation
// reaches the partner's value)
__device__ __forceinline__ float wave_sum_xor(float v) {
  auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(p[0]) + __uint_as_float(p[1]);
  auto q = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(q[0]) + __uint_as_float(q[1]);
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x128, 0xf, 0xf, false));   // row_ror:8
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x124, 0xf, 0xf, false));   // row_ror:4
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xf, 0xf, false));    // quad_perm 2301
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xf, 0xf, false));    // quad_perm 1032
  return v;
}

// the candidate frames of a selection, passed with the launch (no copy to the device ahead of it)
struct CandTable {
  uint16_t frame[kMaxCand];
};

struct SelectArgs {
  const float* feats;      // [n_frames, C], rows L2-normalised
  const int32_t* cand;     // [n_cand] candidate frames, or NULL: the table
  int n_cand, C, k, iters;
  int32_t* reps;           // [k] out: chosen frames ascending, -1 after them
  float* work;             // [8, C] workspace
};

// two candidate rows against the first `live` (at most NQ) rows of `cv`, C floats apart: acc[i][q] is the lane's share of
// row i . cv_q, over e = lane, lane + 64, ... in that order. Both rows' loads go out together, 8 steps at a time.
template <int NQ>
__device__ __forceinline__ void dots(const float* x0, const float* x1, const float* cv, int live, int C, int lane,
                                     float (&acc)[2][NQ]) {
  constexpr int FLY = 8;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int q = 0; q < NQ; ++q) acc[i][q] = 0.0f;
  for (int e0 = lane; e0 < C; e0 += 64 * FLY) {
    float a[FLY], b[FLY];
#pragma unroll
    for (int u = 0; u < FLY; ++u) {
      const int e = min(e0 + 64 * u, C - 1);
      a[u] = x0[e];
      b[u] = x1[e];
    }
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      if (q >= live) break;
      float c[FLY];   // no branch around a load: elements past the row multiply zeros
#pragma unroll
      for (int u = 0; u < FLY; ++u) c[u] = cv[q * C + min(e0 + 64 * u, C - 1)];
#pragma unroll
      for (int u = 0; u < FLY; ++u) {
        const bool in = e0 + 64 * u < C;
        const float cu = in ? c[u] : 0.0f;
        acc[0][q] += (in ? a[u] : 0.0f) * cu;
        acc[1][q] += (in ? b[u] : 0.0f) * cu;
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
}

// first index of the maximum of v[0 .. n), over one wavefront (n >= 1; the same in every lane). NaN entries never win
// over an earlier entry.
__device__ __forceinline__ int wave_argmax(const float* v, int n, int lane) {
  float best = -INFINITY;
  int bi = 0x7fffffff;
  for (int i = lane; i < n; i += 64)
    if (bi == 0x7fffffff || v[i] > best) {   // ascending i per lane: its first maximum
      best = v[i];
      bi = i;
    }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    const float b = __shfl_xor(best, o, 64);
    const int j = __shfl_xor(bi, o, 64);
    if (b > best || (b == best && j < bi)) {
      best = b;
      bi = j;
    }
  }
  return bi < n ? bi : 0;
}

// The whole choice in one workgroup: every pass is a few microseconds of dependent loads from the L2, so the passes are
// few and each keeps many loads in flight: two candidate rows per wavefront and 8 steps of each at once, no branch around
// a load, 16 rows of two columns at once in the member sums (the candidates taken cluster by cluster, so that a row is
// added once and not to each of eight sums), and the similarities of the last assignment serve the medoids. Every sum
// keeps the order of a plain loop over lanes and rows: in a cluster of two, both members are equally similar to their
// mean, so a sum taken in another order would choose the other one.
// 32 candidates x 2048 columns, 4 centres: 157 us (one 4-byte load at a time per thread, a pass over the candidates and
// a block-wide argmax tree per medoid), 81 with the loads batched under branches, sums by selection and shuffles through
// LDS, now 63 (16 steps at once spilled: 71).
__global__ __launch_bounds__(kSelThreads) void frame_select_kernel(SelectArgs g, CandTable table) {
  extern __shared__ __attribute__((aligned(16))) float smem[];
  float* c = smem;                  // [k, C] centres
  float* mrow = g.work;             // [8, C] means of the eight clusters being updated (global workspace)
  __shared__ float dv[kMaxCand];    // per-candidate scores
  __shared__ int z[kMaxCand];       // assignment
  __shared__ int cand[kMaxCand];
  __shared__ int order[kMaxCand];   // the candidates, cluster by cluster
  __shared__ float sv[8 * kSelWaves];
  __shared__ int centre[kMaxK];
  __shared__ int cnt[kMaxK];
  __shared__ int changed;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int nc = g.n_cand, C = g.C, k = g.k;
  for (int n = tid; n < nc; n += kSelThreads) {
    cand[n] = g.cand ? g.cand[n] : table.frame[n];
    dv[n] = INFINITY;
  }
  if (tid == 0) centre[0] = 0;
  __syncthreads();
  auto row = [&](int n) { return g.feats + (int64_t)cand[min(n, nc - 1)] * C; };

  // farthest-point initialisation: centre 0 is candidate 0, then each time the candidate whose nearest chosen
  // centre is farthest (largest 1 - dot)
  for (int m = 1; m < k; ++m) {
    const float* xc = row(centre[m - 1]);
    for (int n = 2 * w; n < nc; n += 2 * kSelWaves) {
      float acc[2][1];
      dots<1>(row(n), row(n + 1), xc, 1, C, lane, acc);
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const float d = 1.0f - wave_sum_xor(acc[i][0]);
        if (lane == 0 && n + i < nc) dv[n + i] = fminf(dv[n + i], d);
      }
    }
    __syncthreads();
    if (w == 0) {
      const int a = wave_argmax(dv, nc, lane);
      if (lane == 0) centre[m] = a;
    }
    __syncthreads();
  }
  for (int i = 0; i < k; ++i) {
    const float* x = row(centre[i]);
    for (int e = tid; e < C; e += kSelThreads) c[i * C + e] = x[e];
  }
  __syncthreads();

  // k-means: z = the most similar centre (first on ties); centre i = normalize(mean of its members), unchanged when
  // it has none; stop when no centre changed. After the loop z belongs to the final centres. Centres are taken eight
  // at a time, so that a candidate row is read once per eight dot products and the member sums of eight clusters
  // (in row order) are one pass over their rows. dv: each candidate's similarity to its centre.
  for (int it = 0;; ++it) {
    for (int n = 2 * w; n < nc; n += 2 * kSelWaves) {
      float best[2] = {0.0f, 0.0f};
      int bi[2] = {0, 0};
      for (int i0 = 0; i0 < k; i0 += 8) {
        float acc[2][8];
        dots<8>(row(n), row(n + 1), c + i0 * C, k - i0, C, lane, acc);
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          if (i0 + q >= k) break;
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            const float d = wave_sum_xor(acc[i][q]);
            if (i0 + q == 0 || d > best[i]) {
              best[i] = d;
              bi[i] = i0 + q;
            }
          }
        }
      }
      if (lane == 0)
#pragma unroll
        for (int i = 0; i < 2; ++i)
          if (n + i < nc) {
            z[n + i] = bi[i];
            dv[n + i] = best[i];
          }
    }
    if (tid < k) cnt[tid] = 0;
    if (tid == 0) changed = 0;
    __syncthreads();
    if (it == g.iters) break;
    for (int n = tid; n < nc; n += kSelThreads) atomicAdd(&cnt[z[n]], 1);
    __syncthreads();
    // the candidates cluster by cluster, ascending within one
    for (int n = tid; n < nc; n += kSelThreads) {
      int place = 0;
      for (int i = 0; i < z[n]; ++i) place += cnt[i];
      for (int m = 0; m < n; ++m) place += z[m] == z[n];
      order[place] = n;
    }
    __syncthreads();
    for (int i0 = 0, p0 = 0; i0 < k; i0 += 8) {
      int p1 = p0;     // positions p0 .. p1 - 1 belong to these eight clusters
      for (int q = 0; q < 8 && i0 + q < k; ++q) p1 += cnt[i0 + q];
      // the means of their columns, two columns per thread and 16 rows of both at a time, whatever their clusters: a sum
      // ends where the next position starts another cluster
      for (int e = tid; e < C; e += 2 * kSelThreads) {
        const int e1 = min(e + kSelThreads, C - 1);   // past the row: not stored
        float s0 = 0.0f, s1 = 0.0f;
        for (int p = p0; p < p1; p += kSelRows) {
          float v0[kSelRows], v1[kSelRows];
#pragma unroll
          for (int u = 0; u < kSelRows; ++u) {
            const float* x = row(order[min(p + u, p1 - 1)]);
            v0[u] = x[e];
            v1[u] = x[e1];
          }
#pragma unroll
          for (int u = 0; u < kSelRows; ++u) {
            if (p + u >= p1) break;
            s0 += v0[u];
            s1 += v1[u];
            const int zi = __builtin_amdgcn_readfirstlane(z[order[p + u]]);
            if (p + u + 1 == p1 || __builtin_amdgcn_readfirstlane(z[order[p + u + 1]]) != zi) {
              const float n = (float)cnt[zi];
              mrow[(zi - i0) * C + e] = s0 / n;
              if (e + kSelThreads < C) mrow[(zi - i0) * C + e1] = s1 / n;
              s0 = s1 = 0.0f;
            }
          }
        }
      }
      float part[8] = {};
      for (int e = tid; e < C; e += kSelThreads)
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          const float mean = i0 + q < k && cnt[i0 + q] ? mrow[q * C + e] : 0.0f;   // this thread's own values
          part[q] += mean * mean;
        }
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        if (i0 + q >= k) break;
        const float p = wave_sum_xor(part[q]);
        if (lane == 0) sv[q * kSelWaves + w] = p;
      }
      __syncthreads();
      for (int q = 0; q < 8 && i0 + q < k; ++q) {
        if (cnt[i0 + q] == 0) continue;   // no members: the centre stays
        float t = 0.0f;
#pragma unroll
        for (int u = 0; u < kSelWaves; ++u) t += sv[q * kSelWaves + u];
        const float nrm = fmaxf(sqrtf(t), 1e-12f);
        float* ci = c + (i0 + q) * C;
        for (int e = tid; e < C; e += kSelThreads) {
          const float nv = mrow[q * C + e] / nrm;
          if (nv != ci[e]) changed = 1;
          ci[e] = nv;
        }
      }
      __syncthreads();
      p0 = p1;
    }
    if (!changed) break;   // z and dv were computed from these (unchanged) centres
    __syncthreads();
  }

  // medoid of each non-empty cluster: the member most similar to its centre, the first on ties (a wavefront per cluster)
  for (int i = w; i < k; i += kSelWaves) {
    float best = -INFINITY;
    int bi = 0x7fffffff;
    for (int n = lane; n < nc; n += 64)
      if (z[n] == i && (bi == 0x7fffffff || dv[n] > best)) {
        best = dv[n];
        bi = n;
      }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
      const float b = __shfl_xor(best, o, 64);
      const int j = __shfl_xor(bi, o, 64);
      if (j != 0x7fffffff && (bi == 0x7fffffff || b > best || (b == best && j < bi))) {
        best = b;
        bi = j;
      }
    }
    if (lane == 0) centre[i] = bi < nc ? cand[bi] : -1;
  }
  __syncthreads();
  // ascending, -1 after the last: a frame's place is the number of smaller ones
  if (tid < k) {
    const int f = centre[tid];
    int place = 0, found = 0;
    for (int i = 0; i < k; ++i) {
      place += centre[i] >= 0 && (centre[i] < f || (centre[i] == f && i < tid));
      found += centre[i] >= 0;
    }
    if (f >= 0) g.reps[place] = f;
    if (tid >= found) g.reps[tid] = -1;
  }
}

}  // namespace
}  // namespace onereel

using namespace onereel;

extern "C" int or_frame_pool(const void* hs, int64_t n_rows, int32_t C, int64_t row_stride, int64_t row0, int32_t T,
                             int32_t n_frames, float* sums, float* counts, void* stream) {
  if (n_rows < 0 || C < 8 || C % 8 || T < 1 || n_frames < 1 || row0 < 0 || row_stride < C)
    return fail_arg("or_frame_pool: need n_rows >= 0, C a multiple of 8, T >= 1, n_frames >= 1, row0 >= 0 and a row "
                    "stride covering C (C=%d T=%d frames=%d)", C, T, n_frames);
  if (n_rows == 0) return 0;
  if (!hs || !sums || !counts) return fail_arg("or_frame_pool: hs, sums and counts are required");
  if ((row0 + n_rows + T - 1) / T > n_frames)
    return fail_arg("or_frame_pool: rows %lld..%lld reach past frame %d", (long long)row0, (long long)(row0 + n_rows),
                    n_frames);
  if (((uintptr_t)hs & 15u) || row_stride % 8) return fail_arg("or_frame_pool: hs must be 16-byte aligned rows");
  PoolArgs g{(const uint16_t*)hs, n_rows, row_stride, row0, C, T, n_frames, sums, counts};
  if (pool_by_wave(std::min<int64_t>(n_frames, n_rows / T + 1), C, T))
    hipLaunchKernelGGL(frame_pool_wave_kernel, dim3((unsigned)((C + 2047) / 2048), (unsigned)n_frames), dim3(kPoolThreads),
                       0, (hipStream_t)stream, g);
  else
    hipLaunchKernelGGL(frame_pool_kernel, dim3((unsigned)((C + 127) / 128), (unsigned)n_frames), dim3(kPoolThreads), 0,
                       (hipStream_t)stream, g);
  return check_hip(hipGetLastError(), "frame_pool_kernel launch");
}

// the candidates from the device (cand) or from the host (table; cand NULL)
static int launch_select(const float* feats, int n_frames, int C, const int32_t* cand, const CandTable& table, int n_cand,
                         int k, int iters, int32_t* reps, float* work, void* stream) {
  if (C < 1 || n_frames < 1 || n_cand < 1 || n_cand > kMaxCand || k < 1 || k > kMaxK || k > n_cand || iters < 0)
    return fail_arg("or_frame_select: need C >= 1, 1 <= n_cand <= %d and 1 <= k <= min(n_cand, %d) (n_cand=%d k=%d)",
                    kMaxCand, kMaxK, n_cand, k);
  if ((int64_t)k * C > kMaxCentreFloats)
    return fail_arg("or_frame_select: k * C = %lld floats of centres exceed %d of LDS", (long long)k * C,
                    kMaxCentreFloats);
  SelectArgs g{feats, cand, n_cand, C, k, iters, reps, work};
  const size_t lds = (size_t)k * C * sizeof(float);
  static thread_local bool attr = false;
  if (!attr) {
    if (int rc = check_hip(hipFuncSetAttribute((const void*)frame_select_kernel,
                                               hipFuncAttributeMaxDynamicSharedMemorySize, kMaxCentreFloats * 4),
                           "hipFuncSetAttribute"))
      return rc;
    attr = true;
  }
  hipLaunchKernelGGL(frame_select_kernel, dim3(1), dim3(kSelThreads), lds, (hipStream_t)stream, g, table);
  return check_hip(hipGetLastError(), "frame_select_kernel launch");
}

extern "C" int or_frame_select(const float* feats, int32_t n_frames, int32_t C, const int32_t* cand, int32_t n_cand,
                               int32_t k, int32_t iters, int32_t* reps, float* work, void* stream) {
  if (!feats || !cand || !reps || !work) return fail_arg("or_frame_select: feats, cand, reps and work are required");
  return launch_select(feats, n_frames, C, cand, CandTable{}, n_cand, k, iters, reps, work, stream);
}

extern "C" int or_frame_select_host(const float* feats, int32_t n_frames, int32_t C, const int32_t* cand,
                                    int32_t n_cand, int32_t k, int32_t iters, int32_t* reps, float* work,
                                    void* stream) {
  if (!feats || !cand || !reps || !work) return fail_arg("or_frame_select_host: feats, cand, reps and work are required");
  CandTable table{};
  for (int i = 0; i < n_cand && i < kMaxCand; ++i) {
    if (cand[i] < 0 || cand[i] >= n_frames || cand[i] > 0xffff)
      return fail_arg("or_frame_select_host: candidate frame %d outside [0, min(%d, 65536))", cand[i], n_frames);
    table.frame[i] = (uint16_t)cand[i];
  }
  return launch_select(feats, n_frames, C, nullptr, table, n_cand, k, iters, reps, work, stream);
}
