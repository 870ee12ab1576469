// Device pieces shared by the IVF router (ivf.hip) and the certified causal cascade (ccc.hip):
// ordering keys, fp64 inner products, workgroup scans, radix top-K threshold and compaction over
// LDS, and the inverted-list build (assignment keys, per-tile ranks, list scatter, centroid
// update). Everything is deterministic: inner products accumulate in fp64 in dimension order and
// round once to fp32, ties go to the lower index, list members stay in ascending order.
#pragma once
#include <math.h>

#include "common.h"

namespace ssa {
namespace {
constexpr int kIvfMaxD = 256;      // head dim: a multiple of 32, at most this
constexpr int kIvfCap = 2048;      // LDS keys per route pass (coarse keys, candidates, the union)
constexpr int kIvfMaxSearch = kIvfCap / 2;
constexpr int kTile = 256;         // block means per rank / scatter workgroup
constexpr int kScoreRows = 128;    // block means per scoring workgroup

inline size_t r256(size_t x) { return (x + 255) & ~size_t(255); }

// Unique, order-preserving key of (score, index): larger score first, then lower index.
__device__ inline unsigned long long ivf_key(float s, int64_t idx) {
  return ((unsigned long long)score_key(s) << 32) |
         (unsigned long long)(0xffffffffu - (unsigned int)idx);
}

__device__ inline int64_t ivf_key_index(unsigned long long k) {
  return (int64_t)(0xffffffffu - (unsigned int)(k & 0xffffffffull));
}

// <q, x> with q in LDS and x[t] at col[t * stride] (d a multiple of 32), accumulated in fp64 in
// dimension order (a product of two fp32 values is exact in fp64, so each step rounds once) and
// rounded once to fp32. Each 32-element chunk of x is loaded in one burst before its fmas.
__device__ inline float dot_strided(const float* q, const float* col, int64_t stride,
                                    int64_t d) {
  double acc = 0.0;
  for (int64_t t0 = 0; t0 < d; t0 += 32) {
    float x[32];
#pragma unroll
    for (int u = 0; u < 32; ++u) x[u] = col[(t0 + u) * stride];
#pragma unroll
    for (int u = 0; u < 32; u += 4) {
      const float4 qq = *reinterpret_cast<const float4*>(q + t0 + u);
      acc = fma((double)qq.x, (double)x[u], acc);
      acc = fma((double)qq.y, (double)x[u + 1], acc);
      acc = fma((double)qq.z, (double)x[u + 2], acc);
      acc = fma((double)qq.w, (double)x[u + 3], acc);
    }
  }
  return (float)acc;
}

// Exclusive prefix of v over a 256-thread workgroup; *total = the sum. ws holds 4 ints.
__device__ inline int ivf_block_scan(int v, int* ws, int* total) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  int x = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int y = __shfl_up(x, o);
    if (lane >= o) x += y;
  }
  if (lane == 63) ws[w] = x;
  __syncthreads();
  int base = 0, tot = 0;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    if (k < w) base += ws[k];
    tot += ws[k];
  }
  __syncthreads();
  *total = tot;
  return base + x - v;
}

// A threshold T with exactly K of the n keys in LDS >= T (0 < K <= n, the K largest keys
// distinct), by an MSB-first radix walk over 8-bit digits that stops once the digit's whole bin
// is taken (T then ends in zero bits). 256 threads; shv holds 3 ints.
__device__ unsigned long long block_kth_largest(const unsigned long long* keys, int n, int K,
                                                unsigned int* hist, unsigned int* shv) {
  const int tid = threadIdx.x, lane = tid & 63;
  unsigned long long prefix = 0ull;
  int need = K;
  for (int shift = 56; shift >= 0; shift -= 8) {
    hist[tid] = 0u;
    __syncthreads();
    const unsigned long long hi = shift == 56 ? 0ull : (~0ull << (shift + 8));
    for (int e = tid; e < n; e += 256) {
      const unsigned long long k = keys[e];
      if ((k & hi) == prefix) atomicAdd(&hist[(k >> shift) & 255u], 1u);
    }
    __syncthreads();
    if (tid < 64) {
      const unsigned int c0 = hist[4 * lane], c1 = hist[4 * lane + 1];
      const unsigned int c2 = hist[4 * lane + 2], c3 = hist[4 * lane + 3];
      const unsigned int s = c0 + c1 + c2 + c3;
      unsigned int suf = s;  // sum over lanes >= this one
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const unsigned int y = __shfl_down(suf, o);
        if (lane + o < 64) suf += y;
      }
      unsigned int above = suf - s;  // keys in the bins above this lane's four
      const unsigned int cb[4] = {c0, c1, c2, c3};
#pragma unroll
      for (int b = 3; b >= 0; --b) {
        if (above < (unsigned int)need && (unsigned int)need <= above + cb[b]) {
          shv[0] = 4u * lane + b;
          shv[1] = (unsigned int)need - above;
          shv[2] = (unsigned int)need == above + cb[b];
        }
        above += cb[b];
      }
    }
    __syncthreads();
    prefix |= (unsigned long long)shv[0] << shift;
    need = (int)shv[1];
    const bool whole = shv[2] != 0u;
    __syncthreads();
    if (whole) break;  // uniform: every key of the bin is taken
  }
  return prefix;
}

// ---- build --------------------------------------------------------------------------------------
// A wave scores 32 block means (a workgroup of four: kScoreRows) against one group of `per_group`
// 16-centroid tiles: pbest = the key of the group's best centroid for each mean (largest inner
// product, ties to the lower centroid). v_mfma_f64_16x16x4_f64 (lane l supplies A[l%16][l/16] and
// B[l/16][l%16]; accumulator r of lane l is C[4r + l/16][l%16]): A = the centroids, B = the means,
// step s the dimensions 4 s .. 4 s + 3, which the unit adds in that order, one rounding each: the
// bits of the fma chain in dimension order. d = 32 NC. A lane loads 16 bytes of a row at a time
// (4 bytes a lane, one per step, fetched each line eight times: 16.2 us) and quarter_transpose
// hands every lane the dimensions of its steps; the means stay in registers, the next tile's
// centroids are loaded while this one's are multiplied, and nothing goes through LDS: as fma chains
// over staged centroids a wave spent its time on the staging's bank conflicts and on four waits for
// its rows. d 64: 8192 means, 90 centroids 20 -> 6.6 us (the matrix rate alone: 1.3); 8192 to 32,768
// means, 181 centroids 23 -> 11.5 on average. What is left is the launch and one wait for the rows.
typedef double ivf_f64x4 __attribute__((ext_vector_type(4)));
typedef float f32x4_u __attribute__((ext_vector_type(4), aligned(4)));  // (a caller's centroids)

// Element e of the lanes of quarter q (lane / 16) <-> element q of the lanes of quarter e.
__device__ inline f32x4 quarter_transpose(const f32x4& x) {
  unsigned int u[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) u[e] = __float_as_uint(x[e]);
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const auto r = __builtin_amdgcn_permlane32_swap(u[e], u[e + 2], false, false);
    u[e] = r[0];
    u[e + 2] = r[1];
  }
#pragma unroll
  for (int e = 0; e < 4; e += 2) {
    const auto r = __builtin_amdgcn_permlane16_swap(u[e], u[e + 1], false, false);
    u[e] = r[0];
    u[e + 1] = r[1];
  }
  return f32x4{__uint_as_float(u[0]), __uint_as_float(u[1]), __uint_as_float(u[2]),
               __uint_as_float(u[3])};
}

template <int NC>
__global__ __launch_bounds__(256) void ivf_score_kernel(
    const float* __restrict__ mu, const float* __restrict__ cent, int64_t nb, int64_t nlist,
    int64_t per_group, unsigned long long* __restrict__ pbest) {
  constexpr int D = 32 * NC, NV = D / 16;  // 16-byte loads of a lane per row
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, col = lane & 15, kq = lane >> 4;
  const int64_t bh = blockIdx.y, g = blockIdx.z;
  const int64_t j0 = (int64_t)blockIdx.x * kScoreRows + 32 * w;
  if (j0 >= nb) return;
  f32x4 b[2][NV];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int64_t j = j0 + 16 * h + col < nb ? j0 + 16 * h + col : nb - 1;
    const float* row = mu + (bh * nb + j) * D + 4 * kq;
#pragma unroll
    for (int v = 0; v < NV; ++v) b[h][v] = *reinterpret_cast<const f32x4*>(row + 16 * v);
  }
  const float* cb = cent + bh * nlist * D + 4 * kq;
  const int tiles = (int)((nlist + 15) / 16);
  const int tbeg = (int)(g * per_group);
  const int tend = tbeg + (int)per_group < tiles ? tbeg + (int)per_group : tiles;
  auto load = [&](int tile, f32x4* a) {  // (rows past the last centroid re-read it: discarded)
    const int64_t c = 16 * (int64_t)tile + col < nlist ? 16 * (int64_t)tile + col : nlist - 1;
#pragma unroll
    for (int v = 0; v < NV; ++v) a[v] = *reinterpret_cast<const f32x4_u*>(cb + c * D + 16 * v);
  };
  unsigned long long best[2] = {0ull, 0ull};
  f32x4 a[NV];
  if (tbeg < tend) load(tbeg, a);
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int v = 0; v < NV; ++v) b[h][v] = quarter_transpose(b[h][v]);
  for (int tile = tbeg; tile < tend; ++tile) {
    f32x4 an[NV];
    load(tile + 1 < tend ? tile + 1 : tile, an);
    ivf_f64x4 acc[2] = {{0.0, 0.0, 0.0, 0.0}, {0.0, 0.0, 0.0, 0.0}};
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      const f32x4 at = quarter_transpose(a[v]);
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int h = 0; h < 2; ++h)
          acc[h] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)at[e], (double)b[h][v][e], acc[h],
                                                        0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int c = 16 * tile + 4 * r + kq;
      if (c < nlist) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const unsigned long long k = ivf_key((float)acc[h][r], c);
          best[h] = k > best[h] ? k : best[h];
        }
      }
    }
#pragma unroll
    for (int v = 0; v < NV; ++v) a[v] = an[v];
  }
#pragma unroll
  for (int h = 0; h < 2; ++h) {
#pragma unroll
    for (int o = 16; o <= 32; o <<= 1) {
      const unsigned long long k = __shfl_xor(best[h], o);
      best[h] = k > best[h] ? k : best[h];
    }
    const int64_t j = j0 + 16 * h + col;
    if (kq == 0 && j < nb) pbest[(bh * gridDim.z + g) * nb + j] = best[h];
  }
}

// How ivf_score_kernel's launch splits the centroids: as many groups as give it about 2048 waves
// (two per SIMD), at most `gmax` and at most one per 16 centroids.
struct ScoreSplit {
  int64_t wgs, groups, per_group;  // workgroups over the means; groups of per_group tiles
  ScoreSplit(int64_t m, int64_t heads, int64_t nlist, int64_t gmax) {
    const int64_t tiles = (nlist + 15) / 16;
    wgs = (m + kScoreRows - 1) / kScoreRows;
    int64_t g = (2048 + 4 * wgs * heads - 1) / (4 * wgs * heads);
    g = g > tiles ? tiles : g;
    g = g > gmax ? gmax : g;
    g = g < 1 ? 1 : g;
    per_group = (tiles + g - 1) / g;
    groups = (tiles + per_group - 1) / per_group;
  }
};

inline int ivf_score(const float* mu, const float* cent, int64_t heads, int64_t m, int64_t d,
                     int64_t nlist, const ScoreSplit& sp, unsigned long long* pbest,
                     hipStream_t s) {
  const dim3 grid((unsigned)sp.wgs, (unsigned)heads, (unsigned)sp.groups);
#define SSA_SCORE(NC)                                                                        \
  case NC:                                                                                   \
    ivf_score_kernel<NC><<<grid, 256, 0, s>>>(mu, cent, m, nlist, sp.per_group, pbest);      \
    break
  switch (d / 32) {  // d: a multiple of 32, at most kIvfMaxD
    SSA_SCORE(1); SSA_SCORE(2); SSA_SCORE(3); SSA_SCORE(4);
    SSA_SCORE(5); SSA_SCORE(6); SSA_SCORE(7); SSA_SCORE(8);
  }
#undef SSA_SCORE
  return launch_status("ivf_score_kernel");
}

// The rank of this thread's centroid a (-1: none) among the threads before it of a 256-thread tile
// that hold the same one, and trow[c] = how many hold centroid c, for c < nlist <= kIvfCap. A wave
// finds the lanes that share a centroid with one ballot per bit; their counts (at most 64) meet in
// wcnt, a byte per (wave, centroid). Walking the tile's 256 centroids in every thread instead took
// 16-20 us at any size (8192 means, 90
// centroids: 20.6 -> 4.7 us for the kernel; 4096 means, 181 centroids 16.2 -> 4.2).
__device__ inline int tile_rank(int a, int64_t nlist, int32_t* __restrict__ trow,
                                unsigned char (*wcnt)[kIvfCap]) {
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int n16 = (int)((nlist + 15) / 16);
  for (int e = tid; e < 4 * n16; e += kTile)
    *reinterpret_cast<u32x4*>(&wcnt[e / n16][16 * (e % n16)]) = u32x4{0u, 0u, 0u, 0u};
  unsigned long long same = __ballot(a >= 0);
  for (int b = 0; (1 << b) < nlist; ++b) {
    const bool one = (a >> b) & 1;
    const unsigned long long v = __ballot(one);
    same &= one ? v : ~v;
  }
  const int before = __popcll(same & ((1ull << lane) - 1));
  __syncthreads();  // the counts are zero
  if (a >= 0 && before == 0) wcnt[w][a] = (unsigned char)__popcll(same);
  __syncthreads();
  for (int64_t c = tid; c < nlist; c += kTile)
    trow[c] = wcnt[0][c] + wcnt[1][c] + wcnt[2][c] + wcnt[3][c];
  int r = before;
  if (a >= 0)
#pragma unroll
    for (int u = 0; u < 3; ++u) r += u < w ? wcnt[u][a] : 0;
  return r;
}

// One workgroup per tile: each block mean joins the best of its groups' centroids; rank = its
// position among the tile's members of that centroid, and the tile's member count of every
// centroid goes to its tcount row (0 for absent ones).
__global__ __launch_bounds__(256) void ivf_rank_kernel(
    const unsigned long long* __restrict__ pbest, int64_t nb, int64_t nlist, int64_t ntiles,
    int64_t groups, int32_t* __restrict__ assign, int32_t* __restrict__ rank,
    int32_t* __restrict__ tcount) {
  __shared__ __align__(16) unsigned char wcnt[4][kIvfCap];
  const int64_t bh = blockIdx.y, tile = blockIdx.x;
  const int64_t j = tile * kTile + threadIdx.x;
  const bool live = j < nb;
  unsigned long long best = 0ull;
  const unsigned long long* pb = pbest + bh * groups * nb + (live ? j : 0);
  for (int64_t g0 = 0; g0 < groups; g0 += 8) {  // 8 loads in flight (clamped to a valid group)
    unsigned long long k[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) k[u] = pb[(g0 + u < groups ? g0 + u : groups - 1) * nb];
#pragma unroll
    for (int u = 0; u < 8; ++u) best = k[u] > best ? k[u] : best;
  }
  const int a = live ? (int)ivf_key_index(best) : -1;
  const int r = tile_rank(a, nlist, tcount + (bh * ntiles + tile) * nlist, wcnt);
  if (live) {
    assign[bh * nb + j] = a;
    rank[bh * nb + j] = r;
  }
}

// One workgroup per (centroid, head): tcount[t] <- the centroid's members in the tiles before t
// (an exclusive prefix over the tiles, in place, 256 tiles per pass) and count = its members in
// all tiles. Work O(tiles x centroids). With gate set, nothing runs unless *gate != 0.
__global__ __launch_bounds__(256) void ivf_tile_prefix_kernel(int32_t* __restrict__ tcount,
                                                               int64_t ntiles, int64_t nlist,
                                                               int32_t* __restrict__ count,
                                                               const int32_t* __restrict__ gate) {
  __shared__ int ws[4];
  if (gate != nullptr && *gate == 0) return;
  const int64_t bh = blockIdx.y, c = blockIdx.x;
  int32_t* col = tcount + bh * ntiles * nlist + c;
  int running = 0;
  for (int64_t t0 = 0; t0 < ntiles; t0 += 256) {
    const int64_t t = t0 + threadIdx.x;
    const int v = t < ntiles ? col[t * nlist] : 0;
    int tot;
    const int ex = ivf_block_scan(v, ws, &tot);
    if (t < ntiles) col[t * nlist] = running + ex;
    running += tot;
  }
  if (threadIdx.x == 0) count[bh * nlist + c] = running;
}

// One thread per block mean: its slot in ids = offset of its list + members of the list in
// earlier tiles (tbase, the prefix of ivf_tile_prefix_kernel) + its rank in its tile. With muL set
// (the last assignment), the mean is also copied to its list's transposed storage: element t of
// member k of list p at d * off[p] + t * size[p] + k. Every workgroup adds up the list sizes for
// itself (nlist <= kIvfCap) and the first one of a head writes off[c] = the members of the centroids
// before c, off[nlist] = all: a launch of its own for that took 2.5 us and a gap beside this kernel's
// 4.8, now 5.5 (1M-token IVF prefill 906 -> 881 us).
__global__ __launch_bounds__(256) void ivf_scatter_kernel(
    const int32_t* __restrict__ assign, const int32_t* __restrict__ rank,
    const int32_t* __restrict__ tbase, int64_t nb, int64_t nlist, int64_t ntiles,
    const int32_t* __restrict__ count, int32_t* __restrict__ off, int32_t* __restrict__ ids,
    const float* __restrict__ mu, int64_t d, float* __restrict__ muL) {
  __shared__ int start[kIvfCap];
  __shared__ int ws[4];
  const int64_t bh = blockIdx.y, tile = blockIdx.x;
  const int64_t j = tile * kTile + threadIdx.x;
  const int a = j < nb ? assign[bh * nb + j] : 0;
  const int r = j < nb ? tbase[(bh * ntiles + tile) * nlist + a] + rank[bh * nb + j] : 0;
  int running = 0;
  for (int64_t c0 = 0; c0 < nlist; c0 += 256) {
    const int64_t c = c0 + threadIdx.x;
    const int v = c < nlist ? count[bh * nlist + c] : 0;
    int tot;
    const int at = running + ivf_block_scan(v, ws, &tot);
    if (c < nlist) {
      start[c] = at;
      if (tile == 0) off[bh * (nlist + 1) + c] = at;
    }
    running += tot;
  }
  if (tile == 0 && threadIdx.x == 0) off[bh * (nlist + 1) + nlist] = running;
  __syncthreads();
  if (j >= nb) return;
  const int o = start[a], pos = o + r;
  ids[bh * nb + pos] = (int32_t)j;
  if (muL != nullptr) {
    const int64_t L = count[bh * nlist + a];
    const float* src = mu + (bh * nb + j) * d;
    float* dst = muL + bh * nb * d + d * (int64_t)o + (pos - o);
    for (int64_t t = 0; t < d; ++t) dst[t * L] = src[t];
  }
}

// The lists of an assignment whose per-tile ranks and counts (tcount) are set: sizes, offsets,
// member ids in ascending order and, with muL, the transposed member storage. tcount is
// overwritten with its prefix over the tiles.
inline int ivf_lists(const int32_t* assign, const int32_t* rank, int32_t* tcount, int64_t BH,
                     int64_t nb, int64_t nlist, int64_t ntiles, int32_t* count, int32_t* off,
                     int32_t* ids, const float* mu, int64_t d, float* muL, hipStream_t s) {
  ivf_tile_prefix_kernel<<<dim3((unsigned)nlist, (unsigned)BH), 256, 0, s>>>(tcount, ntiles,
                                                                             nlist, count, nullptr);
  SSA_TRY(launch_status("ivf_tile_prefix_kernel"));
  ivf_scatter_kernel<<<dim3((unsigned)ntiles, (unsigned)BH), 256, 0, s>>>(
      assign, rank, tcount, nb, nlist, ntiles, count, off, ids, mu, d, muL);
  return launch_status("ivf_scatter_kernel");
}

// centT (BH, d, nlist) = the centroids transposed.
__global__ __launch_bounds__(64) void ivf_transpose_cent_kernel(const float* __restrict__ cent,
                                                                 int64_t d, int64_t nlist,
                                                                 float* __restrict__ centT) {
  const int64_t bh = blockIdx.y, c = blockIdx.x;
  for (int64_t t = threadIdx.x; t < d; t += 64)
    centT[(bh * d + t) * nlist + c] = cent[(bh * nlist + c) * d + t];
}

// Centroid c <- normalised sum of its members (fp64, ascending member order; SPHERICAL), or
// fl32(sum / count), the members' mean (!SPHERICAL); unchanged when it has no members (or, when
// SPHERICAL, their sum is zero). Lane l owns dimensions l + 64 u, u < NU (d <= 64 NU). A list is
// one wave's chain of loads (a member's id, then its row): with 16 members a step, ids and rows loaded
// one after the other, 12.3 us at 8192 means, 90 lists of d 64 and 24.8 at 32,768 means, 181 lists; 8.9
// and 15.9 with the rows one batch and the ids a run ahead.
template <int NU, bool SPHERICAL = true>
__global__ __launch_bounds__(64) void ivf_update_kernel(
    const float* __restrict__ mu, const int32_t* __restrict__ count,
    const int32_t* __restrict__ off, const int32_t* __restrict__ ids, int64_t nb, int64_t d,
    int64_t nlist, float* __restrict__ cent) {
  __shared__ double sd[kIvfMaxD];
  __shared__ double snrm;
  const int64_t bh = blockIdx.y, c = blockIdx.x;
  const int lane = threadIdx.x;
  const int L = count[bh * nlist + c];
  if (L == 0) return;
  const int32_t* mem = ids + bh * nb + off[bh * (nlist + 1) + c];
  const float* mb = mu + bh * nb * d;
  int64_t tt[NU];
#pragma unroll
  for (int u = 0; u < NU; ++u) tt[u] = lane + 64 * u < d ? lane + 64 * u : 0;
  double acc[NU];
#pragma unroll
  for (int u = 0; u < NU; ++u) acc[u] = 0.0;
  // kB members' values are in flight while the kB before them are added in order; a lane holds one
  // member id of a run of 64, and of the run after it
  constexpr int kB = NU == 1 ? 32 : NU == 2 ? 16 : 8;
  int idw = mem[lane < L ? lane : L - 1];
  int idn = mem[64 + lane < L ? 64 + lane : L - 1];
  float va[kB][NU], vb[kB][NU];
  auto load = [&](int k0, float (*v)[NU]) {  // called for k0 = 0, kB, 2 kB, ..
    if (k0 >= L) return;
    if (k0 > 0 && (k0 & 63) == 0) {
      idw = idn;
      idn = mem[k0 + 64 + lane < L ? k0 + 64 + lane : L - 1];
    }
#pragma unroll
    for (int b = 0; b < kB; ++b) {  // (past the last member: it again, not added)
      const int64_t j = __builtin_amdgcn_readlane(idw, (k0 & 63) + b);
#pragma unroll
      for (int u = 0; u < NU; ++u) v[b][u] = mb[j * d + tt[u]];
    }
  };
  auto add = [&](int k0, const float (*v)[NU]) {
#pragma unroll
    for (int b = 0; b < kB; ++b)
      if (b < L - k0) {
#pragma unroll
        for (int u = 0; u < NU; ++u) acc[u] = __dadd_rn(acc[u], (double)v[b][u]);
      }
  };
  load(0, va);
  for (int k0 = 0; k0 < L; k0 += 2 * kB) {
    load(k0 + kB, vb);
    add(k0, va);
    load(k0 + 2 * kB, va);
    add(k0 + kB, vb);
  }
  if constexpr (!SPHERICAL) {
    float* dst = cent + (bh * nlist + c) * d;
#pragma unroll
    for (int u = 0; u < NU; ++u)
      if (lane + 64 * u < d) dst[lane + 64 * u] = (float)(acc[u] / (double)L);
    return;
  }
#pragma unroll
  for (int u = 0; u < NU; ++u)
    if (lane + 64 * u < d) sd[lane + 64 * u] = acc[u];
  __syncthreads();
  if (lane == 0) {
    double nrm = 0.0;
    for (int64_t t = 0; t < d; ++t) nrm = __dadd_rn(nrm, __dmul_rn(sd[t], sd[t]));
    snrm = nrm;
  }
  __syncthreads();
  const double nrm = snrm;
  if (!(nrm > 0.0)) return;
  const double r = sqrt(nrm);
  float* dst = cent + (bh * nlist + c) * d;
  for (int64_t t = lane; t < d; t += 64) dst[t] = (float)(sd[t] / r);
}

// ---- route --------------------------------------------------------------------------------------
// Compacts the entries of v[0..n) (LDS, at most 8 per thread) for which take(entry) holds to
// dst[0..), in any order; returns how many. 256 threads.
template <typename T, typename F>
__device__ inline int block_compact(const T* v, int n, T* dst, int* ws, F take) {
  T mine[kIvfCap / 256];
  bool keep[kIvfCap / 256];
  int cnt = 0;
#pragma unroll
  for (int u = 0; u < kIvfCap / 256; ++u) {
    const int e = threadIdx.x + 256 * u;
    keep[u] = e < n && take(v[e]);
    mine[u] = e < n ? v[e] : T(0);
    cnt += keep[u];
  }
  int total;
  int pos = ivf_block_scan(cnt, ws, &total);  // its barriers order the reads before the writes
#pragma unroll
  for (int u = 0; u < kIvfCap / 256; ++u)
    if (keep[u]) dst[pos++] = mine[u];
  __syncthreads();
  return total;
}

}  // namespace
}  // namespace ssa
