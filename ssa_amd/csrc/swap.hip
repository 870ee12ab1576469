// Tiled forward / backward of the per-row block-sparse softmax attention behind ssa_swap.ssa_masked
// (ssa/ssa_swap.py:32-56), head_dim 64, on v_mfma_f32_32x32x2_f32.
//
// Every query row i has its own selected key blocks (kv_num/kv_idx). The rows are grouped in
// query tiles of 64; row_block_masks_kernel turns the 64 rows' lists into one 64-bit word per
// (query tile, key block): bit r set iff row r of the tile selected the block. The attention
// kernels then walk 64-key tiles and skip a (query tile, key tile) pair whose words are all
// zero; inside a pair a (row, key) entry counts iff the row's bit is set for the key's block and
// key <= row (token causal).
//
//   swap_fwd_kernel   grid (B*Hq*nqt), one 64-row query tile per workgroup: S^T = K Q^T, online
//                     softmax per query column, O^T += V^T P^T; writes O and the row's
//                     natural-log lse.
//   swap_dq_kernel    same grid: recomputes P from lse, dP^T = V dO^T, dS = P (dP - D),
//                     dQ^T += K^T dS^T; also writes D_i = dO_i . O_i for the dk/dv pass.
//   swap_dkdv_kernel  grid (B*Hkv*nkt), one 64-key tile per workgroup, loops the G query heads
//                     and the query tiles at or after the key tile: S = Q K^T, dP = dO V^T,
//                     dV^T += dO^T P, dK^T += Q^T dS.
// Workgroups are issued longest first (the last query tiles, the first key tiles).
// The dq and dk/dv passes each own their outputs (no atomics, deterministic). fp32 inputs:
// products and sums are fp32 (the reference trains the swap in fp32); 16-bit inputs: below.
//
// MFMA operand layout (32x32x2 f32): lane l supplies A[l%32][l/32] and B[l/32][l%32]; the result
// lane l, register r holds C[(r/4)*8 + (l/32)*4 + r%4][l%32]. The contraction index k of a step
// is assigned freely to the two lane halves, as long as A and B agree: head-dim contractions use
// d = 32*(l/32) + t at step t (contiguous 16-byte LDS reads), key/query contractions use the
// rows the previous product's accumulators already hold in each half.
#include <math.h>

#include "common.h"

namespace ssa {

size_t masked_tiled_workspace(int64_t B, int64_t Hq, int64_t n, int64_t block);

namespace {

constexpr int kMaxMaskBlocks = 8192;    // key blocks per sequence (LDS of the mask builder)
constexpr float kLog2eS = 1.4426950408889634f;
constexpr float kLn2S = 0.6931471805599453f;

struct SwapArgs {
  const char* q;
  const char* k;
  const char* v;
  char* o;
  const char* dout;  // strides of o
  float* lse;        // (B*Hq*n)
  float* delta;      // (B*Hq*n)
  void* dq;          // (B, Hq, n, 64) contiguous, fp32 or (grad16) the input type
  void* dk;          // (B, Hkv, n, 64)
  void* dv;
  bool grad16;       // gradients stored in the 16-bit input type (16-bit kernels only)
  int64_t qsb, qsh, qsn, ksb, ksh, ksn, vsb, vsh, vsn, osb, osh, osn;
  int64_t B, Hq, Hkv, G, n, block, nqt, nkt, nb;
  const int32_t* kv_num;
  const int32_t* kv_idx;
  int64_t W;
  unsigned long long* masks;  // (B*Hq, nqt, nb)
  float scale, scale_log2;
};

__device__ inline f32x16 mfma(float a, float b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

// max / sum of a lane and lane ^ 32 (in lane order, so both get the same bits)
__device__ inline float pair_max(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ inline float pair_sum(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// 4 consecutive gradient values of a row: fp32, or rounded to the 16-bit input type DT
template <int DT>
__device__ inline void store_grad4(void* base, int64_t off, const f32x4& v, bool grad16) {
  if (DT != SSA_F32 && grad16) {
    unsigned int w[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
      w[j] = DT == SSA_BF16 ? (unsigned int)__builtin_bit_cast(unsigned short, (__bf16)v[j])
                            : (unsigned int)__builtin_bit_cast(unsigned short, (_Float16)v[j]);
    uint2 u;
    u.x = w[0] | (w[1] << 16);
    u.y = w[2] | (w[3] << 16);
    *reinterpret_cast<uint2*>(static_cast<unsigned short*>(base) + off) = u;
  } else {
    *reinterpret_cast<f32x4*>(static_cast<float*>(base) + off) = v;
  }
}

// 32 consecutive elements [c0, c0 + 32) of one row as fp32 (zeros when !valid).
template <int DT>
__device__ inline void load_row32(const char* base, int64_t off, bool valid, float* out) {
  if constexpr (DT == SSA_F32) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      f32x4 x = {0.0f, 0.0f, 0.0f, 0.0f};
      if (valid) x = *reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(base) + off + 4 * i);
#pragma unroll
      for (int j = 0; j < 4; ++j) out[4 * i + j] = x[j];
    }
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      u32x4 w = {0u, 0u, 0u, 0u};
      if (valid) w = *reinterpret_cast<const u32x4*>(reinterpret_cast<const unsigned short*>(base) + off + 8 * i);
      unpack8(w, out + 8 * i, DT == SSA_BF16);
    }
  }
}

// Stores 4 consecutive fp32 values as DT.
template <int DT>
__device__ inline void store4(char* base, int64_t off, float a, float b, float c, float d) {
  if constexpr (DT == SSA_F32) {
    *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(base) + off) = f32x4{a, b, c, d};
  } else {
    unsigned short u[4];
    const float x[4] = {a, b, c, d};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if constexpr (DT == SSA_BF16) u[j] = __builtin_bit_cast(unsigned short, (__bf16)x[j]);
      else u[j] = __builtin_bit_cast(unsigned short, (_Float16)x[j]);
    }
    typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
    *reinterpret_cast<u32x2*>(reinterpret_cast<unsigned short*>(base) + off) =
        u32x2{(unsigned)u[0] | ((unsigned)u[1] << 16), (unsigned)u[2] | ((unsigned)u[3] << 16)};
  }
}

// Bits [lo, hi) of a 64-bit word (0 <= lo <= hi <= 64).
__device__ inline unsigned long long bit_range(int lo, int hi) {
  if (hi <= lo) return 0ull;
  const unsigned long long upto = hi >= 64 ? ~0ull : ((1ull << hi) - 1ull);
  return upto & ~((1ull << lo) - 1ull);
}

// For the key tile [k0, k0 + 64): OR of the tile's block words of one query tile (`any`), and
// the keys of the tile selected by query-tile row `r` (bit j = key k0 + j; r < 0: none).
// (32-bit: at most 8192 blocks of at most 1024 keys.)
__device__ inline void tile_bits(const unsigned long long* mrow, int64_t k0_, int64_t block_,
                                 int64_t nb_, int r, unsigned long long& any,
                                 unsigned long long& keys) {
  const int k0 = (int)k0_, block = (int)block_, nb = (int)nb_;
  const int c0 = (int)((unsigned)k0 / (unsigned)block);
  any = 0ull;
  keys = 0ull;
  for (int c = c0; c < nb && c * block <= k0 + 63; ++c) {
    const unsigned long long w = mrow[c];
    any |= w;
    if (r >= 0 && ((w >> r) & 1ull)) {
      const int a = c * block - k0, e = a + block;
      keys |= bit_range(a < 0 ? 0 : a, e > 64 ? 64 : e);
    }
  }
}

// grid (B*Hq*nqt), 256 threads: the (query tile, key block) words from the rows' lists.
__global__ __launch_bounds__(256) void row_block_masks_kernel(SwapArgs a) {
  __shared__ unsigned long long mk[kMaxMaskBlocks];
  const int tid = threadIdx.x;
  const int64_t qt = blockIdx.x % a.nqt, bh = blockIdx.x / a.nqt;
  for (int64_t c = tid; c < a.nb; c += 256) mk[c] = 0ull;
  __syncthreads();
  const int64_t q0 = qt * 64;
  for (int64_t idx = tid; idx < 64 * a.W; idx += 256) {
    const int r = (int)(idx / a.W);
    const int64_t j = idx % a.W, row = q0 + r;
    if (row >= a.n) continue;
    const int64_t rid = bh * a.n + row;
    int64_t cnt = a.kv_num[rid];
    if (cnt > a.W) cnt = a.W;
    if (j >= cnt) continue;
    const int64_t c = a.kv_idx[rid * a.W + j];
    if (c < 0 || c >= a.nb || c * a.block > row) continue;  // out of range / not begun: no keys
    atomicOr(&mk[c], 1ull << r);
  }
  __syncthreads();
  unsigned long long* out = a.masks + (bh * a.nqt + qt) * a.nb;
  for (int64_t c = tid; c < a.nb; c += 256) out[c] = mk[c];
}

// Workgroup layout of the three attention kernels: 4 waves, wave w = (x = w & 1, y = w >> 1).
// fwd / dq: x picks the 32 query rows of the 64-row tile, y the 32 keys of each 64-key tile the
// wave contracts over; the two y halves keep separate softmax / gradient state and are merged
// through LDS at the end. dk/dv: x picks the 32 keys, y the 32 query rows of each query tile.

// Cursor over the key tiles of a query tile that hold a selected key: lane t tests tile 64 c + t,
// one round of loads per 64 tiles. The same in every wave of the workgroup.
struct TileCursor {
  const unsigned long long* mrow;
  int block, nb, nkt, chunk;
  unsigned long long act, word;  // word: this lane's tile's rows (any of its blocks)
  __device__ int next(int kt, int lane) {
    while (kt < nkt) {
      const int c0 = kt & ~63;
      if (c0 != chunk) {
        unsigned long long any = 0ull, unused;
        if (c0 + lane < nkt) tile_bits(mrow, (c0 + lane) * 64, block, nb, -1, any, unused);
        act = __ballot(any != 0ull);
        word = any;
        chunk = c0;
      }
      const unsigned long long rest = act & (~0ull << (kt - c0));
      if (rest != 0ull) return c0 + __builtin_ctzll(rest);
      kt = c0 + 64;
    }
    return nkt;
  }
  // the keys of tile kt (the last next()) that row r of the query tile attends, at most key row q
  // (r < 0: none), as the 32 bits from key `from` on. A tile inside one block (block a multiple of
  // 64) needs only the word next() loaded, read from its lane: no memory wait per tile.
  __device__ unsigned int keys(int kt, int r, int q, int from) const {
    unsigned long long any, k;
    if (block % 64 == 0) {
      const unsigned int lo = __builtin_amdgcn_readlane((unsigned int)word, kt - chunk);
      const unsigned int hi = __builtin_amdgcn_readlane((unsigned int)(word >> 32), kt - chunk);
      const unsigned int half = r & 32 ? hi : lo;
      k = r >= 0 && ((half >> (r & 31)) & 1u) ? ~0ull : 0ull;
    } else {
      tile_bits(mrow, kt * 64, block, nb, r, any, k);
    }
    const int past = q - kt * 64;
    if (past < 63) k &= past < 0 ? 0ull : (2ull << past) - 1ull;
    return (unsigned int)(k >> from);
  }
};

// All ones if bit c of bits is set, else 0 (one v_bfe_i32); x where it is, else `other` (v_bfi_b32).
__device__ inline unsigned int bit_mask(unsigned int bits, int c) {
  return (unsigned int)__builtin_amdgcn_sbfe((int)bits, c, 1);
}
__device__ inline float masked(float x, unsigned int mask, float other) {
  return __uint_as_float((__float_as_uint(x) & mask) | (__float_as_uint(other) & ~mask));
}

// Two fp32 64 x 64 tiles side by side, 16 KB each, go from memory to LDS directly
// (global_load_lds) while the previous pair is multiplied. 16-byte chunk c of row r sits at chunk
// c ^ (r & 15): a ds_read_b128 phase (16 rows, one chunk) hits every bank once, and so do the 32
// consecutive head dims of one row that a product along the columns reads 4 bytes a lane.
// One natural copy serves both products (4-byte column reads cost one LDS cycle pair per 64-cycle
// MFMA), so nothing is transposed on the way in. n 1000, B 4, 12 heads, block 64, top_c 4 + local 2:
// forward 103 -> 86 us, dq 129 -> 112, dk / dv 198 -> 141 (matrix rate alone: 47, 71, 95) against
// tiles staged through registers, twice where a transposed copy was needed.
constexpr int kPairTile32 = 64 * 256;
__device__ inline void issue_pair32(const char* x, int64_t xs, const char* y, int64_t ys,
                                    int64_t r0, int64_t nrows, unsigned char* st, int w,
                                    int lane) {
  const float* xb = reinterpret_cast<const float*>(x);
  const float* yb = reinterpret_cast<const float*>(y);
  const float* zero = reinterpret_cast<const float*>(kZeroRow);
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int r = (4 * j + w) * 4 + (lane >> 4);
    const int64_t row = r0 + r;
    const int col = ((lane & 15) ^ (r & 15)) * 4;
    const float* xr = row < nrows ? xb + row * xs : zero;  // past the end: masked entries
    const float* yr = row < nrows ? yb + row * ys : zero;
    __builtin_amdgcn_global_load_lds(xr + col, st + (4 * j + w) * 1024, 16, 0, 0);
    __builtin_amdgcn_global_load_lds(yr + col, st + kPairTile32 + (4 * j + w) * 1024, 16, 0, 0);
  }
}

// LDS offsets of a lane's operands in such a tile, for the 32 rows from row 32 * part: `row[t]` the
// 4 floats of head-dim steps 4 t .. 4 t + 3 of row 32 part + lo; `col[j]` element (row 32 part +
// 8 g + 4 hi + j, head dim 32 dh + lo) for g = dh = 0 (others: col32()).
struct PairOffsets32 {
  uint32_t row[8], col[4];
  __device__ PairOffsets32(int lane, int part) {
    const int hi = lane >> 5, lo = lane & 31, r = 32 * part + lo;
#pragma unroll
    for (int t = 0; t < 8; ++t) row[t] = (uint32_t)(r * 256 + (((8 * hi + t) ^ (r & 15)) * 16));
#pragma unroll
    for (int j = 0; j < 4; ++j)
      col[j] = (uint32_t)((32 * part + 4 * hi + j) * 256 + (((lo >> 2) ^ (4 * hi + j)) * 16) +
                          (lo & 3) * 4);
  }
};
__device__ inline float col32(const unsigned char* st, const PairOffsets32& o, int dh, int g,
                              int j) {
  return *reinterpret_cast<const float*>(st + o.col[j] + g * 2048 + ((dh ^ (g & 1)) * 128));
}
__device__ inline f32x4 row32(const unsigned char* st, const PairOffsets32& o, int t) {
  return *reinterpret_cast<const f32x4*>(st + o.row[t]);
}

__global__ __launch_bounds__(256) void swap_fwd_kernel(SwapArgs a) {
  __shared__ __attribute__((aligned(1024))) unsigned char st0[2 * kPairTile32];  // K, V tiles
  __shared__ __attribute__((aligned(1024))) unsigned char st1[2 * kPairTile32];
  __shared__ float ml[2 * 128];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, hi = lane >> 5, lo = lane & 31;
  const int qh = w & 1, kh = w >> 1;
  const int64_t nbh = a.B * a.Hq;
  const int64_t bh = blockIdx.x % nbh, qt = a.nqt - 1 - blockIdx.x / nbh;  // longest rows first
  const int64_t b = bh / a.Hq, h = bh % a.Hq, kvh = h / a.G;
  const int64_t q0 = qt * 64;
  const int r = 32 * qh + lo;  // this lane's query row in the tile
  const int64_t qi = q0 + r;
  const bool qvalid = qi < a.n;
  float qreg[32];
  load_row32<SSA_F32>(a.q, b * a.qsb + h * a.qsh + qi * a.qsn + 32 * hi, qvalid, qreg);
  const unsigned long long* mrow = a.masks + (bh * a.nqt + qt) * a.nb;
  const char* kb = a.k + (b * a.ksb + kvh * a.ksh) * 4;
  const char* vb = a.v + (b * a.vsb + kvh * a.vsh) * 4;
  const float sl2 = a.scale_log2;

  float m = -INFINITY, l = 0.0f;
  f32x16 o[2];
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int e = 0; e < 16; ++e) o[x][e] = 0.0f;
  int64_t qlast = q0 + 63;
  if (qlast > a.n - 1) qlast = a.n - 1;
  TileCursor cur{mrow, (int)a.block, (int)a.nb, (int)(qlast / 64) + 1, -1, 0ull, 0ull};
  const int nkt = cur.nkt;
  const PairOffsets32 off(lane, kh);
  auto key_bits = [&](int kt) {
    return cur.keys(kt, qvalid ? r : -1, (int)qi, 32 * kh + 4 * hi);
  };
  auto compute = [&](const unsigned char* st, unsigned int keys) {
    if (!__any(keys != 0u)) return;  // no row of the wave attends a key of its half
    f32x16 s;
#pragma unroll
    for (int e = 0; e < 16; ++e) s[e] = 0.0f;
#pragma unroll
    for (int t4 = 0; t4 < 8; ++t4) {
      const f32x4 a4 = row32(st, off, t4);
#pragma unroll
      for (int j = 0; j < 4; ++j) s = mfma(a4[j], qreg[4 * t4 + j], s);
    }
    // key of register e: 32*kh + (e/4)*8 + hi*4 + e%4
    float mx = -INFINITY;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      s[e] = masked(s[e] * sl2, bit_mask(keys, (e >> 2) * 8 + (e & 3)), -INFINITY);
      mx = fmaxf(mx, s[e]);
    }
    const float mnew = fmaxf(m, pair_max(mx));
    if (__any(mnew > m)) {
      const float alpha = mnew > m ? __builtin_amdgcn_exp2f(m - mnew) : 1.0f;
      l *= alpha;
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[x][e] *= alpha;
      m = mnew;
    }
    const float mref = m == -INFINITY ? 0.0f : m;
    float ps = 0.0f;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      s[e] = __builtin_amdgcn_exp2f(s[e] - mref);
      ps += s[e];
    }
    l += ps;
#pragma unroll
    for (int g = 0; g < 4; ++g)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int dh = 0; dh < 2; ++dh)
          o[dh] = mfma(col32(st + kPairTile32, off, dh, g, j), s[4 * g + j], o[dh]);
  };
  int kt = cur.next(0, lane);
  unsigned int keys = 0u;
  if (kt < nkt) {
    keys = key_bits(kt);
    issue_pair32(kb, a.ksn, vb, a.vsn, (int64_t)kt * 64, a.n, st0, w, lane);
  }
  while (kt < nkt) {
    int nxt = cur.next(kt + 1, lane);
    unsigned int nkeys = nxt < nkt ? key_bits(nxt) : 0u;
    dma_barrier();  // st0 has landed for every wave; st1 is no longer read
    if (nxt < nkt) issue_pair32(kb, a.ksn, vb, a.vsn, (int64_t)nxt * 64, a.n, st1, w, lane);
    compute(st0, keys);
    kt = nxt;
    if (kt >= nkt) break;
    keys = nkeys;
    nxt = cur.next(kt + 1, lane);
    nkeys = nxt < nkt ? key_bits(nxt) : 0u;
    dma_barrier();  // st1 has landed; st0 is no longer read
    if (nxt < nkt) issue_pair32(kb, a.ksn, vb, a.vsn, (int64_t)nxt * 64, a.n, st0, w, lane);
    compute(st1, keys);
    kt = nxt;
    keys = nkeys;
  }
  l = pair_sum(l);
  // merge the two key halves: (m, l, O^T) of the kh = 1 waves through LDS
  __syncthreads();
  float* buf = reinterpret_cast<float*>(st0);  // 32 x 128 floats
  const int slot = qh * 64 + lane;
  if (kh == 1) {
    ml[slot] = m;
    ml[128 + slot] = l;
#pragma unroll
    for (int x = 0; x < 32; ++x) buf[x * 128 + slot] = o[x >> 4][x & 15];
  }
  __syncthreads();
  if (kh == 1 || !qvalid) return;
  const float m1 = ml[slot], l1 = ml[128 + slot];
  const float M = fmaxf(m, m1);
  const float a0 = m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m - M);
  const float a1 = m1 == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m1 - M);
  const float lt = l * a0 + l1 * a1;
  const float inv = 1.0f / lt;
  float of[32];
#pragma unroll
  for (int x = 0; x < 32; ++x) of[x] = (o[x >> 4][x & 15] * a0 + buf[x * 128 + slot] * a1) * inv;
  const int64_t ooff = b * a.osb + h * a.osh + qi * a.osn;
#pragma unroll
  for (int dh = 0; dh < 2; ++dh)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int d0 = 32 * dh + 8 * g + 4 * hi, x = 16 * dh + 4 * g;
      store4<SSA_F32>(a.o, ooff + d0, of[x], of[x + 1], of[x + 2], of[x + 3]);
    }
  if (hi == 0) a.lse[bh * a.n + qi] = (M + log2f(lt)) * kLn2S;
}

__global__ __launch_bounds__(256, 2) void swap_dq_kernel(SwapArgs a) {
  __shared__ __attribute__((aligned(1024))) unsigned char st0[2 * kPairTile32];  // K, V tiles
  __shared__ __attribute__((aligned(1024))) unsigned char st1[2 * kPairTile32];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, hi = lane >> 5, lo = lane & 31;
  const int qh = w & 1, kh = w >> 1;
  const int64_t nbh = a.B * a.Hq;
  const int64_t bh = blockIdx.x % nbh, qt = a.nqt - 1 - blockIdx.x / nbh;
  const int64_t b = bh / a.Hq, h = bh % a.Hq, kvh = h / a.G;
  const int64_t q0 = qt * 64;
  const int r = 32 * qh + lo;
  const int64_t qi = q0 + r;
  const bool qvalid = qi < a.n;
  float qreg[32], greg[32];
  load_row32<SSA_F32>(a.q, b * a.qsb + h * a.qsh + qi * a.qsn + 32 * hi, qvalid, qreg);
  const int64_t ooff = b * a.osb + h * a.osh + qi * a.osn + 32 * hi;
  load_row32<SSA_F32>(a.dout, ooff, qvalid, greg);
  float Di;
  {
    float orow[32];
    load_row32<SSA_F32>(a.o, ooff, qvalid, orow);
    float acc = 0.0f;
#pragma unroll
    for (int t = 0; t < 32; ++t) acc = fmaf(greg[t], orow[t], acc);
    Di = pair_sum(acc);
  }
  const int64_t rid = bh * a.n + qi;
  const float lse2 = qvalid ? a.lse[rid] * kLog2eS : 0.0f;
  if (qvalid && kh == 0 && hi == 0) a.delta[rid] = Di;
  const unsigned long long* mrow = a.masks + (bh * a.nqt + qt) * a.nb;
  const char* kb = a.k + (b * a.ksb + kvh * a.ksh) * 4;
  const char* vb = a.v + (b * a.vsb + kvh * a.vsh) * 4;
  const float sl2 = a.scale_log2;

  f32x16 dqa[2];
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int e = 0; e < 16; ++e) dqa[x][e] = 0.0f;
  int64_t qlast = q0 + 63;
  if (qlast > a.n - 1) qlast = a.n - 1;
  TileCursor cur{mrow, (int)a.block, (int)a.nb, (int)(qlast / 64) + 1, -1, 0ull, 0ull};
  const int nkt = cur.nkt;
  const PairOffsets32 off(lane, kh);
  auto key_bits = [&](int kt) {
    return cur.keys(kt, qvalid ? r : -1, (int)qi, 32 * kh + 4 * hi);
  };
  auto compute = [&](const unsigned char* st, unsigned int keys) {
    if (!__any(keys != 0u)) return;  // no row of the wave attends a key of its half
    f32x16 s, dp;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      s[e] = 0.0f;
      dp[e] = 0.0f;
    }
#pragma unroll
    for (int t4 = 0; t4 < 8; ++t4) {
      const f32x4 a4 = row32(st, off, t4);
      const f32x4 b4 = row32(st + kPairTile32, off, t4);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        s = mfma(a4[j], qreg[4 * t4 + j], s);
        dp = mfma(b4[j], greg[4 * t4 + j], dp);
      }
    }
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const float p = masked(__builtin_amdgcn_exp2f(fmaf(s[e], sl2, -lse2)),
                             bit_mask(keys, (e >> 2) * 8 + (e & 3)), 0.0f);
      s[e] = p * (dp[e] - Di);  // dS^T
    }
#pragma unroll
    for (int g = 0; g < 4; ++g)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int dh = 0; dh < 2; ++dh)
          dqa[dh] = mfma(col32(st, off, dh, g, j), s[4 * g + j], dqa[dh]);
  };
  int kt = cur.next(0, lane);
  unsigned int keys = 0u;
  if (kt < nkt) {
    keys = key_bits(kt);
    issue_pair32(kb, a.ksn, vb, a.vsn, (int64_t)kt * 64, a.n, st0, w, lane);
  }
  while (kt < nkt) {
    int nxt = cur.next(kt + 1, lane);
    unsigned int nkeys = nxt < nkt ? key_bits(nxt) : 0u;
    dma_barrier();  // st0 has landed for every wave; st1 is no longer read
    if (nxt < nkt) issue_pair32(kb, a.ksn, vb, a.vsn, (int64_t)nxt * 64, a.n, st1, w, lane);
    compute(st0, keys);
    kt = nxt;
    if (kt >= nkt) break;
    keys = nkeys;
    nxt = cur.next(kt + 1, lane);
    nkeys = nxt < nkt ? key_bits(nxt) : 0u;
    dma_barrier();  // st1 has landed; st0 is no longer read
    if (nxt < nkt) issue_pair32(kb, a.ksn, vb, a.vsn, (int64_t)nxt * 64, a.n, st0, w, lane);
    compute(st1, keys);
    kt = nxt;
    keys = nkeys;
  }
  __syncthreads();
  float* buf = reinterpret_cast<float*>(st0);  // 32 x 128 floats
  const int slot = qh * 64 + lane;
  if (kh == 1) {
#pragma unroll
    for (int x = 0; x < 32; ++x) buf[x * 128 + slot] = dqa[x >> 4][x & 15];
  }
  __syncthreads();
  if (kh == 1 || !qvalid) return;
#pragma unroll
  for (int dh = 0; dh < 2; ++dh)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int d0 = 32 * dh + 8 * g + 4 * hi, x = 16 * dh + 4 * g;
      f32x4 val;
#pragma unroll
      for (int j = 0; j < 4; ++j) val[j] = (dqa[dh][4 * g + j] + buf[(x + j) * 128 + slot]) * a.scale;
      store_grad4<SSA_F32>(a.dq, rid * 64 + d0, val, false);
    }
}

// The next query tile >= qt (in order) holding a selected (row, key) pair of key tile k0 for
// head bh, or a.nqt. The workgroup's 256 threads test 256 tiles at a time into a bitmap in
// LDS (act: 4 words; chunk: the first tile of the bitmap held, -1 at first), so a walk over
// mostly unselected tiles costs one round of loads per 256 tiles. Called uniformly.
__device__ inline int64_t next_active_tile(const SwapArgs& a, int64_t bh, int64_t k0, int64_t qt,
                                           unsigned long long* act, int64_t& chunk) {
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  while (qt < a.nqt) {
    const int64_t c0 = qt & ~int64_t(255);
    if (c0 != chunk) {
      const int64_t t = c0 + tid;
      bool on = false;
      if (t >= k0 / 64 && t < a.nqt) {
        unsigned long long any, unused;
        tile_bits(a.masks + (bh * a.nqt + t) * a.nb, k0, a.block, a.nb, -1, any, unused);
        on = any != 0ull;
      }
      const unsigned long long bal = __ballot(on);
      __syncthreads();  // the previous bitmap is no longer read
      if (lane == 0) act[w] = bal;
      __syncthreads();
      chunk = c0;
    }
    const int r = (int)(qt - c0);
    const unsigned long long rest = act[r >> 6] & (~0ull << (r & 63));
    if (rest != 0ull) return c0 + (r & ~63) + (int64_t)__builtin_ctzll(rest);
    qt = c0 + (r & ~63) + 64;  // no active tile left in this 64-tile word
  }
  return a.nqt;
}

__global__ __launch_bounds__(256, 2) void swap_dkdv_kernel(SwapArgs a) {
  __shared__ __attribute__((aligned(1024))) unsigned char st0[2 * kPairTile32];  // Q, dO tiles
  __shared__ __attribute__((aligned(1024))) unsigned char st1[2 * kPairTile32];
  __shared__ float ld_s[2][2][64];  // [stage][lse, delta][row]
  __shared__ unsigned long long act_s[4];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, hi = lane >> 5, lo = lane & 31;
  const int kq = w & 1, qp = w >> 1;
  const int64_t nbkv = a.B * a.Hkv;
  const int64_t bkv = blockIdx.x % nbkv, kt = blockIdx.x / nbkv;  // most query tiles first
  const int64_t b = bkv / a.Hkv, kvh = bkv % a.Hkv;
  const int64_t k0 = kt * 64;
  const int64_t key = k0 + 32 * kq + lo;
  const bool kvalid = key < a.n;
  float kreg[32], vreg[32];
  load_row32<SSA_F32>(a.k, b * a.ksb + kvh * a.ksh + key * a.ksn + 32 * hi, kvalid, kreg);
  load_row32<SSA_F32>(a.v, b * a.vsb + kvh * a.vsh + key * a.vsn + 32 * hi, kvalid, vreg);
  const int64_t ck = kvalid ? key / a.block : 0;
  const float sl2 = a.scale_log2;

  f32x16 dka[2], dva[2];
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      dka[x][e] = 0.0f;
      dva[x][e] = 0.0f;
    }
  const PairOffsets32 off(lane, qp);
  auto compute = [&](const unsigned char* st, const float (*ld)[64], unsigned int rows) {
    if (!__any(rows != 0u)) return;  // no row of the wave's half attends a key of its half
    f32x16 s, dp;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      s[e] = 0.0f;
      dp[e] = 0.0f;
    }
#pragma unroll
    for (int t4 = 0; t4 < 8; ++t4) {
      const f32x4 a4 = row32(st, off, t4);
      const f32x4 b4 = row32(st + kPairTile32, off, t4);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        s = mfma(a4[j], kreg[4 * t4 + j], s);
        dp = mfma(b4[j], vreg[4 * t4 + j], dp);
      }
    }
    // query row of register e: 32*qp + (e/4)*8 + hi*4 + e%4 of the tile
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int qq = 32 * qp + (e >> 2) * 8 + hi * 4 + (e & 3);
      s[e] = masked(__builtin_amdgcn_exp2f(fmaf(s[e], sl2, -ld[0][qq])),
                    bit_mask(rows, (e >> 2) * 8 + (e & 3)), 0.0f);
      dp[e] = s[e] * (dp[e] - ld[1][qq]);  // dS
    }
#pragma unroll
    for (int g4 = 0; g4 < 4; ++g4)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int dh = 0; dh < 2; ++dh) {
          dva[dh] = mfma(col32(st + kPairTile32, off, dh, g4, j), s[4 * g4 + j], dva[dh]);
          dka[dh] = mfma(col32(st, off, dh, g4, j), dp[4 * g4 + j], dka[dh]);
        }
  };
  // The walk over (query head, query tile) pairs. A pair's mask word and (threads 0..127) its row's
  // lse or delta are loaded one pair before its tiles are, two before it is multiplied.
  struct Pair {
    int64_t g, qt;
    unsigned long long mw;
    float ld;
  };
  int64_t chunk = -1;
  auto next_pair = [&](Pair at) {  // the pair at or after `at`; g == G: none left
    for (; at.g < a.G; ++at.g, at.qt = k0 / 64, chunk = -1) {
      const int64_t bh = b * a.Hq + kvh * a.G + at.g;
      at.qt = next_active_tile(a, bh, k0, at.qt, act_s, chunk);
      if (at.qt < a.nqt) {
        at.mw = kvalid ? a.masks[(bh * a.nqt + at.qt) * a.nb + ck] : 0ull;
        const int64_t row = at.qt * 64 + lane;
        if (tid < 128)  // (rows past the end belong to no list, but an infinity would be NaN)
          at.ld = row < a.n ? (tid < 64 ? a.lse : a.delta)[bh * a.n + row] : 0.0f;
        break;
      }
    }
    return at;
  };
  auto after = [&](Pair at) {
    if (at.g >= a.G) return at;
    ++at.qt;
    return next_pair(at);
  };
  auto issue = [&](const Pair& at, unsigned char* st, float (*ld)[64]) {
    const int64_t hq = kvh * a.G + at.g;
    issue_pair32(a.q + (b * a.qsb + hq * a.qsh) * 4, a.qsn, a.dout + (b * a.osb + hq * a.osh) * 4,
                 a.osn, at.qt * 64, a.n, st, w, lane);
    if (tid < 128) ld[tid >> 6][lane] = tid < 64 ? at.ld * kLog2eS : at.ld;
  };
  // the rows of the lane's half that attend its key, as the 32 bits from row 32 qp + 4 hi on
  auto rows_of = [&](const Pair& at) {
    unsigned long long mw = at.mw;
    const int ahead = (int)(key - at.qt * 64);  // token causal: rows at or after the key
    if (ahead > 0) mw &= ~0ull << ahead;        // (< 64: the walk starts at the key's tile)
    return (unsigned int)(mw >> (32 * qp + 4 * hi));
  };
  Pair at = next_pair(Pair{0, k0 / 64, 0ull, 0.0f});
  if (at.g < a.G) issue(at, st0, ld_s[0]);
  Pair nx = after(at);
  while (at.g < a.G) {
    dma_barrier();  // stage 0 has landed for every wave; stage 1 is no longer read
    if (nx.g < a.G) issue(nx, st1, ld_s[1]);
    Pair nn = after(nx);
    compute(st0, ld_s[0], rows_of(at));
    at = nx;
    nx = nn;
    if (at.g >= a.G) break;
    dma_barrier();  // stage 1 has landed; stage 0 is no longer read
    if (nx.g < a.G) issue(nx, st0, ld_s[0]);
    nn = after(nx);
    compute(st1, ld_s[1], rows_of(at));
    at = nx;
    nx = nn;
  }
  __syncthreads();
  float* bk = reinterpret_cast<float*>(st0);  // 32 x 128 floats each
  float* bv = reinterpret_cast<float*>(st1);
  const int slot = kq * 64 + lane;
  if (qp == 1) {
#pragma unroll
    for (int x = 0; x < 32; ++x) {
      bk[x * 128 + slot] = dka[x >> 4][x & 15];
      bv[x * 128 + slot] = dva[x >> 4][x & 15];
    }
  }
  __syncthreads();
  if (qp == 1 || !kvalid) return;
  const int64_t krow = (bkv * a.n + key) * 64;
#pragma unroll
  for (int dh = 0; dh < 2; ++dh)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int d0 = 32 * dh + 8 * g + 4 * hi, x = 16 * dh + 4 * g;
      f32x4 kv4, vv4;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        kv4[j] = (dka[dh][4 * g + j] + bk[(x + j) * 128 + slot]) * a.scale;
        vv4[j] = dva[dh][4 * g + j] + bv[(x + j) * 128 + slot];
      }
      store_grad4<SSA_F32>(a.dk, krow + d0, kv4, false);
      store_grad4<SSA_F32>(a.dv, krow + d0, vv4, false);
    }
}

// ---- 16-bit inputs: v_mfma_f32_32x32x16_{bf16,f16} ------------------------------------------
// Tiles stay 16-bit in LDS, one copy read along rows and, transposed, along columns; P and dS are
// rounded to the input type for the second products, as flash attention does. Operand layout
// (32x32x16): lane l supplies A[l%32][8*(l/32) + j] and B[8*(l/32) + j][l%32], j = 0..7.
// Head-dim steps t = 0..3 use d = 32*(l/32) + 8t + j; key (query) steps u = 0..1 over a wave's
// 32 accumulator rows use the rows its registers e = 8u + j hold: 16u + 8*(j/4) + 4*(l/32) + j%4.

template <int DT>
struct Mma16;
template <>
struct Mma16<SSA_BF16> {
  typedef bf16x8 vec;
  __device__ static f32x16 mma(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(vec, a),
                                                   __builtin_bit_cast(vec, b), c, 0, 0, 0);
  }
  __device__ static unsigned int bits(float x) { return __builtin_bit_cast(unsigned short, (__bf16)x); }
};
template <>
struct Mma16<SSA_F16> {
  typedef f16x8 vec;
  __device__ static f32x16 mma(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(vec, a),
                                                  __builtin_bit_cast(vec, b), c, 0, 0, 0);
  }
  __device__ static unsigned int bits(float x) { return __builtin_bit_cast(unsigned short, (_Float16)x); }
};

// 8 fp32 values (x[0..7]) rounded and packed as one 16-byte operand
template <int DT>
__device__ inline u32x4 pack8(const float* x) {
  u32x4 r;
#pragma unroll
  for (int i = 0; i < 4; ++i) r[i] = Mma16<DT>::bits(x[2 * i]) | (Mma16<DT>::bits(x[2 * i + 1]) << 16);
  return r;
}

// Two 64 x 64 tiles side by side, 8 KB each, go from memory to LDS directly (global_load_lds)
// while the previous pair is multiplied. 16-byte chunk c of row r sits at chunk c ^ pair_swz(r):
// the 16 rows of a ds_read_b128 phase and the 4 rows x 64 bytes of a transposing read's phase both
// hit every bank once, so one copy of a tile serves the product along its rows and the one along
// its columns.
// What bounds these kernels is a workgroup's chain of tiles (16 at n 1024: memory latency, products,
// exponentials, products), not the matrix rate: tiles are loaded one ahead, masks before them, and
// there are no transposed copies. B 4, 12 heads, n 1024, block 64, top_c 4 + local 2, bf16:
// forward 47 -> 25 us, dq 50 -> 29, dk / dv 53 -> 38 against tiles staged through registers
// between two barriers.
constexpr int kPairTile = 64 * 128;
__device__ inline int pair_swz(int r) { return ((r & 2) << 1) | ((r >> 2) & 3); }

// Issues this wave's share of rows [r0, r0 + 64) of x and y (row strides in elements; rows past the
// last one are zeros: their entries are masked, and 0 times an infinity of a real row read twice
// would be NaN) into st and st + kPairTile. 256 threads.
__device__ inline void issue_pair(const char* x, int64_t xs, const char* y, int64_t ys, int64_t r0,
                                  int64_t nrows, unsigned char* st, int w, int lane) {
  const unsigned short* xb = reinterpret_cast<const unsigned short*>(x);
  const unsigned short* yb = reinterpret_cast<const unsigned short*>(y);
  const unsigned short* zero = reinterpret_cast<const unsigned short*>(kZeroRow);
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int r = (4 * j + w) * 8 + (lane >> 3);
    const int64_t row = r0 + r;
    const int col = ((lane & 7) ^ pair_swz(r)) * 8;
    const unsigned short* xr = row < nrows ? xb + row * xs : zero;
    const unsigned short* yr = row < nrows ? yb + row * ys : zero;
    __builtin_amdgcn_global_load_lds(xr + col, st + (4 * j + w) * 1024, 16, 0, 0);
    __builtin_amdgcn_global_load_lds(yr + col, st + kPairTile + (4 * j + w) * 1024, 16, 0, 0);
  }
}

// LDS offsets of a lane's operands in such a tile, for the 32 rows from row 32 * part: `row[t]`
// the 8 halves of head-dim step t of row 32 part + lo; `col[dh][p]` the transposing reads of the
// rows 32 part + 8 p + 4 hi .. + 3 at head dim 32 dh + lo (step u: + 2048 u).
struct PairOffsets {
  uint32_t row[4], col[2][2];
  __device__ PairOffsets(int lane, int part) {
    const int hi = lane >> 5, r = 32 * part + (lane & 31);
#pragma unroll
    for (int t = 0; t < 4; ++t)
      row[t] = (uint32_t)(r * 128 + (((4 * hi + t) ^ pair_swz(r)) * 16));
    const int a = lane & 15;
#pragma unroll
    for (int dh = 0; dh < 2; ++dh)
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const int k = 32 * part + 8 * p + 4 * hi + (a >> 2);
        const int c = 4 * dh + 2 * ((lane >> 4) & 1) + ((a & 3) >> 1);
        col[dh][p] = (uint32_t)(k * 128 + ((c ^ pair_swz(k)) * 16) + (a & 1) * 8);
      }
  }
};
__device__ inline u32x4 lds16(const unsigned char* p) { return *reinterpret_cast<const u32x4*>(p); }
__device__ inline u32x4 lds_cols(const unsigned char* st, const PairOffsets& o, int dh, int u) {
  const uint2 x = lds_read_tr(st + o.col[dh][0] + 2048 * u);
  const uint2 y = lds_read_tr(st + o.col[dh][1] + 2048 * u);
  return u32x4{x.x, x.y, y.x, y.y};
}

// one row's 32 halves [32*hi, 32*hi + 32) as 4 packed operands (zeros when !valid)
__device__ inline void load_row16(const char* base, int64_t off, bool valid, u32x4* out) {
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    u32x4 w = {0u, 0u, 0u, 0u};
    if (valid) w = *reinterpret_cast<const u32x4*>(reinterpret_cast<const unsigned short*>(base) + off + 8 * t);
    out[t] = w;
  }
}

template <int DT>
__global__ __launch_bounds__(256, 4) void swap_fwd16_kernel(SwapArgs a) {
  __shared__ __attribute__((aligned(1024))) unsigned char st0[2 * kPairTile];  // K, V tiles
  __shared__ __attribute__((aligned(1024))) unsigned char st1[2 * kPairTile];
  __shared__ float ml[2 * 128];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, hi = lane >> 5, lo = lane & 31;
  const int qh = w & 1, kh = w >> 1;
  const int64_t nbh = a.B * a.Hq;
  const int64_t bh = blockIdx.x % nbh, qt = a.nqt - 1 - blockIdx.x / nbh;
  const int64_t b = bh / a.Hq, h = bh % a.Hq, kvh = h / a.G;
  const int64_t q0 = qt * 64;
  const int r = 32 * qh + lo;
  const int64_t qi = q0 + r;
  const bool qvalid = qi < a.n;
  u32x4 qv[4];
  load_row16(a.q, b * a.qsb + h * a.qsh + qi * a.qsn + 32 * hi, qvalid, qv);
  const unsigned long long* mrow = a.masks + (bh * a.nqt + qt) * a.nb;
  const char* kb = a.k + (b * a.ksb + kvh * a.ksh) * 2;
  const char* vb = a.v + (b * a.vsb + kvh * a.vsh) * 2;
  const float sl2 = a.scale_log2;

  float m = -INFINITY, l = 0.0f;
  f32x16 o[2];
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int e = 0; e < 16; ++e) o[x][e] = 0.0f;
  int64_t qlast = q0 + 63;
  if (qlast > a.n - 1) qlast = a.n - 1;
  TileCursor cur{mrow, (int)a.block, (int)a.nb, (int)(qlast / 64) + 1, -1, 0ull, 0ull};
  const int nkt = cur.nkt;
  const PairOffsets off(lane, kh);
  auto key_bits = [&](int kt) {
    return cur.keys(kt, qvalid ? r : -1, (int)qi, 32 * kh + 4 * hi);
  };
  auto compute = [&](const unsigned char* st, unsigned int keys) {
    if (!__any(keys != 0u)) return;  // no row of the wave attends a key of its half
    f32x16 s;
#pragma unroll
    for (int e = 0; e < 16; ++e) s[e] = 0.0f;
#pragma unroll
    for (int t = 0; t < 4; ++t) s = Mma16<DT>::mma(lds16(st + off.row[t]), qv[t], s);
    float mx = -INFINITY;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      s[e] = masked(s[e], bit_mask(keys, (e >> 2) * 8 + (e & 3)), -INFINITY);
      mx = fmaxf(mx, s[e]);
    }
    const float mnew = fmaxf(m, pair_max(mx) * sl2);
    if (__any(mnew > m)) {  // (rare after the first tiles)
      const float alpha = mnew > m ? __builtin_amdgcn_exp2f(m - mnew) : 1.0f;
      l *= alpha;
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[x][e] *= alpha;
      m = mnew;
    }
    const float mref = m == -INFINITY ? 0.0f : m;
    float p[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      p[e] = __builtin_amdgcn_exp2f(fmaf(s[e], sl2, -mref));
      l += p[e];
    }
    const u32x4 p0 = pack8<DT>(p), p1 = pack8<DT>(p + 8);
#pragma unroll
    for (int dh = 0; dh < 2; ++dh) {
      o[dh] = Mma16<DT>::mma(lds_cols(st + kPairTile, off, dh, 0), p0, o[dh]);
      o[dh] = Mma16<DT>::mma(lds_cols(st + kPairTile, off, dh, 1), p1, o[dh]);
    }
  };
  int kt = cur.next(0, lane);
  unsigned int keys = 0u;
  if (kt < nkt) {
    keys = key_bits(kt);
    issue_pair(kb, a.ksn, vb, a.vsn, (int64_t)kt * 64, a.n, st0, w, lane);
  }
  while (kt < nkt) {
    int nxt = cur.next(kt + 1, lane);
    unsigned int nkeys = nxt < nkt ? key_bits(nxt) : 0u;
    dma_barrier();  // st0 has landed for every wave; st1 is no longer read
    if (nxt < nkt) issue_pair(kb, a.ksn, vb, a.vsn, (int64_t)nxt * 64, a.n, st1, w, lane);
    compute(st0, keys);
    kt = nxt;
    if (kt >= nkt) break;
    keys = nkeys;
    nxt = cur.next(kt + 1, lane);
    nkeys = nxt < nkt ? key_bits(nxt) : 0u;
    dma_barrier();  // st1 has landed; st0 is no longer read
    if (nxt < nkt) issue_pair(kb, a.ksn, vb, a.vsn, (int64_t)nxt * 64, a.n, st0, w, lane);
    compute(st1, keys);
    kt = nxt;
    keys = nkeys;
  }
  l = pair_sum(l);
  __syncthreads();
  float* buf = reinterpret_cast<float*>(st0);  // 32 x 128 floats
  const int slot = qh * 64 + lane;
  if (kh == 1) {
    ml[slot] = m;
    ml[128 + slot] = l;
#pragma unroll
    for (int x = 0; x < 32; ++x) buf[x * 128 + slot] = o[x >> 4][x & 15];
  }
  __syncthreads();
  if (kh == 1 || !qvalid) return;
  const float m1 = ml[slot], l1 = ml[128 + slot];
  const float M = fmaxf(m, m1);
  const float a0 = m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m - M);
  const float a1 = m1 == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m1 - M);
  const float lt = l * a0 + l1 * a1;
  const float inv = 1.0f / lt;
  float of[32];
#pragma unroll
  for (int x = 0; x < 32; ++x) of[x] = (o[x >> 4][x & 15] * a0 + buf[x * 128 + slot] * a1) * inv;
  const int64_t ooff = b * a.osb + h * a.osh + qi * a.osn;
#pragma unroll
  for (int dh = 0; dh < 2; ++dh)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int d0 = 32 * dh + 8 * g + 4 * hi, x = 16 * dh + 4 * g;
      store4<DT>(a.o, ooff + d0, of[x], of[x + 1], of[x + 2], of[x + 3]);
    }
  if (hi == 0) a.lse[bh * a.n + qi] = (M + log2f(lt)) * kLn2S;
}

template <int DT>
__global__ __launch_bounds__(256, 3) void swap_dq16_kernel(SwapArgs a) {
  __shared__ __attribute__((aligned(1024))) unsigned char st0[2 * kPairTile];  // K, V tiles
  __shared__ __attribute__((aligned(1024))) unsigned char st1[2 * kPairTile];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, hi = lane >> 5, lo = lane & 31;
  const int qh = w & 1, kh = w >> 1;
  const int64_t nbh = a.B * a.Hq;
  const int64_t bh = blockIdx.x % nbh, qt = a.nqt - 1 - blockIdx.x / nbh;
  const int64_t b = bh / a.Hq, h = bh % a.Hq, kvh = h / a.G;
  const int64_t q0 = qt * 64;
  const int r = 32 * qh + lo;
  const int64_t qi = q0 + r;
  const bool qvalid = qi < a.n;
  u32x4 qv[4], gv[4];
  load_row16(a.q, b * a.qsb + h * a.qsh + qi * a.qsn + 32 * hi, qvalid, qv);
  const int64_t ooff = b * a.osb + h * a.osh + qi * a.osn + 32 * hi;
  load_row16(a.dout, ooff, qvalid, gv);
  float Di;
  {
    float orow[32], grow[32];
    load_row32<DT>(a.o, ooff, qvalid, orow);
#pragma unroll
    for (int t = 0; t < 4; ++t) unpack8(gv[t], grow + 8 * t, DT == SSA_BF16);
    float acc = 0.0f;
#pragma unroll
    for (int t = 0; t < 32; ++t) acc = fmaf(grow[t], orow[t], acc);
    Di = pair_sum(acc);
  }
  const int64_t rid = bh * a.n + qi;
  const float lse2 = qvalid ? a.lse[rid] * kLog2eS : 0.0f;
  if (qvalid && kh == 0 && hi == 0) a.delta[rid] = Di;
  const unsigned long long* mrow = a.masks + (bh * a.nqt + qt) * a.nb;
  const char* kb = a.k + (b * a.ksb + kvh * a.ksh) * 2;
  const char* vb = a.v + (b * a.vsb + kvh * a.vsh) * 2;
  const float sl2 = a.scale_log2;

  f32x16 dqa[2];
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int e = 0; e < 16; ++e) dqa[x][e] = 0.0f;
  int64_t qlast = q0 + 63;
  if (qlast > a.n - 1) qlast = a.n - 1;
  TileCursor cur{mrow, (int)a.block, (int)a.nb, (int)(qlast / 64) + 1, -1, 0ull, 0ull};
  const int nkt = cur.nkt;
  const PairOffsets off(lane, kh);
  auto key_bits = [&](int kt) {
    return cur.keys(kt, qvalid ? r : -1, (int)qi, 32 * kh + 4 * hi);
  };
  auto compute = [&](const unsigned char* st, unsigned int keys) {
    if (!__any(keys != 0u)) return;  // no row of the wave attends a key of its half
    f32x16 s, dp;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      s[e] = 0.0f;
      dp[e] = 0.0f;
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      s = Mma16<DT>::mma(lds16(st + off.row[t]), qv[t], s);
      dp = Mma16<DT>::mma(lds16(st + kPairTile + off.row[t]), gv[t], dp);
    }
    float ds[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const float p = masked(__builtin_amdgcn_exp2f(fmaf(s[e], sl2, -lse2)),
                             bit_mask(keys, (e >> 2) * 8 + (e & 3)), 0.0f);
      ds[e] = p * (dp[e] - Di);
    }
    const u32x4 d0 = pack8<DT>(ds), d1 = pack8<DT>(ds + 8);
#pragma unroll
    for (int dh = 0; dh < 2; ++dh) {
      dqa[dh] = Mma16<DT>::mma(lds_cols(st, off, dh, 0), d0, dqa[dh]);
      dqa[dh] = Mma16<DT>::mma(lds_cols(st, off, dh, 1), d1, dqa[dh]);
    }
  };
  int kt = cur.next(0, lane);
  unsigned int keys = 0u;
  if (kt < nkt) {
    keys = key_bits(kt);
    issue_pair(kb, a.ksn, vb, a.vsn, (int64_t)kt * 64, a.n, st0, w, lane);
  }
  while (kt < nkt) {
    int nxt = cur.next(kt + 1, lane);
    unsigned int nkeys = nxt < nkt ? key_bits(nxt) : 0u;
    dma_barrier();  // st0 has landed for every wave; st1 is no longer read
    if (nxt < nkt) issue_pair(kb, a.ksn, vb, a.vsn, (int64_t)nxt * 64, a.n, st1, w, lane);
    compute(st0, keys);
    kt = nxt;
    if (kt >= nkt) break;
    keys = nkeys;
    nxt = cur.next(kt + 1, lane);
    nkeys = nxt < nkt ? key_bits(nxt) : 0u;
    dma_barrier();  // st1 has landed; st0 is no longer read
    if (nxt < nkt) issue_pair(kb, a.ksn, vb, a.vsn, (int64_t)nxt * 64, a.n, st0, w, lane);
    compute(st1, keys);
    kt = nxt;
    keys = nkeys;
  }
  __syncthreads();
  float* buf = reinterpret_cast<float*>(st0);  // 32 x 128 floats
  const int slot = qh * 64 + lane;
  if (kh == 1) {
#pragma unroll
    for (int x = 0; x < 32; ++x) buf[x * 128 + slot] = dqa[x >> 4][x & 15];
  }
  __syncthreads();
  if (kh == 1 || !qvalid) return;
#pragma unroll
  for (int dh = 0; dh < 2; ++dh)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int dd = 32 * dh + 8 * g + 4 * hi, x = 16 * dh + 4 * g;
      f32x4 val;
#pragma unroll
      for (int j = 0; j < 4; ++j) val[j] = (dqa[dh][4 * g + j] + buf[(x + j) * 128 + slot]) * a.scale;
      store_grad4<DT>(a.dq, rid * 64 + dd, val, a.grad16);
    }
}

template <int DT>
__global__ __launch_bounds__(256, 2) void swap_dkdv16_kernel(SwapArgs a) {
  __shared__ __attribute__((aligned(1024))) unsigned char st0[2 * kPairTile];  // Q, dO tiles
  __shared__ __attribute__((aligned(1024))) unsigned char st1[2 * kPairTile];
  __shared__ float ld_s[2][2][64];  // [stage][lse, delta][row]
  __shared__ unsigned long long act_s[4];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, hi = lane >> 5, lo = lane & 31;
  const int kq = w & 1, qp = w >> 1;
  const int64_t nbkv = a.B * a.Hkv;
  const int64_t bkv = blockIdx.x % nbkv, kt = blockIdx.x / nbkv;
  const int64_t b = bkv / a.Hkv, kvh = bkv % a.Hkv;
  const int64_t k0 = kt * 64;
  const int64_t key = k0 + 32 * kq + lo;
  const bool kvalid = key < a.n;
  u32x4 kv[4], vv[4];
  load_row16(a.k, b * a.ksb + kvh * a.ksh + key * a.ksn + 32 * hi, kvalid, kv);
  load_row16(a.v, b * a.vsb + kvh * a.vsh + key * a.vsn + 32 * hi, kvalid, vv);
  const int64_t ck = kvalid ? key / a.block : 0;
  const float sl2 = a.scale_log2;

  f32x16 dka[2], dva[2];
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      dka[x][e] = 0.0f;
      dva[x][e] = 0.0f;
    }
  const PairOffsets off(lane, qp);
  auto compute = [&](const unsigned char* st, const float (*ld)[64], unsigned int rows) {
    if (!__any(rows != 0u)) return;  // no row of the wave's half attends a key of its half
    f32x16 s, dp;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      s[e] = 0.0f;
      dp[e] = 0.0f;
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      s = Mma16<DT>::mma(lds16(st + off.row[t]), kv[t], s);
      dp = Mma16<DT>::mma(lds16(st + kPairTile + off.row[t]), vv[t], dp);
    }
    float p[16], ds[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int qq = 32 * qp + (e >> 2) * 8 + hi * 4 + (e & 3);
      p[e] = masked(__builtin_amdgcn_exp2f(fmaf(s[e], sl2, -ld[0][qq])),
                    bit_mask(rows, (e >> 2) * 8 + (e & 3)), 0.0f);
      ds[e] = p[e] * (dp[e] - ld[1][qq]);
    }
    const u32x4 p0 = pack8<DT>(p), p1 = pack8<DT>(p + 8);
    const u32x4 d0 = pack8<DT>(ds), d1 = pack8<DT>(ds + 8);
#pragma unroll
    for (int dh = 0; dh < 2; ++dh) {
      dva[dh] = Mma16<DT>::mma(lds_cols(st + kPairTile, off, dh, 0), p0, dva[dh]);
      dva[dh] = Mma16<DT>::mma(lds_cols(st + kPairTile, off, dh, 1), p1, dva[dh]);
      dka[dh] = Mma16<DT>::mma(lds_cols(st, off, dh, 0), d0, dka[dh]);
      dka[dh] = Mma16<DT>::mma(lds_cols(st, off, dh, 1), d1, dka[dh]);
    }
  };
  // The walk over (query head, query tile) pairs. A pair's mask word and (threads 0..127) its row's
  // lse or delta are loaded one pair before its tiles are, two before it is multiplied.
  struct Pair {
    int64_t g, qt;
    unsigned long long mw;
    float ld;
  };
  int64_t chunk = -1;
  auto next_pair = [&](Pair at) {  // the pair at or after `at`; g == G: none left
    for (; at.g < a.G; ++at.g, at.qt = k0 / 64, chunk = -1) {
      const int64_t bh = b * a.Hq + kvh * a.G + at.g;
      at.qt = next_active_tile(a, bh, k0, at.qt, act_s, chunk);
      if (at.qt < a.nqt) {
        at.mw = kvalid ? a.masks[(bh * a.nqt + at.qt) * a.nb + ck] : 0ull;
        const int64_t row = at.qt * 64 + lane;
        if (tid < 128)  // (rows past the end belong to no list, but an infinity would be NaN)
          at.ld = row < a.n ? (tid < 64 ? a.lse : a.delta)[bh * a.n + row] : 0.0f;
        break;
      }
    }
    return at;
  };
  auto after = [&](Pair at) {
    if (at.g >= a.G) return at;
    ++at.qt;
    return next_pair(at);
  };
  auto issue = [&](const Pair& at, unsigned char* st, float (*ld)[64]) {
    const int64_t hq = kvh * a.G + at.g;
    issue_pair(a.q + (b * a.qsb + hq * a.qsh) * 2, a.qsn, a.dout + (b * a.osb + hq * a.osh) * 2,
               a.osn, at.qt * 64, a.n, st, w, lane);
    if (tid < 128) ld[tid >> 6][lane] = tid < 64 ? at.ld * kLog2eS : at.ld;
  };
  // the rows of the lane's half that attend its key, as the 32 bits from row 32 qp + 4 hi on
  auto rows_of = [&](const Pair& at) {
    unsigned long long mw = at.mw;
    const int ahead = (int)(key - at.qt * 64);  // token causal: rows at or after the key
    if (ahead > 0) mw &= ~0ull << ahead;        // (< 64: the walk starts at the key's tile)
    return (unsigned int)(mw >> (32 * qp + 4 * hi));
  };
  Pair at = next_pair(Pair{0, k0 / 64, 0ull, 0.0f});
  if (at.g < a.G) issue(at, st0, ld_s[0]);
  Pair nx = after(at);
  while (at.g < a.G) {
    dma_barrier();  // stage 0 has landed for every wave; stage 1 is no longer read
    if (nx.g < a.G) issue(nx, st1, ld_s[1]);
    Pair nn = after(nx);
    compute(st0, ld_s[0], rows_of(at));
    at = nx;
    nx = nn;
    if (at.g >= a.G) break;
    dma_barrier();  // stage 1 has landed; stage 0 is no longer read
    if (nx.g < a.G) issue(nx, st0, ld_s[0]);
    nn = after(nx);
    compute(st1, ld_s[1], rows_of(at));
    at = nx;
    nx = nn;
  }
  __syncthreads();
  float* bk = reinterpret_cast<float*>(st0);  // 32 x 128 floats each
  float* bv = reinterpret_cast<float*>(st1);
  const int slot = kq * 64 + lane;
  if (qp == 1) {
#pragma unroll
    for (int x = 0; x < 32; ++x) {
      bk[x * 128 + slot] = dka[x >> 4][x & 15];
      bv[x * 128 + slot] = dva[x >> 4][x & 15];
    }
  }
  __syncthreads();
  if (qp == 1 || !kvalid) return;
  const int64_t krow = (bkv * a.n + key) * 64;
#pragma unroll
  for (int dh = 0; dh < 2; ++dh)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int dd = 32 * dh + 8 * g + 4 * hi, x = 16 * dh + 4 * g;
      f32x4 kv4, vv4;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        kv4[j] = (dka[dh][4 * g + j] + bk[(x + j) * 128 + slot]) * a.scale;
        vv4[j] = dva[dh][4 * g + j] + bv[(x + j) * 128 + slot];
      }
      store_grad4<DT>(a.dk, krow + dd, kv4, a.grad16);
      store_grad4<DT>(a.dv, krow + dd, vv4, a.grad16);
    }
}

int fill_args(SwapArgs& a, const void* q, const void* k, const void* v, const void* out,
              int dtype, int64_t B, int64_t Hq, int64_t Hkv, int64_t n, int64_t block,
              const int64_t* strides, const int32_t* kv_num, const int32_t* kv_idx, int64_t W,
              float scale, void* workspace, size_t workspace_bytes) {
  SSA_REQUIRE(aligned16(q) && aligned16(k) && aligned16(v) && aligned16(out), SSA_ERR_UNSUPPORTED,
              "masked_attn: q, k, v and out must be 16-byte aligned");
  a.q = static_cast<const char*>(q);
  a.k = static_cast<const char*>(k);
  a.v = static_cast<const char*>(v);
  a.o = static_cast<char*>(const_cast<void*>(out));
  a.qsb = strides[0]; a.qsh = strides[1]; a.qsn = strides[2];
  a.ksb = strides[3]; a.ksh = strides[4]; a.ksn = strides[5];
  a.vsb = strides[6]; a.vsh = strides[7]; a.vsn = strides[8];
  a.osb = strides[9]; a.osh = strides[10]; a.osn = strides[11];
  a.B = B; a.Hq = Hq; a.Hkv = Hkv; a.G = Hq / Hkv; a.n = n; a.block = block;
  a.nqt = (n + 63) / 64;
  a.nkt = a.nqt;
  a.nb = (n + block - 1) / block;
  a.kv_num = kv_num; a.kv_idx = kv_idx; a.W = W;
  a.scale = scale;
  a.scale_log2 = scale * kLog2eS;
  const size_t need = masked_tiled_workspace(B, Hq, n, block);
  SSA_REQUIRE(workspace && workspace_bytes >= need, SSA_ERR_WORKSPACE,
              "masked_attn: workspace needs %zu bytes", need);
  a.masks = static_cast<unsigned long long*>(workspace);
  a.delta = reinterpret_cast<float*>(static_cast<char*>(workspace) +
                                     (size_t)B * Hq * a.nqt * a.nb * 8u);
  a.lse = nullptr; a.dout = nullptr; a.dq = a.dk = a.dv = nullptr;
  a.grad16 = false;
  SSA_REQUIRE(B * Hq * a.nqt < (1ll << 31) && B * Hkv * a.nkt < (1ll << 31), SSA_ERR_UNSUPPORTED,
              "masked_attn: grid too large");
  return SSA_OK;
}

}  // namespace

bool masked_tiled_ok(int64_t d, int64_t block, int64_t n) {
  return d == 64 && block >= 1 && (n + block - 1) / block <= kMaxMaskBlocks;
}

size_t masked_tiled_workspace(int64_t B, int64_t Hq, int64_t n, int64_t block) {
  const int64_t nqt = (n + 63) / 64, nb = (n + block - 1) / block;
  return (size_t)B * Hq * nqt * nb * 8u + (size_t)B * Hq * n * 4u;
}

int masked_tiled_fwd(const void* q, const void* k, const void* v, void* out, float* lse,
                     int dtype, int64_t B, int64_t Hq, int64_t Hkv, int64_t n, int64_t block,
                     const int64_t* strides, const int32_t* kv_num, const int32_t* kv_idx,
                     int64_t W, float scale, void* workspace, size_t workspace_bytes,
                     hipStream_t st) {
  SwapArgs a;
  SSA_TRY(fill_args(a, q, k, v, out, dtype, B, Hq, Hkv, n, block, strides, kv_num, kv_idx, W,
                    scale, workspace, workspace_bytes));
  a.lse = lse;
  const unsigned grid = (unsigned)(B * Hq * a.nqt);
  row_block_masks_kernel<<<grid, 256, 0, st>>>(a);
  SSA_TRY(launch_status("row_block_masks_kernel"));
  if (dtype == SSA_F32) swap_fwd_kernel<<<grid, 256, 0, st>>>(a);
  else if (dtype == SSA_F16) swap_fwd16_kernel<SSA_F16><<<grid, 256, 0, st>>>(a);
  else swap_fwd16_kernel<SSA_BF16><<<grid, 256, 0, st>>>(a);
  return launch_status("swap_fwd_kernel");
}

int masked_tiled_bwd(const void* q, const void* k, const void* v, const void* out,
                     const void* dout, const float* lse, void* dq, void* dk, void* dv,
                     int dtype, int grad_dtype, int flags, int64_t B, int64_t Hq, int64_t Hkv, int64_t n, int64_t block,
                     const int64_t* strides, const int32_t* kv_num, const int32_t* kv_idx,
                     int64_t W, float scale, void* workspace, size_t workspace_bytes,
                     hipStream_t st) {
  SwapArgs a;
  SSA_TRY(fill_args(a, q, k, v, out, dtype, B, Hq, Hkv, n, block, strides, kv_num, kv_idx, W,
                    scale, workspace, workspace_bytes));
  SSA_REQUIRE(aligned16(dout) && aligned16(dq) && aligned16(dk) && aligned16(dv),
              SSA_ERR_UNSUPPORTED, "masked_attn_bwd: dout, dq, dk, dv must be 16-byte aligned");
  a.dout = static_cast<const char*>(dout);
  a.lse = const_cast<float*>(lse);
  SSA_REQUIRE(grad_dtype == SSA_F32 || grad_dtype == dtype, SSA_ERR_INVALID,
              "masked_attn_bwd: gradients must be fp32 or the input type");
  a.dq = dq; a.dk = dk; a.dv = dv;
  a.grad16 = grad_dtype != SSA_F32;
  const unsigned gq = (unsigned)(B * Hq * a.nqt), gk = (unsigned)(B * Hkv * a.nkt);
  if (!(flags & SSA_MASKED_MASKS_READY)) {  // else the forward's masks are in the workspace
    row_block_masks_kernel<<<gq, 256, 0, st>>>(a);
    SSA_TRY(launch_status("row_block_masks_kernel"));
  }
  if (dtype == SSA_F32) {
    swap_dq_kernel<<<gq, 256, 0, st>>>(a);
    swap_dkdv_kernel<<<gk, 256, 0, st>>>(a);
  } else if (dtype == SSA_F16) {
    swap_dq16_kernel<SSA_F16><<<gq, 256, 0, st>>>(a);
    swap_dkdv16_kernel<SSA_F16><<<gk, 256, 0, st>>>(a);
  } else {
    swap_dq16_kernel<SSA_BF16><<<gq, 256, 0, st>>>(a);
    swap_dkdv16_kernel<SSA_BF16><<<gk, 256, 0, st>>>(a);
  }
  return launch_status("swap_dkdv_kernel");
}

}  // namespace ssa
