// bn_fused_head.hip -- the reference's fused-head attention chain in one launch or two.
//
// Replaces the chain of llama_layers.hpp:83-109 (fp32):
//   K_rep = repeat_kv(K), V_rep = repeat_kv(V)       (:87-89, :131-168)
//   S = Q @ K_rep^T                                    (:96-98, op_mm)
//   S = S * scale                                      (:101, op_multiply)
//   P = softmax(S, causal, seq_offset)                 (:105, op_softmax.cuh:77-151)
//   O = P @ V_rep                                      (:108-109, op_mm)
// Q is [Sq, H*D]; the chain's scores contract over ALL H*D columns, so one
// probability matrix is shared by every head.  With n_rep = H / KV and head
// h reading KV head h / n_rep (:159-163):
//   S[i][j] = sum_g Qsum_g[i] . K_g[j],   Qsum_g[i] = sum_{r < n_rep} Q_{g*n_rep + r}[i]
// a KV*D-wide contraction instead of an H*D-wide one over K_rep, and
//   O[i][h*D + d] = (P @ V_{h / n_rep})[i][d]
// so the n_rep heads of a group receive the same values.  Neither K_rep,
// V_rep nor the Sq x Sk matrices exist here.
//
// Short key ranges and widths other than 256 (the rest: the matrix-core path
// below): a 256-thread workgroup (4 waves) owns R = 4 query rows and walks the
// visible keys in tiles of 64 with an online softmax:
//   1. the rows' Qsum (R x KV*D) is formed once into LDS;
//   2. scores: thread (wave w, lane l) forms the R partial dots of key l over
//      the w-th quarter of the contraction (each K element is loaded once per
//      workgroup and used R times); the quarters meet in LDS;
//   3. softmax: wave r owns row r (max, exponentials and row sum by wave
//      reductions) and publishes P^T and the rescale factor;
//   4. P.V: thread (w, l) accumulates columns 4l.. of every row over the keys
//      j = w mod 4 of the tile (a wave reads whole V rows: coalesced);
//   5. the four key-split partials meet in LDS and every thread writes its
//      share of the R x H*D output, each group's values to its n_rep heads.
// Why VALU and not fp32 MFMA: at the config this chain runs on (Sq = Sk =
// 128, KV*D = 256) the launch is latency-bound -- 17 MFLOP and 2.4 MB of
// algorithmic traffic, i.e. well under a microsecond at either roofline.
// The v_mfma_f32_16x16x4f32 rate is 2x VALU FMA but needs 16-row tiles:
// 4x fewer workgroups (8 at Sq = 128) and 4x the per-workgroup work, so the
// last workgroup would finish later.  Four rows per workgroup also balance
// the K/V bytes a workgroup pulls from L2 against its FMAs (R FMAs per
// loaded float).  Measured (rocprofv3, 300 launches): 13.0 us at Sq = 128
// (2 key tiles on the longest rows), 34.3 us at 512 (8 tiles): ~6 us fixed
// (launch, Q and the first tile's K/V, output) and ~3.5 us per tile, of
// which the dot products take ~0.9 and P.V ~0.4; the rest is the 128 KB of
// K and V each workgroup pulls per tile through one CU.
#include <algorithm>

#include "bn_common.hpp"

namespace bn {
namespace {

constexpr int kRows = 4;      // query rows per workgroup (= waves)
constexpr int kTile = 64;     // keys per tile (= lanes)
constexpr int kMaxKvd = 512;  // KV*D limit: 2 column chunks of 256
constexpr int kRepChunk = 8;  // Q heads summed per batch of loads

struct FusedHeadParams {
  const float *q, *k, *v;
  float *o;
  int64_t ldq, ldk, ldv, ldo;  // row strides in elements (columns contiguous)
  int sq, sk;
  int n_heads, head_dim, kvd, n_rep;
  float scale;
  int causal, seq_offset;
};

__device__ __forceinline__ float4 ld4(const float *p) { return *reinterpret_cast<const float4 *>(p); }
__device__ __forceinline__ float4 zero4() { return float4{0.f, 0.f, 0.f, 0.f}; }

// Max over the wave without an LDS round trip: DPP inside each 16-lane row
// (quad xor 1, quad xor 2, half-row mirror, row mirror: every source lane is
// in the row), then the four row maxima by readlane.
template <int CTRL>
__device__ __forceinline__ float dpp_mov(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL,
                                                               0xf, 0xf, false));
}
__device__ __forceinline__ float lane_of(float v, int lane) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
}
__device__ __forceinline__ float wave_max_dpp(float x) {
  x = fmaxf(x, dpp_mov<0xB1>(x));
  x = fmaxf(x, dpp_mov<0x4E>(x));
  x = fmaxf(x, dpp_mov<0x141>(x));
  x = fmaxf(x, dpp_mov<0x140>(x));
  return fmaxf(fmaxf(lane_of(x, 0), lane_of(x, 16)), fmaxf(lane_of(x, 32), lane_of(x, 48)));
}

// KC = 256-column chunks of KV*D (1: KV*D <= 256, 2: <= 512).  The launch is
// latency-bound, so every phase issues all of its global loads before the
// first use: K and V of tile 0, then Q (the rows' heads) behind them; with
// KC = 1 the K quarter of tile t+1 is in flight during the softmax and P.V of
// tile t, and its V rows during the softmax of tile t+1.
// FQ: the contraction quarter in float4s when fixed at compile time (16 for
// KV*D = 256: no per-load predicates), 0 when read from p.kvd.
template <int KC, int FQ>
__global__ __launch_bounds__(256) void fused_head_attention_kernel(FusedHeadParams p) {
  constexpr int NQ = 4 * KC;   // float4s of one contraction quarter per 256 columns
  // KC = 1: the next tile's K and V stay in registers across a tile (128
  // VGPRs); KC = 2 would need 256, so it loads K, then V, per tile
  constexpr bool kPipe = KC == 1;
  __shared__ float4 qs[kRows][kMaxKvd / 4];       // Qsum rows
  __shared__ float part[4][kRows][kTile];         // quarter partial dots
  __shared__ float4 pt[kTile];                    // P^T: key -> 4 rows
  __shared__ float alpha_s[kRows], lsum_s[kRows];
  __shared__ float4 obuf[4][kRows][kMaxKvd / 4];  // key-split partial O

  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
  const int r0 = blockIdx.x * kRows;
  const int nrows = min(kRows, p.sq - r0);
  const int kvd4 = p.kvd >> 2, D = p.head_dim;
  const int quarter4 = FQ ? FQ : kvd4 >> 2;  // float4s per contraction quarter (<= 4*NQ)

  // visible keys of the block: j < kend (row r also needs j <= r0 + r + off)
  const int last = r0 + nrows - 1;
  int kend = p.sk;
  if (p.causal) kend = (int)min((int64_t)p.sk, max((int64_t)0, (int64_t)last + p.seq_offset + 1));

  // K quarter w of key kb + lane, V rows kb + w + 4u (u < 16) at columns 4*lane + 256*cc
  float4 kx[4 * NQ];
  float4 vx[KC][16];
  auto load_k = [&](int kb) __attribute__((always_inline)) {
    const int j = min(kb + lane, kend - 1);
    const float *kr = p.k + (int64_t)j * p.ldk + 4 * w * quarter4;
#pragma unroll
    for (int i = 0; i < 4 * NQ; ++i) kx[i] = (FQ || i < quarter4) ? ld4(kr + 4 * i) : zero4();
  };
  // Rows past the tile's last key are read at the last key (in bounds, P = 0
  // there): no branch around the loads, so their waits stay counted.
  auto load_v = [&](int kb) __attribute__((always_inline)) {
    const int nk = min(kTile, kend - kb);
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      const float *vr = p.v + (int64_t)(kb + min(w + 4 * u, nk - 1)) * p.ldv;
#pragma unroll
      for (int cc = 0; cc < KC; ++cc) {
        const int c = 4 * lane + 256 * cc;
        vx[cc][u] = (FQ || c < p.kvd) ? ld4(vr + c) : zero4();
      }
    }
  };

  // tile 0's K and V go out first; the Q loads queue behind them
  if (kPipe && kend > 0) {
    load_k(0);
    load_v(0);
  }
  // 1. Qsum: column c = g*D + d sums Q columns (g*n_rep + r)*D + d, r ascending
  for (int e = tid; e < kRows * kvd4; e += 256) {
    const int r = e / kvd4, c = 4 * (e - r * kvd4);
    const int g = c / D, d = c - g * D;
    // rows past the last one and heads past the group re-read a valid
    // element and are weighted 0: the loads need no branch
    float4 acc = zero4();
    const float row_w = r < nrows ? 1.f : 0.f;
    const float *src = p.q + (int64_t)(r0 + min(r, nrows - 1)) * p.ldq + (int64_t)g * p.n_rep * D + d;
    for (int rb = 0; rb < p.n_rep; rb += kRepChunk) {
      float4 x[kRepChunk];
#pragma unroll
      for (int rr = 0; rr < kRepChunk; ++rr) x[rr] = ld4(src + min(rb + rr, p.n_rep - 1) * D);
#pragma unroll
      for (int rr = 0; rr < kRepChunk; ++rr) {
        const float f = rb + rr < p.n_rep ? row_w : 0.f;
        acc.x = fmaf(f, x[rr].x, acc.x);
        acc.y = fmaf(f, x[rr].y, acc.y);
        acc.z = fmaf(f, x[rr].z, acc.z);
        acc.w = fmaf(f, x[rr].w, acc.w);
      }
    }
    qs[r][c >> 2] = acc;
  }
  // row w's state (wave w): running max, and this lane's share of the row sum
  // (the lanes' shares meet once, after the last tile)
  float m_row = -INFINITY, l_lane = 0.f;
  float4 oacc[kRows][KC];
#pragma unroll
  for (int r = 0; r < kRows; ++r)
#pragma unroll
    for (int cc = 0; cc < KC; ++cc) oacc[r][cc] = zero4();
  __syncthreads();

  const int64_t row_lim = (int64_t)(r0 + w) + p.seq_offset;  // wave w runs row r0 + w
  for (int kb = 0; kb < kend; kb += kTile) {
    const int nk = min(kTile, kend - kb);
    if (!kPipe) load_k(kb);
    // 2. partial dots of key kb + lane over quarter w
    {
      float acc[kRows] = {0.f, 0.f, 0.f, 0.f};
      const float4 *qq = &qs[0][w * quarter4];
#pragma unroll
      for (int i = 0; i < 4 * NQ; ++i) {
        if (FQ || i < quarter4) {
#pragma unroll
          for (int r = 0; r < kRows; ++r) {
            const float4 a = qq[r * (kMaxKvd / 4) + i];
            acc[r] = fmaf(a.x, kx[i].x, acc[r]);
            acc[r] = fmaf(a.y, kx[i].y, acc[r]);
            acc[r] = fmaf(a.z, kx[i].z, acc[r]);
            acc[r] = fmaf(a.w, kx[i].w, acc[r]);
          }
        }
      }
#pragma unroll
      for (int r = 0; r < kRows; ++r) part[w][r][lane] = acc[r];
    }
    if (kPipe && kb + kTile < kend) load_k(kb + kTile);  // next tile's K in flight
    if (!kPipe) load_v(kb);
    __syncthreads();
    // 3. online softmax of row w over the tile
    {
      const int j = kb + lane;
      float s = ((part[0][w][lane] + part[1][w][lane]) + part[2][w][lane]) + part[3][w][lane];
      s *= p.scale;
      const bool vis = w < nrows && lane < nk && (!p.causal || (int64_t)j <= row_lim);
      s = vis ? s : -INFINITY;
      const float m_new = fmaxf(m_row, wave_max_dpp(s));
      const float mn = m_new == -INFINITY ? 0.f : m_new;
      const float pj = vis ? expf(s - mn) : 0.f;
      const float alpha = expf(m_row - mn);  // m_row = -inf -> 0 (l and O are 0 then)
      l_lane = fmaf(l_lane, alpha, pj);
      m_row = m_new;
      reinterpret_cast<float *>(&pt[lane])[w] = pj;
      if (lane == 0) alpha_s[w] = alpha;
    }
    __syncthreads();
    // 4. O += P V over keys j = w (mod 4) of the tile
    {
      float al[kRows];
#pragma unroll
      for (int r = 0; r < kRows; ++r) al[r] = alpha_s[r];
#pragma unroll
      for (int r = 0; r < kRows; ++r)
#pragma unroll
        for (int cc = 0; cc < KC; ++cc) {
          oacc[r][cc].x *= al[r];
          oacc[r][cc].y *= al[r];
          oacc[r][cc].z *= al[r];
          oacc[r][cc].w *= al[r];
        }
#pragma unroll
      for (int u = 0; u < 16; ++u) {
        const float4 pp = pt[w + 4 * u];  // 0 past the tile's last key
        const float pr[kRows] = {pp.x, pp.y, pp.z, pp.w};
#pragma unroll
        for (int cc = 0; cc < KC; ++cc)
#pragma unroll
          for (int r = 0; r < kRows; ++r) {
            oacc[r][cc].x = fmaf(pr[r], vx[cc][u].x, oacc[r][cc].x);
            oacc[r][cc].y = fmaf(pr[r], vx[cc][u].y, oacc[r][cc].y);
            oacc[r][cc].z = fmaf(pr[r], vx[cc][u].z, oacc[r][cc].z);
            oacc[r][cc].w = fmaf(pr[r], vx[cc][u].w, oacc[r][cc].w);
          }
      }
    }
    if (kPipe && kb + kTile < kend) load_v(kb + kTile);
  }

  // 5. merge the key-split partials, normalise, write each group to its heads
#pragma unroll
  for (int r = 0; r < kRows; ++r)
#pragma unroll
    for (int cc = 0; cc < KC; ++cc) {
      const int c = 4 * lane + 256 * cc;
      if (c < p.kvd) obuf[w][r][c >> 2] = oacc[r][cc];
    }
  const float l_row = wave_sum(l_lane);
  if (lane == 0) lsum_s[w] = l_row;
  __syncthreads();
  const int hd4 = (p.n_heads * D) >> 2;
  for (int e = tid; e < nrows * hd4; e += 256) {
    const int r = e / hd4, c = 4 * (e - r * hd4);
    const int h = c / D, d = c - h * D;
    const int src = ((h / p.n_rep) * D + d) >> 2;
    const float4 a = obuf[0][r][src], b = obuf[1][r][src], x = obuf[2][r][src],
                 y = obuf[3][r][src];
    const float l = lsum_s[r];
    float4 out = zero4();
    if (l > 0.f) {  // a row with no visible key: the chain's P row is all 0
      const float inv = 1.f / l;
      out.x = (((a.x + b.x) + x.x) + y.x) * inv;
      out.y = (((a.y + b.y) + x.y) + y.y) * inv;
      out.z = (((a.z + b.z) + x.z) + y.z) * inv;
      out.w = (((a.w + b.w) + x.w) + y.w) * inv;
    }
    *reinterpret_cast<float4 *>(p.o + (int64_t)(r0 + r) * p.ldo + c) = out;
  }
}

// ------------------------------------------------------- matrix-core path
// KV*D = 256 (TinyLLaMA's 4 KV heads of 64) on v_mfma_f32_16x16x4f32, one
// launch or two:
//   1. fh_rows_kernel: a workgroup of 8 waves takes 16 query rows and one split
//      of their visible keys.  The rows' group sums Qsum (times c2 = scale *
//      log2 e: scores in log2 units; summed in head order) go to LDS once.  Each
//      wave then walks its own 16-key tiles with an online softmax: S^T = K.Qs^T
//      over the whole contraction (64 MFMAs in four chains), P straight from the
//      score registers as the B operand of O^T += V^T.P^T (64 MFMAs, all 256
//      value columns).  K and V go from memory to registers, no barrier in the
//      loop; the waves meet in LDS once at the end.
//   2. fh_merge_kernel, with more than one split: merges the splits' records.
// What bounds it: at 512 rows nothing but latency (13.6 us: launch, Q, K and V
// one after the other, 3.4 us of MFMAs, the merge of 8 waves; + 4.9 us for the
// second launch); at 2048 rows and more the matrix rate (8256 tiles of 4096
// cycles on 1024 SIMDs: 14 us of 50) and K/V from L2 (32 KB per tile).
// Measured against one 32-row x 128-key block per workgroup with the group sums
// and the merge in launches of their own and an allocation for both, us per
// call: 512 rows 30-36 -> 18.1, 1024 rows 32-36 -> 27.3, 2048 rows 71.7 -> 50,
// 8192 rows 696 -> 350, 512 rows + 1000 past 36 -> 27.6; and against the VALU
// kernel at fewer rows: 200 rows 19.1 -> 13.2, 384 rows 27.1 -> 15.0, 64 rows +
// 1000 past 65 -> 20.  V's first tile fetched before the barrier: 2-10% slower
// (it delays K).
constexpr int FH_KVD = 256, FH_ROWS = 16, FH_TILE = 16, FH_WAVES = 8, FH_SPLITS = 7;

typedef float fh_f32x4 __attribute__((ext_vector_type(4)));

struct FhParams {
  const float *q, *k, *v;
  float *o, *rec;                   // rec: the splits' records, one row per query row
  int64_t ldq, ldk, ldv, ldo, ldr;  // row strides in elements
  int sq, sk, head_dim, n_rep;
  int n_split, ml;  // records per row; first column of a row's (m, l) pairs
  int direct;       // one split: the workgroup writes the output itself
  int nan_rows;     // a row whose sum is NaN: 1 gives NaN, 0 zeros
  int causal, seq_offset;
  float c2;  // scale * log2(e)
};

// visible keys of query row `row`: [0, key_end)
__device__ __forceinline__ int fh_key_end(const FhParams &p, int row) {
  if (!p.causal) return p.sk;
  const int64_t e = (int64_t)row + p.seq_offset + 1;
  return (int)(e < 0 ? 0 : (e > p.sk ? p.sk : e));
}

// keys per split of the row block that ends with key `kend`: whole tiles,
// every row block's own tiles dealt evenly
__device__ __forceinline__ int fh_chunk(const FhParams &p, int kend) {
  const int tiles = (kend + FH_TILE - 1) / FH_TILE;
  return (tiles + p.n_split - 1) / p.n_split * FH_TILE;
}

__device__ __forceinline__ bool fh_finite(float x) { return fabsf(x) < INFINITY; }

// The values of the 4 columns c.. of one row, given its sums: the n_rep heads
// of the KV head they belong to get the same ones.
__device__ __forceinline__ void fh_store(const FhParams &p, int row, int c, float M, float L, float4 A) {
  float4 out = zero4();
  // a row with no visible key: the chain's P row is all 0
  if (p.nan_rows ? M != -INFINITY : L > 0.f) {
    const float inv = 1.f / L;
    out = make_float4(A.x * inv, A.y * inv, A.z * inv, A.w * inv);
  }
  const int g = c / p.head_dim, d = c - g * p.head_dim;
  float *orow = p.o + (int64_t)row * p.ldo + (int64_t)g * p.n_rep * p.head_dim + d;
  for (int h = 0; h < p.n_rep; ++h) *reinterpret_cast<float4 *>(orow + (int64_t)h * p.head_dim) = out;
}

__global__ __launch_bounds__(64 * FH_WAVES, 2) void fh_rows_kernel(FhParams p) {
  constexpr int QS = FH_KVD + 4;   // row stride of the group sums: 16 rows on 64 different banks
  constexpr int OS = FH_KVD / 2 + 4;
  __shared__ float qsum[FH_ROWS * QS];
  __shared__ float2 ml[FH_WAVES][FH_ROWS];
  __shared__ float obuf[FH_WAVES][FH_ROWS * OS];
  __shared__ int odd_values;  // a tile's infinite or NaN values were left out
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, r16 = lane & 15, kq = lane >> 4;
  const int split = blockIdx.x % p.n_split;
  const int n_rt = (p.sq + FH_ROWS - 1) / FH_ROWS;
  const int rt = n_rt - 1 - blockIdx.x / p.n_split;  // the rows that see most keys first
  const int row0 = rt * FH_ROWS;
  const int kend = fh_key_end(p, min(row0 + FH_ROWS, p.sq) - 1);
  const int chunk = fh_chunk(p, kend);
  const int kbeg = split * chunk, kstop = min(kend, kbeg + chunk);
  if (kbeg >= kend && split > 0) return;  // no record: the merge counts them the same way

  // A operand of S^T: key kt + r16, contraction step (4u + e, kq) = column 16u + 4kq + e
  float4 kr[16];
  auto load_k = [&](int kt) __attribute__((always_inline)) {
    const float *kp = p.k + (int64_t)min(kt + r16, kstop - 1) * p.ldk + 4 * kq;
#pragma unroll
    for (int u = 0; u < 16; ++u) kr[u] = ld4(kp + 16 * u);
  };
  int kt = kbeg + FH_TILE * w;
  if (tid == 0) odd_values = 0;

  // the group sums of rows 2w, 2w + 1: lane = 4 columns, heads in order
  {
    const int c = 4 * lane, g = c / p.head_dim, col = c + g * (p.n_rep - 1) * p.head_dim;
    float4 a[2];
    const float *qr[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) qr[i] = p.q + (int64_t)min(row0 + 2 * w + i, p.sq - 1) * p.ldq + col;
    for (int r0 = 0; r0 < p.n_rep; r0 += kRepChunk) {
      float4 x[kRepChunk][2];
#pragma unroll
      for (int r = 0; r < kRepChunk; ++r)
#pragma unroll
        for (int i = 0; i < 2; ++i) x[r][i] = ld4(qr[i] + (int64_t)min(r0 + r, p.n_rep - 1) * p.head_dim);
      if (r0 == 0 && kt < kstop) load_k(kt);
#pragma unroll
      for (int r = 0; r < kRepChunk; ++r) {
        if (r0 + r >= p.n_rep) break;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          if (r0 + r == 0) {
            a[i] = x[r][i];
          } else {
            a[i].x += x[r][i].x; a[i].y += x[r][i].y; a[i].z += x[r][i].z; a[i].w += x[r][i].w;
          }
        }
      }
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
      *reinterpret_cast<float4 *>(&qsum[(2 * w + i) * QS + c]) =
          make_float4(a[i].x * p.c2, a[i].y * p.c2, a[i].z * p.c2, a[i].w * p.c2);
  }
  __syncthreads();

  // O^T: register i of o[t][e] = value column 64t + 16kq + 4i + e of query r16
  fh_f32x4 o[4][4];
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int e = 0; e < 4; ++e) o[t][e] = fh_f32x4{};
  const int kend_row = row0 + r16 < p.sq ? min(fh_key_end(p, row0 + r16), kstop) : 0;
  const int kall = min(fh_key_end(p, row0), kstop);  // keys that every row of the block sees
  float m = -INFINITY, l = 0.f;
  for (; kt < kstop; kt += FH_TILE * FH_WAVES) {
    asm volatile("" ::: "memory");  // the group sums are read again in each step: kept, they would spill
    // A operand of P.V: value column 64t + 4 r16 + e (tile (t, e)), key kt + 4kq + i
    float4 vr[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float *vp = p.v + (int64_t)min(kt + 4 * kq + i, kstop - 1) * p.ldv + 4 * r16;
#pragma unroll
      for (int t = 0; t < 4; ++t) vr[i][t] = ld4(vp + 64 * t);
    }
    fh_f32x4 s4[4] = {fh_f32x4{}, fh_f32x4{}, fh_f32x4{}, fh_f32x4{}};
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      const float4 b = *reinterpret_cast<const float4 *>(&qsum[r16 * QS + 16 * u + 4 * kq]);
      fh_f32x4 &s = s4[u & 3];
      s = __builtin_amdgcn_mfma_f32_16x16x4f32(kr[u].x, b.x, s, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_16x16x4f32(kr[u].y, b.y, s, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_16x16x4f32(kr[u].z, b.z, s, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_16x16x4f32(kr[u].w, b.w, s, 0, 0, 0);
    }
    if (kt + FH_TILE * FH_WAVES < kstop) load_k(kt + FH_TILE * FH_WAVES);
    // register i: key kt + 4kq + i of query r16
    float pr[4], mx = m;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float x = (s4[0][i] + s4[1][i]) + (s4[2][i] + s4[3][i]);
      pr[i] = kt + 4 * kq + i < kend_row ? x : -INFINITY;
      mx = fmaxf(mx, pr[i]);
    }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float mu = mx == -INFINITY ? 0.f : mx;
    const float al = __builtin_amdgcn_exp2f(m - mu);  // no key so far: 0
    m = mx;
    l *= al;  // the lane's own 4 keys of each tile
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      pr[i] = __builtin_amdgcn_exp2f(pr[i] - mu);
      l += pr[i];
    }
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) o[t][e] *= al;
    // P = 0 does not keep an infinite or NaN value of a hidden key (or of the
    // last one, which stands for those past the end) out of a product: a tile
    // that not every row sees whole takes 0 for it, and the merge below adds it
    // to the rows that do see it (the look at a tile's values costs 0-0.3 us a
    // call; 200 rows 13.15 -> 13.45, 512 rows 18.5 either way)
    if (kt + FH_TILE > kall) {
      float4 z = zero4();  // 0 * x is 0 for a finite x alone
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int t = 0; t < 4; ++t)
          z = make_float4(fmaf(0.f, vr[i][t].x, z.x), fmaf(0.f, vr[i][t].y, z.y), fmaf(0.f, vr[i][t].z, z.z),
                          fmaf(0.f, vr[i][t].w, z.w));
      if (__builtin_amdgcn_ballot_w64(!((z.x + z.y) + (z.z + z.w) == 0.f)) != 0) {
        if (lane == 0) odd_values = 1;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            vr[i][t].x = fh_finite(vr[i][t].x) ? vr[i][t].x : 0.f;
            vr[i][t].y = fh_finite(vr[i][t].y) ? vr[i][t].y : 0.f;
            vr[i][t].z = fh_finite(vr[i][t].z) ? vr[i][t].z : 0.f;
            vr[i][t].w = fh_finite(vr[i][t].w) ? vr[i][t].w : 0.f;
          }
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        o[t][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(vr[i][t].x, pr[i], o[t][0], 0, 0, 0);
        o[t][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(vr[i][t].y, pr[i], o[t][1], 0, 0, 0);
        o[t][2] = __builtin_amdgcn_mfma_f32_16x16x4f32(vr[i][t].z, pr[i], o[t][2], 0, 0, 0);
        o[t][3] = __builtin_amdgcn_mfma_f32_16x16x4f32(vr[i][t].w, pr[i], o[t][3], 0, 0, 0);
      }
  }
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  if (kq == 0) ml[w][r16] = make_float2(m, l);

  // the waves' shares meet in LDS, half of the columns at a time; thread =
  // 4 columns of one row (a wave: two rows)
  const int row = tid >> 5, c = 4 * (tid & 31);
  float M = -INFINITY, L = 0.f, f[FH_WAVES];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    if (h) __syncthreads();
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        *reinterpret_cast<float4 *>(&obuf[w][r16 * OS + 64 * t + 16 * kq + 4 * i]) =
            make_float4(o[2 * h + t][0][i], o[2 * h + t][1][i], o[2 * h + t][2][i], o[2 * h + t][3][i]);
    __syncthreads();
    if (h == 0) {
      float2 x[FH_WAVES];
#pragma unroll
      for (int j = 0; j < FH_WAVES; ++j) x[j] = ml[j][row];
#pragma unroll
      for (int j = 0; j < FH_WAVES; ++j) M = fmaxf(M, x[j].x);
      const float mu = M == -INFINITY ? 0.f : M;
#pragma unroll
      for (int j = 0; j < FH_WAVES; ++j) {
        f[j] = __builtin_amdgcn_exp2f(x[j].x - mu);
        L = fmaf(x[j].y, f[j], L);
      }
    }
    float4 A = zero4();
#pragma unroll
    for (int j = 0; j < FH_WAVES; ++j) {
      const float4 a = *reinterpret_cast<const float4 *>(&obuf[j][row * OS + c]);
      A.x = fmaf(a.x, f[j], A.x); A.y = fmaf(a.y, f[j], A.y);
      A.z = fmaf(a.z, f[j], A.z); A.w = fmaf(a.w, f[j], A.w);
    }
    if (row0 + row >= p.sq) continue;
    if (odd_values) {  // (their P is positive: the sum is what they make it)
      const int seen = min(fh_key_end(p, row0 + row), kstop);
      for (int key = max(kall - FH_TILE + 1, kbeg); key < seen; ++key) {
        if (key - (key - kbeg) % FH_TILE + FH_TILE <= kall) continue;  // (a tile that kept its own)
        const float4 x = ld4(p.v + (int64_t)key * p.ldv + 128 * h + c);
        A.x += fh_finite(x.x) ? 0.f : x.x; A.y += fh_finite(x.y) ? 0.f : x.y;
        A.z += fh_finite(x.z) ? 0.f : x.z; A.w += fh_finite(x.w) ? 0.f : x.w;
      }
    }
    if (p.direct) {
      fh_store(p, row0 + row, 128 * h + c, M, L, A);
    } else {
      float *rec = p.rec + (int64_t)(row0 + row) * p.ldr;
      *reinterpret_cast<float4 *>(rec + FH_KVD * split + 128 * h + c) = A;
      if (h == 0 && c == 0) *reinterpret_cast<float2 *>(rec + p.ml + 2 * split) = make_float2(M, L);
    }
  }
}

// One wave per row (lane = 4 columns): all of the row's records are in
// registers before its first store, so they may lie in the row itself.
__global__ __launch_bounds__(256) void fh_merge_kernel(FhParams p) {
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6), c = 4 * (threadIdx.x & 63);
  if (row >= p.sq) return;
  const int kend = fh_key_end(p, min(row / FH_ROWS * FH_ROWS + FH_ROWS, p.sq) - 1);
  const int chunk = fh_chunk(p, kend);
  const int n = kend > 0 ? (kend + chunk - 1) / chunk : 1;  // the splits that wrote a record
  const float *rec = p.rec + (int64_t)row * p.ldr;
  float2 x[FH_SPLITS];
  float4 a[FH_SPLITS];
#pragma unroll
  for (int j = 0; j < FH_SPLITS; ++j) {
    const int b = min(j, n - 1);
    x[j] = *reinterpret_cast<const float2 *>(rec + p.ml + 2 * b);
    a[j] = ld4(rec + FH_KVD * b + c);
  }
  float M = -INFINITY, L = 0.f;
#pragma unroll
  for (int j = 0; j < FH_SPLITS; ++j) M = fmaxf(M, x[j].x);
  const float mu = M == -INFINITY ? 0.f : M;
  float4 A = zero4();
#pragma unroll
  for (int j = 0; j < FH_SPLITS; ++j) {
    if (j >= n) break;
    const float f = __builtin_amdgcn_exp2f(x[j].x - mu);  // a split the row cannot see: 0
    L = fmaf(x[j].y, f, L);
    A.x = fmaf(a[j].x, f, A.x); A.y = fmaf(a[j].y, f, A.y);
    A.z = fmaf(a[j].z, f, A.z); A.w = fmaf(a[j].w, f, A.w);
  }
  fh_store(p, row, c, M, L, A);
}

// Bytes that a view's elements cover, [lo, hi).
struct Extent {
  uintptr_t lo, hi;
};
Extent extent(const bn_view *v) {
  if (v->h == 0 || v->w == 0) return {0, 0};
  const int64_t first = v->offset, rows = (int64_t)(v->h - 1) * v->stride_h;
  const int64_t lo = first + std::min<int64_t>(rows, 0), hi = first + std::max<int64_t>(rows, 0) + v->w;
  const uintptr_t base = reinterpret_cast<uintptr_t>(v->data);
  return {base + lo * sizeof(float), base + hi * sizeof(float)};
}
bool overlaps(const bn_view *a, const bn_view *b) {
  const Extent x = extent(a), y = extent(b);
  return x.lo < y.hi && y.lo < x.hi;
}

// From this many rows a call may take pool memory, and a row whose sum is NaN
// comes out as NaN; shorter calls take none and give zeros, as the VALU kernel.
constexpr int kPoolRows = 512;
// Up to this many keys a call shorter than that stays with the VALU kernel: two
// key tiles there take less than a second launch (128 rows of 128 keys 12.4 us
// against 13.0; of 140 keys 15.6 against 12.9).
constexpr int kValuKeys = 128;

// Splits of a row block's keys.  Up to 36 row blocks, all of them at seven
// splits are on the card at once; more row blocks fill it with fewer splits,
// and four (two) are left for their unequal lengths under the causal mask.
// Measured, us per call, no past, 7 / 6 / 4 / 2 / 1 splits: 384 rows 15.0 /
// 16.6 / 16.7 / 19.5 / 25.3; 600 rows - / 19.4 / 20.4 / 25.7 / 34.3; 1024
// rows 29.8 / 28.6 / 27.3 / 35.3 / 49.4; 2048 rows 66 / 60 / 50 / 59 / 89;
// 4096 rows - / 153 / 132 / 115 / 166; 8192 rows - / 453 / 408 / 375 / 350.
int fh_splits(int n_rt, int tiles) {
  const int n = n_rt <= 36 ? 7 : n_rt <= 42 ? 6 : n_rt <= 160 ? 4 : n_rt < 512 ? 2 : 1;
  return std::max(1, std::min(n, tiles));
}

int launch_rows(const bn_view *q, const bn_view *k, const bn_view *v, const bn_view *o, int head_dim,
                int n_rep, float scale, int causal, int seq_offset, hipStream_t s, bool alias) {
  FhParams f;
  f.q = reinterpret_cast<const float *>(q->data) + q->offset;
  f.k = reinterpret_cast<const float *>(k->data) + k->offset;
  f.v = reinterpret_cast<const float *>(v->data) + v->offset;
  f.o = reinterpret_cast<float *>(o->data) + o->offset;
  f.ldq = q->stride_h; f.ldk = k->stride_h; f.ldv = v->stride_h; f.ldo = o->stride_h;
  f.sq = q->h; f.sk = k->h;
  f.head_dim = head_dim; f.n_rep = n_rep;
  f.causal = causal ? 1 : 0;
  f.seq_offset = seq_offset;
  f.c2 = scale * 1.4426950408889634f;
  f.nan_rows = q->h >= kPoolRows;
  const int n_rt = (q->h + FH_ROWS - 1) / FH_ROWS, tiles = (k->h + FH_TILE - 1) / FH_TILE;
  const int want = fh_splits(n_rt, tiles);
  // The records lie in the output's own rows ([split][256], the last 256 for
  // the (m, l) pairs): an allocation and its release cost 13 us per call.  Pool
  // memory only where the output overlaps an input, or where the rows' room
  // leaves fewer splits than wanted and those cost more (a round of the 8 waves
  // takes 4.6 us: 512 rows + 8000 past, 328 us at one split and 67 at seven).
  const int room = std::max(1, n_rep - 1);
  const bool mem = alias || (q->h >= kPoolRows && want > room &&
                             (int64_t)tiles * (want - room) > 24 * (int64_t)want * room);
  f.n_split = mem ? want : std::min(want, room);
  f.direct = f.n_split == 1 && !alias;
  f.rec = f.o; f.ldr = f.ldo;
  f.ml = FH_KVD * (mem ? f.n_split : room);
  void *ws = nullptr;
  int st;
  if (mem && !f.direct) {
    f.ldr = f.ml + 2 * FH_SPLITS + 2;
    if ((st = bn_alloc(&ws, (size_t)q->h * f.ldr * sizeof(float), s))) return st;
    f.rec = (float *)ws;
  }
  hipLaunchKernelGGL(fh_rows_kernel, dim3((unsigned)((int64_t)n_rt * f.n_split)), dim3(64 * FH_WAVES), 0, s, f);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess && !f.direct) {
    hipLaunchKernelGGL(fh_merge_kernel, dim3((unsigned)((q->h + 3) / 4)), dim3(256), 0, s, f);
    e = hipGetLastError();
  }
  st = e == hipSuccess ? BN_OK : hip_fail(e, __FILE__, __LINE__);
  if (!ws) return st;
  const int st2 = bn_free(ws, s);
  return st ? st : st2;
}

// A view the kernel can read with float4 loads: fp32, columns contiguous,
// every row on a 16-byte boundary.
bool vec4_rows(const bn_view *v) { return rows_aligned(v, 16); }

}  // namespace
}  // namespace bn

using namespace bn;

extern "C" int bn_fused_head_attention(const bn_view *q, const bn_view *k, const bn_view *v,
                                       const bn_view *o, int n_heads, int n_kv_heads,
                                       int head_dim, float scale, int causal, int seq_offset,
                                       void *stream) {
  const char *op = "Fused-head attention";
  const unsigned mask = 1u << BN_F32;
  int st;
  if ((st = check_view(q, op, "query", mask))) return st;
  if ((st = check_view(k, op, "key", mask))) return st;
  if ((st = check_view(v, op, "value", mask))) return st;
  if ((st = check_view(o, op, "output", mask))) return st;
  if (n_heads <= 0 || n_kv_heads <= 0 || head_dim <= 0 || n_heads % n_kv_heads != 0)
    return fail(BN_ERR_SHAPE, std::string(op) + ": n_heads must be a positive multiple of n_kv_heads");
  const int64_t hd = (int64_t)n_heads * head_dim, kvd = (int64_t)n_kv_heads * head_dim;
  if (q->w != hd || o->w != hd || o->h != q->h)
    return fail(BN_ERR_SHAPE, std::string(op) + ": query and output must be [seq_q, n_heads*head_dim]");
  if (k->w != kvd || v->w != kvd || v->h != k->h)
    return fail(BN_ERR_SHAPE, std::string(op) + ": key and value must be [seq_kv, n_kv_heads*head_dim]");
  if (head_dim % 4 != 0 || kvd % 16 != 0 || kvd > kMaxKvd)
    return fail(BN_ERR_UNSUPPORTED,
                std::string(op) + ": needs head_dim % 4 == 0, n_kv_heads*head_dim % 16 == 0 and <= " +
                    std::to_string(kMaxKvd) + " (got head_dim " + std::to_string(head_dim) +
                    ", n_kv_heads*head_dim " + std::to_string(kvd) + ")");
  if ((st = require_device(op, {q, k, v, o}))) return st;
  if (!vec4_rows(q) || !vec4_rows(k) || !vec4_rows(v) || !vec4_rows(o))
    return fail(BN_ERR_UNSUPPORTED,
                std::string(op) + ": views need contiguous columns and rows on 16-byte boundaries");
  if ((st = ensure_device())) return st;
  if (q->h == 0) return BN_OK;
  const bool alias = overlaps(o, q) || overlaps(o, k) || overlaps(o, v) || std::abs(o->stride_h) < hd;
  if (kvd == FH_KVD && (q->h >= kPoolRows || (k->h > kValuKeys && !alias)))
    return launch_rows(q, k, v, o, head_dim, n_heads / n_kv_heads, scale, causal, seq_offset,
                       as_stream(stream), alias);
  FusedHeadParams p;
  p.q = reinterpret_cast<const float *>(q->data) + q->offset;
  p.k = reinterpret_cast<const float *>(k->data) + k->offset;
  p.v = reinterpret_cast<const float *>(v->data) + v->offset;
  p.o = reinterpret_cast<float *>(o->data) + o->offset;
  p.ldq = q->stride_h;
  p.ldk = k->stride_h;
  p.ldv = v->stride_h;
  p.ldo = o->stride_h;
  p.sq = q->h;
  p.sk = k->h;
  p.n_heads = n_heads;
  p.head_dim = head_dim;
  p.kvd = (int)kvd;
  p.n_rep = n_heads / n_kv_heads;
  p.scale = scale;
  p.causal = causal ? 1 : 0;
  p.seq_offset = seq_offset;
  const dim3 grid((q->h + kRows - 1) / kRows);
  if (kvd == 256)
    hipLaunchKernelGGL((fused_head_attention_kernel<1, 16>), grid, dim3(256), 0, as_stream(stream), p);
  else if (kvd < 256)
    hipLaunchKernelGGL((fused_head_attention_kernel<1, 0>), grid, dim3(256), 0, as_stream(stream), p);
  else
    hipLaunchKernelGGL((fused_head_attention_kernel<2, 0>), grid, dim3(256), 0, as_stream(stream), p);
  BN_LAUNCH_CHECK();
  return BN_OK;
}
