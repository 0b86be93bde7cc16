// bn_decode.hip -- KV-cache decode attention: one new query token per
// sequence against a contiguous per-sequence cache, split-K over the cache.
//
// The reference has no KV cache: generate() re-runs the whole prefix
// (llama_model.py:135-141) and the new token is the last row of the causal
// softmax with seq_offset = L-1 (op_softmax.cuh:89-99).  This kernel computes
// exactly that row for every query head h against KV head
// g = h / (n_heads/n_kv_heads) (llama_layers.hpp:159-163).
//
// Decode is HBM-bound (each cached K/V byte is used by G query heads and
// nothing else), so the design goal is one coalesced pass over the cache:
//   * one workgroup = (sequence b, KV head g, chunk of CH keys); its 4 waves
//     split the chunk; all G query heads of the group are served by the same
//     loads, so every cached byte is read once;
//   * a wave reads 8 (bf16) or 4 (fp32) whole 128/256-byte key rows per
//     16-byte-per-lane load instruction: LPK lanes own one key, each lane 16
//     bytes of it; the q.k partial dot products are reduced across the LPK
//     lanes with xor shuffles;
//   * every lane group keeps its own running (max, sum, acc) per head, updated
//     once per tile of NT keys, and the groups, waves and chunks are merged
//     with the log-sum-exp rule: in-wave by shuffles, in-workgroup through LDS,
//     across chunks over (m, l, acc) partials, by a small combine kernel (fp32)
//     or by a cache's last split to finish (bf16).
// Scores live in the log2 domain: s = (q.k) * scale*log2(e), p = exp2(s - m).

#include <algorithm>
#include <atomic>
#include <cstdlib>
#include <mutex>
#include <vector>

#include "bn_common.hpp"

// Chunk partials of bn_gqa_decode_noalloc: a file-scope device array, one
// copy per GPU, held until the process ends.  Host code never passes its name
// to a kernel (on the host the name is only a stand-in); it uses the device
// address hipGetSymbolAddress returns for the current device.
static __device__ __align__(256) float scratch[BN_GQA_DECODE_SCRATCH_BYTES / sizeof(float)];

// Per-(sequence, query head) split counters of the short-cache decode's
// in-launch merge: slots of kShortMaxUnits counters, zero at load time, a
// host-side ring of slots; each unit's last split clears its counter.
static __device__ __align__(256) uint32_t short_counters[16 * 256];

// bf16 K/V cache loads are non-temporal (streamed once, kept out of L2/MALL):
// +24% on config 3 against plain loads.

namespace bn {
namespace {

constexpr int HD = 64;
constexpr int NT = 8;  // keys per lane group between softmax rescales
// short-cache split (DEC_SHORT): keys per lane group per round (one round
// covers a 640-key cache's 160-key splits: 4 waves x 4 lane groups x 10),
// waves per workgroup and query heads per workgroup
constexpr int kShortNT = 10, kShortWV = 4, kShortG = 1;

template <typename T> struct DecVec;
template <> struct DecVec<float> {
  static constexpr int VEC = 4;
  __device__ static __forceinline__ void load(const float *p, float (&v)[4]) {
    const float4 t = *reinterpret_cast<const float4 *>(p);
    v[0] = t.x; v[1] = t.y; v[2] = t.z; v[3] = t.w;
  }
};

// Sum over each group of N (8 or 16) consecutive lanes with DPP moves inside
// a 16-lane row (no LDS round trip): quad xor 1, quad xor 2, half-row mirror
// (lane i <-> 7 - i), row mirror (lane i <-> 15 - i); every lane gets the sum.
template <int CTRL>
__device__ __forceinline__ float dpp_mov(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL,
                                                               0xf, 0xf, false));
}
template <int N>
__device__ __forceinline__ float row_sum(float x) {
  static_assert(N == 8 || N == 16, "8 or 16 lanes");
  x += dpp_mov<0xB1>(x);   // quad_perm 1,0,3,2
  x += dpp_mov<0x4E>(x);   // quad_perm 2,3,0,1
  x += dpp_mov<0x141>(x);  // row_half_mirror
  if (N == 16) x += dpp_mov<0x140>(x);  // row_mirror
  return x;
}

// Largest of the wave's values (not negative), uniform, without an LDS round
// trip: DPP moves inside each 16-lane row, then the rows' by readlane.
template <int CTRL>
__device__ __forceinline__ int dpp_max(int v) {
  return max(v, __builtin_amdgcn_update_dpp(0, v, CTRL, 0xf, 0xf, false));
}
__device__ __forceinline__ int wave_max_i32(int v) {
  v = dpp_max<0x140>(dpp_max<0x141>(dpp_max<0x4E>(dpp_max<0xB1>(v))));
  return max(max(__builtin_amdgcn_readlane(v, 0), __builtin_amdgcn_readlane(v, 16)),
             max(__builtin_amdgcn_readlane(v, 32), __builtin_amdgcn_readlane(v, 48)));
}

struct DecodeParams {
  const void *q, *k, *v;
  const int32_t *lens;
  void *o;
  float *ws;  // partials: [batch*n_heads][n_split][HD + 2]
  int batch, max_len, n_heads, n_kv_heads, n_split, chunk;
  int min_split = 1;  // pieces of a cache at least (n_split: at most)
  int groups = 0;     // dealt batches: workgroups per KV head (0: pieces per cache)
  float c;        // scale * log2(e)
  int hlen = -1;  // >= 0: every sequence's length, from the host (lens not read)
  // cache strides in elements: sequence, KV head, key row (a contiguous
  // [batch, max_len, n_kv_heads, 64] cache: max_len*n_kv_heads*64, 64,
  // n_kv_heads*64; a head-major [batch, n_kv_heads, max_len, 64] one:
  // n_kv_heads*max_len*64, max_len*64, 64)
  int64_t kv_bs = 0, kv_hs = 0, kv_rs = 0;
  // DEC_SHORT: per-(sequence, query head) counters (zero at launch, cleared
  // again by each unit's last split): the last split to arrive merges the
  // unit's records and writes the output in the same launch; null: the
  // records are left for a combine
  uint32_t *cnt = nullptr;
  // split whole-cache kernel: two arrival words per (sequence, KV head) below
  // arrive_end (any contents before the launch), and the launch's 48-bit tag
  unsigned long long *arrive_end = nullptr;
  unsigned long long tag = 0;
};

// WV waves per workgroup; MODE:
//   DEC_SPLIT: one workgroup per (sequence, KV head, chunk of p.chunk keys)
//     serving the KV head's G query heads; the waves interleave blocks of
//     KPI*NT keys over the chunk; writes the chunk's partial records.
//   DEC_SHORT: one workgroup per (sequence, G query heads of one KV head,
//     split); split s takes keys [s*chunk, (s+1)*chunk) of the sequence's
//     length with chunk = short_split_chunk(len, n_split), each wave a
//     contiguous part; writes the split's partial records.  For short caches
//     and few sequences, where one workgroup per query head is bound by what
//     one compute unit can stream (every workgroup reads the whole cache).
// The workgroups that read the same cache rows (the query heads of one KV
// head, in SHORT) get consecutive unit numbers, and units are
// numbered so that consecutive ones go to one XCD (workgroups are dealt to
// the 8 XCDs in turn): they read those rows from one L2.
constexpr int DEC_SPLIT = 0, DEC_SHORT = 1;
template <typename T, int G, int WV, int MODE>
__global__ __launch_bounds__(64 * WV) void decode_split_kernel(DecodeParams p) {
  constexpr bool CONTIG = MODE == DEC_SHORT;
  constexpr int VEC = DecVec<T>::VEC;
  constexpr int NT = CONTIG ? kShortNT : bn::NT;
  constexpr int LPK = HD / VEC;  // lanes per key
  constexpr int KPI = 64 / LPK;  // keys per wave per load instruction
  __shared__ float red_m[WV][G], red_l[WV][G];
  __shared__ float red_o[WV][G][HD];

  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int sub = lane % LPK;  // 16-byte slice of the key row
  const int grp = lane / LPK;  // key slot within the wave
  int u = blockIdx.x;
  if (CONTIG && (gridDim.x & 7) == 0) u = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  int b, g, h0, split = 0;
  if constexpr (MODE == DEC_SPLIT) {
    split = u % p.n_split;
    const int bg = u / p.n_split;
    b = bg / p.n_kv_heads;
    g = bg % p.n_kv_heads;
    h0 = g * G;
  } else {  // units (sequence, KV head, split, query-head group), the last fastest
    const int qpg = p.n_heads / p.n_kv_heads / G;  // query-head groups per KV head
    const int qg = u % qpg;
    u /= qpg;
    split = u % p.n_split;
    u /= p.n_split;
    g = u % p.n_kv_heads;
    b = u / p.n_kv_heads;
    h0 = g * (p.n_heads / p.n_kv_heads) + qg * G;
  }

  // this lane's slice of the G query vectors, pre-scaled into the log2
  // domain; requested before the length (its loads do not wait for it)
  float qv[G][VEC];
#pragma unroll
  for (int h = 0; h < G; ++h) {
    const T *qp = (const T *)p.q + ((int64_t)b * p.n_heads + h0 + h) * HD + sub * VEC;
    DecVec<T>::load(qp, qv[h]);
  }
  int len = p.hlen >= 0 ? p.hlen : p.lens[b];
  len = len < 0 ? 0 : (len > p.max_len ? p.max_len : len);
  const int chunk = MODE == DEC_SHORT ? short_split_chunk(len, p.n_split) : p.chunk;
  const int k_begin = split * chunk;
  if (k_begin >= len) {  // the combine ignores chunks past len
    if (MODE == DEC_SHORT && p.cnt && len == 0 && split == 0)  // no key, no merge: zeros
      for (int idx = tid; idx < G * HD; idx += 64 * WV)
        Elem<T>::store((T *)p.o + ((int64_t)b * p.n_heads + h0) * HD + idx, 0.f);
    return;
  }
  const int k_end = min(k_begin + chunk, len);
  // CONTIG: wave w takes keys [kw0, kw1), a contiguous range; else the waves
  // interleave blocks of KPI*NT keys over the chunk
  const int per = ((k_end - k_begin + WV - 1) / WV + KPI - 1) / KPI * KPI;
  const int kw0 = CONTIG ? k_begin + wave * per : k_begin + wave * KPI * NT;
  const int kw1 = CONTIG ? min(kw0 + per, k_end) : k_end;

  const int64_t kv_rs = p.kv_rs;
  const T *Kb = (const T *)p.k + b * p.kv_bs + g * p.kv_hs + sub * VEC;
  const T *Vb = (const T *)p.v + b * p.kv_bs + g * p.kv_hs + sub * VEC;

#pragma unroll
  for (int h = 0; h < G; ++h)
#pragma unroll
    for (int e = 0; e < VEC; ++e) qv[h][e] *= p.c;

  float m[G], l[G], acc[G][VEC];
#pragma unroll
  for (int h = 0; h < G; ++h) {
    m[h] = -INFINITY;
    l[h] = 0.f;
#pragma unroll
    for (int e = 0; e < VEC; ++e) acc[h][e] = 0.f;
  }

  const int step = CONTIG ? KPI * NT : WV * KPI * NT;
  for (int base = kw0; base < kw1; base += step) {
    // K and V of the NT keys of this lane group are requested together (one
    // memory round trip per NT keys); keys past the chunk read the chunk's
    // last row (initialised data, finite) and are masked to P = 0
    float s[G][NT];
    float kk[NT][VEC], vv[NT][VEC];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int key = min(base + t * KPI + grp, kw1 - 1);
      DecVec<T>::load(Kb + (int64_t)key * kv_rs, kk[t]);
      DecVec<T>::load(Vb + (int64_t)key * kv_rs, vv[t]);
    }
    // contiguous ranges: every load of the round is issued before any is
    // consumed.  Left alone, the scheduler trades them for registers (load,
    // wait, use, next: one round trip per key).
    if constexpr (CONTIG) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int key = base + t * KPI + grp;
#pragma unroll
      for (int h = 0; h < G; ++h) {
        float d = 0.f;
#pragma unroll
        for (int e = 0; e < VEC; ++e) d = fmaf(qv[h][e], kk[t][e], d);
        d = row_sum<LPK>(d);
        s[h][t] = key < kw1 ? d : -INFINITY;
      }
    }
#pragma unroll
    for (int h = 0; h < G; ++h) {
      float mx = s[h][0];
#pragma unroll
      for (int t = 1; t < NT; ++t) mx = fmaxf(mx, s[h][t]);
      const float m_new = fmaxf(m[h], mx);
      const float m_use = m_new == -INFINITY ? 0.f : m_new;
      const float alpha = __builtin_amdgcn_exp2f(m[h] - m_use);
      m[h] = m_new;
      float pt[NT], ps = 0.f;
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        pt[t] = __builtin_amdgcn_exp2f(s[h][t] - m_use);
        ps += pt[t];
      }
      l[h] = l[h] * alpha + ps;
#pragma unroll
      for (int e = 0; e < VEC; ++e) {
        float a = acc[h][e] * alpha;
#pragma unroll
        for (int t = 0; t < NT; ++t) a = fmaf(pt[t], vv[t][e], a);
        acc[h][e] = a;
      }
    }
  }

  // merge the KPI lane groups of this wave (lanes differing in bits >= log2(LPK))
#pragma unroll
  for (int h = 0; h < G; ++h) {
    float mw = m[h];
#pragma unroll
    for (int msk = LPK; msk < 64; msk <<= 1) mw = fmaxf(mw, __shfl_xor(mw, msk, 64));
    const float mu = mw == -INFINITY ? 0.f : mw;
    const float f = __builtin_amdgcn_exp2f(m[h] - mu);
    float lw = l[h] * f;
#pragma unroll
    for (int msk = LPK; msk < 64; msk <<= 1) lw += __shfl_xor(lw, msk, 64);
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
      float a = acc[h][e] * f;
#pragma unroll
      for (int msk = LPK; msk < 64; msk <<= 1) a += __shfl_xor(a, msk, 64);
      acc[h][e] = a;
    }
    if (lane == 0) {
      red_m[wave][h] = mw;
      red_l[wave][h] = lw;
    }
    if (grp == 0) {
#pragma unroll
      for (int e = 0; e < VEC; ++e) red_o[wave][h][sub * VEC + e] = acc[h][e];
    }
  }
  __syncthreads();

  // merge the waves and write this chunk's partial (m, l, acc[HD]) per head
  for (int idx = tid; idx < G * HD; idx += 64 * WV) {
    const int h = idx / HD, d = idx % HD;
    float M = red_m[0][h];
#pragma unroll
    for (int w2 = 1; w2 < WV; ++w2) M = fmaxf(M, red_m[w2][h]);
    const float Mu = M == -INFINITY ? 0.f : M;
    float L = 0.f, A = 0.f;
#pragma unroll
    for (int w2 = 0; w2 < WV; ++w2) {
      const float f = __builtin_amdgcn_exp2f(red_m[w2][h] - Mu);
      L += red_l[w2][h] * f;
      A += red_o[w2][h][d] * f;
    }
    float *part = p.ws + (((int64_t)b * p.n_heads + h0 + h) * p.n_split + split) * kDecRec;
    if (MODE == DEC_SHORT && p.cnt) {  // through to memory: another workgroup merges them
      __hip_atomic_store(part + 2 + d, A, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      if (d == 0) {
        __hip_atomic_store(part, M, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        __hip_atomic_store(part + 1, L, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      }
      continue;
    }
    part[2 + d] = A;
    if (d == 0) {
      part[0] = M;
      part[1] = L;
    }
  }
  if constexpr (MODE == DEC_SHORT) {
    if (!p.cnt) return;
    // the unit's splits holding keys count themselves; the last to arrive
    // reads their records past the caches and merges them as the combine
    // kernel does (DecMerge), so the output has the combine's bits
    __shared__ bool s_last;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this thread's record stores done
    __syncthreads();
    if (tid == 0) {
      const int unit = (b * p.n_heads + h0) / G;
      const uint32_t nvalid = (uint32_t)((len + chunk - 1) / chunk);
      const uint32_t seen = __hip_atomic_fetch_add(p.cnt + unit, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const bool last = seen == nvalid - 1;
      if (last) __hip_atomic_store(p.cnt + unit, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      s_last = last;
    }
    __syncthreads();
    if (!s_last) return;
    const int nvalid = (len + chunk - 1) / chunk;
    for (int idx = tid; idx < G * HD / 4; idx += 64 * WV) {
      const int h = idx / (HD / 4), d0 = (idx % (HD / 4)) * 4;
      const float *part = p.ws + ((int64_t)b * p.n_heads + h0 + h) * p.n_split * kDecRec;
      DecMerge mg;
      mg.load8<true>(part, p.n_split, 0, d0);
      mg.start();
      mg.merge8(0, nvalid);
      for (int s0 = 8; s0 < nvalid; s0 += 8) {
        mg.load8<true>(part, p.n_split, s0, d0);
        mg.merge8(s0, nvalid);
      }
      const float4 r = mg.result();
      T *out = (T *)p.o + ((int64_t)b * p.n_heads + h0 + h) * HD + d0;
      Elem<T>::store(out + 0, r.x);
      Elem<T>::store(out + 1, r.y);
      Elem<T>::store(out + 2, r.z);
      Elem<T>::store(out + 3, r.w);
    }
  }
}

// bf16 caches run on the matrix cores.  Per wave, tiles of 32 keys:
//   S^T[key][head] = K[key][:] . Q[head][:]   two v_mfma_f32_16x16x32_bf16 per
//     16 keys; the K tile is the A operand (lane: key l%16, 16 bytes of d), the
//     G query heads are the B operand columns (padded to 16);
//   online softmax per head column (4 keys per lane, 4 lane groups);
//   O^T[d][head] += V^T[d][key] . P^T[key][head]  one MFMA per 16 d; V^T by
//     transposed LDS reads, P^T straight from registers.
typedef __bf16 dbf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 dbf16x4_t __attribute__((ext_vector_type(4)));
typedef float df32x4_t __attribute__((ext_vector_type(4)));
constexpr int TK = 32;   // keys per wave tile
typedef short ds4_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ dbf16x4_t lds_read_tr16(const bf16_t *p) {
  const ds4_t r = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) ds4_t *)(__attribute__((address_space(3))) void *)p);
  return __builtin_bit_cast(dbf16x4_t, r);
}

// bf16 cache, one workgroup per (sequence, KV head) over the whole cache:
// no partials in memory and no combine launch.  Chosen when there are at
// least as many (sequence, KV head) pairs as compute units, so every CU has a
// workgroup.  Wave w of the WWV takes the 32-key tiles w, w + WWV, ... and
// streams them through a private LDS tile (no workgroup barrier in the loop):
// 16-byte loads of the head's 128-byte cache rows, 8 rows per instruction,
// the next tile register-staged; the scores and P V on
// v_mfma_f32_16x16x32_bf16 as above.  The waves'
// (m, l, acc) are merged through LDS at the end and the workgroup writes the
// G output rows.  Four waves stream a cache (8 measured 8% slower on config
// 3, 2 3% slower).  When a KV head's rows are contiguous (row stride
// head_dim: a head-major cache) the workgroup has WWX waves and a cache more
// than 1.25x the batch's mean length uses all of them (once the other caches
// are done, one CU streams a long cache faster with more waves: config 3's
// ragged draw -4%, a few long caches among short ones -12%; uniform lengths
// keep four); token-major caches stream slower with more waves and keep four.
constexpr int WWV = 4;  // streaming waves per workgroup
constexpr int WWX = 6;  // waves of an adaptive whole-cache workgroup, active for a long cache
constexpr int WW1 = 8;  // waves of the split kernel's unsplit pairs
constexpr int kMeanBatchMax = 512;  // longer batches: four waves for every cache
constexpr int WKP = HD + 8;  // tile row pitch, 144 B: b128 K reads of 16 rows and tr16 V
                             // reads of 4 rows x 32 B hit distinct banks

// a cache up to this length is one split's (500 keys: 5.8 us, in 2-8 splits 6.9)
constexpr int kSplitMinLen = 512;
// how caches are dealt to workgroups: whole, each in up to n_split equal pieces,
// in pieces by its own length, or the batch in equal shares
constexpr int kWhole = 0, kSplit = 1, kByLength = 2, kDealt = 3;
constexpr int kPieceMinLen = 1024;  // keys of each piece of a cache in more than min_split
constexpr int kShareMin = 8;        // tiles of a share at least
constexpr int kUneven = 40;         // tiles over a share that the longest cache's piece may have
constexpr unsigned long long kArrive = 0x5bd1e995a93c71d4ull;
// keys per split of a cache: whole rounds of the workgroup's four tiles
template <int NW>
__device__ __forceinline__ int split_chunk(int len, int n_split) {
  if (len <= kSplitMinLen) return max(len, 1);
  const int c = (len + n_split - 1) / n_split;
  return max((c + NW * TK - 1) / (NW * TK), 1) * (NW * TK);
}

// NW waves per workgroup: WWV, or WWX with the long-cache adaptation.
// SPLIT (fewer (sequence, KV head) pairs than compute units): a cache in pieces,
// so that a few caches have most of their loads in flight at once; bound by
// latencies (launch, one or two memory round trips, the merge).  kSplit, kByLength:
// up to n_split workgroups per pair, each over a run of the cache.  kDealt: the
// sequences' tiles in a row, an equal share of it per workgroup, which takes the
// caches in it one after another, so that long and uneven batches end together
// (dealt_groups).  A split writes its merged (m, l,
// acc) record through to memory, waits for it, and counts itself in on the
// pair's arrival word; the last one to arrive merges the records and writes
// the output, in the same launch.  Measured (graph replay, B=1 / 4 KV heads, G
// 8) against the former chunk kernel over 4 KV heads' whole rows with its
// combine launch: one cache of 1543 keys 9.9 -> 7.0 us, of 200 8.5 -> 4.5, of
// 8000 18.0 -> 11.0; 12 caches of 200..4000 keys 16.9 -> 11.2, 32 of 500..2000
// 17.5 -> 13.0, 48 of 500..4000 34.4 -> 25.2.
// The arrival words stand at the workspace's end.  The first holds kArrive
// between calls and counts up from it: one atomic.  Anything else there (a
// fresh workspace) sends every split of the launch to the second word, where a
// count starts under the launch's tag: a load, for the first splits a
// compare-exchange, and an add (words overwritten before every call, whose
// fill is in the time: one cache of 1530 keys 10.2 us, 14066 keys 18.6, four of
// 4203..7439 16.4; with a compare-exchange per arrival, which all retry while
// others arrive, 11.6, 20.1 and 18.2; the former chunk kernel 11.5, 22.7 and
// 18.0).  A finished count clears the second word, and the last
// arrival leaves kArrive, so neither a fresh workspace nor a replayed graph
// needs a clearing pass.
template <int G, int NW, int DEAL>
__global__ __launch_bounds__(64 * NW) void decode_bf16_whole_kernel(DecodeParams p) {
  constexpr bool SPLIT = DEAL != kWhole;
  __shared__ __attribute__((aligned(16))) bf16_t KT[NW][TK * WKP];
  __shared__ __attribute__((aligned(16))) bf16_t VT[NW][TK * WKP];
  __shared__ float red_m[NW][G], red_l[NW][G];
  __shared__ float red_o[NW][G][HD];
  __shared__ int last_split;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, grp = lane >> 4;
  // the KV heads of a sequence's (split's) rows next to each other
  const int g = blockIdx.x % p.n_kv_heads, bs = blockIdx.x / p.n_kv_heads;
  auto clamp_len = [&](int x) { return x < 0 ? 0 : (x > p.max_len ? p.max_len : x); };

  // One piece: keys [k0, kw1) of sequence b, by nw waves; piece q of the
  // pieces() that hold the cache's keys (a division, left until the loads are
  // through).  bin0: the group of a dealt cache's first piece.
  auto run = [&](const int b, const int k0, const int kw1, const int nw, auto pieces, const int q,
                 const int bin0) __attribute__((always_inline)) {
    bf16_t *const out = (bf16_t *)p.o + ((int64_t)b * p.n_heads + (int64_t)g * G) * HD;
    // wave w < nw takes the 32-key tiles w, w + nw, w + 2*nw, ...: the waves of
    // a workgroup stream adjacent tiles (a contiguous key range per wave, or the
    // KV heads of one sequence placed on one XCD, measured 3-4% slower)
    const int all_tiles = (kw1 - k0 + TK - 1) / TK;
    const int kw0 = k0 + TK * wave;
    const int tstride = TK * nw;  // keys between a wave's tiles
    const int ntiles = wave < nw && all_tiles > wave ? (all_tiles - wave + nw - 1) / nw : 0;

    const int64_t kv_rs = p.kv_rs;
    const bf16_t *Kr = (const bf16_t *)p.k + b * p.kv_bs + g * p.kv_hs;
    const bf16_t *Vr = (const bf16_t *)p.v + b * p.kv_bs + g * p.kv_hs;

    dbf16x8_t qb[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      if (l16 < G)
        qb[t] = *(const dbf16x8_t *)((const bf16_t *)p.q +
                                     ((int64_t)b * p.n_heads + g * G + l16) * HD + 8 * grp + 32 * t);
      else
        qb[t] = dbf16x8_t{};
    }

    // lane's 16-byte chunks of a tile: rows crow + 8i (i = 0..3), columns ccol..ccol+7
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    struct RegTile {
      u32x4 k0, k1, k2, k3, v0, v1, v2, v3;
    };
    const int crow = lane >> 3, ccol = (lane & 7) * 8;
    auto gload = [&](RegTile &r, int ti) __attribute__((always_inline)) {
      const int kb = kw0 + tstride * min(ti, ntiles - 1);  // clamped: same load count on every path
      const int last = min(kb + TK, kw1) - 1;  // past the end: a valid row, masked to P = 0
      const int64_t o0 = (int64_t)min(kb + crow, last) * kv_rs + ccol;
      const int64_t o1 = (int64_t)min(kb + crow + 8, last) * kv_rs + ccol;
      const int64_t o2 = (int64_t)min(kb + crow + 16, last) * kv_rs + ccol;
      const int64_t o3 = (int64_t)min(kb + crow + 24, last) * kv_rs + ccol;
      // streamed once: non-temporal loads
      r.k0 = __builtin_nontemporal_load((const u32x4 *)(Kr + o0)); r.v0 = __builtin_nontemporal_load((const u32x4 *)(Vr + o0));
      r.k1 = __builtin_nontemporal_load((const u32x4 *)(Kr + o1)); r.v1 = __builtin_nontemporal_load((const u32x4 *)(Vr + o1));
      r.k2 = __builtin_nontemporal_load((const u32x4 *)(Kr + o2)); r.v2 = __builtin_nontemporal_load((const u32x4 *)(Vr + o2));
      r.k3 = __builtin_nontemporal_load((const u32x4 *)(Kr + o3)); r.v3 = __builtin_nontemporal_load((const u32x4 *)(Vr + o3));
    };
    bf16_t *const kt = KT[wave], *const vt = VT[wave];
    auto lstore = [&](const RegTile &r) __attribute__((always_inline)) {
      *(u32x4 *)(kt + crow * WKP + ccol) = r.k0;
      *(u32x4 *)(kt + (crow + 8) * WKP + ccol) = r.k1;
      *(u32x4 *)(kt + (crow + 16) * WKP + ccol) = r.k2;
      *(u32x4 *)(kt + (crow + 24) * WKP + ccol) = r.k3;
      *(u32x4 *)(vt + crow * WKP + ccol) = r.v0;
      *(u32x4 *)(vt + (crow + 8) * WKP + ccol) = r.v1;
      *(u32x4 *)(vt + (crow + 16) * WKP + ccol) = r.v2;
      *(u32x4 *)(vt + (crow + 24) * WKP + ccol) = r.v3;
    };

    float m = -INFINITY, l = 0.f;
    df32x4_t o[4] = {df32x4_t{}, df32x4_t{}, df32x4_t{}, df32x4_t{}};
    const float c = p.c;
    // one 32-key tile from this wave's LDS tile; keys kb .. kb + 31
    auto compute = [&](int kb) __attribute__((always_inline)) {
      const bf16_t *kl = kt + 8 * grp;
      df32x4_t s[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const bf16_t *kp = kl + (16 * u + l16) * WKP;
        s[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const dbf16x8_t *)(kp), qb[0], df32x4_t{},
                                                       0, 0, 0);
        s[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const dbf16x8_t *)(kp + 32), qb[1], s[u],
                                                       0, 0, 0);
      }
      // s[u][i] = score of key kb + 16u + 4grp + i for query head g*G + l16
      if (kb + TK > kw1) {
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (kb + 16 * u + 4 * grp + i >= kw1) s[u][i] = -INFINITY;
      }
      float mx = fmaxf(fmaxf(fmaxf(s[0][0], s[0][1]), fmaxf(s[0][2], s[0][3])),
                       fmaxf(fmaxf(s[1][0], s[1][1]), fmaxf(s[1][2], s[1][3])));
      mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
      mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
      const float m_new = fmaxf(m, mx);  // -inf while every key so far scores -inf
      const float mc = (m_new == -INFINITY ? 0.f : m_new) * c;
      const float alpha = __builtin_amdgcn_exp2f(m * c - mc);  // m = -inf -> 0
      float rs = 0.f;
      dbf16x8_t pb;
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float e = __builtin_amdgcn_exp2f(fmaf(s[u][i], c, -mc));
          rs += e;
          pb[4 * u + i] = (__bf16)e;  // k-slot (grp, 4u+i) = key 16u + 4grp + i
        }
      l = l * alpha + rs;
      m = m_new;
      // V^T operand: slot j of lane (grp, l16) = V[key 16(j/4) + 4grp + j%4][16dt + l16];
      // transpose read: local lane n supplies V[key 4grp + n/4 (+16)][16dt + 4(n%4) .. +3]
      const bf16_t *vp = vt + (4 * grp + (l16 >> 2)) * WKP + 4 * (l16 & 3);
#pragma unroll
      for (int dt = 0; dt < 4; ++dt) {
        o[dt] *= alpha;
        const dbf16x4_t lo = lds_read_tr16(vp + 16 * dt);
        const dbf16x4_t hi = lds_read_tr16(vp + 16 * WKP + 16 * dt);
        const dbf16x8_t a = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, pb, o[dt], 0, 0, 0);
      }
    };

    // The wave's tile ti goes through one register tile (loaded one tile ahead)
    // and the wave's LDS tile.  LDS instructions of one wave execute in order,
    // so a tile's writes follow the previous tile's reads (already consumed) and
    // precede its own reads with no barrier; wave_barrier keeps the compiler
    // from moving LDS accesses across.  One tile in flight per wave (4 KB of K
    // and of V; 32 KB per CU at 4 waves) streams best: two tiles ahead measured
    // 8% slower on config 3, more waves per workgroup slower still.
    if (ntiles > 0) {  // wave-uniform
      RegTile ta;
      gload(ta, 0);
      lstore(ta);
      gload(ta, 1);
      __builtin_amdgcn_wave_barrier();
      for (int ti = 0; ti < ntiles; ++ti) {
        compute(kw0 + tstride * ti);
        if (ti + 1 < ntiles) {
          __builtin_amdgcn_wave_barrier();
          lstore(ta);
          gload(ta, ti + 2);
          __builtin_amdgcn_wave_barrier();
        }
      }
    }

    // merge the waves: o[dt][i] = O^T[d = 16dt + 4grp + i][head g*G + l16]
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    if (l16 < G) {
#pragma unroll
      for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int i = 0; i < 4; ++i) red_o[wave][l16][16 * dt + 4 * grp + i] = o[dt][i];
      if (grp == 0) {
        red_m[wave][l16] = m * c;  // -inf for a wave without keys
        red_l[wave][l16] = l;
      }
    }
    __syncthreads();
    const int nvalid = pieces();
    __builtin_assume(nvalid >= 1);
    // query head h's record of piece n: of a dealt cache in its workgroup's second
    // place for the cache's first piece (the workgroup's last), else in its first
    auto rec_of = [&](int h, int n) __attribute__((always_inline)) {
      if (DEAL == kDealt) return p.ws + ((int64_t)((2 * (bin0 + n) + (n == 0)) * p.n_kv_heads + g) * G + h) * kDecRec;
      return p.ws + (((int64_t)b * p.n_heads + (int64_t)g * G + h) * p.n_split + n) * kDecRec;
    };
    for (int idx = tid; idx < G * HD; idx += 64 * NW) {
      const int h = idx / HD, d = idx - h * HD;
      float M = red_m[0][h];
#pragma unroll
      for (int w = 1; w < NW; ++w) M = fmaxf(M, red_m[w][h]);
      const float Mu = M == -INFINITY ? 0.f : M;  // no key above -inf: every weight 0
      float L = 0.f, A = 0.f;
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        const float wt = __builtin_amdgcn_exp2f(red_m[w][h] - Mu);
        L += red_l[w][h] * wt;
        A += red_o[w][h][d] * wt;
      }
      if (!SPLIT || nvalid == 1) {
        out[idx] = f32_to_bf16(L == 0.f ? 0.f : A / L);
      } else {
        float *rec = rec_of(h, q);
        auto wr = [](float *q, float v) { __hip_atomic_store(q, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM); };
        wr(rec + 2 + d, A);
        if (d == 0) {
          wr(rec, M);
          wr(rec + 1, L);
        }
      }
    }
    if constexpr (SPLIT) {
      if (nvalid == 1) return;
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the record's stores have reached memory
      __syncthreads();
      if (tid == 0) {
        unsigned long long *word = p.arrive_end - 2 * ((int64_t)b * p.n_kv_heads + g + 1);
        unsigned long long old = __hip_atomic_fetch_add(word, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        bool last = old - kArrive == (unsigned long long)(nvalid - 1);
        if (old - kArrive >= (unsigned long long)nvalid) {
          // one split puts the tag there, then every split adds
          old = __hip_atomic_load(word + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          while (old >> 16 != p.tag &&
                 !__hip_atomic_compare_exchange_strong(word + 1, &old, p.tag << 16, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                       __HIP_MEMORY_SCOPE_AGENT)) {
          }
          const unsigned long long next =
              __hip_atomic_fetch_add(word + 1, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1;
          last = (int)(next & 0xffff) == nvalid;
          // a replay has the same tag: nothing of this count may be left for one
          // that finds only the first word overwritten
          if (last) __hip_atomic_store(word + 1, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        if (last) __hip_atomic_store(word, kArrive, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        last_split = last;
      }
      __syncthreads();
      if (!last_split) return;
      for (int idx = tid; idx < G * (HD / 4); idx += 64 * NW) {
        const int h = idx / (HD / 4), d0 = 4 * (idx % (HD / 4));
        DecMerge mg;
        mg.start();
        for (int s0 = 0; s0 < nvalid; s0 += 8) {
          if constexpr (DEAL == kDealt)
            mg.load8_from([&](int n) { return rec_of(h, n); }, nvalid, s0, d0);
          else
            mg.load8<true>(rec_of(h, 0), p.n_split, s0, d0);
          mg.merge8(s0, nvalid);
        }
        const float4 r = mg.result();
        const uint32_t lo = (uint32_t)f32_to_bf16(r.x) | ((uint32_t)f32_to_bf16(r.y) << 16);
        const uint32_t hi = (uint32_t)f32_to_bf16(r.z) | ((uint32_t)f32_to_bf16(r.w) << 16);
        bf16_t *const od = out + h * HD + d0;
        if (((uintptr_t)out & 7) == 0) {
          *(uint2 *)od = make_uint2(lo, hi);
        } else {  // (o is the caller's: any element may be its first)
          od[0] = (bf16_t)lo; od[1] = (bf16_t)(lo >> 16);
          od[2] = (bf16_t)hi; od[3] = (bf16_t)(hi >> 16);
        }
      }
    }
  };
  auto zeros = [&](int b) {  // a sequence without keys
    bf16_t *const out = (bf16_t *)p.o + ((int64_t)b * p.n_heads + (int64_t)g * G) * HD;
    for (int idx = tid; idx < G * HD; idx += 64 * NW) out[idx] = f32_to_bf16(0.f);
  };

  if constexpr (DEAL == kWhole) {
    // the batch's total length (batches up to kMeanBatchMax sequences), summed
    // by every wave itself (no barrier), read with this sequence's length
    const bool adapt = NW > WWV && p.batch <= kMeanBatchMax;
    int part = 0;
    if (adapt)
      for (int i = lane; i < p.batch; i += 64) part += clamp_len(p.lens[i]);
    const int len = clamp_len(p.lens[bs]);
    if (len == 0) return zeros(bs);
    int nw = WWV;  // streaming waves of this workgroup (uniform)
    if (adapt) {
#pragma unroll
      for (int o2 = 32; o2 > 0; o2 >>= 1) part += __shfl_xor(part, o2, 64);
      const int total = __builtin_amdgcn_readfirstlane(part);  // <= 512 * max_len
      if ((int64_t)len * p.batch * 4 > (int64_t)total * 5) nw = NW;
    }
    run(bs, 0, len, nw, [] { return 1; }, 0, 0);
  } else if constexpr (DEAL == kSplit || DEAL == kByLength) {
    const int b = bs / p.n_split, q = bs - b * p.n_split;
    const int len = clamp_len(p.lens[b]);
    // (in eights past min_split: records merge eight at a time)
    const int pieces =
        DEAL == kSplit ? p.n_split : min(max(len / kPieceMinLen & ~7, p.min_split), p.n_split);
    const int chunk = split_chunk<NW>(len, pieces), k0 = q * chunk;
    if (q > 0 && k0 >= len) return;
    if (len == 0) return zeros(b);
    run(b, k0, min(k0 + chunk, len), NW, [&] { return (int)((uint32_t)(len + chunk - 1) / (uint32_t)chunk); }, q, 0);
  } else {
    // every wave scans the batch's tiles for itself (lane: 4 sequences)
    int t[4], own = 0, most = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int n = 4 * lane + i < p.batch ? clamp_len(p.lens[4 * lane + i]) : 0;
      t[i] = (n >> 5) + ((n & 31) != 0);
      own += t[i];
      most = max(most, t[i]);
    }
    static_assert(TK == 32, "tiles of 32 keys");
    int upto = own;  // tiles of the sequences up to and with this lane's
#pragma unroll
    for (int o2 = 1; o2 < 64; o2 <<= 1) {
      const int x = __shfl_up(upto, o2, 64);
      upto += lane >= o2 ? x : 0;
    }
    const int total = __builtin_amdgcn_readlane(upto, 63);
    most = wave_max_i32(most);
    for (int b = bs; b < p.batch; b += p.groups)
      if (clamp_len(p.lens[b]) == 0) zeros(b);
    const int share = max((int)((uint32_t)total / (uint32_t)p.groups) + 1, kShareMin);
    // Equal pieces (min_split a cache) end with the longest cache's.  Where that
    // isn't far past a share, they take less time than shares over the ends of
    // caches and the merges that those need: with 0 / 32 / 48 / 80 in kUneven's
    // place, 86 batches of 65..128 pairs and 6000..9000 rows took 0.83 / 0.77 /
    // 0.78 / 0.85 of the former chunk kernel's time, 22 short caches (13..829 keys,
    // 8 KV heads) 14.8 / 9.5 / 9.5 / 9.5 us.
    if (most <= (share + max(share / 4, kUneven)) * (int64_t)p.min_split) {
      const int b = bs / p.min_split, q = bs - b * p.min_split;
      const int len = b < p.batch ? clamp_len(p.lens[b]) : 0;
      const int chunk = split_chunk<NW>(len, p.min_split), k0 = q * chunk;
      auto n = [&] { return (int)((uint32_t)(len + chunk - 1) / (uint32_t)chunk); };
      if (k0 < len) run(b, k0, min(k0 + chunk, len), NW, n, q, b * p.min_split);
      return;
    }
    const int end = min((bs + 1) * share, total);
    for (int pos = bs * share; pos < end;) {
      const int src = __builtin_ctzll(__builtin_amdgcn_ballot_w64(upto > pos));
      int b = 4 * src, first = __builtin_amdgcn_readlane(upto - own, src);  // b's first tile
      int tb = __builtin_amdgcn_readlane(t[0], src);
#pragma unroll
      for (int i = 1; i < 4; ++i) {
        const int ti = __builtin_amdgcn_readlane(t[i], src);
        if (pos >= first + tb) {
          first += tb;
          tb = ti;
          ++b;
        }
      }
      const int stop = min(first + tb, end), len = clamp_len(p.lens[b]);
      const int bin0 = (int)((uint32_t)first / (uint32_t)share);
      auto n = [&] { return (int)((uint32_t)(first + tb - 1) / (uint32_t)share) - bin0 + 1; };
      run(b, TK * (pos - first), min(TK * (stop - first), len), NW, n, bs - bin0, bin0);
      pos = stop;
      __syncthreads();  // the next piece's LDS writes follow this one's reads
    }
  }
}

// Planned ragged decode (bn_gqa_decode_planned): the lengths are known on
// the host, which deals the batch's 32-key tiles -- units (sequence, KV head)
// in order -- into equal contiguous shares, one per workgroup and compute
// unit, so that every compute unit streams the same number of bytes and a
// long cache is cut across neighbouring workgroups instead of one compute
// unit streaming it alone after the others have finished.  A workgroup's
// share touches a few units (segments); its waves take the share's tiles in
// turn (tile i -> wave i % 4, the loads running on across segment
// boundaries), keep one (m, l, acc) per segment, and merge them through LDS
// at the end.  A unit lying wholly in the share is written directly.  A cut
// unit's head (its first tiles: the LAST segment of the share where it
// starts) merges it; every later part is the FIRST segment of its share, so
// its waves finish it early and hand their states to a fifth wave of the
// workgroup (through LDS and a workgroup counter), which merges them and
// writes the part's (m, l, acc) record to memory while the four stream on
// (written through to memory, a store holds up the wave that issued it, so
// none of the streaming waves issues one) -- every 64-bit word holding a
// value and this launch's epoch, so a reader knows a word is this launch's
// without any ordering between words, counters or waits.  At the end the
// head loads the records (one round trip: they were written while the rest
// of the shares streamed), merges and writes the output.  A record not yet this launch's
// is polled again a bounded number of times; past that the head streams the
// unit's remaining keys itself (never needed when the launch's workgroups
// run side by side, which 256 of them on 256 compute units do), so no
// workgroup waits on another without limit.
constexpr int kPlanBins = 256;   // workgroups of a planned launch, at most
constexpr int kPlanUnits = 256;  // (sequence, KV head) units, at most
constexpr int kPlanSeg = 8;      // units one share may touch, at most
constexpr int kPlanPolls = 1 << 14;  // re-polls of a record before the head streams the keys itself
// a part's record, G query heads: acc[G][HD], then m[G] (log2 units), l[G]
// (64-bit words; the writer wave's store instructions cover 512 contiguous bytes)
template <int G> constexpr int rec_words() { return G * HD + 2 * G; }

struct PlanParams {
  const void *q, *k, *v;
  void *o;
  uint64_t *rec;  // part records [record][rec_words<G>()], epoch in bits 32..63 of each word
  int batch, max_len, n_heads, n_kv_heads, n_units, share, total;  // share: sequence tiles per group
  float c;                         // scale * log2(e)
  uint32_t epoch;                  // this launch's tag (never 0; a fresh workspace may hold anything)
  int max_polls;                   // kPlanPolls; -1: ignore records, the heads stream every key
  int64_t kv_bs, kv_hs, kv_rs;     // cache strides (elements): sequence, KV head, key row
  uint32_t wg_start[kPlanBins];    // group: first sequence (bits 0..15), its first tile (16..31)
  uint32_t unit[kPlanUnits];       // record base (0..11), first group (12..23), parts (24..31)
  int32_t len[kPlanUnits];         // per sequence: length, clamped to [0, max_len]
};

// WWV streaming waves and one record-writer wave per workgroup
constexpr int kPlanThreads = 64 * (WWV + 1);

template <int G>
__global__ __launch_bounds__(kPlanThreads) void decode_bf16_planned_kernel(PlanParams p) {
  __shared__ __attribute__((aligned(16))) bf16_t KT[WWV][TK * WKP];
  __shared__ __attribute__((aligned(16))) bf16_t VT[WWV][TK * WKP];
  __shared__ float red_m[kPlanSeg][WWV][G], red_l[kPlanSeg][WWV][G];
  __shared__ float red_o[kPlanSeg][WWV][G][HD];
  __shared__ uint32_t seg0_done;  // streaming waves that have handed over segment 0

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool streamer = wave < WWV;  // wave WWV writes segment 0's record
  const int l16 = lane & 15, grp = lane >> 4;
  const int bin = blockIdx.x, Hkv = p.n_kv_heads;
  // workgroups come in groups of Hkv, one per KV head, that walk the same
  // share of the batch's sequences together (consecutive ids: dispatched at
  // the same time), so the KV heads' slices of a cache row are read close in
  // time, as in the whole-cache kernel
  const int grp_id = bin / Hkv, gh = bin - grp_id * Hkv;
  const int64_t kv_rs = p.kv_rs;
  auto tiles_of = [&](int b) { return (p.len[b] + TK - 1) / TK; };

  // units with no key at all: zeros, each written by workgroup u % gridDim.x
  for (int u = bin; u < p.n_units; u += gridDim.x) {
    if (p.len[u / Hkv] == 0) {
      bf16_t *out = (bf16_t *)p.o + ((int64_t)(u / Hkv) * p.n_heads + (int64_t)(u % Hkv) * G) * HD;
      for (int idx = tid; idx < G * HD; idx += kPlanThreads) out[idx] = f32_to_bf16(0.f);
    }
  }
  if (tid == 0) seg0_done = 0;
  __syncthreads();
  // This group's share [grp_id * share, +ntile) of the batch's sequence
  // tiles, as segments (one sequence each, sequences with keys in order) of
  // this workgroup's KV head.  Every wave walks them itself in scalar
  // registers -- no table, no barrier before the first loads -- forward only,
  // since a wave's tiles increase.
  const int ntile = min(p.share, p.total - grp_id * p.share);
  struct Seg {
    int s, b, end, kb0, len;  // sequence b; keys of local tile i: kb0 + 32 * i
    const bf16_t *kr, *vr;
  };
  auto seg_set = [&](Seg &x, int b, int lb, int t) __attribute__((always_inline)) {
    const int g = gh;
    x.b = b;
    x.len = p.len[b];
    x.end = min(ntile, lb + (x.len + TK - 1) / TK - t);
    x.kb0 = TK * (t - lb);
    x.kr = (const bf16_t *)p.k + b * p.kv_bs + g * p.kv_hs;
    x.vr = (const bf16_t *)p.v + b * p.kv_bs + g * p.kv_hs;
  };
  auto seg_first = [&](Seg &x) __attribute__((always_inline)) {
    x.s = 0;
    seg_set(x, (int)(p.wg_start[grp_id] & 0xffffu), 0, (int)(p.wg_start[grp_id] >> 16));
  };
  auto seg_next = [&](Seg &x) __attribute__((always_inline)) {
    int b = x.b + 1;
    while (b + 1 < p.batch && tiles_of(b) == 0) ++b;  // sequences without keys hold no tile
    ++x.s;
    seg_set(x, b, x.end, 0);
  };
  auto seg_adv = [&](Seg &x, int i) __attribute__((always_inline)) {
    while (i >= x.end && x.end < ntile) seg_next(x);
  };
  int nseg = 0;
  if (ntile > 0) {
    Seg x;
    seg_first(x);
    while (x.end < ntile && x.s + 1 < kPlanSeg) seg_next(x);
    nseg = x.s + 1;
  }

  typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
  struct RegTile {
    u32x4 k0, k1, k2, k3, v0, v1, v2, v3;
  };
  const int crow = lane >> 3, ccol = (lane & 7) * 8;
  auto gload = [&](RegTile &r, int i, const Seg &x) __attribute__((always_inline)) {
    const int kb = x.kb0 + TK * i, kw1 = x.len;
    const bf16_t *Kr = x.kr, *Vr = x.vr;
    const int last = min(kb + TK, kw1) - 1;  // past the end: a valid row, masked to P = 0
    const int64_t o0 = (int64_t)min(kb + crow, last) * kv_rs + ccol;
    const int64_t o1 = (int64_t)min(kb + crow + 8, last) * kv_rs + ccol;
    const int64_t o2 = (int64_t)min(kb + crow + 16, last) * kv_rs + ccol;
    const int64_t o3 = (int64_t)min(kb + crow + 24, last) * kv_rs + ccol;
    r.k0 = __builtin_nontemporal_load((const u32x4 *)(Kr + o0)); r.v0 = __builtin_nontemporal_load((const u32x4 *)(Vr + o0));
    r.k1 = __builtin_nontemporal_load((const u32x4 *)(Kr + o1)); r.v1 = __builtin_nontemporal_load((const u32x4 *)(Vr + o1));
    r.k2 = __builtin_nontemporal_load((const u32x4 *)(Kr + o2)); r.v2 = __builtin_nontemporal_load((const u32x4 *)(Vr + o2));
    r.k3 = __builtin_nontemporal_load((const u32x4 *)(Kr + o3)); r.v3 = __builtin_nontemporal_load((const u32x4 *)(Vr + o3));
  };
  // the query rows of a segment's unit: lane (grp, l16) holds head l16's
  // d = 8grp .. +7 and 32 + 8grp .. +7 (the MFMA B operand)
  auto gload_q = [&](dbf16x8_t (&qv)[2], const Seg &x) __attribute__((always_inline)) {
    const int b = x.b, g = gh;
#pragma unroll
    for (int t = 0; t < 2; ++t)
      qv[t] = l16 < G ? *(const dbf16x8_t *)((const bf16_t *)p.q +
                                            ((int64_t)b * p.n_heads + g * G + l16) * HD + 8 * grp + 32 * t)
                      : dbf16x8_t{};
  };
  // the writer wave (wave WWV) has no tile of its own and never uses these
  bf16_t *const kt = KT[streamer ? wave : 0], *const vt = VT[streamer ? wave : 0];
  auto lstore = [&](const RegTile &r) __attribute__((always_inline)) {
    *(u32x4 *)(kt + crow * WKP + ccol) = r.k0;
    *(u32x4 *)(kt + (crow + 8) * WKP + ccol) = r.k1;
    *(u32x4 *)(kt + (crow + 16) * WKP + ccol) = r.k2;
    *(u32x4 *)(kt + (crow + 24) * WKP + ccol) = r.k3;
    *(u32x4 *)(vt + crow * WKP + ccol) = r.v0;
    *(u32x4 *)(vt + (crow + 8) * WKP + ccol) = r.v1;
    *(u32x4 *)(vt + (crow + 16) * WKP + ccol) = r.v2;
    *(u32x4 *)(vt + (crow + 24) * WKP + ccol) = r.v3;
  };

  float m = -INFINITY, l = 0.f;
  df32x4_t o[4] = {df32x4_t{}, df32x4_t{}, df32x4_t{}, df32x4_t{}};
  dbf16x8_t qb[2], qn[2];
  const float c = p.c;
  // one 32-key tile from this wave's LDS tile: keys kb .. kb + 31 of a unit of kw1 keys
  auto compute = [&](int kb, int kw1) __attribute__((always_inline)) {
    const bf16_t *kl = kt + 8 * grp;
    df32x4_t s[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const bf16_t *kp = kl + (16 * u + l16) * WKP;
      s[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const dbf16x8_t *)(kp), qb[0], df32x4_t{},
                                                     0, 0, 0);
      s[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const dbf16x8_t *)(kp + 32), qb[1], s[u],
                                                     0, 0, 0);
    }
    if (kb + TK > kw1) {
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (kb + 16 * u + 4 * grp + i >= kw1) s[u][i] = -INFINITY;
    }
    float mx = fmaxf(fmaxf(fmaxf(s[0][0], s[0][1]), fmaxf(s[0][2], s[0][3])),
                     fmaxf(fmaxf(s[1][0], s[1][1]), fmaxf(s[1][2], s[1][3])));
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float m_new = fmaxf(m, mx);  // -inf while every key so far scores -inf
    const float mr = m_new * c, mc = mr == -INFINITY ? 0.f : mr;
    const float alpha = __builtin_amdgcn_exp2f(m * c - mc);  // m = -inf -> 0
    float rs = 0.f;
    dbf16x8_t pb;
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float e = __builtin_amdgcn_exp2f(fmaf(s[u][i], c, -mc));
        rs += e;
        pb[4 * u + i] = (__bf16)e;
      }
    l = l * alpha + rs;
    m = m_new;
    const bf16_t *vp = vt + (4 * grp + (l16 >> 2)) * WKP + 4 * (l16 & 3);
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) {
      o[dt] *= alpha;
      const dbf16x4_t lo = lds_read_tr16(vp + 16 * dt);
      const dbf16x4_t hi = lds_read_tr16(vp + 16 * WKP + 16 * dt);
      const dbf16x8_t a = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, pb, o[dt], 0, 0, 0);
    }
  };
  // segment 0 of the share is a later part of a cut unit (not its head):
  // every wave writes its state of it to the part's record as it moves on
  uint64_t *rec0 = nullptr;
  if (ntile > 0) {
    const int b0 = (int)(p.wg_start[grp_id] & 0xffffu);
    const uint32_t info0 = p.unit[b0 * Hkv + gh];
    const int parts0 = (int)(info0 >> 24), part0 = grp_id - (int)((info0 >> 12) & 0xfffu);
    if (parts0 > 1 && part0 > 0 && part0 < parts0)
      rec0 = p.rec + (int64_t)((info0 & 0xfffu) + part0) * rec_words<G>();
  }
  const uint64_t tag = (uint64_t)p.epoch << 32;
  auto put = [&](uint64_t *a, float v) __attribute__((always_inline)) {
    __hip_atomic_store(a, tag | __builtin_bit_cast(uint32_t, v), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_SYSTEM);
  };
  // this wave's state of segment s into LDS slot ls (o[dt][i] = O^T[16dt + 4grp + i][head l16])
  auto flush_to = [&](int s, int ls) __attribute__((always_inline)) {
    float lt = l + __shfl_xor(l, 16, 64);
    lt += __shfl_xor(lt, 32, 64);
    if (l16 < G) {
#pragma unroll
      for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int i = 0; i < 4; ++i) red_o[ls][wave][l16][16 * dt + 4 * grp + i] = o[dt][i];
      if (grp == 0) {
        red_m[ls][wave][l16] = m * c;  // -inf: no key of s in this wave
        red_l[ls][wave][l16] = lt;
      }
    }
    if (s == 0 && rec0) {  // segment 0 handed to the writer wave (LDS writes first)
      __builtin_amdgcn_wave_barrier();
      if (lane == 0) __hip_atomic_fetch_add(&seg0_done, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
  };
  auto flush = [&](int s) __attribute__((always_inline)) { flush_to(s, s); };
  auto reset = [&]() __attribute__((always_inline)) {
    m = -INFINITY;
    l = 0.f;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) o[dt] = df32x4_t{};
  };

  // One register tile ahead per wave, as the whole-cache kernel: cur is the
  // segment of the tile computed, pre that of the tile in the registers;
  // when pre enters a new segment its query rows are loaded into qn, taken
  // over by qb when the wave's tiles reach that segment.
  int sc = -1;  // segment of the wave's running state
  if (streamer && wave < ntile) {  // wave-uniform
    Seg cur, pre;
    seg_first(cur);
    seg_adv(cur, wave);
    gload_q(qb, cur);
    RegTile ta;
    gload(ta, wave, cur);
    lstore(ta);
    pre = cur;
    if (wave + WWV < ntile) {
      seg_adv(pre, wave + WWV);
      if (pre.s != cur.s) gload_q(qn, pre);
      gload(ta, wave + WWV, pre);
    }
    __builtin_amdgcn_wave_barrier();
    for (int i = wave; i < ntile; i += WWV) {
      if (cur.s != sc) {  // a new segment: the previous one's state to LDS, a fresh state
        if (sc >= 0) flush(sc);
        for (int x = sc + 1; x < cur.s; ++x) {
          reset();
          flush(x);
        }
        reset();
        sc = cur.s;
      }
      compute(cur.kb0 + TK * i, cur.len);
      if (i + WWV < ntile) {
        __builtin_amdgcn_wave_barrier();
        lstore(ta);
        if (pre.s != cur.s) {
          qb[0] = qn[0];
          qb[1] = qn[1];
        }
        cur = pre;
        if (i + 2 * WWV < ntile) {
          const int s0 = pre.s;
          seg_adv(pre, i + 2 * WWV);
          if (pre.s != s0) gload_q(qn, pre);
          gload(ta, i + 2 * WWV, pre);
        }
        __builtin_amdgcn_wave_barrier();
      }
    }
  }
  if (streamer) {
    if (sc >= 0) flush(sc);
    reset();
    for (int x = sc + 1; x < nseg; ++x) flush(x);
  } else if (rec0) {
    // the writer wave: once the streaming waves have handed over segment 0
    // (bounded wait inside this workgroup; without the record the head
    // streams the keys itself), merge their states and write the record
    int polls = 0;
    while (__hip_atomic_load(&seg0_done, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP) < (uint32_t)WWV &&
           polls < kPlanPolls) {
      __builtin_amdgcn_s_sleep(2);
      ++polls;
    }
    if (polls < kPlanPolls) {
      for (int idx = lane; idx < G * HD; idx += 64) {
        const int h = idx / HD, d = idx - h * HD;
        // (a part whose keys all score -inf: a finite M whose sums are 0, so
        // that the merges subtract finite numbers)
        float M = fmaxf(red_m[0][0][h], -__FLT_MAX__);
#pragma unroll
        for (int w = 1; w < WWV; ++w) M = fmaxf(M, red_m[0][w][h]);
        float L = 0.f, A = 0.f;
#pragma unroll
        for (int w = 0; w < WWV; ++w) {
          const float wt = __builtin_amdgcn_exp2f(red_m[0][w][h] - M);
          L += red_l[0][w][h] * wt;
          A += red_o[0][w][h][d] * wt;
        }
        put(rec0 + idx, A);
        if (d == 0) {
          put(rec0 + G * HD + h, M);
          put(rec0 + G * HD + G + h, L);
        }
      }
    }
  }
  __syncthreads();

  // Merge the waves of each segment.  A unit wholly in this share is written.
  // A cut unit's later parts wrote their records from the waves (above); its
  // head -- the share's last segment -- loads them past the caches
  // (system-scope loads), each word tagged with this launch's epoch, merges
  // and writes the output.
  Seg x;
  if (nseg > 0) seg_first(x);
  for (int s = 0; s < nseg; ++s) {
    if (s > 0) seg_next(x);
    const int b = x.b, g = gh, u = b * Hkv + g;
    const uint32_t info = p.unit[u];
    const int parts = (int)(info >> 24), part = grp_id - (int)((info >> 12) & 0xfffu);
    if (parts > 1 && part != 0) continue;  // a later part: its record is written
    bf16_t *out = (bf16_t *)p.o + ((int64_t)b * p.n_heads + (int64_t)g * G) * HD;
    // this share's waves: (M, L, A) of output idx from LDS slot ls
    auto own = [&](int ls, int idx, float &M, float &L, float &A) __attribute__((always_inline)) {
      const int h = idx / HD, d = idx - h * HD;
      M = fmaxf(red_m[ls][0][h], -__FLT_MAX__);  // finite, as the records'
#pragma unroll
      for (int w = 1; w < WWV; ++w) M = fmaxf(M, red_m[ls][w][h]);
      L = 0.f;
      A = 0.f;
#pragma unroll
      for (int w = 0; w < WWV; ++w) {
        const float wt = __builtin_amdgcn_exp2f(red_m[ls][w][h] - M);
        L += red_l[ls][w][h] * wt;
        A += red_o[ls][w][h][d] * wt;
      }
    };
    if (parts <= 1) {
      for (int idx = tid; idx < G * HD; idx += kPlanThreads) {
        float M, L, A;
        own(s, idx, M, L, A);
        out[idx] = f32_to_bf16(L == 0.f ? 0.f : A / L);
      }
      continue;
    }
    // the head of a cut unit: this share holds its first tiles, the later
    // parts the rest; each thread merges its outputs from its own loads
    constexpr int NO = (G * HD + kPlanThreads - 1) / kPlanThreads;  // outputs per thread
    const uint64_t *recb = p.rec + (int64_t)(info & 0xfffu) * rec_words<G>();
    float Mv[NO], Lv[NO], Av[NO];
    bool ok = true;
    auto gather = [&]() __attribute__((always_inline)) {
      ok = true;
#pragma unroll
      for (int j = 0; j < NO; ++j) {
        const int idx = min(tid + kPlanThreads * j, G * HD - 1);  // past G*HD: a repeat, not stored
        own(s, idx, Mv[j], Lv[j], Av[j]);
      }
      // one part at a time, every word of the part requested before any is
      // used: one round trip per later part
      for (int q = 1; q < parts; ++q) {
        const uint64_t *r = recb + (int64_t)q * rec_words<G>();
        uint64_t wm[NO], wl[NO], wa[NO];
#pragma unroll
        for (int j = 0; j < NO; ++j) {
          const int idx = min(tid + kPlanThreads * j, G * HD - 1);
          const int h = idx / HD;
          wm[j] = __hip_atomic_load(r + G * HD + h, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
          wl[j] = __hip_atomic_load(r + G * HD + G + h, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
          wa[j] = __hip_atomic_load(r + idx, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
#pragma unroll
        for (int j = 0; j < NO; ++j) {
          ok = ok && (wm[j] >> 32) == p.epoch && (wl[j] >> 32) == p.epoch && (wa[j] >> 32) == p.epoch;
          const float mq = __builtin_bit_cast(float, (uint32_t)wm[j]);
          const float m2 = fmaxf(Mv[j], mq);
          const float a1 = __builtin_amdgcn_exp2f(Mv[j] - m2), a2 = __builtin_amdgcn_exp2f(mq - m2);
          Lv[j] = Lv[j] * a1 + __builtin_bit_cast(float, (uint32_t)wl[j]) * a2;
          Av[j] = Av[j] * a1 + __builtin_bit_cast(float, (uint32_t)wa[j]) * a2;
          Mv[j] = m2;
        }
      }
    };
    bool all_ok = false;
    if (p.max_polls >= 0) {
      gather();
      all_ok = __syncthreads_and(ok);
      for (int poll = 0; !all_ok && poll < p.max_polls; ++poll) {
        __builtin_amdgcn_s_sleep(4);
        gather();
        all_ok = __syncthreads_and(ok);
      }
    }
    if (!all_ok) {
      // Fallback: stream the unit's keys past this share's tiles here, into a
      // free LDS slot (slot 0 is finished when s > 0; slot 1 is unused when
      // the share holds this segment only), and merge with this share's part.
      const int ls = s == 0 ? 1 : 0;
      // local tile i of x holds keys x.kb0 + 32 i, so the later parts start
      // at the unit's tile x.kb0 / 32 + x.end
      const int first_rest = x.kb0 / TK + x.end;
      const int rest = tiles_of(b) - first_rest;
      Seg y = x;
      y.kb0 = TK * first_rest;  // local tile i of y: keys kb0 + 32 i
      if (streamer) {
        reset();
        if (wave < rest) {
          dbf16x8_t qf[2];
          gload_q(qf, y);
          qb[0] = qf[0];
          qb[1] = qf[1];
          for (int i = wave; i < rest; i += WWV) {
            RegTile r;
            gload(r, i, y);
            __builtin_amdgcn_wave_barrier();
            lstore(r);
            __builtin_amdgcn_wave_barrier();
            compute(y.kb0 + TK * i, y.len);
            __builtin_amdgcn_wave_barrier();
          }
        }
        flush_to(-1, ls);
      }
      __syncthreads();
#pragma unroll
      for (int j = 0; j < NO; ++j) {
        const int idx = min(tid + kPlanThreads * j, G * HD - 1);
        float M, L, A, M2, L2, A2;
        own(s, idx, M, L, A);
        own(ls, idx, M2, L2, A2);
        const float mm = fmaxf(M, M2);
        const float a1 = __builtin_amdgcn_exp2f(M - mm), a2 = __builtin_amdgcn_exp2f(M2 - mm);
        Mv[j] = mm;
        Lv[j] = L * a1 + L2 * a2;
        Av[j] = A * a1 + A2 * a2;
      }
    }
#pragma unroll
    for (int j = 0; j < NO; ++j) {
      const int idx = tid + kPlanThreads * j;
      if (idx < G * HD) out[idx] = f32_to_bf16(Lv[j] == 0.f ? 0.f : Av[j] / Lv[j]);
    }
    __syncthreads();  // the fallback's LDS slot and state are reused by the next segment
  }
}

// One thread per (b, head, d): merge the chunks [0, ceil(len/chunk)) in one
// pass (running log-sum-exp), four chunks' loads in flight at a time.
template <typename T>
__global__ __launch_bounds__(256) void decode_combine_kernel(DecodeParams p) {
  // one thread per 4 consecutive d of one (sequence, head); the partial loads
  // of 8 chunks are issued together with the length load (slots past the
  // valid chunks read an in-range record and are skipped in the merge).
  // chunk 0: the short-cache split's chunk, derived from the length.
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= (int64_t)p.batch * p.n_heads * (HD / 4)) return;
  const int d0 = (int)(idx % (HD / 4)) * 4;
  const int64_t bh = idx / (HD / 4);
  const int b = (int)(bh / p.n_heads);
  const float *part = p.ws + bh * p.n_split * kDecRec;
  DecMerge mg;
  int len = p.hlen >= 0 ? p.hlen : p.lens[b];
  mg.load8(part, p.n_split, 0, d0);
  len = len < 0 ? 0 : (len > p.max_len ? p.max_len : len);
  const int chunk = p.chunk > 0 ? p.chunk : short_split_chunk(len, p.n_split);
  const int nvalid = (len + chunk - 1) / chunk;  // chunks holding keys (finite max)
  mg.start();
  mg.merge8(0, nvalid);  // the first 8 chunks need no branch on the length
  for (int s0 = 8; s0 < nvalid; s0 += 8) {
    mg.load8(part, p.n_split, s0, d0);
    mg.merge8(s0, nvalid);
  }
  const float4 r = mg.result();
  T *out = (T *)p.o + bh * HD + d0;
  Elem<T>::store(out + 0, r.x);
  Elem<T>::store(out + 1, r.y);
  Elem<T>::store(out + 2, r.z);
  Elem<T>::store(out + 3, r.w);
}

// workgroup targets of the fp32 chunks, and of the chunks of four KV heads in
// which the no-allocation call counts a bf16 call's size: its limit is the
// caller's to rely on, so it does not follow the pieces, which need less
// (17.3 MB at most of the 32)
constexpr int kMinWg = 2048, kRowsMinWg = 512;
int choose_chunk(int batch, int max_len, int units, int min_wg) {
  // enough workgroups to cover the 256 CUs several times over (a partial last
  // round of resident workgroups costs a whole round), chunks >= 128 keys
  int chunk = 1024;
  while (chunk > 128 && (int64_t)batch * units * ((max_len + chunk - 1) / chunk) < min_wg)
    chunk >>= 1;
  return chunk;
}

bool rows_path(const DecodeParams &p, bool bf16) { return bf16 && p.n_kv_heads % 4 == 0; }

void launch_short(const DecodeParams &p, hipStream_t s) {
  const dim3 grid((unsigned)((int64_t)p.batch * p.n_heads / kShortG * p.n_split));
  hipLaunchKernelGGL((decode_split_kernel<float, kShortG, kShortWV, DEC_SHORT>), grid, dim3(64 * kShortWV),
                     0, s, p);
}

// fp32 caches past the short split: chunks, then the combine
int launch_decode(const DecodeParams &p, int G, hipStream_t s) {
  const dim3 grid((unsigned)((int64_t)p.batch * p.n_kv_heads * p.n_split));
  switch (G) {
    case 1: hipLaunchKernelGGL((decode_split_kernel<float, 1, 4, DEC_SPLIT>), grid, dim3(256), 0, s, p); break;
    case 2: hipLaunchKernelGGL((decode_split_kernel<float, 2, 4, DEC_SPLIT>), grid, dim3(256), 0, s, p); break;
    case 4: hipLaunchKernelGGL((decode_split_kernel<float, 4, 4, DEC_SPLIT>), grid, dim3(256), 0, s, p); break;
    default: hipLaunchKernelGGL((decode_split_kernel<float, 8, 4, DEC_SPLIT>), grid, dim3(256), 0, s, p);
  }
  BN_LAUNCH_CHECK();
  const int64_t n = (int64_t)p.batch * p.n_heads * (HD / 4);
  hipLaunchKernelGGL(decode_combine_kernel<float>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, p);
  BN_LAUNCH_CHECK();
  return BN_OK;
}

}  // namespace

bool short_path_ok(int dtype, int batch, int max_len, int n_heads) {
  return dtype == BN_F32 && batch > 0 && max_len > 0 && max_len <= kShortMaxLen &&
         (int64_t)batch * n_heads <= kShortMaxUnits;
}

int decode_short_partials(const float *q, const float *k_cache, const float *v_cache,
                          const int32_t *seq_lens, int host_len, float *part, int batch, int max_len,
                          int n_heads, int n_kv_heads, float scale, hipStream_t s) {
  DecodeParams p;
  p.q = q; p.k = k_cache; p.v = v_cache; p.lens = seq_lens; p.o = nullptr; p.ws = part;
  p.hlen = host_len;
  p.batch = batch; p.max_len = max_len; p.n_heads = n_heads; p.n_kv_heads = n_kv_heads;
  p.kv_rs = (int64_t)n_kv_heads * HD;  // contiguous [batch, max_len, n_kv_heads, 64]
  p.kv_hs = HD;
  p.kv_bs = (int64_t)max_len * p.kv_rs;
  p.n_split = kShortSplits;
  p.chunk = 0;
  p.c = scale * 1.4426950408889634f;
  launch_short(p, s);
  BN_LAUNCH_CHECK();
  return BN_OK;
}

// Device address of `scratch` per device, looked up once per device by
// bn_init (with that device current).  Each GPU holds its own copy of the
// array at its own address.
constexpr int kMaxScratchDevices = 64;
static std::mutex g_scratch_mu;
static void *g_scratch_ptr[kMaxScratchDevices];

// the planned decode's launch epochs (the tag of every record word a launch
// writes; never 0)
static std::atomic<uint32_t> g_plan_epoch{0};
static void *g_short_cnt_ptr[kMaxScratchDevices];
static std::atomic<uint32_t> g_short_next{0};

int decode_scratch_setup(int device) {
  if (device < 0 || device >= kMaxScratchDevices)
    return fail(BN_ERR_UNSUPPORTED, "bn_init: device " + std::to_string(device) +
                                        " above the decode scratch table (" +
                                        std::to_string(kMaxScratchDevices) + " devices)");
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (g_scratch_ptr[device]) return BN_OK;
  void *ptr = nullptr;
  BN_HIP_TRY(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
  if (!ptr) return fail(BN_ERR_HIP, "bn_init: decode scratch has no device address");
  void *scnt = nullptr;  // the short-cache decode's split counters
  BN_HIP_TRY(hipGetSymbolAddress(&scnt, HIP_SYMBOL(short_counters)));
  if (!scnt) return fail(BN_ERR_HIP, "bn_init: short decode counters have no device address");
  g_scratch_ptr[device] = ptr;
  g_short_cnt_ptr[device] = scnt;
  return BN_OK;
}

namespace {
void *decode_scratch(int device) {
  if (device < 0 || device >= kMaxScratchDevices) return nullptr;
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  return g_scratch_ptr[device];
}
// the next planned-decode launch epoch (never 0)
uint32_t next_plan_epoch() {
  uint32_t e = g_plan_epoch.fetch_add(1) + 1;
  if (e == 0) e = g_plan_epoch.fetch_add(1) + 1;
  return e;
}
// Splits per (sequence, KV head) pair of the split whole-cache kernel: about
// one workgroup per compute unit, at most 8 records to merge (us, by splits:
// one cache of 1543 keys 1 / 4 / 8 / 12 11.2 / 8.1 / 7.0 / 7.1; 12 caches of
// 200..4000 4 / 5 / 8 12.4 / 11.2 / 12.0; 16 of 4000, 4 KV heads, 2 / 4 / 8
// 19.3 / 13.9 / 16.7; 32 of 500..2000 1 / 2 / 4 16.1 / 13.0 / 15.0; 48 of
// 500..4000 1 / 2 28.4 / 28.8), and one fewer than the cache's 128-key chunks,
// so that the records and the arrival words fit the workspace that
// bn_gqa_decode_workspace_size() asks for.  Unsplit pairs have eight waves
// (48 caches: 28.4 -> 25.2; 60 of 100..1000 11.6 -> 11.0), split ones four.
int whole_splits(int units, int max_len) {
  return std::max(1, std::min({256 / units, 8, (max_len + 127) / 128 - 1}));
}
// Where caches can be longer than those lines were drawn for:
//  - below 32 pairs a cache's pieces follow its own length (the most of them
//    returned, 0: equal pieces as above): a piece per 1024 keys.  us, former chunk
//    kernel / equal pieces / by length, 4 KV heads: one cache of 16384 keys 23.4
//    / 16.8 / 13.4, of 131072 86 / 94 / 32, with 8 KV heads 74 / 97 / 44; of 1543
//    in 131072 rows 11.8 / 6.9 / 6.9
int pieces_by_length(int units, int max_len) {
  return units < 32 && max_len >= 16384 ? std::min({256 / units, 64, max_len / kPieceMinLen & ~7}) : 0;
}
//  - from there the batch's tiles are dealt in equal shares (kDealt) to the
//    workgroups per KV head returned (0: as above), one per compute unit.  1500
//    drawn batches in both layouts (equal, ragged and mixed lengths, one long
//    cache, all short), equal pieces / dealt as ratios to the former chunk kernel,
//    mean and worst: 65..255 pairs from 8192 rows 1.08 and 4.4 / 0.72 and 1.04, of
//    4096..8191 0.85 and 2.6 / 0.77 and 1.18, of 2500..4095 0.74 and 1.65 / 0.77
//    and 1.31; 32..64 pairs from 20000 rows 0.80 and 1.78 / 0.74 and 1.03, of
//    10240..19999 0.70 and 1.28 / 0.70 and 1.01, of 4000..6999 0.63 and 0.91 /
//    0.69 and 0.98.  us, chunk kernel / equal pieces / dealt, 4 KV heads: 33
//    token-major caches of 707..8103 keys 48 / 51 / 32, all of 8192 61 / 58 / 49, 40
//    of 1269..16128 91 / 104 / 66, 32 of 618..15604 58 / 58 / 46, 24 of 4079..30201
//    102 / 103 / 75, one of 16384 among 39 of 500 53 / 92 / 19.  The scan over the
//    lengths costs 0.6 us: 8 of 16384 34.7 / 23.9 / 24.5.
int dealt_groups(int batch, int n_kv_heads, int max_len) {
  const int64_t units = (int64_t)batch * n_kv_heads;
  // a lane scans four sequences (units < 256), and tiles are counted in 31 bits
  if (units < 32 || units >= 256 || (int64_t)batch * max_len > ((int64_t)1 << 34)) return 0;
  // Two records a workgroup, at most 512 / n_kv_heads of a head, and the arrival
  // words fit the 128-key chunks' workspace: over 2000 / n_kv_heads records.
  return max_len >= (units > 64 ? 4096 : 10240) ? 256 / n_kv_heads : 0;
}
// a launch's 48-bit tag: a mixed counter (SplitMix64's finaliser), so that
// no plausible memory contents look like this launch's arrivals
std::atomic<uint64_t> g_split_launch{0};
unsigned long long next_split_tag() {
  uint64_t z = (g_split_launch.fetch_add(1) + 1) * 0x9e3779b97f4a7c15ull;
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
  return (z ^ (z >> 31)) >> 16 | 1;
}
// the next counter slot of the short-cache decode on `device` (null: not set up)
constexpr int kShortSlots = 16;
static_assert(kShortSlots * kShortMaxUnits == 16 * 256, "short_counters holds kShortSlots slots");
uint32_t *short_counter_slot(int device) {
  if (device < 0 || device >= kMaxScratchDevices) return nullptr;
  void *base;
  {
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    base = g_short_cnt_ptr[device];
  }
  if (!base) return nullptr;
  return (uint32_t *)base + (g_short_next.fetch_add(1) % kShortSlots) * kShortMaxUnits;
}
}  // namespace
}  // namespace bn

using namespace bn;

extern "C" {

size_t bn_gqa_decode_workspace_size(int batch, int max_len, int n_heads, int head_dim) {
  if (batch <= 0 || max_len <= 0 || n_heads <= 0 || head_dim != HD) return 0;
  // n_split does not depend on n_kv_heads by more than the chunk choice; size
  // for the smallest chunk (most splits) so any n_kv_heads fits
  int64_t n_split = (max_len + 127) / 128;
  if (short_path_ok(BN_F32, batch, max_len, n_heads)) n_split = std::max<int64_t>(n_split, kShortSplits);
  return (size_t)batch * n_heads * n_split * kDecRec * sizeof(float);
}

}  // extern "C"

namespace bn {
namespace {
// bn_gqa_decode and bn_gqa_decode_noalloc: the same validation, kernels and
// launch shapes; they differ only in where the split-K partials live (the
// caller's workspace or the pool, against the file-scope scratch array).
// strides: the caches' element strides (sequence, KV head, key row), or null
// for a contiguous [batch, max_len, n_kv_heads, head_dim] cache.
int gqa_decode_impl(int dtype, const void *q, const void *k_cache, const void *v_cache,
                    const int32_t *seq_lens, void *o, int batch, int max_len, int n_heads,
                    int n_kv_heads, int head_dim, float scale, void *workspace,
                    size_t workspace_bytes, bool noalloc, void *stream,
                    const int64_t *strides = nullptr) {
  const char *op = noalloc ? "GQA decode (no allocation)" : strides ? "GQA decode (strided)" : "GQA decode";
  if (dtype != BN_F32 && dtype != BN_BF16)
    return fail(BN_ERR_UNSUPPORTED, std::string(op) + ": dtype must be F32 or BF16");
  if (batch < 0 || max_len < 0)
    return fail(BN_ERR_SHAPE, std::string(op) + ": negative batch or cache length");
  if (n_heads <= 0 || n_kv_heads <= 0 || n_heads % n_kv_heads != 0)
    return fail(BN_ERR_SHAPE, std::string(op) + ": num_heads must be a positive multiple of num_kv_heads");
  const int G = n_heads / n_kv_heads;
  if (G != 1 && G != 2 && G != 4 && G != 8)
    return fail(BN_ERR_UNSUPPORTED, std::string(op) + ": heads per KV head must be 1, 2, 4 or 8");
  if (head_dim != HD) return fail(BN_ERR_UNSUPPORTED, std::string(op) + ": head_dim must be 64");
  if (!(scale > 0.f) || !std::isfinite(scale))
    return fail(BN_ERR_INVALID_ARG, std::string(op) + ": scale must be positive and finite");
  if (batch == 0) return BN_OK;
  if (max_len == 0) return fail(BN_ERR_SHAPE, std::string(op) + ": max_len must be positive");
  if (strides) {
    // every key row starts 16-byte aligned (the kernels load 16 bytes per lane)
    const int64_t align = dtype == BN_BF16 ? 8 : 4;
    for (int i = 0; i < 3; ++i)
      if (strides[i] <= 0 || strides[i] % align != 0 || strides[i] > ((int64_t)1 << 40))
        return fail(BN_ERR_INVALID_ARG, std::string(op) + ": cache strides must be positive multiples of " +
                                            std::to_string(align) + " elements (16 bytes)");
  }
  if (!q || !k_cache || !v_cache || !seq_lens || !o)
    return fail(BN_ERR_INVALID_ARG, std::string(op) + ": NULL pointer");
  if (((uintptr_t)q | (uintptr_t)k_cache | (uintptr_t)v_cache) & 15u)
    return fail(BN_ERR_UNSUPPORTED, std::string(op) + ": q and caches must be 16-byte aligned");
  // a caller's workspace must hold what bn_gqa_decode_workspace_size() asks
  // for, whichever kernel the call takes (checked before any device work)
  if (workspace) {
    const size_t want = bn_gqa_decode_workspace_size(batch, max_len, n_heads, head_dim);
    if (workspace_bytes < want)
      return fail(BN_ERR_INVALID_ARG, std::string(op) + ": workspace of " +
                                          std::to_string(workspace_bytes) + " bytes, need " +
                                          std::to_string(want));
  }
  DecodeParams p;
  p.q = q; p.k = k_cache; p.v = v_cache; p.lens = seq_lens; p.o = o;
  p.batch = batch; p.max_len = max_len; p.n_heads = n_heads; p.n_kv_heads = n_kv_heads;
  p.kv_bs = strides ? strides[0] : (int64_t)max_len * n_kv_heads * HD;
  p.kv_hs = strides ? strides[1] : HD;
  p.kv_rs = strides ? strides[2] : (int64_t)n_kv_heads * HD;
  const bool short_split = short_path_ok(dtype, batch, max_len, n_heads);
  if (!short_split && dtype == BN_BF16) {  // one workgroup per (sequence, KV head) when that fills the CUs
    int st = ensure_device();
    if (st) return st;
    const int cus = device_cu_count();
    if (cus > 0 && (int64_t)batch * n_kv_heads >= cus) {
      p.ws = nullptr;
      p.n_split = 1;
      p.chunk = max_len;
      p.c = scale * 1.4426950408889634f;
      hipStream_t s = as_stream(stream);
      // a KV head's rows contiguous: long caches may take more waves
      const bool wide = p.kv_rs == HD && batch <= kMeanBatchMax;
      const dim3 grid((unsigned)((int64_t)batch * n_kv_heads)), block(64 * (wide ? WWX : WWV));
#define BN_WHOLE(GG)                                                                        \
  do {                                                                                      \
    if (wide)                                                                               \
      hipLaunchKernelGGL((decode_bf16_whole_kernel<GG, WWX, kWhole>), grid, block, 0, s, p);        \
    else                                                                                    \
      hipLaunchKernelGGL((decode_bf16_whole_kernel<GG, WWV, kWhole>), grid, block, 0, s, p);        \
  } while (0)
      switch (G) {
        case 1: BN_WHOLE(1); break;
        case 2: BN_WHOLE(2); break;
        case 4: BN_WHOLE(4); break;
        default: BN_WHOLE(8); break;
      }
#undef BN_WHOLE
      BN_LAUNCH_CHECK();
      return BN_OK;
    }
  }
  if (short_split) {  // kShortSplits splits of the length; the combine derives the chunk
    p.chunk = 0;
    p.n_split = kShortSplits;
  } else {
    p.chunk = rows_path(p, dtype == BN_BF16)
                  ? choose_chunk(batch, max_len, n_kv_heads / 4, kRowsMinWg)
                  : choose_chunk(batch, max_len, n_kv_heads, kMinWg);
    p.n_split = (max_len + p.chunk - 1) / p.chunk;
  }
  p.c = scale * 1.4426950408889634f;
  const bool bsplit = !short_split && dtype == BN_BF16;  // split whole-cache kernel
  size_t need = (size_t)batch * n_heads * p.n_split * (HD + 2) * sizeof(float);
  if (noalloc && need > (size_t)BN_GQA_DECODE_SCRATCH_BYTES)
    return fail(BN_ERR_UNSUPPORTED, std::string(op) + ": the call needs " + std::to_string(need) +
                                        " bytes of chunk partials, above the " +
                                        std::to_string((size_t)BN_GQA_DECODE_SCRATCH_BYTES) +
                                        "-byte scratch");
  size_t words = 0;
  if (bsplit) {  // (the no-allocation limit above stays that of the chunks' partials)
    const int units = batch * n_kv_heads;
    p.min_split = whole_splits(units, max_len);
    p.n_split = std::max(p.min_split, pieces_by_length(units, max_len));
    p.groups = dealt_groups(batch, n_kv_heads, max_len);
    const size_t records = p.groups ? 2 * p.groups * (size_t)n_heads : (size_t)batch * n_heads * p.n_split;
    words = p.groups || p.n_split > 1 ? (size_t)units * 16 + 8 : 0;
    need = words ? records * kDecRec * sizeof(float) + words : 0;
  }
  int st = ensure_device();
  if (st) return st;
  hipStream_t s = as_stream(stream);
  void *ws = workspace;
  bool own = false;
  if (noalloc) {
    // every record the combine reads is written by this call's split kernel
    // first, so the scratch needs no clearing
    ws = decode_scratch(library_device());
    if (!ws) return fail(BN_ERR_HIP, std::string(op) + ": scratch address not set up for device " +
                                         std::to_string(library_device()));
  } else if (!ws && need > 0) {
    if ((st = bn_alloc(&ws, need, stream))) return st;
    own = true;
  }
  p.ws = (float *)ws;
  if (bsplit) {  // one launch: a pair's last split merges its records
    if (words) {
      const size_t bytes = noalloc ? (size_t)BN_GQA_DECODE_SCRATCH_BYTES : own ? need : workspace_bytes;
      p.arrive_end = (unsigned long long *)(((uintptr_t)ws + bytes) & ~(uintptr_t)7);
      p.tag = next_split_tag();
    }
    const dim3 grid((unsigned)(p.groups ? p.groups * n_kv_heads : batch * n_kv_heads * p.n_split));
    const bool by_length = p.n_split > p.min_split, eight = !p.groups && p.n_split == 1;  // (waves)
#define BN_SPLIT(GG)                                                                                        \
  do {                                                                                                      \
    if (p.groups)                                                                                           \
      hipLaunchKernelGGL((decode_bf16_whole_kernel<GG, WWV, kDealt>), grid, dim3(64 * WWV), 0, s, p);       \
    else if (by_length)                                                                                     \
      hipLaunchKernelGGL((decode_bf16_whole_kernel<GG, WWV, kByLength>), grid, dim3(64 * WWV), 0, s, p);    \
    else if (eight)                                                                                         \
      hipLaunchKernelGGL((decode_bf16_whole_kernel<GG, WW1, kSplit>), grid, dim3(64 * WW1), 0, s, p);       \
    else                                                                                                    \
      hipLaunchKernelGGL((decode_bf16_whole_kernel<GG, WWV, kSplit>), grid, dim3(64 * WWV), 0, s, p);       \
  } while (0)
    switch (G) {
      case 1: BN_SPLIT(1); break;
      case 2: BN_SPLIT(2); break;
      case 4: BN_SPLIT(4); break;
      default: BN_SPLIT(8); break;
    }
#undef BN_SPLIT
    const hipError_t e = hipGetLastError();
    st = e == hipSuccess ? BN_OK : hip_fail(e, __FILE__, __LINE__);
  } else if (short_split) {  // one launch: the unit's last split merges its records
    p.cnt = short_counter_slot(library_device());
    if (!p.cnt) {
      st = fail(BN_ERR_HIP, std::string(op) + ": split counters not set up for device " +
                                std::to_string(library_device()));
    } else {
      launch_short(p, s);
      const hipError_t e = hipGetLastError();
      st = e == hipSuccess ? BN_OK : hip_fail(e, __FILE__, __LINE__);
    }
  } else {
    st = launch_decode(p, G, s);
  }
  if (own) {
    int st2 = bn_free(ws, stream);
    if (st == BN_OK) st = st2;
  }
  return st;
}
// The planned launch's share plan from the host lengths: groups of
// n_kv_heads workgroups (one per KV head) split the batch's sequence tiles
// into equal contiguous shares.  False when the batch is not worth planning
// (longest sequence within 1.25x of the mean: the whole-cache kernel is
// balanced already) or does not fit the plan's limits.
bool build_plan(const int32_t *h_lens, int batch, int max_len, int n_kv_heads, int n_heads, int cus,
                PlanParams &pl, int &bins, int &records) {
  (void)n_heads;
  const int units = batch * n_kv_heads;
  if (units > kPlanUnits || batch > kPlanUnits || cus <= 0) return false;
  std::vector<int> tiles(batch);
  int64_t total = 0;
  int tmax = 0;
  for (int b = 0; b < batch; ++b) {
    const int len = h_lens[b] < 0 ? 0 : (h_lens[b] > max_len ? max_len : h_lens[b]);
    pl.len[b] = len;
    tiles[b] = (len + TK - 1) / TK;
    total += tiles[b];
    tmax = std::max(tmax, tiles[b]);
  }
  if (total == 0 || total > 0xffffff || (int64_t)tmax * batch * 4 <= total * 5) return false;
  const int groups0 = (int)std::min<int64_t>(std::min(cus, kPlanBins) / n_kv_heads, total);
  if (groups0 <= 0) return false;
  const int share = (int)((total + groups0 - 1) / groups0);
  const int groups = (int)((total + share - 1) / share);
  bins = groups * n_kv_heads;
  if (share > 0xffff || tmax > 0xffff) return false;
  // prefix of each sequence's tiles; group k takes tiles [k*share, (k+1)*share)
  std::vector<int64_t> pre(batch + 1, 0);
  for (int b = 0; b < batch; ++b) pre[b + 1] = pre[b] + tiles[b];
  int b = 0;
  for (int k = 0; k < groups; ++k) {
    const int64_t g0 = (int64_t)k * share;
    while (b < batch && pre[b] + tiles[b] <= g0) ++b;  // skips empty sequences
    pl.wg_start[k] = (uint32_t)b | ((uint32_t)(g0 - pre[b]) << 16);
    // the sequences this share touches (with keys), at most kPlanSeg
    int n = 0;
    for (int v = b; v < batch && pre[v] < g0 + share; ++v) n += tiles[v] > 0;
    if (n > kPlanSeg) return false;
  }
  records = 0;
  for (int v = 0; v < batch; ++v) {
    int c0 = 0, parts = 1;
    if (tiles[v] > 0) {
      c0 = (int)(pre[v] / share);
      parts = (int)((pre[v] + tiles[v] - 1) / share) - c0 + 1;
    }
    for (int g = 0; g < n_kv_heads; ++g) {  // each KV head's unit: parts in the same groups
      const int base = parts > 1 ? records : 0;
      if (parts > 1) records += parts;
      if (records > 0xfff || c0 > 0xfff || parts > 0xff) return false;
      pl.unit[v * n_kv_heads + g] = (uint32_t)base | ((uint32_t)c0 << 12) | ((uint32_t)parts << 24);
    }
  }
  pl.share = share;
  pl.total = (int)total;
  pl.n_units = units;
  return true;
}
}  // namespace
}  // namespace bn

extern "C" {

int bn_gqa_decode(int dtype, const void *q, const void *k_cache, const void *v_cache,
                  const int32_t *seq_lens, void *o, int batch, int max_len, int n_heads,
                  int n_kv_heads, int head_dim, float scale, void *workspace,
                  size_t workspace_bytes, void *stream) {
  return gqa_decode_impl(dtype, q, k_cache, v_cache, seq_lens, o, batch, max_len, n_heads,
                         n_kv_heads, head_dim, scale, workspace, workspace_bytes, false, stream);
}

int bn_gqa_decode_noalloc(int dtype, const void *q, const void *k_cache, const void *v_cache,
                          const int32_t *seq_lens, void *o, int batch, int max_len, int n_heads,
                          int n_kv_heads, int head_dim, float scale, void *stream) {
  return gqa_decode_impl(dtype, q, k_cache, v_cache, seq_lens, o, batch, max_len, n_heads,
                         n_kv_heads, head_dim, scale, nullptr, 0, true, stream);
}

int bn_gqa_decode_strided(int dtype, const void *q, const void *k_cache, const void *v_cache,
                          const int32_t *seq_lens, void *o, int batch, int max_len, int n_heads,
                          int n_kv_heads, int head_dim, int64_t cache_seq_stride,
                          int64_t cache_head_stride, int64_t cache_row_stride, float scale,
                          void *workspace, size_t workspace_bytes, void *stream) {
  const int64_t strides[3] = {cache_seq_stride, cache_head_stride, cache_row_stride};
  return gqa_decode_impl(dtype, q, k_cache, v_cache, seq_lens, o, batch, max_len, n_heads,
                         n_kv_heads, head_dim, scale, workspace, workspace_bytes, false, stream,
                         strides);
}

size_t bn_gqa_decode_planned_workspace_size(int batch, int max_len, int n_heads, int n_kv_heads,
                                            int head_dim) {
  if (batch <= 0 || max_len <= 0 || n_heads <= 0 || n_kv_heads <= 0 || n_heads % n_kv_heads ||
      head_dim != HD)
    return 0;
  // the unplanned fallback's partials, or the plan's part records (at most
  // one per unit plus one per workgroup boundary; each holds every wave's
  // state as epoch-tagged 64-bit words)
  const size_t recs = ((size_t)batch * n_kv_heads + kPlanBins) *
                      ((size_t)(n_heads / n_kv_heads) * HD + 2 * (n_heads / n_kv_heads)) * sizeof(uint64_t);
  return std::max(bn_gqa_decode_workspace_size(batch, max_len, n_heads, head_dim), recs);
}

}  // extern "C"

namespace bn {
namespace {
// bn_gqa_decode_planned and bn_gqa_decode_planned_strided (strides: null for
// a contiguous [batch, max_len, n_kv_heads, 64] cache)
int gqa_decode_planned_impl(int dtype, const void *q, const void *k_cache, const void *v_cache,
                            const int32_t *seq_lens, const int32_t *h_seq_lens, void *o, int batch,
                            int max_len, int n_heads, int n_kv_heads, int head_dim, float scale,
                            void *workspace, size_t workspace_bytes, void *stream,
                            const int64_t *strides) {
  const char *op = "GQA decode (planned)";
  if (batch > 0 && !h_seq_lens)
    return fail(BN_ERR_INVALID_ARG, std::string(op) + ": NULL host lengths");
  if (workspace && batch > 0) {
    const size_t want = bn_gqa_decode_planned_workspace_size(batch, max_len, n_heads, n_kv_heads, head_dim);
    if (want && workspace_bytes < want)
      return fail(BN_ERR_INVALID_ARG, std::string(op) + ": workspace of " +
                                          std::to_string(workspace_bytes) + " bytes, need " +
                                          std::to_string(want));
  }
  // the plan applies to bf16 caches of 1, 2, 4 or 8 query heads per KV head
  // with at least as many units as compute units; anything else (and every
  // argument check) is bn_gqa_decode's
  const int G = n_kv_heads > 0 ? n_heads / n_kv_heads : 0;
  bool planned = dtype == BN_BF16 && head_dim == HD && batch > 0 && max_len > 0 && n_kv_heads > 0 &&
                 n_heads % n_kv_heads == 0 && (G == 1 || G == 2 || G == 4 || G == 8) &&
                 (scale > 0.f) && std::isfinite(scale) && q && k_cache && v_cache && seq_lens && o &&
                 !(((uintptr_t)q | (uintptr_t)k_cache | (uintptr_t)v_cache) & 15u);
  if (strides)
    for (int i = 0; i < 3; ++i)
      planned = planned && strides[i] > 0 && strides[i] % 8 == 0 && strides[i] <= ((int64_t)1 << 40);
  int st;
  PlanParams pl;
  int bins = 0, records = 0;
  if (planned) {
    if ((st = ensure_device())) return st;
    const int cus = device_cu_count();
    planned = (int64_t)batch * n_kv_heads >= cus &&
              build_plan(h_seq_lens, batch, max_len, n_kv_heads, n_heads, cus, pl, bins, records);
  }
  if (!planned)
    return gqa_decode_impl(dtype, q, k_cache, v_cache, seq_lens, o, batch, max_len, n_heads, n_kv_heads,
                           head_dim, scale, workspace, workspace_bytes, false, stream, strides);
  pl.q = q; pl.k = k_cache; pl.v = v_cache; pl.o = o;
  pl.batch = batch; pl.max_len = max_len; pl.n_heads = n_heads; pl.n_kv_heads = n_kv_heads;
  pl.kv_bs = strides ? strides[0] : (int64_t)max_len * n_kv_heads * HD;
  pl.kv_hs = strides ? strides[1] : HD;
  pl.kv_rs = strides ? strides[2] : (int64_t)n_kv_heads * HD;
  pl.c = scale * 1.4426950408889634f;
  pl.epoch = next_plan_epoch();
  // BN_PLAN_FALLBACK=1 (tests): the heads ignore the records and stream the
  // later parts' keys themselves -- the path a head takes if a record never
  // arrives
  const char *fb = std::getenv("BN_PLAN_FALLBACK");
  pl.max_polls = (fb && fb[0] == '1') ? -1 : kPlanPolls;
  hipStream_t s = as_stream(stream);
  void *ws = workspace;
  bool own = false;
  const size_t need = (size_t)std::max(records, 1) * ((size_t)G * HD + 2 * G) * sizeof(uint64_t);
  if (!ws && records > 0) {
    if ((st = bn_alloc(&ws, need, stream))) return st;
    own = true;
  }
  pl.rec = (uint64_t *)ws;
  const dim3 grid((unsigned)bins), block(kPlanThreads);
  switch (G) {
    case 1: hipLaunchKernelGGL(decode_bf16_planned_kernel<1>, grid, block, 0, s, pl); break;
    case 2: hipLaunchKernelGGL(decode_bf16_planned_kernel<2>, grid, block, 0, s, pl); break;
    case 4: hipLaunchKernelGGL(decode_bf16_planned_kernel<4>, grid, block, 0, s, pl); break;
    default: hipLaunchKernelGGL(decode_bf16_planned_kernel<8>, grid, block, 0, s, pl); break;
  }
  st = BN_OK;
  {
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) st = hip_fail(e, __FILE__, __LINE__);
  }
  if (own) {
    int st2 = bn_free(ws, stream);
    if (st == BN_OK) st = st2;
  }
  return st;
}
}  // namespace
}  // namespace bn

extern "C" {

int bn_gqa_decode_planned(int dtype, const void *q, const void *k_cache, const void *v_cache,
                          const int32_t *seq_lens, const int32_t *h_seq_lens, void *o, int batch,
                          int max_len, int n_heads, int n_kv_heads, int head_dim, float scale,
                          void *workspace, size_t workspace_bytes, void *stream) {
  return gqa_decode_planned_impl(dtype, q, k_cache, v_cache, seq_lens, h_seq_lens, o, batch, max_len,
                                 n_heads, n_kv_heads, head_dim, scale, workspace, workspace_bytes,
                                 stream, nullptr);
}

int bn_gqa_decode_planned_strided(int dtype, const void *q, const void *k_cache,
                                  const void *v_cache, const int32_t *seq_lens,
                                  const int32_t *h_seq_lens, void *o, int batch, int max_len,
                                  int n_heads, int n_kv_heads, int head_dim,
                                  int64_t cache_seq_stride, int64_t cache_head_stride,
                                  int64_t cache_row_stride, float scale, void *workspace,
                                  size_t workspace_bytes, void *stream) {
  const int64_t strides[3] = {cache_seq_stride, cache_head_stride, cache_row_stride};
  return gqa_decode_planned_impl(dtype, q, k_cache, v_cache, seq_lens, h_seq_lens, o, batch, max_len,
                                 n_heads, n_kv_heads, head_dim, scale, workspace, workspace_bytes,
                                 stream, strides);
}

}  // extern "C"
