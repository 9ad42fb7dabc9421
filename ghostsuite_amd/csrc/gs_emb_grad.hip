// Embedding train gradient and dot products, gfx950.  The gradient:
//
//   grad[v] = scale * sum over the train tokens t with id_t = v of g_t        grad: [vocab, d]
//
// The train tokens are listed by id, so every id's tokens form one run, in index order, of a
// sorted token list; sums run over that list in a fixed order, so the result is the same bits on
// every run, and every step's work is linear in the number of tokens however often an id repeats.
// Launches:
//   1. eg_bucket_kernel  -- the list, its length and the presence bitmap of the ids, for up to
//                           131072 tokens and 524288 ids; beyond that in two launches:
//      eg_sort_kernel    -- chunks of EG_CHUNK tokens sorted in registers and LDS (bitonic);
//                           per-chunk counts of in-range ids; the id-presence bitmap cleared.
//   2. eg_merge_kernel   -- every key's place in the whole list = its place in its chunk plus
//                           the number of smaller keys in each other chunk (binary search);
//                           the presence bitmap set.
//   3. eg_window_kernel  -- one wave per window of EG_WIN places: each run inside the window
//                           is summed in index order and its row written (scaled, added to
//                           the old row when accumulating); a run crossing a window boundary
//                           leaves its part of the window as an fp32 partial.  In overwrite
//                           mode further waves write zeros to the rows of absent ids.
//   4. eg_combine_kernel -- per run that crosses windows, its partials summed in a fixed
//                           order and the row written: by one wave for a run of a few
//                           windows, by the 16 waves of a workgroup for a longer one, and by
//                           the workgroups whose windows it covers, a share of the features
//                           each, for a run of hundreds of tokens or more.
// Token ids outside [0, vocab) take no part.
//
// The dots, dot_i = sum_t <g_it, V[x_it]> with V[v] the sum of the val rows of id v, for up to 8192
// val tokens: the val tokens' list (with a table of runs per id) in launch 1, the sums of runs of
// two tokens or more (eg_runs) in the launch of the windows, then
//   eg_dot_kernel     -- each train token's row against its run's sum or its id's only val row
//                        (with a gradient: in launch 4, eg_combine_dot_kernel).
//   eg_dot_sum_kernel -- the parts of a train row added.
// Either alone, or both in shared launches.  Measured on MI355X (GPT-2 wte, 16 + 4 rows of 1024
// tokens, d = 768, bf16; 80 us before): lists 14.9 us, runs and windows 23.0 (102 MB written and
// read: the rate of a copy), combine and dots 7.5 + 3.9; a padded batch of 65536 train tokens with
// one id on 59k of them and 4096 val tokens likewise, d = 256: lists 57, windows 38, combine
// and dots 48 + 4.7 (1870 before).

#include <algorithm>

#include "gs_common.h"

namespace gs {
namespace {

constexpr int EG_CHUNK = 2048;                  // keys per sort workgroup
constexpr int EG_SORT_THREADS = 1024;
constexpr int EG_KPT = EG_CHUNK / EG_SORT_THREADS;  // keys per thread (2)
constexpr int EG_WIN = 8;                       // list places per window (one wave)
constexpr int EG_BATCH = 8;                     // rows of a window loaded together
constexpr int EG_THREADS = 256;                 // window / zero / combine workgroups
constexpr unsigned long long EG_NONE = ~0ull;   // key of an out-of-range id (sorts last)

__device__ __forceinline__ int64_t key_id(unsigned long long k) {
  return static_cast<int64_t>(k >> 32);
}
__device__ __forceinline__ int64_t key_tok(unsigned long long k) {
  return static_cast<int64_t>(k & 0xffffffffull);
}

// Physical row of token q of a row set (tokens numbered in row order): the set is contiguous but
// for the samples it skips, so one compare, not a division by the row length.
struct EgRows {
  int64_t M, off, cut, skip;   // tokens; row of token 0; first token past the skip; rows skipped
  __device__ int64_t operator()(int64_t q) const { return q + off + (q >= cut ? skip : 0); }
};
EgRows eg_rows(const RowMap& m) {
  const int64_t M = m.total();
  return EgRows{M, m.seg_offset * m.seglen, m.skip_at >= m.nseg ? M : m.skip_at * m.seglen,
                m.skip_n * m.seglen};
}

// An id's order in the token list.  Bucketed (shift >= 0): the list is ordered by (id % nb, id /
// nb) for nb = 2^nbits buckets, whose number `(id % nb) << shift | id / nb` takes the id's place
// in the keys; presence bits lie in whole words per bucket.  Otherwise (shift < 0): by the id.
struct EgOrder {
  int shift, nbits;
  __device__ int64_t of(int64_t v) const {
    return shift < 0 ? v : (v & ((int64_t{1} << nbits) - 1)) << shift | v >> nbits;
  }
  __device__ int64_t id(int64_t o) const {
    return shift < 0 ? o : (o & ((int64_t{1} << shift) - 1)) << nbits | o >> shift;
  }
  __host__ __device__ int64_t bucket_words() const { return ((int64_t{1} << shift) + 31) / 32; }
  __device__ bool present(const uint32_t* __restrict__ bits, int64_t v) const {
    if (shift < 0) return (bits[v >> 5] >> (v & 31)) & 1u;
    const int64_t b = v & ((int64_t{1} << nbits) - 1), l = v >> nbits;
    return (bits[b * bucket_words() + (l >> 5)] >> (l & 31)) & 1u;
  }
};

// The token list of one row set and what is made from it.
struct EgList {
  EgRows rows;
  EgOrder order;
  int64_t chunks, windows;        // entries of cnt; windows of the list at its full length
  unsigned long long* ck;         // the sorted chunks (not bucketed)
  unsigned long long* sk;         // the list: order << 32 | token
  int32_t* cnt;                   // in-range tokens, per chunk (bucketed: one number)
  uint32_t* present;              // presence bits of the ids, or null
  uint2* table;                   // null, or per id (in list order): its run's first place, length
  float* part;                    // [windows][2][d] sums of runs that cross windows, or null
};

// Lane l's value of v, as a wave-uniform value (l a compile-time or uniform lane index).
__device__ __forceinline__ unsigned long long readlane_u64(unsigned long long v, int l) {
  const unsigned lo = static_cast<unsigned>(
      __builtin_amdgcn_readlane(static_cast<int>(v & 0xffffffffull), l));
  const unsigned hi = static_cast<unsigned>(__builtin_amdgcn_readlane(static_cast<int>(v >> 32), l));
  return (static_cast<unsigned long long>(hi) << 32) | lo;
}

__device__ __forceinline__ int64_t readlane_i64(int64_t v, int l) {
  return static_cast<int64_t>(readlane_u64(static_cast<unsigned long long>(v), l));
}

__device__ __forceinline__ unsigned long long shfl_xor_u64(unsigned long long v, int m) {
  const int lo = __shfl_xor(static_cast<int>(v & 0xffffffffull), m, 64);
  const int hi = __shfl_xor(static_cast<int>(v >> 32), m, 64);
  return (static_cast<unsigned long long>(static_cast<unsigned>(hi)) << 32) |
         static_cast<unsigned>(lo);
}

// Sort keys of chunk c: (id << 11 | index within the chunk) as 32 bits while every id is
// below 2^20, else (id << 32 | token index) as 64 bits; an out-of-range id (and the tail past
// M) is the largest key.  Both orders are (id, token index) within a chunk.
template <class K>
struct EgKey;
template <>
struct EgKey<uint32_t> {
  static constexpr uint32_t NONE = ~0u;
  __device__ static uint32_t make(int64_t id, int64_t q, int64_t q0) {
    return (static_cast<uint32_t>(id) << 11) | static_cast<uint32_t>(q - q0);
  }
  __device__ static int64_t id(uint32_t k) { return k >> 11; }
  __device__ static int64_t tok(uint32_t k, int64_t q0) { return q0 + (k & 2047u); }
  // keys of another chunk that precede (id, q): ids below `id` (chunk after q's), or ids up
  // to `id` (chunk before q's) -- the count of keys below the returned bound
  __device__ static uint32_t bound(int64_t id, bool earlier_chunk) {
    return earlier_chunk ? ((static_cast<uint32_t>(id) + 1u) << 11)
                         : (static_cast<uint32_t>(id) << 11);
  }
};
template <>
struct EgKey<unsigned long long> {
  static constexpr unsigned long long NONE = ~0ull;
  __device__ static unsigned long long make(int64_t id, int64_t q, int64_t) {
    return (static_cast<unsigned long long>(id) << 32) | static_cast<unsigned long long>(q);
  }
  __device__ static int64_t id(unsigned long long k) { return static_cast<int64_t>(k >> 32); }
  __device__ static int64_t tok(unsigned long long k, int64_t) {
    return static_cast<int64_t>(k & 0xffffffffull);
  }
  __device__ static unsigned long long bound(int64_t id, bool earlier_chunk) {
    return earlier_chunk ? (static_cast<unsigned long long>(id + 1) << 32)
                         : (static_cast<unsigned long long>(id) << 32);
  }
};
constexpr int64_t EG_KEY32_VOCAB = int64_t(1) << 20;

__device__ __forceinline__ uint32_t shfl_xor_key(uint32_t v, int m) {
  return static_cast<uint32_t>(__shfl_xor(static_cast<int>(v), m, 64));
}
__device__ __forceinline__ unsigned long long shfl_xor_key(unsigned long long v, int m) {
  return shfl_xor_u64(v, m);
}

// Chunk c (tokens [c * EG_CHUNK, ...)): its keys sorted ascending into ck[c][0, EG_CHUNK),
// the number of in-range keys into cnt[c]; the workgroups also clear the presence bitmap.
// Key u of thread t is element t + 1024 u of the chunk: compare-exchange partners at distance
// j = 1024 are in the same thread, at j < 64 in the same wave (lane shuffles), the others go
// through LDS; sixteen waves per workgroup hide each other's shuffle and LDS latency.
template <class K>
__global__ void __launch_bounds__(EG_SORT_THREADS) eg_sort_kernel(
    const int64_t* __restrict__ ids, EgRows tr, int64_t vocab, K* __restrict__ ck,
    int32_t* __restrict__ cnt, uint32_t* __restrict__ present, int64_t present_words) {
  __shared__ K xs[EG_CHUNK];
  __shared__ int32_t wcount[EG_SORT_THREADS / 64];
  const int t = threadIdx.x, lane = t & 63;
  const int64_t M = tr.M;
  const int64_t q0 = static_cast<int64_t>(blockIdx.x) * EG_CHUNK;
  for (int64_t w = static_cast<int64_t>(blockIdx.x) * EG_SORT_THREADS + t; w < present_words;
       w += static_cast<int64_t>(gridDim.x) * EG_SORT_THREADS)
    present[w] = 0u;
  K key[EG_KPT];
  int valid = 0;
#pragma unroll
  for (int u = 0; u < EG_KPT; ++u) {
    const int64_t q = q0 + t + EG_SORT_THREADS * u;
    K k = EgKey<K>::NONE;
    if (q < M) {
      const int64_t id = ids[tr(q)];
      if (id >= 0 && id < vocab) {
        k = EgKey<K>::make(id, q, q0);
        ++valid;
      }
    }
    key[u] = k;
  }
  for (int k = 2; k <= EG_CHUNK; k <<= 1) {
    for (int j = k >> 1; j > 0; j >>= 1) {
      if (j >= EG_SORT_THREADS) {
        const int uj = j / EG_SORT_THREADS;
#pragma unroll
        for (int u = 0; u < EG_KPT; ++u) {
          if (u & uj) continue;
          const int i = t + EG_SORT_THREADS * u;
          const bool asc = (i & k) == 0;
          const K a = key[u], b = key[u | uj];
          const K lo = a < b ? a : b, hi = a < b ? b : a;
          key[u] = asc ? lo : hi;
          key[u | uj] = asc ? hi : lo;
        }
        continue;
      }
      K other[EG_KPT];
      if (j >= 64) {
        __syncthreads();   // earlier readers of xs are done
#pragma unroll
        for (int u = 0; u < EG_KPT; ++u) xs[t + EG_SORT_THREADS * u] = key[u];
        __syncthreads();
#pragma unroll
        for (int u = 0; u < EG_KPT; ++u) other[u] = xs[(t ^ j) + EG_SORT_THREADS * u];
      } else {
#pragma unroll
        for (int u = 0; u < EG_KPT; ++u) other[u] = shfl_xor_key(key[u], j);
      }
#pragma unroll
      for (int u = 0; u < EG_KPT; ++u) {
        const int i = t + EG_SORT_THREADS * u;
        const bool asc = (i & k) == 0, lower = (i & j) == 0;
        const K a = key[u], b = other[u];
        // the lower element keeps the minimum when ascending, the upper one the maximum
        key[u] = (lower == asc) ? (a < b ? a : b) : (a < b ? b : a);
      }
    }
  }
  K* out = ck + static_cast<int64_t>(blockIdx.x) * EG_CHUNK;
#pragma unroll
  for (int u = 0; u < EG_KPT; ++u) out[t + EG_SORT_THREADS * u] = key[u];
  // in-range keys of the chunk: a fixed-order integer sum
  for (int off = 32; off > 0; off >>= 1) valid += __shfl_xor(valid, off, 64);
  if (lane == 0) wcount[t >> 6] = valid;
  __syncthreads();
  if (t == 0) {
    int s = 0;
    for (int w = 0; w < EG_SORT_THREADS / 64; ++w) s += wcount[w];
    cnt[blockIdx.x] = s;
  }
}

// sk[place] = (id << 32 | token index), place = the key's index in its chunk + the keys of
// every other chunk that precede it; present[id] set.  One thread per chunk slot, a
// workgroup per 256 consecutive slots of one chunk (slots holding the largest key do
// nothing).  The keys of other chunks that precede a key depend only on its id, so only the
// first slot of each id within the workgroup (its run head) needs them, and the slots after
// it take the head's count from LDS: an id that fills the chunk is searched for once per
// workgroup, not once per token.  The (run head, other chunk) binary searches are spread over
// all the workgroup's threads, eight per thread advancing together so their loads are in
// flight at once; each adds its count to the head's total (integer adds: any order gives the
// same total).  With SAMP (32-bit keys, at most EG_SAMP_CHUNKS chunks) the workgroup first
// copies every EG_SAMP-th key of every chunk into LDS; a search then narrows the range to
// EG_SAMP - 1 keys among the samples in LDS and finishes over global memory in 5 steps
// instead of 12 (the global loads, each a trip to L2, are what the searches wait on).
constexpr int EG_SAMP = 32, EG_NSAMP = EG_CHUNK / EG_SAMP;  // 64 samples per chunk
constexpr int64_t EG_SAMP_CHUNKS = 128;                      // 32 KiB of samples at most

template <class K, bool SAMP>
__global__ void __launch_bounds__(EG_THREADS) eg_merge_kernel(
    const K* __restrict__ ck, int64_t chunks, unsigned long long* __restrict__ sk,
    uint32_t* __restrict__ present) {
  // STEPS halvings take an interval of 2^(STEPS - 1) = EG_CHUNK slots down to empty;
  // sampled: SSTEPS over the EG_NSAMP samples (EG_NSAMP + 1 outcomes), then GSTEPS over an
  // interval of EG_SAMP - 1 keys
  constexpr int G = 8, STEPS = 12, SSTEPS = 7, GSTEPS = 5;
  static_assert((1 << (STEPS - 1)) == EG_CHUNK, "search steps");
  static_assert((1 << (SSTEPS - 1)) == EG_NSAMP && (1 << GSTEPS) == EG_SAMP, "sampled steps");
  static_assert(!SAMP || sizeof(K) == 4, "samples of 32-bit keys");
  extern __shared__ __attribute__((aligned(16))) unsigned char eg_samples[];
  static_assert(EG_CHUNK % EG_THREADS == 0, "a merge workgroup stays inside one chunk");
  __shared__ int64_t kid[EG_THREADS];  // ids of the workgroup's slots (-1: none)
  __shared__ int before[EG_THREADS];   // at run heads: keys of other chunks preceding (< 2^31)
  __shared__ int hslot[EG_THREADS];    // the run heads' slots, in slot order
  __shared__ K hkey[EG_THREADS];       // and their keys
  __shared__ int wheads[EG_THREADS / 64];
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  const int64_t s = static_cast<int64_t>(blockIdx.x) * EG_THREADS + t;
  const int64_t c = static_cast<int64_t>(blockIdx.x) * EG_THREADS / EG_CHUNK, q0 = c * EG_CHUNK;
  const K k = ck[s];
  const bool valid = k != EgKey<K>::NONE;
  const int64_t id = valid ? EgKey<K>::id(k) : -1;
  kid[t] = id;
  before[t] = 0;
  const K* samp = reinterpret_cast<const K*>(eg_samples);
  if constexpr (SAMP) {
    K* w = reinterpret_cast<K*>(eg_samples);
    for (int64_t x = t; x < chunks * EG_NSAMP; x += EG_THREADS)
      w[x] = ck[(x / EG_NSAMP) * EG_CHUNK + (x % EG_NSAMP) * EG_SAMP];
  }
  __syncthreads();
  const bool head = valid && (t == 0 || kid[t - 1] != id);
  const unsigned long long hb = __ballot(head);
  if (lane == 0) wheads[wv] = __popcll(hb);
  __syncthreads();
  int hbase = 0, nh = 0;
#pragma unroll
  for (int v = 0; v < EG_THREADS / 64; ++v) {
    const int x = wheads[v];
    hbase += v < wv ? x : 0;
    nh += x;
  }
  if (head) {
    const int h = hbase + __popcll(hb & ((1ull << lane) - 1ull));
    hslot[h] = t;
    hkey[h] = k;
  }
  __syncthreads();
  // pair p = (head p / chunks, chunk p % chunks); thread t takes pairs t + EG_THREADS j
  // (fewer than 2^28 pairs: chunks < 2^20, as the entry point takes fewer than 2^31 tokens)
  const unsigned nc = static_cast<unsigned>(chunks), cc = static_cast<unsigned>(c);
  const unsigned pairs = static_cast<unsigned>(nh) * nc;
  for (unsigned p0 = t; p0 < pairs; p0 += G * EG_THREADS) {
    int lo[G], hi[G], hh[G];
    K bnd[G];
    int64_t oo[G];
#pragma unroll
    for (int u = 0; u < G; ++u) {
      const unsigned p = p0 + u * EG_THREADS;
      const unsigned h = p < pairs ? p / nc : 0u;
      const unsigned o = p < pairs ? p - h * nc : cc;
      hh[u] = static_cast<int>(h);
      oo[u] = o;
      const K hk = hkey[h];
      // 64-bit keys hold the token index: the plain order of keys; 32-bit keys compare ids
      // only across chunks (every token of an earlier chunk precedes, of a later one follows)
      bnd[u] = sizeof(K) == 8 ? hk : EgKey<K>::bound(EgKey<K>::id(hk), o < cc);
      lo[u] = 0;
      hi[u] = o != cc ? (SAMP ? EG_NSAMP : EG_CHUNK) : 0;
    }
    if constexpr (SAMP) {
      // samples below the bound: s of them means keys [0, EG_SAMP (s - 1)] are below it and
      // the keys from EG_SAMP s on are not, so the count lies in (EG_SAMP (s - 1), EG_SAMP s]
#pragma unroll
      for (int step = 0; step < SSTEPS; ++step) {
#pragma unroll
        for (int u = 0; u < G; ++u) {
          if (lo[u] >= hi[u]) continue;
          const int mid = (lo[u] + hi[u]) >> 1;
          if (samp[oo[u] * EG_NSAMP + mid] < bnd[u]) lo[u] = mid + 1; else hi[u] = mid;
        }
      }
#pragma unroll
      for (int u = 0; u < G; ++u) {
        const int sb = lo[u];
        lo[u] = sb == 0 ? 0 : (sb - 1) * EG_SAMP + 1;
        hi[u] = sb * EG_SAMP;
      }
    }
#pragma unroll
    for (int step = 0; step < (SAMP ? GSTEPS : STEPS); ++step) {
#pragma unroll
      for (int u = 0; u < G; ++u) {
        if (lo[u] >= hi[u]) continue;
        const int mid = (lo[u] + hi[u]) >> 1;
        if (ck[oo[u] * EG_CHUNK + mid] < bnd[u]) lo[u] = mid + 1; else hi[u] = mid;
      }
    }
#pragma unroll
    for (int u = 0; u < G; ++u)
      if (lo[u] != 0) atomicAdd(&before[hslot[hh[u]]], lo[u]);
  }
  __syncthreads();
  if (!valid) return;
  // the run head of this slot's id in the workgroup: the first slot with the id (ids sorted)
  int lo = 0, hi = t;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (kid[mid] < id) lo = mid + 1; else hi = mid;
  }
  const int64_t place = (s - q0) + before[lo];
  sk[place] = (static_cast<unsigned long long>(id) << 32) |
              static_cast<unsigned long long>(EgKey<K>::tok(k, q0));
  // Presence bits: the workgroup's first slot of each bitmap word ORs the bits of the ids
  // that follow it in that word (the slots are in id order), so a word takes one atomic per
  // workgroup, not one per id (position ids put a chunk's 1024 ids in 32 words).
  const int64_t word = id >> 5;
  if (t == 0 || (kid[t - 1] >> 5) != word) {
    uint32_t bits = 0;
    bool more = true;
    for (int u0 = t; more && u0 < EG_THREADS; u0 += 8) {   // 8 independent LDS reads a round
      int64_t v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = u0 + j < EG_THREADS ? kid[u0 + j] : -1;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        more = more && v[j] >= 0 && (v[j] >> 5) == word;
        if (more) bits |= 1u << (v[j] & 31);
      }
    }
    atomicOr(present + word, bits);
  }
}

// The token lists of one or two row sets (lists a and c, of one order) in one launch: bucket b of a
// list holds the ids congruent to b modulo the number of buckets (256, or 1024 beyond 131072 ids),
// and its workgroup reads every id of the set.
// The tokens of lower buckets, counted in passing, are where the bucket's part of the list
// begins, so no workgroup waits for another; taking ids by remainder spreads the frequent low ids
// of a real vocabulary over the buckets.  Each of the 16 (8) waves takes a contiguous share of the
// tokens and keeps the bucket's in LDS (a wave in whose share the bucket has more than
// EG_BUCKET_KEEP, a padded batch, reads its ids a second time instead).  Counts per (wave, id) in
// LDS, where tokens of one id among 64 are found by a ballot per bit of the id, become places by
// a scan over (id, wave); the keys (order << 32 | token) are written in the order (bucket, id,
// token).  Also writes the bucket's presence bits and the length of the list (cnt[0], by the last
// bucket).  Bound by the latency of its two or three trips to L2 for small batches and by the
// 256-fold reading of the ids for large ones.  Measured on MI355X against the sort and merge below
// (whole gradient call, us): 16384 tokens of 50257 ids 53.9 -> 35.2 (11 in this kernel, 29 in
// those two), with 90% of them one id 70.8 -> 53.9; 65536 tokens 101 -> 52.7, 90% one id 125 ->
// 108; 131072 tokens 225 -> 86, 90% one id 240 -> 177; 192 tokens 40 -> 27.
constexpr int EG_BUCKET_SHIFT = 9, EG_BUCKET_KEEP = 384, EG_SHARE_BITS = 13;
constexpr int64_t EG_BUCKET_TOKENS = int64_t{16} << EG_SHARE_BITS;
template <int NW>
__global__ void __launch_bounds__(64 * NW, 8) eg_bucket_kernel(
    const int64_t* __restrict__ ids, EgList a, EgList c, int64_t vocab) {
  constexpr int U = 8, SHARE_BITS = EG_SHARE_BITS;
  static_assert(64 * NW >= 1 << EG_BUCKET_SHIFT, "a thread for every id of a bucket");
  extern __shared__ int eg_counts[];   // [NW][R]
  __shared__ uint32_t eg_kept[NW][EG_BUCKET_KEEP];   // id of the bucket << SHARE_BITS | place
  __shared__ int wbase[NW], wtot[NW];
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  const EgOrder order = a.order;
  const int nb = 1 << order.nbits, R = 1 << order.shift;
  const EgList& list = static_cast<int>(blockIdx.x) < nb ? a : c;
  const int b = blockIdx.x & (nb - 1);
  const int M = static_cast<int>(list.rows.M);
  const int share = ((M + NW - 1) / NW + 63) & ~63;
  const int q_begin = std::min(M, wv * share), q_end = std::min(M, q_begin + share);
  const unsigned nv = static_cast<unsigned>(vocab);
  int* const mine = eg_counts + wv * R;
  uint32_t* const kept = eg_kept[wv];
  for (int x = lane; x < R; x += 64) mine[x] = 0;
  // f(v, q) for the wave's tokens, 64 at a time: v is the id of the lane's token q, or a number
  // past the vocabulary.  The loads of the next U groups are in flight meanwhile.
  const auto scan = [&](auto&& f) {
    int64_t next[U];
    const auto load = [&](int q) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int x = q + 64 * u + lane;
        next[u] = x < q_end ? ids[list.rows(x)] : -1;
      }
    };
    load(q_begin);
    for (int q = q_begin; q < q_end; q += 64 * U) {
      unsigned v[U];
#pragma unroll
      for (int u = 0; u < U; ++u)
        v[u] = next[u] >= 0 && next[u] < vocab ? static_cast<unsigned>(next[u]) : ~0u;
      load(q + 64 * U);
#pragma unroll
      for (int u = 0; u < U; ++u) f(v[u], q + 64 * u + lane);
    }
  };
  // The lanes of `in` whose token has this lane's id of the bucket.
  const auto same_id = [&](unsigned long long in, int lid) {
    const int one = __builtin_amdgcn_readlane(lid, __builtin_ctzll(in));
    if ((__ballot(lid == one) & in) == in) return in;
    for (int bit = 0; bit < order.shift; ++bit) {
      const unsigned long long set = __ballot((lid >> bit) & 1);
      in &= ((lid >> bit) & 1) ? set : ~set;
    }
    return in;
  };
  const auto count = [&](bool hit, int lid) {
    const unsigned long long same = same_id(__ballot(hit), lid);
    if (hit && __builtin_ctzll(same) == lane) atomicAdd(mine + lid, __popcll(same));
  };
  int below = 0, n = 0;
  scan([&](unsigned v, int q) {
    below += __popcll(__ballot(v < nv && static_cast<int>(v & (nb - 1)) < b));
    const bool hit = v < nv && static_cast<int>(v & (nb - 1)) == b;
    const unsigned long long hits = __ballot(hit);
    if (hits == 0) return;
    const int lid = static_cast<int>(v >> order.nbits), n0 = n;
    n += __popcll(hits);
    if (n <= EG_BUCKET_KEEP) {
      if (hit)
        kept[n0 + __popcll(hits & ((1ull << lane) - 1ull))] =
            static_cast<uint32_t>(lid) << SHARE_BITS | static_cast<uint32_t>(q - q_begin);
    } else {
      if (n0 <= EG_BUCKET_KEEP)   // count what was kept, once
        for (int x = lane; x - lane < n0; x += 64)
          count(x < n0, x < n0 ? static_cast<int>(kept[x] >> SHARE_BITS) : 0);
      count(hit, lid);
    }
  });
  if (n <= EG_BUCKET_KEEP)
    for (int x = lane; x - lane < n; x += 64)
      count(x < n, x < n ? static_cast<int>(kept[x] >> SHARE_BITS) : 0);
  if (lane == 0) wbase[wv] = below;
  __syncthreads();
  // Counts to places: thread t owns id t of the bucket.
  int total = 0;
  if (t < R)
    for (int w = 0; w < NW; ++w) total += eg_counts[w * R + t];
  int incl = total;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int x = __shfl_up(incl, off, 64);
    if (lane >= off) incl += x;
  }
  if (lane == 63) wtot[wv] = incl;
  __syncthreads();
  int place = incl - total, all = 0;
  for (int w = 0; w < NW; ++w) {
    place += wbase[w] + (w < wv ? wtot[w] : 0);
    all += wbase[w] + wtot[w];
  }
  if (b == nb - 1 && t == 0) list.cnt[0] = all;
  const unsigned long long present = __ballot(total > 0);
  const int words = static_cast<int>(order.bucket_words());
  if (list.present != nullptr && (lane & 31) == 0 && (t >> 5) < words)
    list.present[b * words + (t >> 5)] = static_cast<uint32_t>(present >> lane);
  if (list.table != nullptr && t < R)
    list.table[(b << order.shift) + t] =
        make_uint2(static_cast<unsigned>(place), static_cast<unsigned>(total));
  if (t < R)
    for (int w = 0; w < NW; ++w) {
      const int x = eg_counts[w * R + t];
      eg_counts[w * R + t] = place;
      place += x;
    }
  __syncthreads();
  const uint32_t o = static_cast<uint32_t>(b) << order.shift;
  const auto write = [&](bool hit, int lid, int q) {
    const unsigned long long same = same_id(__ballot(hit), lid);
    const int lead = hit ? __builtin_ctzll(same) : lane;
    int first = 0;
    if (hit && lead == lane) first = atomicAdd(mine + lid, __popcll(same));
    first = __shfl(first, lead, 64);
    if (hit)
      list.sk[first + __popcll(same & ((1ull << lane) - 1ull))] =
          static_cast<unsigned long long>(o | static_cast<uint32_t>(lid)) << 32 |
          static_cast<unsigned long long>(q);
  };
  if (n <= EG_BUCKET_KEEP) {
    for (int x = lane; x - lane < n; x += 64) {
      const uint32_t k = x < n ? kept[x] : 0u;
      write(x < n, static_cast<int>(k >> SHARE_BITS),
            q_begin + static_cast<int>(k & ((1u << SHARE_BITS) - 1u)));
    }
  } else {
    scan([&](unsigned v, int q) {
      const bool hit = v < nv && static_cast<int>(v & (nb - 1)) == b;
      if (__ballot(hit) != 0) write(hit, hit ? static_cast<int>(v >> order.nbits) : 0, q);
    });
  }
}

// Sum of cnt[0, chunks): the number of in-range keys, the length of the sorted list.
__device__ __forceinline__ int64_t list_length(const int32_t* __restrict__ cnt, int64_t chunks) {
  const int lane = threadIdx.x & 63;
  int n = 0;   // below 2^31 (checked by the entry point)
  for (int64_t c = lane; c < chunks; c += 64) n += cnt[c];
  for (int off = 32; off > 0; off >>= 1) n += __shfl_xor(n, off, 64);
  return n;
}

template <class E>
struct EgVec {
  static constexpr int VE = 16 / sizeof(E);  // elements per 16-byte chunk
  union U {
    uint4 u;
    E e[VE];
  };
};

// Loads the VE elements at f0 of a row (zeros past d); whole 16 bytes when `full`.
template <class E>
__device__ __forceinline__ uint4 eg_load(const E* __restrict__ row, int64_t f0, int64_t d,
                                         bool full) {
  typename EgVec<E>::U x;
  if (full) {
    x.u = *reinterpret_cast<const uint4*>(row + f0);
  } else {
#pragma unroll
    for (int i = 0; i < EgVec<E>::VE; ++i) x.e[i] = f0 + i < d ? row[f0 + i] : E(0);
  }
  return x.u;
}

// Writes scale * acc (+ the old row when accumulating) at f0 of an output row.
template <class GE, int VE>
__device__ __forceinline__ void eg_store(GE* __restrict__ out, int64_t f0, int64_t d,
                                         const float (&acc)[VE], float scale, int accumulate,
                                         bool full) {
  constexpr int NV = VE * static_cast<int>(sizeof(GE)) / 16;  // whole 16-byte vectors
  if (NV > 0 && full) {
    union { uint4 u[NV > 0 ? NV : 1]; GE e[VE]; } o;
    if (accumulate) {
#pragma unroll
      for (int c = 0; c < NV; ++c) o.u[c] = reinterpret_cast<const uint4*>(out + f0)[c];
    }
#pragma unroll
    for (int i = 0; i < VE; ++i) {
      float x = scale * acc[i];
      if (accumulate) x += to_f32<GE>(o.e[i]);
      o.e[i] = from_f32<GE>(x);
    }
#pragma unroll
    for (int c = 0; c < NV; ++c) reinterpret_cast<uint4*>(out + f0)[c] = o.u[c];
  } else {
#pragma unroll
    for (int i = 0; i < VE; ++i) {
      if (f0 + i >= d) break;
      float x = scale * acc[i];
      if (accumulate) x += to_f32<GE>(out[f0 + i]);
      out[f0 + i] = from_f32<GE>(x);
    }
  }
}

// Waves [0, windows): window w = list places [w EG_WIN, (w + 1) EG_WIN).  Lanes own 16-byte
// chunks of the feature row (several passes when d > 64 VE); per pass a lane loads its chunk
// of every row of the window (all in flight), then walks the window's runs in place order,
// summing in fp32.  A run wholly inside the window writes its row; the run holding the
// window's first place, when it began in an earlier window, goes to part[w][0], and the run
// holding the last place, when it continues into the next window (and began in this one),
// to part[w][1] (fp32, [windows][2][d]).
// Waves [windows, windows + zero_waves), overwrite mode: 16 table rows each; rows whose id is
// absent from the list are written as zeros.
template <class E, class GE>
__device__ __forceinline__ void eg_window(const E* __restrict__ G, const EgList& list, int64_t d,
                                          int64_t vocab, int64_t block, float scale,
                                          int accumulate, int vec, GE* __restrict__ grad) {
  constexpr int VE = EgVec<E>::VE;
  const unsigned long long* __restrict__ sk = list.sk;
  float* __restrict__ part = list.part;
  const EgOrder order = list.order;
  const int64_t windows = list.windows;
  const int lane = threadIdx.x & 63;
  const int64_t w = block * (EG_THREADS / 64) + (threadIdx.x >> 6);
  if (w >= windows) {
    // absent rows, overwrite mode only (the last workgroup's surplus waves land here in
    // both modes): 16 rows, lanes over chunks
    const int64_t v0 = (w - windows) * 16;
    if (accumulate || v0 >= vocab) return;
    const unsigned long long bits =
        __ballot(lane < 16 && v0 + lane < vocab && order.present(list.present, v0 + lane));
    for (int r = 0; r < 16 && v0 + r < vocab; ++r) {
      if ((bits >> r) & 1u) continue;
      GE* out = grad + (v0 + r) * d;
      for (int64_t f0 = static_cast<int64_t>(lane) * VE; f0 < d; f0 += 64 * VE) {
        float z[VE];
#pragma unroll
        for (int i = 0; i < VE; ++i) z[i] = 0.f;
        eg_store<GE, VE>(out, f0, d, z, 0.f, 0, vec && f0 + VE <= d);
      }
    }
    return;
  }
  const int64_t n_list = list_length(list.cnt, list.chunks);
  const int64_t r0 = w * EG_WIN;
  if (r0 >= n_list) return;
  const int n = static_cast<int>(std::min<int64_t>(EG_WIN, n_list - r0));
  // lane i < n: the key at place r0 + i, its id and G row; read as wave-uniform values below
  const unsigned long long k = lane < n ? sk[r0 + lane] : EG_NONE;
  const int64_t my_id = key_id(k);
  const int64_t my_row = lane < n ? list.rows(key_tok(k)) : 0;
  const bool from_before = r0 > 0 && key_id(sk[r0 - 1]) == readlane_i64(my_id, 0);
  const bool into_next = r0 + n < n_list && key_id(sk[r0 + n]) == readlane_i64(my_id, n - 1);
  // two feature passes per round (lanes own chunks f0 and f0 + 64 VE); the window's rows in
  // batches, each batch's loads of both passes issued together, the sums carried across
  // batches
  for (int64_t fb = static_cast<int64_t>(lane) * VE; fb < d; fb += 128 * VE) {
    float acc[2][VE];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int e = 0; e < VE; ++e) acc[h][e] = 0.f;
    bool first_run = true;
#pragma unroll
    for (int b0 = 0; b0 < EG_WIN; b0 += EG_BATCH) {
      if (b0 >= n) break;   // wave-uniform
      uint4 x[2][EG_BATCH];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int64_t f0 = fb + h * 64 * VE;
        const bool full = vec && f0 + VE <= d;
#pragma unroll
        for (int i = 0; i < EG_BATCH; ++i)
          x[h][i] = b0 + i < n && f0 < d
                        ? eg_load<E>(G + readlane_i64(my_row, b0 + i) * d, f0, d, full)
                        : make_uint4(0u, 0u, 0u, 0u);
      }
#pragma unroll
      for (int i = 0; i < EG_BATCH; ++i) {
        const int p = b0 + i;
        if (p < n) {   // wave-uniform
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            typename EgVec<E>::U u;
            u.u = x[h][i];
#pragma unroll
            for (int e = 0; e < VE; ++e) acc[h][e] += to_f32<E>(u.e[e]);
          }
          const int64_t id_p = readlane_i64(my_id, p);
          const bool last_run = p == n - 1;
          const bool ends = last_run || (p + 1 < EG_WIN && readlane_i64(my_id, p + 1) != id_p);
          if (ends) {
            float* pp = nullptr;
            if (first_run && from_before)
              pp = part + (w * 2) * d;        // began in an earlier window
            else if (last_run && into_next)
              pp = part + (w * 2 + 1) * d;    // continues into the next window
#pragma unroll
            for (int h = 0; h < 2; ++h) {
              const int64_t f0 = fb + h * 64 * VE;
              if (f0 < d) {
                if (pp != nullptr) {
#pragma unroll
                  for (int e = 0; e < VE; ++e)
                    if (f0 + e < d) pp[f0 + e] = acc[h][e];
                } else {
                  eg_store<GE, VE>(grad + order.id(id_p) * d, f0, d, acc[h], scale, accumulate,
                                   vec && f0 + VE <= d);
                }
              }
#pragma unroll
              for (int e = 0; e < VE; ++e) acc[h][e] = 0.f;
            }
            first_run = false;
          }
        }
      }
    }
  }
}

// Run sums of a list with a table: the sum of every run of two tokens or more, in fp32, goes to row
// (first place) / 2 of S (the first places of two such runs differ by two or more).  Workgroup
// `block` looks at four places, one a wave.  A run of at most EG_SHORT tokens is summed in list
// order by the wave of its first place.  The workgroups that a longer run covers share its features,
// 64 bytes of a row each: 64 groups of threads take every 64th token, and their sums are added in a
// fixed order.  (90% of 4096 val tokens one id, d = 768, bf16: 56 us for a whole dot against 1.8 ms when
// the workgroup of the first place walked the run; of 8192, d = 1024, fp32, 54 against 6.9 ms.)
constexpr int EG_SHORT = 64;
template <class E>
struct EgRunsShared {
  static constexpr int W = 64 / sizeof(E), NG = EG_THREADS / 4;   // features; groups of threads
  float red[NG][W];
  float red2[EG_THREADS];
  int start[EG_THREADS / 64], count[EG_THREADS / 64];
};

template <class E>
__device__ __forceinline__ void eg_runs(const E* __restrict__ G, const EgList& list, int64_t d,
                                        int64_t block, int vec, EgRunsShared<E>& sh,
                                        float* __restrict__ S) {
  constexpr int VE = EgVec<E>::VE, B = 8, W = EgRunsShared<E>::W, NG = EgRunsShared<E>::NG;
  const unsigned long long* __restrict__ sk = list.sk;
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  const int64_t p = block * (EG_THREADS / 64) + wv;
  int start = 0, count = 0;
  if (p < list.cnt[0]) {
    const uint2 e = list.table[key_id(sk[p])];
    start = static_cast<int>(e.x);
    count = static_cast<int>(e.y);
  }
  if (lane == 0) {
    sh.start[wv] = start;
    sh.count[wv] = count;
  }
  if (count >= 2 && count <= EG_SHORT && p == start) {
    for (int64_t f_base = 0; f_base < d; f_base += 128 * VE) {   // every lane, for the rows below
      const int64_t fb = f_base + static_cast<int64_t>(lane) * VE;
      float acc[2][VE] = {};
      for (int r0 = 0; r0 < count; r0 += B) {
        const int n = std::min(B, count - r0);
        const int64_t my_row =
            (lane & (B - 1)) < n ? list.rows(key_tok(sk[start + r0 + (lane & (B - 1))])) : 0;
        uint4 x[2][B];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int64_t f0 = fb + h * 64 * VE;
#pragma unroll
          for (int i = 0; i < B; ++i)
            x[h][i] = i < n && f0 < d ? eg_load<E>(G + readlane_i64(my_row, i) * d, f0, d,
                                                   vec && f0 + VE <= d)
                                      : make_uint4(0u, 0u, 0u, 0u);
        }
#pragma unroll
        for (int i = 0; i < B; ++i)
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            typename EgVec<E>::U u;
            u.u = x[h][i];
#pragma unroll
            for (int e = 0; e < VE; ++e)
              if (i < n) acc[h][e] += to_f32<E>(u.e[e]);
          }
      }
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int64_t f0 = fb + h * 64 * VE;
        if (f0 < d)
          eg_store<float, VE>(S + (static_cast<int64_t>(start) >> 1) * d, f0, d, acc[h], 1.f, 0,
                              vec && f0 + VE <= d);
      }
    }
  }
  __syncthreads();
  for (int q = 0; q < EG_THREADS / 64; ++q) {
    const int len = sh.count[q], first = sh.start[q];
    // (the same for the whole workgroup, which may see the end of one run and another's start)
    if (len <= EG_SHORT || (q > 0 && sh.start[q - 1] == first && sh.count[q - 1] == len)) continue;
    const int b_lo = first / (EG_THREADS / 64), b_hi = (first + len - 1) / (EG_THREADS / 64);
    const int64_t step = static_cast<int64_t>(b_hi - b_lo + 1) * W;
    for (int64_t f0 = (block - b_lo) * W; f0 < d; f0 += step) {
      const int col = t & 3, g = t >> 2;
      const int64_t f = f0 + col * VE;
      float acc[VE] = {};
      if (f < d) {
        unsigned tok[B];   // tokens of the next rows, loaded ahead of them
        const auto tokens = [&](int r0) {
#pragma unroll
          for (int i = 0; i < B; ++i)
            tok[i] = r0 + i * NG < len ? static_cast<unsigned>(sk[first + r0 + i * NG]) : 0u;
        };
        tokens(g);
        for (int r0 = g; r0 < len; r0 += B * NG) {
          uint4 x[B];
#pragma unroll
          for (int i = 0; i < B; ++i)
            x[i] = r0 + i * NG < len
                       ? eg_load<E>(G + list.rows(tok[i]) * d, f, d, vec && f + VE <= d)
                       : make_uint4(0u, 0u, 0u, 0u);
          tokens(r0 + B * NG);
#pragma unroll
          for (int i = 0; i < B; ++i) {
            typename EgVec<E>::U u;
            u.u = x[i];
#pragma unroll
            for (int e = 0; e < VE; ++e)
              if (r0 + i * NG < len) acc[e] += to_f32<E>(u.e[e]);
          }
        }
      }
#pragma unroll
      for (int e = 0; e < VE; ++e) sh.red[g][col * VE + e] = acc[e];
      __syncthreads();
      constexpr int H = EG_THREADS / W, PER = NG / H;
      const int e = t % W, h = t / W;
      float a = sh.red[h * PER][e];
      for (int x = 1; x < PER; ++x) a += sh.red[h * PER + x][e];
      sh.red2[t] = a;
      __syncthreads();
      if (t < W && f0 + t < d) {
        for (int x = 1; x < H; ++x) a += sh.red2[x * W + t];
        S[(static_cast<int64_t>(first) >> 1) * d + f0 + t] = a;
      }
      __syncthreads();   // red is used again
    }
  }
}

// The first val_blocks workgroups: the run sums of the val list into S; the others: the train
// gradient's rows.
template <class E, class GE>
__global__ void __launch_bounds__(EG_THREADS) eg_window_kernel(
    const E* __restrict__ G, EgList val, EgList train, unsigned val_blocks, int64_t d,
    int64_t vocab, float scale, int accumulate, int vec, float* __restrict__ S,
    GE* __restrict__ grad) {
  __shared__ EgRunsShared<E> sh;
  if (blockIdx.x < val_blocks)
    eg_runs<E>(G, val, d, blockIdx.x, vec, sh, S);
  else
    eg_window<E, GE>(G, train, d, vocab, blockIdx.x - val_blocks, scale, accumulate, vec, grad);
}

// Workgroup b looks at windows [16 b, 16 b + 16), one wave each.  A window whose last run
// began in it and continues into the next window owns that run; its partials are part[w][1],
// part[w + 1][0], ..., part[w_end][0] (w_end: the window of the run's last place).
//  - At most EG_LIGHT partials: the owning wave sums them and writes the row.
//  - A run whose windows cover the whole range of fewer than EG_SPREAD other workgroups (at
//    most 48 partials): handed over in window order through LDS; the owner's workgroup splits
//    the partials into 16 contiguous shares summed by its 16 waves, combines the shares in
//    wave order and writes the row.
//  - A longer run: the workgroups whose whole range it covers (b_lo = w / 16 + 1 ..
//    b_hi = w_end / 16 - 1; such a workgroup owns no run) sum it, each a share of the
//    features over all the partials in a fixed order.  Every workgroup works alone: a run of
//    59k tokens is summed by hundreds of workgroups, and none waits for another.
constexpr int EG_COMBINE_WAVES = 16;
constexpr int EG_LIGHT = 8, EG_SPREAD = 2;

// Features [j sw, (j + 1) sw) of row `out` for a long run, sw = the row split evenly over the
// nb covering workgroups (whole float4s), but at least 16 features: 64-byte pieces of the
// partial rows (measured at GPT-2 width, d = 768, and a 59k-token run: 34 us with 48
// workgroups reading 64-byte pieces, 46 us with 192 reading 16-byte ones; a run covering few
// workgroups gives each a wide share in one pass).  In passes of at most 4096 features, a pass of
// `cols` float4 columns has ng = 1024 / cols groups of threads, group g summing partials g,
// g + ng, ... of its column in order; the ng group sums are combined in a fixed tree (sixteen
// at a time, then those results), and the row's features written.
template <class GE>
__device__ void eg_spread_sum(const float* __restrict__ part, int64_t ws, int64_t parts,
                              int64_t d, GE* __restrict__ out, int64_t j, int64_t nb, float scale,
                              int accumulate, float* __restrict__ red) {
  constexpr int NT = EG_COMBINE_WAVES * 64, B = 8, PASS = 4 * NT;
  const int t = threadIdx.x;
  const bool v4 = (d & 3) == 0;   // rows of whole float4s (part is 256-byte aligned)
  const int64_t sw = std::max<int64_t>(16, ((d + nb - 1) / nb + 3) & ~int64_t(3));
  const int64_t f_begin = j * sw, f_end = std::min(d, f_begin + sw);
  float* red2 = red + PASS;   // the tree's first level: at most 4096 + 256 floats
  for (int64_t fp = f_begin; fp < f_end; fp += PASS) {
    const int width = static_cast<int>(std::min<int64_t>(PASS, f_end - fp));
    const int cols = (width + 3) / 4, w4 = 4 * cols;
    const int ng = NT / cols;   // at least 1
    const int col = t % cols, g = t / cols;
    if (g < ng) {
      const int64_t f = fp + 4 * col;
      float a[4] = {0.f, 0.f, 0.f, 0.f};
      for (int64_t p0 = g; p0 < parts; p0 += static_cast<int64_t>(B) * ng) {
        float4 x[B];
#pragma unroll
        for (int u = 0; u < B; ++u) {
          const int64_t p = p0 + static_cast<int64_t>(u) * ng;
          x[u] = make_float4(0.f, 0.f, 0.f, 0.f);
          if (p < parts) {
            const float* src = part + ((ws + p) * 2 + (p == 0 ? 1 : 0)) * d + f;
            if (v4) {
              x[u] = *reinterpret_cast<const float4*>(src);
            } else {
              x[u].x = src[0];
              if (f + 1 < f_end) x[u].y = src[1];
              if (f + 2 < f_end) x[u].z = src[2];
              if (f + 3 < f_end) x[u].w = src[3];
            }
          }
        }
#pragma unroll
        for (int u = 0; u < B; ++u) {
          a[0] += x[u].x;
          a[1] += x[u].y;
          a[2] += x[u].z;
          a[3] += x[u].w;
        }
      }
      *reinterpret_cast<float4*>(red + g * w4 + 4 * col) = make_float4(a[0], a[1], a[2], a[3]);
    }
    __syncthreads();
    const int n1 = (ng + 15) / 16;
    for (int i = t; i < n1 * w4; i += NT) {
      const int h = i / w4, e = i - h * w4, g_end = std::min(ng, 16 * h + 16);
      float s = red[(16 * h) * w4 + e];
      for (int gg = 16 * h + 1; gg < g_end; ++gg) s += red[gg * w4 + e];
      red2[h * w4 + e] = s;
    }
    __syncthreads();
    for (int e = t; e < width; e += NT) {
      float s = red2[e];
      for (int h = 1; h < n1; ++h) s += red2[h * w4 + e];
      float x = scale * s;
      if (accumulate) x += to_f32<GE>(out[fp + e]);
      out[fp + e] = from_f32<GE>(x);
    }
    __syncthreads();   // red is reused by the next pass
  }
}

constexpr int EG_COMBINE_BLOCK = 1024;   // features per block
struct EgCombineShared {
  __attribute__((aligned(16))) float red[EG_COMBINE_WAVES][EG_COMBINE_BLOCK];
  int64_t run_w[EG_COMBINE_WAVES], run_end[EG_COMBINE_WAVES], run_row[EG_COMBINE_WAVES];
  int flags[EG_COMBINE_WAVES];
  int n_runs;
};

template <class GE>
__device__ __forceinline__ void eg_combine(const EgList& list, int64_t d, float scale,
                                           int accumulate, int64_t block, EgCombineShared& sh,
                                           GE* __restrict__ grad) {
  constexpr int NW = EG_COMBINE_WAVES, CB = EG_COMBINE_BLOCK;
  static_assert(NW * 64 == CB, "one feature of a block per thread");
  const unsigned long long* __restrict__ sk = list.sk;
  const float* __restrict__ part = list.part;
  const EgOrder order = list.order;
  const int64_t windows = list.windows;
  auto& red = sh.red;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int64_t n_list = list_length(list.cnt, list.chunks);
  {
    // A workgroup whose whole range of places lies inside one run that began before it and
    // continues after it (every thread decides alike): its share of that run if the run is
    // spread, else nothing (its windows own no run).
    constexpr int64_t SPAN = static_cast<int64_t>(NW) * EG_WIN;
    const int64_t r0 = block * SPAN;
    if (r0 > 0 && r0 + SPAN < n_list) {
      const int64_t id0 = key_id(sk[r0]);
      if (key_id(sk[r0 - 1]) == id0 && key_id(sk[r0 + SPAN]) == id0) {
        const unsigned long long k_lo = static_cast<unsigned long long>(id0) << 32;
        const unsigned long long k_hi = k_lo | 0xffffffffull;
        int64_t lo = 0, hi = r0 - 1;   // the run's first place
        while (lo < hi) {
          const int64_t mid = (lo + hi) >> 1;
          if (sk[mid] < k_lo) lo = mid + 1; else hi = mid;
        }
        const int64_t first = lo;
        lo = r0 + SPAN + 1;             // one past its last place
        hi = n_list;
        while (lo < hi) {
          const int64_t mid = (lo + hi) >> 1;
          if (sk[mid] <= k_hi) lo = mid + 1; else hi = mid;
        }
        const int64_t ws = first / EG_WIN, w_end = (lo - 1) / EG_WIN;
        const int64_t b_lo = ws / NW + 1, nb = w_end / NW - 1 - b_lo + 1;
        if (nb >= EG_SPREAD)
          eg_spread_sum<GE>(part, ws, w_end - ws + 1, d,
                            grad + order.id(id0) * d, block - b_lo, nb, scale, accumulate,
                            &red[0][0]);
        return;
      }
    }
  }
  if (threadIdx.x == 0) sh.n_runs = 0;
  __syncthreads();
  const int64_t w = block * NW + wid;
  bool found = false;
  int64_t id = 0, end = 0, row = 0;
  const int64_t r0 = w * EG_WIN;
  if (w < windows && r0 + EG_WIN < n_list) {   // a next window exists
    const int64_t r_last = r0 + EG_WIN - 1;
    id = key_id(sk[r_last]);
    // the last run continues, and began in this window (at r0 or after an id change)
    if (key_id(sk[r_last + 1]) == id &&
        !(key_id(sk[r0]) == id && r0 > 0 && key_id(sk[r0 - 1]) == id)) {
      // the run's end: the first place past r_last with a larger id -- among the next 64
      // places (one load per lane), else by binary search beyond them
      const int64_t r = r_last + 1 + lane;
      const unsigned long long past = __ballot(r >= n_list || key_id(sk[r]) != id);
      if (past != 0) {
        end = r_last + 1 + __builtin_ctzll(past);
      } else {
        int64_t lo = r_last + 65, hi = n_list;
        const unsigned long long bnd =
            (static_cast<unsigned long long>(id) << 32) | 0xffffffffull;
        while (lo < hi) {
          const int64_t mid = (lo + hi) >> 1;
          if (sk[mid] <= bnd) lo = mid + 1; else hi = mid;
        }
        end = lo;
      }
      row = order.id(id);
      // a spread run is left to the workgroups it covers
      const int64_t w_end = (end - 1) / EG_WIN;
      found = (w_end / NW - 1) - (w / NW + 1) + 1 < EG_SPREAD;
    }
  }
  // A run of at most EG_LIGHT partials is summed by the wave that found it; longer runs are
  // handed over in window order (wave v's run to slot = longer runs of waves below v) and
  // summed by the whole workgroup.
  const int64_t parts_found = found ? (end - 1) / EG_WIN - w + 1 : 0;
  if (found && parts_found <= EG_LIGHT) {
    GE* out = grad + row * d;
    for (int64_t f = static_cast<int64_t>(lane) * 4; f < d; f += 256) {
      float4 x[EG_LIGHT];
#pragma unroll
      for (int p = 0; p < EG_LIGHT; ++p) {
        x[p] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (p < parts_found) {
          const float* src = part + ((w + p) * 2 + (p == 0 ? 1 : 0)) * d + f;
          if ((d & 3) == 0) {
            x[p] = *reinterpret_cast<const float4*>(src);
          } else {
            x[p].x = src[0];
            if (f + 1 < d) x[p].y = src[1];
            if (f + 2 < d) x[p].z = src[2];
            if (f + 3 < d) x[p].w = src[3];
          }
        }
      }
      float t[4] = {x[0].x, x[0].y, x[0].z, x[0].w};
#pragma unroll
      for (int p = 1; p < EG_LIGHT; ++p) {
        if (p < parts_found) {
          t[0] += x[p].x;
          t[1] += x[p].y;
          t[2] += x[p].z;
          t[3] += x[p].w;
        }
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (f + e >= d) break;
        float v = scale * t[e];
        if (accumulate) v += to_f32<GE>(out[f + e]);
        out[f + e] = from_f32<GE>(v);
      }
    }
  }
  const bool heavy = found && parts_found > EG_LIGHT;
  if (lane == 0) sh.flags[wid] = heavy ? 1 : 0;
  __syncthreads();
  if (lane == 0 && heavy) {
    int slot = 0;
    for (int v = 0; v < wid; ++v) slot += sh.flags[v];
    sh.run_w[slot] = w;
    sh.run_end[slot] = end;
    sh.run_row[slot] = row;
    atomicAdd(&sh.n_runs, 1);
  }
  __syncthreads();
  const int runs = sh.n_runs;
  for (int r = 0; r < runs; ++r) {
    const int64_t ws = sh.run_w[r];
    const int64_t w_end = (sh.run_end[r] - 1) / EG_WIN;   // window of the run's last place
    const int64_t parts = w_end - ws + 1;   // part[ws][1], then part[ws + 1 .. w_end][0]
    const int64_t share = (parts + NW - 1) / NW;
    const int64_t p_begin = std::min<int64_t>(parts, wid * share);
    const int64_t p_end = std::min<int64_t>(parts, p_begin + share);
    GE* out = grad + sh.run_row[r] * d;
    const bool v4 = (d & 3) == 0;   // rows of whole float4s (part is 256-byte aligned)
    // feature blocks of CB = 4 x 256: lane l owns features 4 l + 256 j, j < 4, so a partial
    // row's block is one round of loads
    for (int64_t c0 = 0; c0 < d; c0 += CB) {
      float4 sum[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) sum[j] = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll 4
      for (int64_t p = p_begin; p < p_end; ++p) {
        const float* src = part + ((ws + p) * 2 + (p == 0 ? 1 : 0)) * d;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int64_t f = c0 + 256 * j + lane * 4;
          if (f >= d) continue;
          if (v4) {
            const float4 x = *reinterpret_cast<const float4*>(src + f);
            sum[j].x += x.x;
            sum[j].y += x.y;
            sum[j].z += x.z;
            sum[j].w += x.w;
          } else {
            sum[j].x += src[f];
            if (f + 1 < d) sum[j].y += src[f + 1];
            if (f + 2 < d) sum[j].z += src[f + 2];
            if (f + 3 < d) sum[j].w += src[f + 3];
          }
        }
      }
#pragma unroll
      for (int j = 0; j < 4; ++j)
        *reinterpret_cast<float4*>(&red[wid][256 * j + lane * 4]) = sum[j];
      __syncthreads();
      // the block's features, one per thread: shares added in wave order
      const int e = threadIdx.x;
      if (c0 + e < d) {
        float t = red[0][e];
        for (int v = 1; v < NW; ++v) t += red[v][e];
        float x = scale * t;
        if (accumulate) x += to_f32<GE>(out[c0 + e]);
        out[c0 + e] = from_f32<GE>(x);
      }
      __syncthreads();
    }
  }
}

// part[i * chunks + c] = sum over train row i's tokens in chunk c of <g_it, run sum of x_it>.  One
// lane looks up each token; the tokens whose id the val rows have are taken by the half-waves in
// turn, lanes over 16-byte feature chunks, all chunks of up to 1024 features (bf16) in flight.  A
// run of two tokens or more is read from S, a single one straight from that val token's row of G.
// (Letting a row's last workgroup add the parts in place of a launch: 15 us against 7 + 3.5, and 56
// against 15 + 4.5 for 64 chunks a row; the release to the other XCDs costs every workgroup.)
constexpr int EG_TOK = 32;   // tokens per unit of EG_THREADS threads
struct EgDotShared {
  float red[EG_THREADS / 64];
  int64_t rows[EG_TOK], src[EG_TOK];   // src: row of S, or -1 - row of G
  int hits;
};
// Thread `tid` of unit i * chunks + c; units past n_t * chunks only keep the barriers.
template <class E>
__device__ __forceinline__ void eg_dot(const int64_t* __restrict__ ids, const E* __restrict__ G,
                                       const EgRows& train, int64_t n_t, int64_t T,
                                       const EgList& val, int64_t d, int64_t vocab,
                                       const float* __restrict__ S, int vec, int64_t chunks,
                                       int64_t unit, int tid, EgDotShared& sh,
                                       float* __restrict__ part) {
  constexpr int VE = EgVec<E>::VE, P = 4;
  auto& rows = sh.rows;
  auto& src = sh.src;
  const int64_t i = unit / chunks, c = unit - i * chunks;
  if (tid < 64) {
    const int64_t t = c * EG_TOK + tid;
    const bool in = tid < EG_TOK && t < T && i < n_t;
    const int64_t row = in ? train(i * T + t) : 0;
    const int64_t id = in ? ids[row] : -1;
    const uint2 e = id >= 0 && id < vocab ? val.table[val.order.of(id)] : make_uint2(0u, 0u);
    const unsigned long long found = __ballot(e.y != 0);
    if (e.y != 0) {
      const int h = __popcll(found & ((1ull << tid) - 1ull));
      rows[h] = row;
      src[h] = e.y > 1 ? static_cast<int64_t>(e.x >> 1) : -1 - val.rows(key_tok(val.sk[e.x]));
    }
    if (tid == 0) sh.hits = __popcll(found);
  }
  __syncthreads();
  const int hl = tid & 31, n = sh.hits;
  float s = 0.f;
  for (int h = tid >> 5; h < n; h += EG_THREADS / 32) {
    const E* g = G + rows[h] * d;
    const int64_t sr = src[h];
    for (int64_t fb = static_cast<int64_t>(hl) * VE; fb < d; fb += P * 32 * VE) {
      typename EgVec<E>::U x[P];
#pragma unroll
      for (int p = 0; p < P; ++p) {
        const int64_t f = fb + p * 32 * VE;
        x[p].u = f < d ? eg_load<E>(g, f, d, vec && f + VE <= d) : make_uint4(0u, 0u, 0u, 0u);
      }
      if (sr >= 0) {
        const float* v = S + sr * d;
        float4 y[P][VE / 4];
#pragma unroll
        for (int p = 0; p < P; ++p) {
          const int64_t f = fb + p * 32 * VE;
#pragma unroll
          for (int e = 0; e < VE / 4; ++e)
            y[p][e] = f + 4 * e < d
                          ? __builtin_bit_cast(float4, eg_load<float>(v, f + 4 * e, d,
                                                                      vec && f + VE <= d))
                          : make_float4(0.f, 0.f, 0.f, 0.f);
        }
#pragma unroll
        for (int p = 0; p < P; ++p)
#pragma unroll
          for (int e = 0; e < VE / 4; ++e)
            s += to_f32<E>(x[p].e[4 * e]) * y[p][e].x + to_f32<E>(x[p].e[4 * e + 1]) * y[p][e].y +
                 to_f32<E>(x[p].e[4 * e + 2]) * y[p][e].z + to_f32<E>(x[p].e[4 * e + 3]) * y[p][e].w;
      } else {
        const E* v = G + (-1 - sr) * d;
        typename EgVec<E>::U y[P];
#pragma unroll
        for (int p = 0; p < P; ++p) {
          const int64_t f = fb + p * 32 * VE;
          y[p].u = f < d ? eg_load<E>(v, f, d, vec && f + VE <= d) : make_uint4(0u, 0u, 0u, 0u);
        }
#pragma unroll
        for (int p = 0; p < P; ++p)
#pragma unroll
          for (int e = 0; e < VE; ++e) s += to_f32<E>(x[p].e[e]) * to_f32<E>(y[p].e[e]);
      }
    }
  }
  s = wave_sum(s);
  if ((tid & 63) == 0) sh.red[tid >> 6] = s;
  __syncthreads();
  if (tid == 0 && i < n_t) {
    float tot = 0.f;
    for (int w = 0; w < EG_THREADS / 64; ++w) tot += sh.red[w];
    part[unit] = tot;
  }
}

// What the train tokens' dots read.
template <class E>
struct EgDots {
  const int64_t* ids;
  const E* G;
  EgRows train;
  int64_t n_t, T, vocab, chunks;
  const float* S;
  int vec;
  float* part;
};

template <class E>
__global__ void __launch_bounds__(EG_THREADS) eg_dot_kernel(EgDots<E> q, EgList val, int64_t d) {
  __shared__ EgDotShared sh;
  eg_dot<E>(q.ids, q.G, q.train, q.n_t, q.T, val, d, q.vocab, q.S, q.vec, q.chunks, blockIdx.x,
            threadIdx.x, sh, q.part);
}

template <class GE>
__global__ void __launch_bounds__(EG_COMBINE_WAVES * 64) eg_combine_kernel(
    EgList list, int64_t d, float scale, int accumulate, GE* __restrict__ grad) {
  __shared__ EgCombineShared sh;
  eg_combine<GE>(list, d, scale, accumulate, blockIdx.x, sh, grad);
}

// Both need the window launch alone, and each leaves most of the chip waiting for its chains of
// loads: the first dot_blocks workgroups take four units of dots each, the others combine.
// GPT-2 wte, 16 + 4 rows of 1024 tokens, d = 768: 7.5 us against 6.4 + 6.6 apart, the hook 56.5 ->
// 50.3; 8 + 4 rows of 2048, d = 2048: 128 -> 119; 2 + 2 rows of 64: 34.5 -> 31.5; 90% of 65536
// tokens one id: 143.9 -> 143.5.
constexpr int EG_DOT_UNITS = EG_COMBINE_WAVES * 64 / EG_THREADS;
template <class E, class GE>
__global__ void __launch_bounds__(EG_COMBINE_WAVES * 64) eg_combine_dot_kernel(
    EgDots<E> q, EgList val, unsigned dot_blocks, EgList list, int64_t d, float scale,
    int accumulate, GE* __restrict__ grad) {
  __shared__ union {
    EgCombineShared combine;
    EgDotShared dot[EG_DOT_UNITS];
  } sh;
  if (blockIdx.x < dot_blocks) {
    const int u = threadIdx.x / EG_THREADS;
    eg_dot<E>(q.ids, q.G, q.train, q.n_t, q.T, val, d, q.vocab, q.S, q.vec, q.chunks,
              static_cast<int64_t>(blockIdx.x) * EG_DOT_UNITS + u, threadIdx.x % EG_THREADS,
              sh.dot[u], q.part);
    return;
  }
  eg_combine<GE>(list, d, scale, accumulate, blockIdx.x - dot_blocks, sh.combine, grad);
}

__global__ void __launch_bounds__(EG_THREADS) eg_dot_sum_kernel(const float* __restrict__ part,
                                                                int64_t chunks,
                                                                float* __restrict__ out) {
  __shared__ float red[EG_THREADS / 64];
  const int64_t i = blockIdx.x;
  float s = 0.f;
  for (int64_t c = threadIdx.x; c < chunks; c += blockDim.x) s += part[i * chunks + c];
  s = block_sum(s, red);
  if (threadIdx.x == 0) out[i] = s;
}

int64_t eg_cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

// One call: the dots (val list, its run sums S, parts of the dots), the train gradient (train
// list), or both.
struct EgCall {
  int64_t N, n_val, val_start, T, d, vocab;
  bool dot, grad;
  EgList val, train;
  float* S;
  float* parts;
};

// The bucketed list where its counters and a wave's places fit (131072 tokens, 524288 ids): there
// it was the faster one at every size measured (figures at eg_bucket_kernel).  Sort and merge
// beyond.
EgOrder eg_order(int64_t M, int64_t vocab) {
  EgOrder o{-1, 8};
  if (M > EG_BUCKET_TOKENS || vocab > (int64_t{1024} << EG_BUCKET_SHIFT)) return o;
  if (vocab > (int64_t{256} << EG_BUCKET_SHIFT)) o.nbits = 10;
  o.shift = 0;
  while ((int64_t{1} << (o.nbits + o.shift)) < vocab) ++o.shift;
  return o;
}

template <class S>
void carve_list(S& c, EgList& l, const EgRows& rows, int64_t vocab) {
  l = EgList{};
  l.rows = rows;
  l.order = eg_order(rows.M, vocab);
  const bool bucketed = l.order.shift >= 0;
  l.chunks = bucketed ? 1 : eg_cdiv(rows.M, EG_CHUNK);
  l.windows = eg_cdiv(rows.M, EG_WIN);
  if (!bucketed) l.ck = c.template take<unsigned long long>(l.chunks * EG_CHUNK);
  l.sk = c.template take<unsigned long long>(rows.M);
  l.cnt = c.template take<int32_t>(l.chunks);
}

template <class S>
void carve_call(S& c, EgCall& e) {
  if (e.dot) {   // always bucketed: at most 8192 tokens and 2^19 ids
    carve_list(c, e.val, eg_rows(val_rows(e.n_val, e.val_start, e.T)), e.vocab);
    e.val.table = c.template take<uint2>(size_t{1} << (e.val.order.nbits + e.val.order.shift));
    e.S = c.template take<float>((e.n_val * e.T / 2 + 1) * e.d);
    e.parts = c.template take<float>((e.N - e.n_val) * eg_cdiv(e.T, EG_TOK));
  }
  if (e.grad) {
    EgList& l = e.train;
    carve_list(c, l, eg_rows(train_rows(e.N, e.n_val, e.val_start, e.T)), e.vocab);
    l.present = c.template take<uint32_t>(
        l.order.shift >= 0 ? l.order.bucket_words() << l.order.nbits : eg_cdiv(e.vocab, 32));
    l.part = c.template take<float>(l.windows * 2 * e.d);
  }
}

int build_bucketed(const int64_t* ids, const EgList& a, const EgList* c, int64_t vocab,
                   hipStream_t s) {
  const dim3 grid((c != nullptr ? 2u : 1u) << a.order.nbits);
  const int64_t M = std::max(a.rows.M, c != nullptr ? c->rows.M : 0);
  const EgList& b = c != nullptr ? *c : a;
  // Half the waves where a share is short anyway or the buckets are many (measured as the whole
  // dot, us: 4096 val tokens of 50257 ids 22.1 -> 21.0, 2048 of 300000 27.8 -> 21.3).
  if (M <= (int64_t{8} << EG_SHARE_BITS) && (a.order.nbits > 8 || M <= 8192))
    hipLaunchKernelGGL(eg_bucket_kernel<8>, grid, dim3(512), 8 * sizeof(int) << a.order.shift, s,
                       ids, a, b, vocab);
  else
    hipLaunchKernelGGL(eg_bucket_kernel<16>, grid, dim3(1024), 16 * sizeof(int) << a.order.shift,
                       s, ids, a, b, vocab);
  return check_launch("eg_bucket_kernel");
}

int build_list(const int64_t* ids, const EgList& l, int64_t vocab, hipStream_t s) {
  if (l.order.shift >= 0) return build_bucketed(ids, l, nullptr, vocab, s);
  const dim3 mgrid(static_cast<unsigned>(eg_cdiv(l.chunks * EG_CHUNK, EG_THREADS)));
  const dim3 sgrid(static_cast<unsigned>(l.chunks));
  const int64_t words = eg_cdiv(vocab, 32);
  if (vocab <= EG_KEY32_VOCAB) {
    uint32_t* ck32 = reinterpret_cast<uint32_t*>(l.ck);
    hipLaunchKernelGGL(eg_sort_kernel<uint32_t>, sgrid, dim3(EG_SORT_THREADS), 0, s, ids, l.rows,
                       vocab, ck32, l.cnt, l.present, words);
    if (l.chunks <= EG_SAMP_CHUNKS)
      hipLaunchKernelGGL((eg_merge_kernel<uint32_t, true>), mgrid, dim3(EG_THREADS),
                         static_cast<unsigned>(l.chunks * EG_NSAMP * sizeof(uint32_t)), s, ck32,
                         l.chunks, l.sk, l.present);
    else
      hipLaunchKernelGGL((eg_merge_kernel<uint32_t, false>), mgrid, dim3(EG_THREADS), 0, s, ck32,
                         l.chunks, l.sk, l.present);
  } else {
    hipLaunchKernelGGL(eg_sort_kernel<unsigned long long>, sgrid, dim3(EG_SORT_THREADS), 0, s,
                       ids, l.rows, vocab, l.ck, l.cnt, l.present, words);
    hipLaunchKernelGGL((eg_merge_kernel<unsigned long long, false>), mgrid, dim3(EG_THREADS), 0,
                       s, l.ck, l.chunks, l.sk, l.present);
  }
  return check_launch("eg_sort_kernel / eg_merge_kernel");
}

template <class E, class GE>
int run_call(const EgCall& c, const int64_t* ids, const void* Gv, float* out_dot, float scale,
             int accumulate, int vec, void* gradv, hipStream_t s) {
  const E* G = static_cast<const E*>(Gv);
  GE* grad = static_cast<GE*>(gradv);
  int rc = 0;
  if (c.dot && c.grad && c.val.order.shift >= 0 && c.train.order.shift >= 0) {
    rc = build_bucketed(ids, c.val, &c.train, c.vocab, s);
  } else {
    if (c.dot) rc = build_list(ids, c.val, c.vocab, s);
    if (!rc && c.grad) rc = build_list(ids, c.train, c.vocab, s);
  }
  if (rc) return rc;
  const auto blocks = [](int64_t waves, int64_t per) {
    return static_cast<unsigned>(eg_cdiv(waves, per));
  };
  const int64_t zero_waves = accumulate ? 0 : eg_cdiv(c.vocab, 16);
  const unsigned vw = c.dot ? blocks(c.n_val * c.T, EG_THREADS / 64) : 0;
  const unsigned tw = c.grad ? blocks(c.train.windows + zero_waves, EG_THREADS / 64) : 0;
  hipLaunchKernelGGL((eg_window_kernel<E, GE>), dim3(vw + tw), dim3(EG_THREADS), 0, s, G, c.val,
                     c.train, vw, c.d, c.vocab, scale, accumulate, vec, c.S, grad);
  const int64_t n_t = c.N - c.n_val, chunks = eg_cdiv(c.T, EG_TOK);
  const unsigned cb = c.grad ? blocks(c.train.windows, EG_COMBINE_WAVES) : 0;
  if (!c.dot) {
    hipLaunchKernelGGL((eg_combine_kernel<GE>), dim3(cb), dim3(EG_COMBINE_WAVES * 64), 0, s,
                       c.train, c.d, scale, accumulate, grad);
    return check_launch("eg_window_kernel / eg_combine_kernel");
  }
  const EgDots<E> q{ids, G, eg_rows(train_rows(c.N, c.n_val, c.val_start, c.T)), n_t, c.T, c.vocab,
                    chunks, c.S, vec, c.parts};
  if (c.grad) {
    const unsigned db = blocks(n_t * chunks, EG_DOT_UNITS);
    hipLaunchKernelGGL((eg_combine_dot_kernel<E, GE>), dim3(db + cb), dim3(EG_COMBINE_WAVES * 64),
                       0, s, q, c.val, db, c.train, c.d, scale, accumulate, grad);
  } else {
    hipLaunchKernelGGL(eg_dot_kernel<E>, dim3(static_cast<unsigned>(n_t * chunks)),
                       dim3(EG_THREADS), 0, s, q, c.val, c.d);
  }
  hipLaunchKernelGGL(eg_dot_sum_kernel, dim3(static_cast<unsigned>(n_t)), dim3(EG_THREADS), 0, s,
                     c.parts, chunks, out_dot);
  return check_launch("eg_window_kernel / eg_dot_kernel");
}

// grad_dtype: any when there is no gradient.
int start_call(EgCall& c, const char* name, const int64_t* ids, const void* G, int dtype,
               float* out_dot, float scale, void* grad, int grad_dtype, int accumulate,
               void* workspace, size_t workspace_bytes, hipStream_t s) {
  Sizer sz;
  carve_call(sz, c);
  if (workspace == nullptr || workspace_bytes < sz.used)
    return fail(GS_ERR_WORKSPACE, std::string(name) + ": workspace too small");
  Carver cv(workspace, workspace_bytes);
  carve_call(cv, c);
  const size_t esz = elem_size(dtype), gsz = c.grad ? elem_size(grad_dtype) : 4;
  const int vec = (reinterpret_cast<uintptr_t>(G) % 16 == 0) &&
                  (reinterpret_cast<uintptr_t>(grad) % 16 == 0) &&
                  (c.d * static_cast<int64_t>(esz)) % 16 == 0 &&
                  (c.d * static_cast<int64_t>(gsz)) % 16 == 0;
  const bool half = c.grad && grad_dtype == GS_DTYPE_BF16;
  const int acc = accumulate ? 1 : 0;
  if (dtype == GS_DTYPE_BF16)
    return half ? run_call<uint16_t, uint16_t>(c, ids, G, out_dot, scale, acc, vec, grad, s)
                : run_call<uint16_t, float>(c, ids, G, out_dot, scale, acc, vec, grad, s);
  return half ? run_call<float, uint16_t>(c, ids, G, out_dot, scale, acc, vec, grad, s)
              : run_call<float, float>(c, ids, G, out_dot, scale, acc, vec, grad, s);
}

EgCall eg_call(int64_t N, int64_t n_val, int64_t val_start, int64_t T, int64_t d, int64_t vocab,
               bool dot, bool grad) {
  EgCall c{};
  c.N = N, c.n_val = n_val, c.val_start = val_start, c.T = T, c.d = d, c.vocab = vocab;
  c.dot = dot, c.grad = grad;
  return c;
}

size_t call_workspace(EgCall c) {
  Sizer sz;
  carve_call(sz, c);
  return sz.used + 256;
}

int grad_args_ok(const char* name, const int64_t* ids, const void* G, int dtype, int64_t N,
                 int64_t n_val, int64_t val_start, int64_t T, int64_t d, int64_t vocab,
                 const void* grad, int grad_dtype) {
  if (dtype != GS_DTYPE_BF16 && dtype != GS_DTYPE_F32)
    return fail(GS_ERR_DTYPE, std::string(name) + ": dtype must be bf16 or fp32");
  if (grad_dtype != GS_DTYPE_BF16 && grad_dtype != GS_DTYPE_F32)
    return fail(GS_ERR_DTYPE, std::string(name) + ": grad_dtype must be bf16 or fp32");
  if (ids == nullptr || G == nullptr || grad == nullptr || N <= 0 || n_val < 0 || n_val >= N ||
      val_start < 0 || val_start + n_val > N || T <= 0 || d <= 0 || vocab <= 0)
    return fail(GS_ERR_INVALID, std::string(name) + ": invalid arguments");
  if ((N - n_val) * T >= INT32_MAX || vocab >= INT32_MAX)
    return fail(GS_ERR_UNSUPPORTED, std::string(name) + ": 2^31 or more tokens or ids");
  return 0;
}

}  // namespace

// The dots through the val tokens' list (gs_embedding_dot checks the arguments and the sizes).
size_t embedding_dot_listed_workspace(int64_t N, int64_t n_val, int64_t T, int64_t d,
                                      int64_t vocab) {
  return call_workspace(eg_call(N, n_val, 0, T, d, vocab, true, false));
}
int embedding_dot_listed(const int64_t* ids, const void* G, int dtype, int64_t N, int64_t n_val,
                         int64_t val_start, int64_t T, int64_t d, int64_t vocab, float* out_dot,
                         void* workspace, size_t workspace_bytes, hipStream_t s) {
  EgCall c = eg_call(N, n_val, val_start, T, d, vocab, true, false);
  return start_call(c, "gs_embedding_dot", ids, G, dtype, out_dot, 0.f, nullptr, GS_DTYPE_F32, 0,
                    workspace, workspace_bytes, s);
}
}  // namespace gs

using namespace gs;

extern "C" size_t gs_embedding_train_grad_workspace(int64_t N, int64_t n_val, int64_t T,
                                                    int64_t d, int64_t vocab) {
  if (N <= 0 || n_val < 0 || n_val >= N || T <= 0 || d <= 0 || vocab <= 0) return 0;
  return call_workspace(eg_call(N, n_val, 0, T, d, vocab, false, true));
}

extern "C" int gs_embedding_train_grad(const int64_t* ids, const void* G, int dtype, int64_t N,
                                       int64_t n_val, int64_t val_start, int64_t T, int64_t d,
                                       int64_t vocab, float scale, void* grad, int grad_dtype,
                                       int accumulate, void* workspace, size_t workspace_bytes,
                                       void* stream) {
  if (int rc = grad_args_ok("gs_embedding_train_grad", ids, G, dtype, N, n_val, val_start, T, d,
                            vocab, grad, grad_dtype))
    return rc;
  EgCall c = eg_call(N, n_val, val_start, T, d, vocab, false, true);
  return start_call(c, "gs_embedding_train_grad", ids, G, dtype, nullptr, scale, grad, grad_dtype,
                    accumulate, workspace, workspace_bytes, static_cast<hipStream_t>(stream));
}

extern "C" size_t gs_embedding_layer_pass_workspace(int64_t N, int64_t n_val, int64_t T, int64_t d,
                                                    int64_t vocab) {
  if (N <= 0 || n_val <= 0 || n_val >= N || T <= 0 || d <= 0 || vocab <= 0 ||
      !embedding_dot_is_listed(n_val, T, vocab))
    return 0;
  return call_workspace(eg_call(N, n_val, 0, T, d, vocab, true, true));
}

extern "C" int gs_embedding_layer_pass(const int64_t* ids, const void* G, int dtype, int64_t N,
                                       int64_t n_val, int64_t val_start, int64_t T, int64_t d,
                                       int64_t vocab, float* out_dot, float scale, void* grad,
                                       int grad_dtype, int accumulate, void* workspace,
                                       size_t workspace_bytes, void* stream) {
  if (int rc = grad_args_ok("gs_embedding_layer_pass", ids, G, dtype, N, n_val, val_start, T, d,
                            vocab, grad, grad_dtype))
    return rc;
  if (n_val == 0 || out_dot == nullptr)
    return fail(GS_ERR_INVALID, "gs_embedding_layer_pass: invalid arguments");
  if (!embedding_dot_is_listed(n_val, T, vocab))
    return fail(GS_ERR_UNSUPPORTED, "gs_embedding_layer_pass: more than 8192 val tokens or 2^19 ids");
  EgCall c = eg_call(N, n_val, val_start, T, d, vocab, true, true);
  return start_call(c, "gs_embedding_layer_pass", ids, G, dtype, out_dot, scale, grad, grad_dtype,
                    accumulate, workspace, workspace_bytes, static_cast<hipStream_t>(stream));
}
