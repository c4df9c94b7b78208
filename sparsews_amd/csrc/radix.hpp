// Stable LSD radix sort of (key, FP64 value) pairs on the device, up to 9
// bits per pass.
//
// The key bits are split evenly over ceil(bits / 9) passes (34 bits: 9, 9,
// 8, 8).  Per pass, three steps over tiles of kSortTile keys:
//   1. k_radix_hist     per-tile digit histogram (LDS atomics), a row of
//                       counts per tile: hist[t * digits + d].
//   2. k_radix_chunks   the rows of a chunk of tiles become what the chunk's
//                       earlier tiles hold of each digit, and the chunk's
//                       total a row; k_radix_digits does the same to the
//                       chunks' rows, with the digits' totals as last row.
//                       (Few tiles: neither, the scatter sums the rows.)
//   3. k_radix_scatter  adds the digits before (a scan of the totals), the
//                       chunks before and the tiles before into the tile's
//                       offset of each digit; stable tile-local ranks by wavefront multisplit:
//                       each wave walks its contiguous quarter of the tile
//                       64 keys at a time; one ballot per digit bit gives
//                       the lanes holding the same digit, the group's rank
//                       is the running per-wave digit count (LDS) plus the
//                       lanes before it.  Keys, then values, are staged in
//                       LDS in digit order (one buffer, two rounds) and
//                       written out so that consecutive threads store
//                       consecutive addresses of each digit's run.
// Every row is read and written by consecutive threads.  (With the counts of a
// digit side by side instead, one scan made every offset, but a tile stored
// and loaded each of its 512 counts in a cache line of its own, shared with
// tiles on other chiplets.  200,000 x 200,000 with 32 per row, two passes:
// scatter 142 us, histogram 32, scans 28; rows: 131, 21, 25.)
//
// Where the pairs of the first pass come from and where those of the last go
// is a template parameter each, so that keys made from a sparse structure are
// never stored before they are first moved, nor stored as keys when the caller
// wants them in parts.  (20M nonzeros of a CSF: the key pass took 95 us and
// two launches; the first scatter that makes them takes 20 us more than one
// that reads them.)
#pragma once
#include "common.hpp"

namespace spws {

// Tiles of the LSD method's own run and reduce kernels (spgemm_outer.hip).
constexpr int kRadixBlock = 256;
constexpr int kRadixItems = 8;
constexpr int kRadixTile = kRadixBlock * kRadixItems;  // keys per workgroup tile

// The sort: tiles of kSortTile keys, passes of at most kSortDigitMax bits
// (the key bits are split evenly over ceil(bits / kSortDigitMax) passes).
constexpr int kSortBlock = 256;
constexpr int kSortItems = 16;
constexpr int kSortTile = kSortBlock * kSortItems;
constexpr int kSortDigitMax = 9;
constexpr int kSortBucketsMax = 1 << kSortDigitMax;

// Tiles per chunk: 32 row reads are in flight at once; up to 128 tiles are one
// chunk, which needs no second launch.
constexpr int kSortChunk = 32;
constexpr int kSortChunkOnly = 128;

// int32 entries of ctx->radix_hist that one pass over n keys uses at most: a
// row of digits per tile, one per chunk of tiles, and the totals.
inline size_t radix_hist_entries(int64_t n) {
  const int64_t tiles = div_up(n > 0 ? n : 1, kSortTile);
  return (size_t)(tiles + div_up(tiles, kSortChunk) + 1) * kSortBucketsMax;
}

// Sorts keys[0, n) by bits [begin_bit, end_bit) carrying vals along, using
// keys_alt / vals_alt as the ping-pong buffers.  On return *in_alt says
// whether the sorted data ended up in the _alt buffers.  K is uint32_t or
// uint64_t.  Uses ctx->radix_hist.  With vals_first, the values are read from
// there instead of vals (which then needs no copy of them; it is still filled
// when no pass runs).
template <class K>
int radix_sort_pairs(spws_ctx* ctx, K* keys, double* vals, K* keys_alt, double* vals_alt, int64_t n, int begin_bit,
                     int end_bit, bool* in_alt, const double* vals_first = nullptr);

inline int radix_passes(int bits) { return (bits + kSortDigitMax - 1) / kSortDigitMax; }

// ------------------------------------------------------------ segment owners

// s[e] = the last s in [0, n) with pos[s] <= x[e] (pos[0] <= x[e], pos
// nondecreasing), by the whole wavefront: 64 probes a round for each, the same
// ones as long as both lie between the same two.
template <class PosT>
__device__ __forceinline__ void last_at_or_before(const PosT* __restrict__ pos, int32_t n, const int64_t (&x)[2],
                                                  int32_t (&s)[2]) {
  int32_t lo[2] = {0, 0}, hi[2] = {n, n};
  while (max(hi[0] - lo[0], hi[1] - lo[1]) > 1) {
    PosT v[2];
    int32_t step[2];
    const bool same = lo[0] == lo[1] && hi[0] == hi[1];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      step[e] = (hi[e] - lo[e] + kWave - 1) / kWave;
      const int64_t at = lo[e] + (int64_t)lane_id() * step[e];
      v[e] = v[0];
      if (e == 0 || !same) v[e] = at < hi[e] ? pos[at] : std::numeric_limits<PosT>::max();
    }
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      lo[e] += (kWave - 1 - __builtin_clzll(__ballot((int64_t)v[e] <= x[e]))) * step[e];  // lane 0 always holds
      hi[e] = min(hi[e], lo[e] + step[e]);
    }
  }
  s[0] = lo[0];
  s[1] = lo[1];
}

// owner[r] = the segment s with pos[s] <= e < pos[s + 1] of item
// e = base + w * kSub + r * 64 + lane (w: the wavefront, kSub = 64 * ITEMS),
// for the items of one workgroup's tile [base, end).  Segments mark their
// first item in LDS (`marks`: a uint32 per item of the tile), and a max-scan
// carries each mark to the items after it.  Ends with a barrier after the last
// use of `marks`; every thread of the workgroup calls it.
//
// The marks cost the tile a look at every segment that starts in it, empty
// ones too, BLOCK at a time, about 0.2 us each time.  A tile of more than
// eight times as many segments as items searches each item's segment instead:
// 100k entries transposed with 6M empty rows between two of them take 89 us so
// and 9,660 walked; with 900k rows spread between them (ten segments an item)
// 88 searched and 95 walked, with 300k 97 and 67.  The search for the first
// item's segment finds the last one's with it: looked up after it, the number
// of segments cost small calls up to 6 us.
constexpr int kOwnerWalk = 8;    // segments walked per item of a tile at most
constexpr int kOwnerSearch = 8;  // items searched together
template <int BLOCK, int ITEMS, class PosT>
__device__ __forceinline__ void tile_owners(const PosT* __restrict__ pos, int32_t nseg, int64_t base, int64_t end,
                                            uint32_t* __restrict__ marks, int32_t (&owner)[ITEMS]) {
  constexpr int kWaves = BLOCK / kWave;
  static_assert(ITEMS % kOwnerSearch == 0, "items in whole groups of a search");
  __shared__ uint32_t top[kWaves];
  const int lane = lane_id();
  const int w = threadIdx.x / kWave;
  int32_t edge[2];  // the first and the last item's segments
  last_at_or_before(pos, nseg, {base, end - 1}, edge);
  const int32_t s0 = edge[0];
  const uint32_t span = (uint32_t)(edge[1] - s0);
  if (span >= (uint32_t)(kOwnerWalk * BLOCK * ITEMS)) {  // uniform
    uint32_t top_step = 1;
    while (top_step <= span >> 1) top_step <<= 1;
#pragma unroll
    for (int q = 0; q < ITEMS; q += kOwnerSearch) {
#pragma unroll
      for (int r = q; r < q + kOwnerSearch; ++r) owner[r] = s0;
      for (uint32_t step = top_step; step > 0; step >>= 1) {
#pragma unroll
        for (int r = q; r < q + kOwnerSearch; ++r) {
          const int64_t e = min(base + (w * ITEMS + r) * kWave + lane, end - 1);
          const uint32_t s = (uint32_t)owner[r] + step;
          if (s <= (uint32_t)edge[1] && (int64_t)pos[s] <= e) owner[r] = (int32_t)s;
        }
      }
    }
    return;
  }
  for (int e = threadIdx.x; e < BLOCK * ITEMS; e += BLOCK) marks[e] = 0;
  __syncthreads();
  for (uint32_t s = threadIdx.x; s <= span; s += BLOCK) {
    const int64_t p = (int64_t)pos[s0 + s];
    if ((int64_t)pos[s0 + s + 1] > p) marks[p > base ? p - base : 0] = s + 1;
  }
  __syncthreads();
  uint32_t m[ITEMS];
  uint32_t mine = 0;
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) {
    m[r] = marks[(w * ITEMS + r) * kWave + lane];
    mine = max(mine, m[r]);
  }
  mine = wave_max(mine);
  if (lane == 0) top[w] = mine;
  __syncthreads();
  uint32_t carry = 0;
#pragma unroll
  for (int q = 0; q < kWaves; ++q)
    if (q < w) carry = max(carry, top[q]);
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) {
    const uint32_t x = max(wave_incl_max(m[r]), carry);
    owner[r] = s0 + (int32_t)x - 1;
    carry = wave_last(x);
  }
}

// ------------------------------------------------------------ sources and sinks

// A source gives pair idx of the first pass: its value, and raw(idx), from
// which key() makes the key.  With kOwners, key() also gets the item's segment,
// found by owners() while the raw parts and values are in flight.
// digit_bits(raw) holds the first digit's bits, all the histogram needs; with
// kOwnedDigits that takes the segment too, and the histogram calls key().
template <class K>
struct PairSource {
  static constexpr bool kOwners = false, kOwnedDigits = false;
  using Raw = K;
  const K* __restrict__ keys;
  const double* __restrict__ vals;
  __device__ K raw(int64_t idx) const { return keys[idx]; }
  __device__ double val(int64_t idx) const { return vals[idx]; }
  __device__ K digit_bits(K k) const { return k; }
  __device__ K key(K k, int32_t) const { return k; }
};

// A sink takes the key and the value that belong at position `at`.
template <class K>
struct PairSink {
  K* __restrict__ keys;
  double* __restrict__ vals;
  __device__ void key(int64_t at, K k) const { keys[at] = k; }
  __device__ void val(int64_t at, double v) const { vals[at] = v; }
};

template <class K>
__device__ __forceinline__ int radix_digit(K key, int shift, uint32_t mask) {
  return (int)((key >> shift) & (K)mask);
}

// h[d] += 1 for every lane's digit d (d < 0: none); the first lane's digit is
// added once for all the lanes that hold it.
__device__ __forceinline__ void radix_count_common(int32_t* h, int d) {
  uint64_t left = __ballot(d >= 0);
  if (left == 0) return;  // uniform
  const int lead = __builtin_ctzll(left);
  const uint64_t same = __ballot(d == __builtin_amdgcn_readlane(d, lead));
  if (lane_id() == lead) atomicAdd(&h[d], (int32_t)__popcll(same));
  left &= ~same;
  if (left >> lane_id() & 1) atomicAdd(&h[d], 1);
}

template <class K, class Source>
__global__ __launch_bounds__(kSortBlock) void k_radix_hist(Source in, int64_t n, int shift, uint32_t mask,
                                                           int32_t* __restrict__ hist) {
  __shared__ int32_t h[kSortBucketsMax];
  const int nb = (int)mask + 1;
  for (int d = threadIdx.x; d < nb; d += kSortBlock) h[d] = 0;
  __syncthreads();
  const int64_t base = (int64_t)blockIdx.x * kSortTile;
  typename Source::Raw raw[kSortItems];
  if constexpr (Source::kOwnedDigits) {
    __shared__ uint32_t marks[kSortTile];
    int32_t owner[kSortItems];
    in.owners(base, base + kSortTile < n ? base + kSortTile : n, marks, owner);
#pragma unroll
    for (int r = 0; r < kSortItems; ++r) {
      const int64_t idx = base + (int64_t)((threadIdx.x / kWave) * kSortItems + r) * kWave + lane_id();
      if (idx < n) atomicAdd(&h[radix_digit(in.key(in.raw(idx), owner[r]), shift, mask)], 1);
    }
  } else {
#pragma unroll
    for (int it = 0; it < kSortItems; ++it) {
      const int64_t idx = base + (int64_t)it * kSortBlock + threadIdx.x;
      if (idx < n) raw[it] = in.raw(idx);
    }
    int dig[kSortItems];
#pragma unroll
    for (int it = 0; it < kSortItems; ++it) {
      const int64_t idx = base + (int64_t)it * kSortBlock + threadIdx.x;
      dig[it] = idx < n ? radix_digit<K>(in.digit_bits(raw[it]), shift, mask) : -1;
    }
    // Adds to one counter follow one another: where digits are often equal,
    // the first lane's is added once for all.  Neighbouring lanes show it: a
    // digit of share p makes them equal p^2 of the time (6 of these 256 lanes:
    // p = 0.15; 512 even digits: half a lane).  10M nonzeros of power-law
    // coordinates, four passes: 134 us without, 74 with; 6.4M even columns, two
    // passes: 22 either way (25 when every item looks for its own).
    int equal = 0;
#pragma unroll
    for (int it = 0; it < kSortItems; it += kSortItems / 4)
      equal += __popcll(__ballot(dig[it] >= 0 && dig[it] == __builtin_amdgcn_mov_dpp(dig[it], 0xB1, 0xF, 0xF, true)));
    if (equal >= 6) {  // uniform
#pragma unroll
      for (int it = 0; it < kSortItems; ++it) radix_count_common(h, dig[it]);
    } else {
#pragma unroll
      for (int it = 0; it < kSortItems; ++it)
        if (dig[it] >= 0) atomicAdd(&h[dig[it]], 1);
    }
  }
  __syncthreads();
  for (int d = threadIdx.x; d < nb; d += kSortBlock) hist[(int64_t)blockIdx.x * nb + d] = h[d];
}

// Up to 64 tiles the scatter sums the rows itself, 16 reads in flight, and the
// launch of one workgroup's width goes: 49 tiles, three passes, scatters 50 us
// and 21 for the chunks' launches, 55 without them (whole call 180 -> 166 us);
// four tiles, two passes, whole call 164 -> 149.  Reads grow with the square of
// the tiles: at 128 tiles every tile would read 256 KB.
constexpr int kSortDirect = 64;
inline int64_t radix_chunk_tiles(int64_t ntiles) { return ntiles <= kSortChunkOnly ? ntiles : kSortChunk; }

// hist's rows of nb counts, one per tile, in place to what the earlier tiles of
// their chunk hold, and the chunks' rows in chunk likewise, with the totals
// behind them (a single chunk's row is the totals).
int radix_offsets(spws_ctx* ctx, int32_t* hist, int64_t ntiles, int nb, int32_t* chunk);

template <class K, class Source, class Sink>
__global__ __launch_bounds__(kSortBlock, 4) void k_radix_scatter(Source in, Sink out, int64_t n, int shift,
                                                                 uint32_t mask, int nbits,
                                                                 const int32_t* __restrict__ hist,
                                                                 const int32_t* __restrict__ chunk, int64_t chunks,
                                                                 int64_t per) {
  constexpr int kWaves = kSortBlock / kWave;
  constexpr int kSub = kSortTile / kWaves;  // keys per wave
  static_assert(kSortBucketsMax == 2 * kSortBlock, "two digits per thread in the prefix step");
  static_assert(sizeof(K) <= sizeof(double), "one staging buffer for keys and values");
  __shared__ double stage[kSortTile];  // keys, then values, in digit order
  // per (wavefront, digit): counts, then where in the tile the wavefront's
  // pairs of the digit start (at most kSortTile = 4096, so 16 bits: 39.0 KB of
  // LDS in all, four workgroups per CU)
  __shared__ uint16_t wcnt[kWaves][kSortBucketsMax];
  static_assert(kSortTile < 65536, "per-wavefront digit prefixes fit 16 bits");
  __shared__ int32_t goff[kSortBucketsMax];  // position of a digit's pairs, less their place in the tile
  __shared__ int64_t scan_sh[kSortBlock / kWave + 1];
  K* sk = reinterpret_cast<K*>(stage);

  const int lane = lane_id();
  const int w = threadIdx.x / kWave;
  const int nb = (int)mask + 1;
  const int64_t base = (int64_t)blockIdx.x * kSortTile;
  const int64_t wbase = base + (int64_t)w * kSub;
  const uint64_t lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  typename Source::Raw raw[kSortItems];
  K key[kSortItems];
  double val[kSortItems];
  int32_t rank[kSortItems];
#pragma unroll
  for (int r = 0; r < kSortItems; ++r) {
    const int64_t idx = wbase + (int64_t)r * kWave + lane;
    raw[r] = {};
    val[r] = 0.0;
    if (idx < n) {
      raw[r] = in.raw(idx);
      val[r] = in.val(idx);
    }
  }
  // digits 2t and 2t + 1 of thread t: their pairs in earlier tiles, and in all
  int32_t before[2] = {}, all[2] = {};
  if (chunks == 0) {  // few tiles: their rows summed here (nb is even)
    if (2 * (int)threadIdx.x < nb) {
#pragma unroll 16
      for (int t = 0; t < (int)gridDim.x; ++t) {
        const int2 c = *reinterpret_cast<const int2*>(hist + (int64_t)t * nb + 2 * threadIdx.x);
        before[0] += t < (int)blockIdx.x ? c.x : 0;
        before[1] += t < (int)blockIdx.x ? c.y : 0;
        all[0] += c.x;
        all[1] += c.y;
      }
    }
  } else {
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int d = 2 * threadIdx.x + e;
      if (d < nb) {
        before[e] = hist[(int64_t)blockIdx.x * nb + d];
        all[e] = chunk[(chunks > 1 ? chunks * nb : 0) + d];  // a single chunk's row is the totals
        if (chunks > 1) before[e] += chunk[((int64_t)blockIdx.x / per) * nb + d];
      }
    }
  }
  int32_t owner[kSortItems] = {};
  if constexpr (Source::kOwners)
    in.owners(base, base + kSortTile < n ? base + kSortTile : n, reinterpret_cast<uint32_t*>(stage), owner);
  for (int d = threadIdx.x; d < kWaves * kSortBucketsMax; d += kSortBlock) (&wcnt[0][0])[d] = 0;
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kSortItems; ++r) key[r] = in.key(raw[r], owner[r]);
#pragma unroll
  for (int r = 0; r < kSortItems; ++r) {
    const int64_t idx = wbase + (int64_t)r * kWave + lane;
    const bool valid = idx < n;
    const int d = radix_digit(key[r], shift, mask);
    uint64_t match = __ballot(valid);
#pragma unroll
    for (int b = 0; b < kSortDigitMax; ++b) {
      if (b < nbits) {  // uniform
        const bool bit = (d >> b) & 1;
        const uint64_t m = __ballot(bit);
        match &= bit ? m : ~m;
      }
    }
    rank[r] = 0;
    if (valid) {
      const int before = __popcll(match & lt);
      const int32_t old = wcnt[w][d];
      rank[r] = old + before;
      if (before == 0) wcnt[w][d] = (uint16_t)(old + __popcll(match));
    }
  }
  __syncthreads();
  {
    // thread t: digits 2t and 2t + 1: exclusive prefixes over the digits of
    // the tile's counts and (from bit 16) of all, then over the waves
    int32_t c[2][kWaves], tot[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int d = 2 * threadIdx.x + e;
      tot[e] = 0;
#pragma unroll
      for (int q = 0; q < kWaves; ++q) {
        c[e][q] = d < nb ? wcnt[q][d] : 0;
        tot[e] += c[e][q];
      }
    }
    int64_t sum;
    const int64_t st = block_excl_scan<int64_t, kSortBlock>(
        (((int64_t)all[0] + all[1]) << 16) + tot[0] + tot[1], scan_sh, &sum);
    int32_t in_tile = (int32_t)(st & 0xffff);  // the tile's counts sum to at most kSortTile
    int32_t in_all = (int32_t)(st >> 16);
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int d = 2 * threadIdx.x + e;
      if (d < nb) {
        goff[d] = in_all + before[e] - in_tile;
        int32_t run = in_tile;
#pragma unroll
        for (int q = 0; q < kWaves; ++q) {
          wcnt[q][d] = (uint16_t)run;
          run += c[e][q];
        }
      }
      in_tile += tot[e];
      in_all += all[e];
    }
  }
  __syncthreads();
  const int64_t remain = n - base;
  const int tile_n = remain < kSortTile ? (int)remain : kSortTile;
  // round 1: keys in digit order, written out; their destinations kept
#pragma unroll
  for (int r = 0; r < kSortItems; ++r) {
    const int64_t idx = wbase + (int64_t)r * kWave + lane;
    if (idx < n) {
      const int d = radix_digit(key[r], shift, mask);
      rank[r] += wcnt[w][d];
      sk[rank[r]] = key[r];
    }
  }
  __syncthreads();
  int32_t dst[kSortItems];
#pragma unroll
  for (int it = 0; it < kSortItems; ++it) {
    const int i = it * kSortBlock + threadIdx.x;
    dst[it] = 0;
    if (i < tile_n) {
      const K k = sk[i];
      dst[it] = goff[radix_digit(k, shift, mask)] + i;
      out.key(dst[it], k);
    }
  }
  __syncthreads();
  // round 2: the values through the same buffer
#pragma unroll
  for (int r = 0; r < kSortItems; ++r) {
    const int64_t idx = wbase + (int64_t)r * kWave + lane;
    if (idx < n) stage[rank[r]] = val[r];
  }
  __syncthreads();
#pragma unroll
  for (int it = 0; it < kSortItems; ++it) {
    const int i = it * kSortBlock + threadIdx.x;
    if (i < tile_n) out.val(dst[it], stage[i]);
  }
}

// One pass over n pairs (below 2^31) on `nbits` bits from `shift`.
template <class K, class Source, class Sink>
int radix_pass(spws_ctx* ctx, const Source& in, const Sink& out, int64_t n, int shift, int nbits) {
  const int64_t ntiles = div_up(n, kSortTile);
  int rc = ctx->radix_hist.ensure(radix_hist_entries(n) * sizeof(int32_t));
  if (rc) return rc;
  int32_t* hist = ctx->radix_hist.as<int32_t>();
  int32_t* chunk = hist + ntiles * kSortBucketsMax;
  const uint32_t mask = (1u << nbits) - 1u;
  const int nb = 1 << nbits;
  const int64_t per = radix_chunk_tiles(ntiles), chunks = ntiles <= kSortDirect ? 0 : div_up(ntiles, per);
  SPWS_LAUNCH(ctx, "radix_hist", (k_radix_hist<K, Source>), dim3((unsigned)ntiles), dim3(kSortBlock), 0, in, n, shift,
              mask, hist);
  if (chunks > 0 && (rc = radix_offsets(ctx, hist, ntiles, nb, chunk))) return rc;
  SPWS_LAUNCH(ctx, "radix_scatter", (k_radix_scatter<K, Source, Sink>), dim3((unsigned)ntiles), dim3(kSortBlock), 0,
              in, out, n, shift, mask, nbits, (const int32_t*)hist, (const int32_t*)chunk, chunks, per);
  return SPWS_OK;
}

// Sorts n pairs (0 < n < 2^31) from `in` by bits [begin_bit, end_bit), at
// least one, into `out`: pass p writes buffer p mod 2 (keys[], vals[], n
// entries each; the second only from three passes on), the last one `out`,
// which may be the buffer whose turn it is.
template <class K, class Source, class Sink>
int radix_sort_from(spws_ctx* ctx, const Source& in, K* const (&keys)[2], double* const (&vals)[2], const Sink& out,
                    int64_t n, int begin_bit, int end_bit) {
  const int passes = radix_passes(end_bit - begin_bit);
  int shift = begin_bit;
  for (int p = 0; p < passes; ++p) {
    // the remaining bits split evenly over the remaining passes
    const int nbits = (int)div_up(end_bit - shift, passes - p);
    const PairSource<K> from{keys[(p + 1) & 1], vals[(p + 1) & 1]};
    const PairSink<K> to{keys[p & 1], vals[p & 1]};
    int rc;
    if (p == 0 && passes == 1) rc = radix_pass<K>(ctx, in, out, n, shift, nbits);
    else if (p == 0) rc = radix_pass<K>(ctx, in, to, n, shift, nbits);
    else if (p + 1 == passes) rc = radix_pass<K>(ctx, from, out, n, shift, nbits);
    else rc = radix_pass<K>(ctx, from, to, n, shift, nbits);
    if (rc) return rc;
    shift += nbits;
  }
  return SPWS_OK;
}

}  // namespace spws
