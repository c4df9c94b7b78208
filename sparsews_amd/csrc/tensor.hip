// Sparse tensor kernels over 3-level CSF inputs: MTTKRP and TTM.
//
// MTTKRP  M(i,r) = sum_{j,k} X(i,j,k) * Bf(j,r) * Cf(k,r)   (output mode i)
//   Input CSF levels (j, k, i): the output mode is the leaf, as in the
//   reference (B(k,l,i) in benchmark/MTTKRP/COO_CSF_DCSR_DCSR_hash_free.h:233;
//   its C and D factors are Bf and Cf here, given dense, row-major R wide).
//   Bucket workspace over output rows:
//     1. k_seg_owner        fiber -> root owners (with factor masks also
//                           leaf -> fiber owners, and k_mttkrp_keys).
//     2. radix sort         of packed keys (i << (bj+bk) | j << bk | k), stable
//                           on the i bits only: the buckets are the output
//                           rows, CSF (j,k) order kept inside each.  Its first
//                           pass makes the keys from the CSF itself
//                           (CsfSource); they are not stored unsorted.
//     3. k_mttkrp_accum     each group of 16 or 32 lanes (a rank per lane)
//                           walks a segment of the bucketed nonzeros, loading
//                           factor rows Bf(j,:), Cf(k,:) as coalesced rows
//                           (Bf(j,:) only when j changes: within a row the
//                           nonzeros come in (j, k) order) and accumulating
//                           the rank-R fiber in registers; a row inside one
//                           segment is stored, rows over several segments of
//                           a workgroup meet in LDS, and only rows that reach
//                           other workgroups are added with atomics.
//     4. k_rows_present + scan + k_rows_compact: the sorted list of rows that
//                           hold a nonzero (the reference's COO output rows).
//   The product is (X * Bf) * Cf, the reference's B_vals * C_vals * D_vals
//   (:296), and each segment sums in CSF order.
//
// TTM  Y(i,j,r) = sum_k X(i,k,j) * U(k,r)   (contracted mode k)
//   Input CSF levels (i, k, j): the contracted coordinate is the middle
//   level, as in the reference's hash_il (B(k,i,j) in
//   benchmark/TTM/COO_CSF_DCSR_hash_il.h:247), whose hash workspace is keyed
//   on the output fiber (i,j).  Here the fibers are grouped by sorting:
//     1. k_seg_owner        fiber -> root owners (with a U row mask also
//                           leaf -> fiber owners, and k_ttm_direct_keys).
//     2. radix sort         of packed (i, j, k) keys, stable, on the (i, j)
//                           bits only: each fiber's nonzeros end up together
//                           and keep the CSF order, increasing k -- the order
//                           hash_il sums them.  Its first pass makes the keys
//                           and takes the values from the CSF itself.
//     3. k_ttm_seg_starts + scan: fiber starts per segment of 32 to 128
//                           nonzeros, so each segment knows its first fiber.
//     4. k_ttm_accum        one 16-lane group per segment sums X * U(k,:) in
//                           order and writes each fiber that starts there,
//                           with its coordinates; segments inside a longer
//                           fiber write partial sums that k_ttm_fixup adds in
//                           order (no atomics; deterministic).
//   When i, j and k need more than 64 bits together, the fibers are found
//   through an open-addressing table in HBM (k_ttm_insert, 64-bit keys
//   (i << bj) | j, atomicCAS), collected and sorted (k_ttm_occupied,
//   k_ttm_collect, radix sort, k_ttm_rank), and the nonzeros are then
//   sorted by fiber rank (k_ttm_keys) before steps 3 and 4.
//   Output: semi-sparse -- the sorted fiber list (i,j) with a dense length-R
//   vector each.
#include <algorithm>
#include <climits>

#include "radix.hpp"
#include "tensor.hpp"

namespace spws {

// owner[e] = s for e in [pos[s], pos[s+1]), s in [0, nseg); pos[nseg] =
// nitems; a tile of items per workgroup.
constexpr int kOwnBlock = 256;
constexpr int kOwnItems = 8;
constexpr int kOwnTile = kOwnBlock * kOwnItems;

// What k_seg_owner does with item e of segment s: store s.
struct OwnerOut {
  int32_t* __restrict__ owner;
  __device__ void operator()(int64_t e, int32_t s) const { owner[e] = s; }
};

// Or, over a CSF's fibers (s = the fiber's root): its part of the sort key.
struct FiberKeyOut {
  const int32_t* __restrict__ l1_crd;
  const int32_t* __restrict__ l2_crd;
  int root_shift;
  uint64_t* __restrict__ fiber_key;
  __device__ void operator()(int64_t f, int32_t s) const {
    fiber_key[f] = ((uint64_t)(uint32_t)l1_crd[s] << root_shift) | (uint32_t)l2_crd[f];
  }
};

template <class Out>
__global__ __launch_bounds__(kOwnBlock) void k_seg_owner(const int32_t* __restrict__ pos, int32_t nseg, int64_t nitems,
                                                         Out out) {
  __shared__ uint32_t marks[kOwnTile];
  const int64_t base = (int64_t)blockIdx.x * kOwnTile;
  int32_t own[kOwnItems];
  tile_owners<kOwnBlock, kOwnItems>(pos, nseg, base, base + kOwnTile < nitems ? base + kOwnTile : nitems, marks, own);
#pragma unroll
  for (int r = 0; r < kOwnItems; ++r) {
    const int64_t e = base + ((threadIdx.x / kWave) * kOwnItems + r) * kWave + lane_id();
    if (e < nitems) out(e, own[r]);
  }
}

template <class Out>
static int seg_owner(spws_ctx* ctx, const int32_t* pos, int32_t nseg, int64_t nitems, Out out) {
  if (nitems <= 0) return SPWS_OK;
  SPWS_LAUNCH(ctx, "seg_owner", k_seg_owner<Out>, dim3((unsigned)div_up(nitems, kOwnTile)), dim3(kOwnBlock), 0, pos,
              nseg, nitems, out);
  return SPWS_OK;
}

// A CSF's nonzeros as the sort's first pass reads them: nonzero e of fiber f
// has the key (hi << (bj + bk)) | (mid << bk) | k with k = the fiber's
// coordinate and, for TTM, hi = the root's and mid = the leaf's coordinate;
// for MTTKRP the other way round.  The sort starts at the leaf's bits, so the
// first pass's histogram reads the leaves' coordinates alone, unless its digit
// reaches into the root's (kRootDigits: TTM with fewer leaf bits than that).
template <bool kMttkrp, bool kRootDigits>
struct CsfSource {
  static constexpr bool kOwners = true, kOwnedDigits = kRootDigits;
  using Raw = uint32_t;
  const uint64_t* __restrict__ fiber_key;  // per fiber, the key's part from its root and its own coordinate
  const int32_t* __restrict__ l3_pos;
  const int32_t* __restrict__ l3_crd;
  const double* __restrict__ vals;
  int32_t nfibers;
  int leaf_shift;  // the leaf's bits in the key
  __device__ uint32_t raw(int64_t e) const { return (uint32_t)l3_crd[e]; }
  __device__ double val(int64_t e) const { return vals[e]; }
  __device__ uint64_t digit_bits(uint32_t leaf) const { return (uint64_t)leaf << leaf_shift; }
  __device__ void owners(int64_t base, int64_t end, uint32_t* marks, int32_t (&own)[kSortItems]) const {
    tile_owners<kSortBlock, kSortItems>(l3_pos, nfibers, base, end, marks, own);
  }
  __device__ uint64_t key(uint32_t leaf, int32_t f) const { return fiber_key[f] | ((uint64_t)leaf << leaf_shift); }
};

static int bits_of(int64_t v) {  // bits for values in [0, v)
  int b = 0;
  while (b < 63 && ((int64_t)1 << b) < v) ++b;
  return b;
}

// ------------------------------------------------------------------ MTTKRP

// With factor row masks (bit r: column r of the factor row is stored), a
// nonzero whose two rows share no stored column takes no part (the
// reference's co-iteration never reaches it): it gets the row key `drop_i`,
// past every output row, so the sort moves it to the end, and is counted.
__global__ __launch_bounds__(256) void k_mttkrp_keys(int64_t nnz, const int32_t* __restrict__ leaf_fiber,
                                                     const int32_t* __restrict__ fiber_root,
                                                     const int32_t* __restrict__ l1_crd,
                                                     const int32_t* __restrict__ l2_crd,
                                                     const int32_t* __restrict__ l3_crd, int bj, int bk,
                                                     uint64_t* __restrict__ keys, const uint64_t* __restrict__ mB,
                                                     const uint64_t* __restrict__ mC, uint64_t drop_i,
                                                     unsigned long long* __restrict__ dropped) {
  unsigned long long nd = 0;
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < nnz; e += (int64_t)gridDim.x * blockDim.x) {
    const int32_t f = leaf_fiber[e];
    const uint64_t j = (uint32_t)l1_crd[fiber_root[f]];
    const uint64_t k = (uint32_t)l2_crd[f];
    uint64_t i = (uint32_t)l3_crd[e];
    if ((mB[j] & mC[k]) == 0) {
      i = drop_i;
      ++nd;
    }
    keys[e] = (i << (bj + bk)) | (j << bk) | k;
  }
  nd = wave_sum(nd);
  if (lane_id() == 0 && nd) atomicAdd(dropped, nd);
}

// The bucketed nonzeros in tiles of one workgroup, `seg` consecutive ones per
// group of G lanes; the lanes cover ranks lane, lane + G, ... (S slices).
// A group loads G keys and values at once (coalesced, the next G in flight
// while these are used), stages them in LDS, and walks them kAccU at a time,
// each nonzero's record one 16-byte broadcast read; the factor rows of kAccU
// nonzeros are loaded before any is used, so their latencies overlap.  The
// sums run in bucket order.
//
// A row that starts and ends inside a group's segment is stored at once: no
// other group holds a part of it.  The segments' first and last rows meet in
// LDS after the walk; only the tile's own first and last rows are added into
// M with atomics, one per tile.  With one per segment of 128 the atomics of
// the skewed rows bounded the kernel: a row of 2M nonzeros was 15,600 adds to
// the same two lines, about 50 ns each across the XCDs.  50k x 40k x 30k,
// 20M nonzeros, R = 32: 1,204 us with an atomic per segment and row, 518 us
// with one per tile, 470 us with the factors' byte offsets made once per
// nonzero by the lane that loads it (64 VGPRs, 8 wavefronts per SIMD); now
// the gathered factor rows (about 8 GB from the L2) bound it.
constexpr int kAccBlock = 256;
constexpr int kAccU = 4;
constexpr int kAccSegMax = 256;  // nonzeros per group at most
constexpr int kAccSegMin = 32;

// kMask: per row, the OR of its nonzeros' shared stored factor columns
// (mB[j] & mC[k]) is or-ed into rmask[i], the row's stored output columns.
template <int G, int S, bool kMask, bool kOff32>
__global__ __launch_bounds__(kAccBlock, S == 1 && !kMask ? 8 : 4) void k_mttkrp_accum(
    int64_t nnz, int seg, const uint64_t* __restrict__ keys, const double* __restrict__ vals, int bj, int bk, int R,
    const double* __restrict__ Bf, const double* __restrict__ Cf, double* __restrict__ M,
    int32_t* __restrict__ present, const uint64_t* __restrict__ mB, const uint64_t* __restrict__ mC,
    unsigned long long* __restrict__ rmask) {
  constexpr int NG = kAccBlock / G;
  // a nonzero as the walk reads it: its factor rows' byte offsets (kOff32:
  // both factors below 4 GiB) or its j and k, its value, and its row with
  // the top bit set where j differs from the previous nonzero's
  struct alignas(16) Rec {
    uint32_t j, k;
    double val;
  };
  __shared__ Rec recs[kAccBlock];
  __shared__ uint32_t rows[kAccBlock];
  // per group: its segment's first row (slot 2g) and, if another, its last
  // (slot 2g + 1): row (-1: none) and sums
  __shared__ int32_t brow[2 * NG];
  __shared__ double bsum[2 * NG][S * G];
  __shared__ uint64_t bmask[kMask ? 2 * NG : 1];
  const int g = threadIdx.x / G;
  const int r0 = threadIdx.x % G;
  const int64_t e0 = ((int64_t)blockIdx.x * NG + g) * seg;
  const int64_t e1 = e0 + seg < nnz ? e0 + seg : nnz;
  const uint64_t jm = (1ull << bj) - 1, km = (1ull << bk) - 1;
  uint32_t rr[S];  // in-range ranks for the loads
#pragma unroll
  for (int q = 0; q < S; ++q) rr[q] = r0 + q * G < R ? r0 + q * G : 0;
  const auto factor = [&](const double* __restrict__ f, uint32_t x, int q) -> double {
    if (kOff32) return *reinterpret_cast<const double*>(reinterpret_cast<const char*>(f) + (x + rr[q] * 8u));
    return f[(int64_t)x * R + rr[q]];
  };
  int32_t cur = -1;
  bool first = true;  // cur is the segment's first row
  double acc[S];
#pragma unroll
  for (int q = 0; q < S; ++q) acc[q] = 0.0;
  uint64_t rowm = 0;
  // Bf(j,:) of the last nonzero: within a row the nonzeros come in (j, k)
  // order, so runs of equal j reuse it instead of gathering it again
  double bp[S];
#pragma unroll
  for (int q = 0; q < S; ++q) bp[q] = 0.0;
  const auto to_slot = [&](int slot) {
#pragma unroll
    for (int q = 0; q < S; ++q) bsum[slot][r0 + q * G] = acc[q];
    if (r0 == 0) brow[slot] = cur;
    if (kMask && r0 == 0) bmask[slot] = rowm;
  };
  const uint32_t unit = kOff32 ? (uint32_t)R * 8u : 1u;
  uint64_t nkey = 0;
  double nval = 0.0;
  if (e0 + r0 < e1) {
    nkey = keys[e0 + r0];
    nval = vals[e0 + r0];
  }
  uint32_t jlast = ~0u;  // j of the last nonzero of the previous G
  Rec* const mine = recs + g * G;
  uint32_t* const mrow = rows + g * G;
  for (int64_t base = e0; base < e1; base += G) {  // uniform per group
    const int cnt = (int)(e1 - base < G ? e1 - base : G);
    {
      const uint32_t j = (uint32_t)((nkey >> bk) & jm);
      const uint32_t jb = (uint32_t)__shfl_up((int)j, 1, G);
      mine[r0].j = j * unit;
      mine[r0].k = (uint32_t)(nkey & km) * unit;
      mine[r0].val = nval;
      mrow[r0] = (uint32_t)(nkey >> (bj + bk)) | (j != (r0 ? jb : jlast) ? 0x80000000u : 0u);
      jlast = (uint32_t)__shfl((int)j, G - 1, G);
    }
    __builtin_amdgcn_wave_barrier();
    if (base + G + r0 < e1) {
      nkey = keys[base + G + r0];
      nval = vals[base + G + r0];
    }
    for (int t = 0; t < cnt; t += kAccU) {
      uint32_t rw[kAccU];
      double xv[kAccU], bv[kAccU][S], cv[kAccU][S];
      uint64_t mk[kAccU];
#pragma unroll
      for (int u = 0; u < kAccU; ++u) {
        const int p = t + u < cnt ? t + u : cnt - 1;
        const Rec rec = mine[p];
        rw[u] = mrow[p];
        xv[u] = rec.val;
        if ((int32_t)rw[u] < 0) {  // uniform per group
#pragma unroll
          for (int q = 0; q < S; ++q) bv[u][q] = factor(Bf, rec.j, q);
        }
#pragma unroll
        for (int q = 0; q < S; ++q) cv[u][q] = factor(Cf, rec.k, q);
        if (kMask) mk[u] = mB[rec.j / unit] & mC[rec.k / unit];
      }
#pragma unroll
      for (int u = 0; u < kAccU; ++u) {
        if (t + u >= cnt) break;  // uniform per group
        const int32_t i = (int32_t)(rw[u] & 0x7FFFFFFFu);
        if ((int32_t)rw[u] < 0) {
#pragma unroll
          for (int q = 0; q < S; ++q) bp[q] = bv[u][q];
        }
        if (i != cur) {
          if (cur >= 0) {
            if (first) {
              to_slot(2 * g);
            } else {
#pragma unroll
              for (int q = 0; q < S; ++q)
                if (r0 + q * G < R) M[(int64_t)cur * R + r0 + q * G] = acc[q];
              if (r0 == 0) present[cur] = 1;
              if (kMask && r0 == 0) rmask[cur] = rowm;
            }
            first = false;
          }
          cur = i;
#pragma unroll
          for (int q = 0; q < S; ++q) acc[q] = 0.0;
          rowm = 0;
        }
        if (kMask) rowm |= mk[u];
#pragma unroll
        for (int q = 0; q < S; ++q) acc[q] += (xv[u] * bp[q]) * cv[u][q];
      }
    }
  }
  // the segment's last row, and the slots that hold none
  if (cur < 0 || first) {
    if (r0 == 0) brow[2 * g + 1] = -1;
    if (cur < 0 && r0 == 0) brow[2 * g] = -1;
  }
  if (cur >= 0) to_slot(first ? 2 * g : 2 * g + 1);
  __syncthreads();
  // runs of equal rows over the slots: the group owning a run's first slot
  // sums it
  int lo = 0, hi = 2 * NG - 1;  // the tile's first and last slots that hold a row
  while (lo < 2 * NG && brow[lo] < 0) ++lo;
  while (hi >= 0 && brow[hi] < 0) --hi;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int s0 = 2 * g + h;
    const int32_t row = brow[s0];
    if (row < 0) continue;
    int before = s0 - 1;
    while (before >= lo && brow[before] < 0) --before;
    if (before >= lo && brow[before] == row) continue;
    double sum[S];
#pragma unroll
    for (int q = 0; q < S; ++q) sum[q] = 0.0;
    uint64_t msum = 0;
    for (int s = s0; s <= hi; ++s) {
      if (brow[s] < 0) continue;
      if (brow[s] != row) break;
#pragma unroll
      for (int q = 0; q < S; ++q) sum[q] += bsum[s][r0 + q * G];
      if (kMask) msum |= bmask[s];
    }
    const bool shared = row == brow[lo] || row == brow[hi];  // other tiles may hold parts of it
#pragma unroll
    for (int q = 0; q < S; ++q) {
      const int r = r0 + q * G;
      if (r < R) {
        if (shared) atomicAdd(&M[(int64_t)row * R + r], sum[q]);
        else M[(int64_t)row * R + r] = sum[q];
      }
    }
    if (r0 == 0) present[row] = 1;
    if (kMask && r0 == 0) atomicOr(&rmask[row], (unsigned long long)msum);
  }
}

__global__ __launch_bounds__(256) void k_rows_compact(int32_t n, const int32_t* __restrict__ present,
                                                      const int32_t* __restrict__ off, int32_t* __restrict__ rows,
                                                      const unsigned long long* __restrict__ rmask,
                                                      uint64_t* __restrict__ rows_mask) {
  const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n && present[i]) {
    rows[off[i]] = i;
    if (rmask) rows_mask[off[i]] = rmask[i];
  }
}

// ------------------------------------------------------------------ TTM

constexpr uint64_t kEmptyKey = ~0ull;

__device__ __forceinline__ uint64_t mix64(uint64_t x) {
  x ^= x >> 31;
  x *= 0x7fb5d329728ea185ull;
  x ^= x >> 27;
  x *= 0x81dadef4bc2dd44dull;
  x ^= x >> 33;
  return x;
}

__global__ __launch_bounds__(256) void k_ttm_insert(int64_t nnz, const int32_t* __restrict__ leaf_fiber,
                                                    const int32_t* __restrict__ fiber_root,
                                                    const int32_t* __restrict__ l1_crd,
                                                    const int32_t* __restrict__ l3_crd, int bj,
                                                    unsigned long long* __restrict__ table, uint64_t mask,
                                                    int32_t* __restrict__ leaf_slot) {
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < nnz; e += (int64_t)gridDim.x * blockDim.x) {
    const uint64_t i = (uint32_t)l1_crd[fiber_root[leaf_fiber[e]]];
    const uint64_t j = (uint32_t)l3_crd[e];
    const uint64_t key = (i << bj) | j;
    uint64_t h = mix64(key) & mask;
    for (;;) {
      unsigned long long cur = __hip_atomic_load(&table[h], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (cur == kEmptyKey) {
        cur = atomicCAS(&table[h], (unsigned long long)kEmptyKey, (unsigned long long)key);
        if (cur == kEmptyKey) cur = key;
      }
      if (cur == key) break;
      h = (h + 1) & mask;
    }
    leaf_slot[e] = (int32_t)h;
  }
}

__global__ __launch_bounds__(256) void k_ttm_occupied(int64_t T, const unsigned long long* __restrict__ table,
                                                      int32_t* __restrict__ flag) {
  for (int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; s < T; s += (int64_t)gridDim.x * blockDim.x)
    flag[s] = table[s] != kEmptyKey ? 1 : 0;
}

__global__ __launch_bounds__(256) void k_ttm_collect(int64_t T, const unsigned long long* __restrict__ table,
                                                     const int32_t* __restrict__ off, uint64_t* __restrict__ keys,
                                                     double* __restrict__ slot_payload) {
  for (int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; s < T; s += (int64_t)gridDim.x * blockDim.x) {
    const unsigned long long key = table[s];
    if (key != kEmptyKey) {
      const int32_t q = off[s];
      keys[q] = key;
      slot_payload[q] = __longlong_as_double((long long)s);
    }
  }
}

__global__ __launch_bounds__(256) void k_ttm_rank(int64_t F, const uint64_t* __restrict__ keys,
                                                  const double* __restrict__ slot_payload, int bj,
                                                  int32_t* __restrict__ rank_of_slot, int32_t* __restrict__ out_i,
                                                  int32_t* __restrict__ out_j) {
  const uint64_t jm = (1ull << bj) - 1;
  for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < F; q += (int64_t)gridDim.x * blockDim.x) {
    const int64_t s = (int64_t)__double_as_longlong(slot_payload[q]);
    rank_of_slot[s] = (int32_t)q;
    out_i[q] = (int32_t)(keys[q] >> bj);
    out_j[q] = (int32_t)(keys[q] & jm);
  }
}

// Nonzeros keyed by their fiber's rank and their contracted coordinate:
// key = q << bk | k, value = X.  A stable sort on the q bits groups each
// fiber's nonzeros, still in CSF order (increasing k) inside the fiber, the
// order in which the reference's hash workspace accumulates them.
__global__ __launch_bounds__(256) void k_ttm_keys(int64_t nnz, const int32_t* __restrict__ leaf_fiber,
                                                  const int32_t* __restrict__ l2_crd,
                                                  const double* __restrict__ xvals,
                                                  const int32_t* __restrict__ leaf_slot,
                                                  const int32_t* __restrict__ rank_of_slot, int bk,
                                                  uint64_t* __restrict__ keys, double* __restrict__ vals) {
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < nnz; e += (int64_t)gridDim.x * blockDim.x) {
    const uint64_t q = (uint32_t)rank_of_slot[leaf_slot[e]];
    const uint64_t k = (uint32_t)l2_crd[leaf_fiber[e]];
    keys[e] = (q << bk) | k;
    vals[e] = xvals[e];
  }
}

// Per-fiber sums over the nonzeros grouped by fiber (the keys' high bits are
// the fiber, the low bk bits k; within a fiber k increases), in segments of
// consecutive nonzeros, one segment per group of 16 lanes (a DPP row; a rank
// per lane, S slices of 16 ranks, further ranks on blockIdx.y).
//
// A fiber belongs to the group in whose segment it starts, which follows it
// for kTtmReach nonzeros beyond the segment, so a fiber of at most kTtmReach
// nonzeros is summed by one group from 0.0 in order and stored at once.  A
// longer fiber may fill whole segments beyond that: their groups write
// partial sums, which k_ttm_fixup adds in order (no atomics: the result does
// not depend on timing).  seg_off = exclusive prefix of the fiber starts per
// segment gives each group its first fiber's index, so no list of fibers or
// work items is built.
//
// A group reads 16 keys and values at once (the next 16 in flight while these
// are used) and stages them in LDS with the byte offset of each U row; the U
// rows of 8 / S nonzeros are in flight together (68 VGPRs, 7 wavefronts per
// SIMD: 205 us; 16 in flight at 5 per SIMD 246 us, 4 at 8 per SIMD 211 us, on
// 10M nonzeros in 1.16M fibers, R = 16).  It is bound by the issue of the
// gathers from L2.  One work item per fiber padded to 16 nonzeros took 373 us,
// and its item lists and their combination 130 us more
// where the starts and the fixup now take 35 us.
constexpr int kTtmLanes = 16;
constexpr int kTtmBlock = 256;
constexpr int kTtmGroups = kTtmBlock / kTtmLanes;
constexpr int kTtmReach = 128;
// log2 of the segment: 128 nonzeros, or down to 32 where that leaves fewer
// groups than the chip holds (a group walks its segment one batch after
// another: 200k nonzeros, R = 24, 46 us in segments of 128 and 29 in 32)
constexpr int kTtmSegLogMin = 5, kTtmSegLogMax = 7;
constexpr int kTtmWgPerCu = 7;
constexpr int kTtmInFlight = 8;  // U values per lane in flight
constexpr int kTtmStartRounds = 16;  // strides of 64 nonzeros per wavefront of k_ttm_seg_starts

// Fiber starts per segment of 2^segl nonzeros (nonzero p starts a fiber when
// its key's high bits differ from p - 1's).
__global__ __launch_bounds__(256) void k_ttm_seg_starts(int64_t nnz, int segl, int64_t nseg,
                                                        const uint64_t* __restrict__ keys, int bk,
                                                        int32_t* __restrict__ cnt) {
  const int lane = lane_id();
  const int64_t p0 = ((int64_t)blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave) * (kTtmStartRounds * kWave);
  // the nonzero before each row of 16 lanes, loaded by its first lane; the
  // others take theirs from the lane before
  uint64_t key[kTtmStartRounds], edge[kTtmStartRounds];
#pragma unroll
  for (int u = 0; u < kTtmStartRounds; ++u) {
    const int64_t p = p0 + u * kWave + lane;
    key[u] = p < nnz ? keys[p] : 0;
    edge[u] = (lane & 15) == 0 && p > 0 && p < nnz ? keys[p - 1] : 0;
  }
  uint64_t starts[kTtmStartRounds];  // uniform
#pragma unroll
  for (int u = 0; u < kTtmStartRounds; ++u) {
    const int64_t p = p0 + u * kWave + lane;
    const uint64_t left = dpp_move<0x111, 0xF>(key[u], edge[u]);  // row_shr:1
    starts[u] = __ballot(p < nnz && (p == 0 || (key[u] >> bk) != (left >> bk)));
  }
  // 32-nonzero counts of the wavefront's rounds, a lane each, then the sums
  // of 2^(segl - 5) neighbours
  static_assert(2 * kTtmStartRounds <= kWave, "a lane per 32 nonzeros");
  int32_t c = 0;
#pragma unroll
  for (int u = 0; u < kTtmStartRounds; ++u) {
    if (lane == 2 * u) c = __popc((uint32_t)starts[u]);
    if (lane == 2 * u + 1) c = __popc((uint32_t)(starts[u] >> 32));
  }
  for (int d = 1; d < 1 << (segl - 5); d <<= 1) c += __shfl_down(c, d, kWave);
  const int64_t seg = (p0 + (int64_t)lane * 32) >> segl;
  if (lane < 2 * kTtmStartRounds && (lane & ((1 << (segl - 5)) - 1)) == 0 && seg < nseg) cnt[seg] = c;
}

// kMask: every fiber's fmask is or-ed with the U row masks of its nonzeros.
template <int S, bool kOff32, bool kMask>
__global__ __launch_bounds__(kTtmBlock, kMask ? 4 : 7) void k_ttm_accum(int64_t nnz, int segl, int64_t nseg, int R,
                                                         const uint64_t* __restrict__ keys,
                                                         const double* __restrict__ vals, int bj, int bk,
                                                         const int32_t* __restrict__ seg_off,
                                                         const double* __restrict__ U, double* __restrict__ Y,
                                                         double* __restrict__ part, int32_t* __restrict__ out_i,
                                                         int32_t* __restrict__ out_j,
                                                         const uint64_t* __restrict__ umask,
                                                         unsigned long long* __restrict__ fmask) {
  constexpr int kU = kTtmInFlight / S;  // nonzeros whose U rows are in flight together
  // a nonzero as the sums read it: its U row's byte offset (kOff32: U below
  // 4 GiB) or its k, and its value; one pad record per group keeps the four
  // groups of a wavefront in different LDS banks
  struct alignas(16) Rec {
    uint32_t k, pad;
    double val;
  };
  __shared__ Rec recs[kTtmGroups][kTtmLanes + 1];
  const int g = threadIdx.x / kTtmLanes;
  const int l = threadIdx.x % kTtmLanes;
  const int64_t s = (int64_t)blockIdx.x * kTtmGroups + g;
  if (s >= nseg) return;  // uniform per group; no barrier follows
  const int r0 = blockIdx.y * (S * kTtmLanes) + l;
  const bool lead_block = blockIdx.y == 0;
  const uint32_t km = (uint32_t)((1ull << bk) - 1);  // k < 2^31
  const uint64_t jm = (1ull << bj) - 1;
  const uint32_t unit = kOff32 ? (uint32_t)R * 8u : 1u;
  uint32_t rr[S];  // in-range ranks for the loads
#pragma unroll
  for (int q = 0; q < S; ++q) rr[q] = (uint32_t)min(r0 + q * kTtmLanes, R - 1);
  const int64_t e0 = s << segl;
  const int64_t e1 = min(e0 + (1 << segl), nnz);
  const int64_t lim = min(e1 + kTtmReach, nnz);
  const int32_t q0 = seg_off[s] - 1;  // the fiber running into this segment
  // that fiber is this group's to sum (as a partial sum) when the segments
  // within reach before this one have no start: its own group ends there
  const int back = kTtmReach >> segl;
  const bool filled = s >= back && seg_off[s - back] == q0 + 1;
  uint64_t fprev = e0 > 0 ? keys[e0 - 1] >> bk : ~0ull;
  uint64_t key = 0;
  double val = 0.0;
  if (e0 + l < lim) {
    key = keys[e0 + l];
    val = vals[e0 + l];
  }
  constexpr int32_t kDrop = -1, kPart = -2;
  int32_t dest = filled ? kPart : kDrop;
  int32_t q = q0;
  double acc[S];
#pragma unroll
  for (int x = 0; x < S; ++x) acc[x] = 0.0;
  uint64_t rowm = 0;
  const auto flush = [&]() {
    if (dest == kDrop) return;
    double* const to = dest >= 0 ? Y + (int64_t)dest * R : part + s * R;
#pragma unroll
    for (int x = 0; x < S; ++x)
      if (r0 + x * kTtmLanes < R) to[r0 + x * kTtmLanes] = acc[x];
    if (kMask && l == 0 && lead_block) atomicOr(&fmask[dest >= 0 ? dest : q0], (unsigned long long)rowm);
  };
  Rec* const mine = recs[g];
  for (int64_t base = e0; base < lim; base += kTtmLanes) {  // uniform per group
    const bool beyond = base >= e1;  // following the last fiber out of the segment
    if (beyond && dest < 0) break;
    const uint64_t f = base + l < lim ? key >> bk : fprev;
    const uint64_t left = dpp_move<0x111, 0xF>(f, fprev);  // row_shr:1; lane 0: the nonzero before
    const bool start = base + l < lim && (f != left || base + l == 0);
    const uint32_t hm = (uint32_t)(__ballot(start) >> (threadIdx.x & (kWave - kTtmLanes))) & 0xFFFFu;
    int cnt = (int)min((int64_t)kTtmLanes, lim - base);
    if (beyond && hm) cnt = __builtin_ctz(hm);  // the fiber ends here
    mine[l].k = ((uint32_t)key & km) * unit;
    mine[l].val = val;
    if (!beyond && lead_block && out_i && start) {
      const int32_t at = q + __popc(hm & ((2u << l) - 1u));
      out_i[at] = (int32_t)(f >> bj);
      out_j[at] = (int32_t)(f & jm);
    }
    fprev = row_lane(f, kTtmLanes - 1);
    __builtin_amdgcn_wave_barrier();
    if (base + kTtmLanes + l < lim) {
      key = keys[base + kTtmLanes + l];
      val = vals[base + kTtmLanes + l];
    }
    for (int t = 0; t < cnt; t += kU) {
      double xv[kU], uv[kU][S];
      uint64_t mk[kU];
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        const Rec rec = mine[t + u < cnt ? t + u : cnt - 1];
        xv[u] = rec.val;
#pragma unroll
        for (int x = 0; x < S; ++x) {
          if (kOff32)
            uv[u][x] = *reinterpret_cast<const double*>(reinterpret_cast<const char*>(U) + (rec.k + rr[x] * 8u));
          else
            uv[u][x] = U[(int64_t)rec.k * R + rr[x]];
        }
        if (kMask) mk[u] = umask[rec.k / unit];
      }
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        if (t + u >= cnt) break;  // uniform per group
        if ((hm >> (t + u)) & 1u) {
          flush();
          dest = ++q;
#pragma unroll
          for (int x = 0; x < S; ++x) acc[x] = 0.0;
          rowm = 0;
        }
#pragma unroll
        for (int x = 0; x < S; ++x) acc[x] += xv[u] * uv[u][x];
        if (kMask) rowm |= mk[u];
      }
    }
    if (beyond && hm) break;
  }
  flush();
}

// Fibers longer than their group's reach: Y(q,:) += the partial sums of the
// segments beyond it, in order.  A lane looks at each segment; the first such
// segments of the fibers are listed in LDS and taken by groups of 16 lanes, a
// slice of 16 ranks each, with 16 parts in flight.  20 fibers of 50,000
// nonzeros, R = 64: 90 us; all slices by one group with 4 in flight 457.
__global__ __launch_bounds__(kTtmBlock) void k_ttm_fixup(int segl, int64_t nseg, int R,
                                                         const uint64_t* __restrict__ keys, int bk,
                                                         const int32_t* __restrict__ seg_off,
                                                         const double* __restrict__ part, double* __restrict__ Y) {
  __shared__ int32_t list[kTtmBlock];
  __shared__ int32_t count;
  if (threadIdx.x == 0) count = 0;
  __syncthreads();
  const int back = kTtmReach >> segl;
  const int64_t s0 = back + 1 + (int64_t)blockIdx.x * kTtmBlock;
  // a segment whose leading nonzeros were summed into part: no fiber starts
  // in the segments within reach before it and the fiber goes on
  const auto runs_on = [&](int64_t t) {
    return t < nseg && seg_off[t] == seg_off[t - back] &&
           (keys[t << segl] >> bk) == (keys[(t << segl) - 1] >> bk);
  };
  const int64_t mine = s0 + threadIdx.x;
  if (mine < nseg && seg_off[mine - back] != seg_off[mine - back - 1] && runs_on(mine))
    list[atomicAdd(&count, 1)] = threadIdx.x;
  __syncthreads();
  const int l = threadIdx.x % kTtmLanes;
  const int slices = (R + kTtmLanes - 1) / kTtmLanes;
  for (int c = threadIdx.x / kTtmLanes; c < count * slices; c += kTtmGroups) {  // uniform per group
    const int64_t s = s0 + list[c / slices];
    const int64_t q = seg_off[s] - 1;
    int64_t end = s + 1;
    for (;;) {  // 16 segments looked at together
      const uint32_t stop =
          (uint32_t)(__ballot(!runs_on(end + l)) >> (threadIdx.x & (kWave - kTtmLanes))) & 0xFFFFu;
      end += stop ? __builtin_ctz(stop) : kTtmLanes;
      if (stop) break;
    }
    const int r = c % slices * kTtmLanes + l;
    if (r < R) {
      double acc = Y[q * R + r];
#pragma unroll 16
      for (int64_t t = s; t < end; ++t) acc += part[t * R + r];
      Y[q * R + r] = acc;
    }
  }
}

// ------------------------------------------------------------------ drivers

// Direct TTM grouping: the nonzeros carry packed (i, j, k) keys, and one
// stable radix sort on the (i, j) bits puts each output fiber together, in
// (i, j) order, with its nonzeros in increasing k (the CSF order (i, k, j)
// has them so within a root) -- the order hash_il accumulates them
// (COO_CSF_DCSR_hash_il.h:247-377).
// With a U row mask (bit r: U(k, r) stored), a nonzero whose U row stores
// nothing takes no part (the reference's co-iteration of the contracted
// level with U's rows skips it): it gets the fiber key of row `drop_i`, past
// every root, so the sort moves it to the end, and is counted.
__global__ __launch_bounds__(256) void k_ttm_direct_keys(int64_t nnz, const int32_t* __restrict__ leaf_fiber,
                                                         const int32_t* __restrict__ fiber_root,
                                                         const int32_t* __restrict__ l1_crd,
                                                         const int32_t* __restrict__ l2_crd,
                                                         const int32_t* __restrict__ l3_crd, int bj, int bk,
                                                         uint64_t* __restrict__ keys,
                                                         const uint64_t* __restrict__ umask, uint64_t drop_i,
                                                         unsigned long long* __restrict__ dropped) {
  unsigned long long nd = 0;
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < nnz; e += (int64_t)gridDim.x * blockDim.x) {
    const int32_t f = leaf_fiber[e];
    uint64_t i = (uint32_t)l1_crd[fiber_root[f]];
    const uint64_t k = (uint32_t)l2_crd[f];
    const uint64_t j = (uint32_t)l3_crd[e];
    if (umask[k] == 0) {
      i = drop_i;
      ++nd;
    }
    keys[e] = (i << (bj + bk)) | (j << bk) | k;
  }
  nd = wave_sum(nd);
  if (lane_id() == 0 && nd) atomicAdd(dropped, nd);
}

static int csf_owners(spws_ctx* ctx, const Csf3& x, int32_t** leaf_fiber, int32_t** fiber_root) {
  int rc;
  if ((rc = ctx->obuf[0].ensure((size_t)(x.nnz > 0 ? x.nnz : 1) * 4)) ||
      (rc = ctx->obuf[1].ensure((size_t)(x.nfibers > 0 ? x.nfibers : 1) * 4)))
    return rc;
  *leaf_fiber = ctx->obuf[0].as<int32_t>();
  *fiber_root = ctx->obuf[1].as<int32_t>();
  if ((rc = seg_owner(ctx, x.l3_pos, x.nfibers, x.nnz, OwnerOut{*leaf_fiber}))) return rc;
  return seg_owner(ctx, x.l2_pos, x.nroots, x.nfibers, OwnerOut{*fiber_root});
}

// The nonzeros (at least one) sorted by the key's bits [begin_bit, end_bit)
// straight from the CSF, with no array of unsorted keys: into ctx->keys[i] and
// ctx->vals[i] for the *i returned.
template <bool kMttkrp>
static int csf_sort(spws_ctx* ctx, const Csf3& x, int bj, int bk, int begin_bit, int end_bit, int* i) {
  int rc;
  if ((rc = ctx->obuf[1].ensure((size_t)(x.nfibers > 0 ? x.nfibers : 1) * 8))) return rc;
  uint64_t* fiber_key = ctx->obuf[1].as<uint64_t>();
  const int leaf_shift = kMttkrp ? bj + bk : bk;
  if ((rc = seg_owner(ctx, x.l2_pos, x.nroots, x.nfibers,
                      FiberKeyOut{x.l1_crd, x.l2_crd, kMttkrp ? bk : bj + bk, fiber_key})))
    return rc;
  uint64_t* const keys[2] = {ctx->keys[0].as<uint64_t>(), ctx->keys[1].as<uint64_t>()};
  double* const vals[2] = {ctx->vals[0].as<double>(), ctx->vals[1].as<double>()};
  const int passes = radix_passes(end_bit - begin_bit);
  *i = (passes - 1) & 1;
  const PairSink<uint64_t> out{keys[*i], vals[*i]};
  if (!kMttkrp && div_up(end_bit - begin_bit, passes) > bj)
    return radix_sort_from<uint64_t>(
        ctx, CsfSource<kMttkrp, !kMttkrp>{fiber_key, x.l3_pos, x.l3_crd, x.vals, x.nfibers, leaf_shift}, keys, vals,
        out, x.nnz, begin_bit, end_bit);
  return radix_sort_from<uint64_t>(
      ctx, CsfSource<kMttkrp, false>{fiber_key, x.l3_pos, x.l3_crd, x.vals, x.nfibers, leaf_shift}, keys, vals, out,
      x.nnz, begin_bit, end_bit);
}

// mB / mC (device, J and K entries; both null or both set): per factor row,
// its stored columns as bits (the factors are given dense, zero where not
// stored).  With masks, the rows' stored output columns go to
// ctx->obuf[7] (one uint64 per listed row).
static int mttkrp_run(spws_ctx* ctx, const Csf3& x, int32_t I, int32_t J, int32_t K, int32_t R, const double* Bf,
                      const double* Cf, const uint64_t* mB, const uint64_t* mC, int32_t* nrows_out) {
  int rc = ctx_activate(ctx);
  if (rc) return rc;
  SPWS_REQUIRE(I >= 0 && J >= 0 && K >= 0 && R >= 1 && R <= 64, SPWS_ERR_INVALID,
               "MTTKRP needs non-negative dimensions and 1 <= R <= 64");
  SPWS_REQUIRE((mB == nullptr) == (mC == nullptr), SPWS_ERR_INVALID, "give both factor masks or neither");
  const bool masked = mB != nullptr;
  // with masks, row I is the key of the nonzeros that take no part
  const int bi = bits_of(masked ? (int64_t)I + 1 : (I > 1 ? I : 2)), bj = bits_of(J > 1 ? J : 2),
            bk = bits_of(K > 1 ? K : 2);
  SPWS_REQUIRE(bi + bj + bk <= 64, SPWS_ERR_UNSUPPORTED, "tensor dimensions exceed the 64-bit packed key");
  hipStream_t s = ctx->stream;
  memset(&ctx->stats, 0, sizeof(ctx->stats));
  const size_t nz = (size_t)(x.nnz > 0 ? x.nnz : 1);
  const size_t ii = (size_t)(I > 0 ? I : 1);
  if ((rc = ctx->out_val.ensure(ii * R * 8)) || (rc = ctx->out_aux.ensure(ii * 4 * 2 + 8)) ||
      (rc = ctx->out_crd.ensure(ii * 4)) || (rc = ctx->keys[0].ensure(nz * 8)) || (rc = ctx->keys[1].ensure(nz * 8)) ||
      (rc = ctx->vals[0].ensure(nz * 8)) || (rc = ctx->vals[1].ensure(nz * 8)))
    return rc;
  if (masked && ((rc = ctx->obuf[6].ensure(ii * 8 + 256)) || (rc = ctx->obuf[7].ensure(ii * 8)))) return rc;
  double* M = ctx->out_val.as<double>();
  int32_t* present = ctx->out_aux.as<int32_t>();
  int32_t* poff = present + ii;
  unsigned long long* rmask = masked ? ctx->obuf[6].as<unsigned long long>() : nullptr;
  unsigned long long* dropped = masked ? rmask + ii : nullptr;
  SPWS_HIP(hipMemsetAsync(M, 0, ii * R * 8, s));
  SPWS_HIP(hipMemsetAsync(present, 0, ii * 4, s));
  if (masked) SPWS_HIP(hipMemsetAsync(rmask, 0, ii * 8 + 8, s));
  int64_t kept = x.nnz;
  if (x.nnz > 0) {
    int in = 0;  // which of the two buffers holds the sorted nonzeros
    if (masked) {
      int32_t *leaf_fiber, *fiber_root;
      if ((rc = csf_owners(ctx, x, &leaf_fiber, &fiber_root))) return rc;
      const unsigned g = (unsigned)std::min<int64_t>(div_up(x.nnz, 256), 65536);
      SPWS_LAUNCH(ctx, "mttkrp_keys", k_mttkrp_keys, dim3(g), dim3(256), 0, x.nnz, leaf_fiber, fiber_root,
                  x.l1_crd, x.l2_crd, x.l3_crd, bj, bk, ctx->keys[0].as<uint64_t>(), mB, mC, (uint64_t)I, dropped);
      bool in_alt = false;
      if ((rc = radix_sort_pairs<uint64_t>(ctx, ctx->keys[0].as<uint64_t>(), ctx->vals[0].as<double>(),
                                           ctx->keys[1].as<uint64_t>(), ctx->vals[1].as<double>(), x.nnz, bj + bk,
                                           bj + bk + bi, &in_alt, x.vals)))
        return rc;
      in = in_alt ? 1 : 0;
    } else if ((rc = csf_sort<true>(ctx, x, bj, bk, bj + bk, bj + bk + bi, &in))) {
      return rc;
    }
    const uint64_t* keys = ctx->keys[in].as<uint64_t>();
    const double* vals = ctx->vals[in].as<double>();
    if (masked) {
      // the nonzeros that take part come first after the sort
      int64_t* hd = ctx->host_meta.as<int64_t>();
      SPWS_HIP(hipMemcpyAsync(hd, dropped, 8, hipMemcpyDeviceToHost, s));
      SPWS_HIP(hipStreamSynchronize(s));
      kept = x.nnz - *hd;
    }
    // 16 lanes per group up to rank 16; segments long enough for few atomics,
    // short enough for 8 workgroups per CU (the 32-lane kernel's occupancy)
    const int lanes = R <= 16 ? 16 : 32;
    const int groups = kAccBlock / lanes;
    int cus = 0;
    SPWS_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, ctx->device));
    const int64_t fill = kept / ((int64_t)std::max(cus, 1) * 8 * groups) / 32 * 32;
    const int seg = (int)std::min<int64_t>(kAccSegMax, std::max<int64_t>(kAccSegMin, fill));
    const unsigned ga = (unsigned)div_up(kept, (int64_t)seg * groups);
    // both factors addressed with 32-bit byte offsets while they are below 4 GiB
    const bool off32 = std::max<int64_t>(J, K) * R * 8 <= (int64_t)UINT32_MAX;
#define SPWS_MTTKRP_ACCUM(G, S, MASK)                                                                               \
  do {                                                                                                              \
    if (off32)                                                                                                      \
      SPWS_LAUNCH(ctx, "mttkrp_accum", (k_mttkrp_accum<G, S, MASK, true>), dim3(ga), dim3(kAccBlock), 0, kept, seg, \
                  keys, vals, bj, bk, R, Bf, Cf, M, present, mB, mC, rmask);                                        \
    else                                                                                                            \
      SPWS_LAUNCH(ctx, "mttkrp_accum", (k_mttkrp_accum<G, S, MASK, false>), dim3(ga), dim3(kAccBlock), 0, kept,     \
                  seg, keys, vals, bj, bk, R, Bf, Cf, M, present, mB, mC, rmask);                                   \
  } while (0)
    if (kept > 0) {
      if (R <= 16 && masked) SPWS_MTTKRP_ACCUM(16, 1, true);
      else if (R <= 16) SPWS_MTTKRP_ACCUM(16, 1, false);
      else if (R <= 32 && masked) SPWS_MTTKRP_ACCUM(32, 1, true);
      else if (R <= 32) SPWS_MTTKRP_ACCUM(32, 1, false);
      else if (masked) SPWS_MTTKRP_ACCUM(32, 2, true);
      else SPWS_MTTKRP_ACCUM(32, 2, false);
    }
#undef SPWS_MTTKRP_ACCUM
    ctx->stats.products = kept * (int64_t)R;
  }
  if ((rc = exclusive_scan<int32_t, int32_t>(ctx, present, poff, I))) return rc;
  if (I > 0)
    SPWS_LAUNCH(ctx, "rows_compact", k_rows_compact, dim3((unsigned)div_up(I, 256)), dim3(256), 0, I, present, poff,
                ctx->out_crd.as<int32_t>(), (const unsigned long long*)rmask,
                masked ? ctx->obuf[7].as<uint64_t>() : (uint64_t*)nullptr);
  int32_t* hm = ctx->host_meta.as<int32_t>();
  SPWS_HIP(hipMemcpyAsync(hm, poff + I, 4, hipMemcpyDeviceToHost, s));
  SPWS_HIP(hipStreamSynchronize(s));
  *nrows_out = *hm;
  ctx->stats.nnz = (int64_t)(*hm) * R;
  return SPWS_OK;
}

// Fiber starts per segment (2^*segl nonzeros) of the grouped nonzeros into
// obuf[2] and their prefix into obuf[5], whose last entry is the number of
// fibers.
static int ttm_seg_offsets(spws_ctx* ctx, int64_t nnz, const uint64_t* nkeys, int bk, int* segl) {
  int rc, cus = 0;
  SPWS_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, ctx->device));
  int l = kTtmSegLogMin;
  while (l < kTtmSegLogMax && (nnz >> (l + 1)) >= (int64_t)cus * kTtmWgPerCu * kTtmGroups) ++l;
  *segl = l;
  const int64_t nseg = div_up(nnz, (int64_t)1 << l);
  if ((rc = ctx->obuf[2].ensure((size_t)nseg * 4 + 4)) || (rc = ctx->obuf[5].ensure(((size_t)nseg + 1) * 4))) return rc;
  int32_t* cnt = ctx->obuf[2].as<int32_t>();
  if (nseg > 0)
    SPWS_LAUNCH(ctx, "ttm_starts", k_ttm_seg_starts, dim3((unsigned)div_up(nnz, 256 * kTtmStartRounds)), dim3(256), 0,
                nnz, l, nseg, nkeys, bk, cnt);
  return exclusive_scan<int32_t, int32_t>(ctx, cnt, ctx->obuf[5].as<int32_t>(), nseg);
}

// Per-fiber sums over the grouped nonzeros (after ttm_seg_offsets) into Y,
// and, with out_i, the fibers' coordinates.  umask and fmask: both or neither
// (fmask zero on entry).
static int ttm_accumulate(spws_ctx* ctx, int64_t nnz, int segl, int32_t R, int bj, int bk, const uint64_t* nkeys,
                          const double* nvals, const double* U, double* Y, int32_t* out_i, int32_t* out_j,
                          const uint64_t* umask, unsigned long long* fmask) {
  int rc;
  const int64_t nseg = div_up(nnz, (int64_t)1 << segl);
  if ((rc = ctx->obuf[3].ensure((size_t)nseg * R * 8))) return rc;
  double* part = ctx->obuf[3].as<double>();
  const int32_t* seg_off = ctx->obuf[5].as<int32_t>();
  const bool off32 = ((int64_t)1 << bk) * R * 8 <= (int64_t)UINT32_MAX;  // every U offset fits in 32 bits
  const int slices = R <= 16 ? 1 : R <= 32 ? 2 : 4;
  const dim3 grid((unsigned)div_up(nseg, kTtmGroups), (unsigned)div_up(R, slices * kTtmLanes));
#define SPWS_TTM_ACCUM(S, OFF32, MASK)                                                                            \
  SPWS_LAUNCH(ctx, "ttm_accum", (k_ttm_accum<S, OFF32, MASK>), grid, dim3(kTtmBlock), 0, nnz, segl, nseg, R, nkeys, \
              nvals, bj, bk, seg_off, U, Y, part, out_i, out_j, umask, fmask)
#define SPWS_TTM_ACCUM_S(S)                       \
  do {                                            \
    if (umask && off32) SPWS_TTM_ACCUM(S, true, true);        \
    else if (umask) SPWS_TTM_ACCUM(S, false, true); \
    else if (off32) SPWS_TTM_ACCUM(S, true, false); \
    else SPWS_TTM_ACCUM(S, false, false);         \
  } while (0)
  switch (slices) {
    case 1: SPWS_TTM_ACCUM_S(1); break;
    case 2: SPWS_TTM_ACCUM_S(2); break;
    default: SPWS_TTM_ACCUM_S(4); break;
  }
#undef SPWS_TTM_ACCUM_S
#undef SPWS_TTM_ACCUM
  const int64_t late = nseg - (kTtmReach >> segl) - 1;  // segments beyond the first group's reach
  if (late > 0)
    SPWS_LAUNCH(ctx, "ttm_fixup", k_ttm_fixup, dim3((unsigned)div_up(late, kTtmBlock)), dim3(kTtmBlock), 0, segl,
                nseg, R, nkeys, bk, seg_off, (const double*)part, Y);
  return SPWS_OK;
}

// umask (device, K entries, or null): per U row, its stored columns as bits
// (U given dense, zero where not stored); the fibers' stored output columns
// then go to ctx->obuf[6] after its first 256 bytes (one uint64 per fiber).
static int ttm_run(spws_ctx* ctx, const Csf3& x, int32_t I, int32_t J, int32_t K, int32_t R, const double* U,
                   const uint64_t* umask, int64_t* nfib_out) {
  int rc = ctx_activate(ctx);
  if (rc) return rc;
  SPWS_REQUIRE(I >= 0 && J >= 0 && K >= 0 && R >= 1 && R <= 256, SPWS_ERR_INVALID,
               "TTM needs non-negative dimensions and 1 <= R <= 256");
  const bool masked = umask != nullptr;
  SPWS_REQUIRE(!masked || R <= 64, SPWS_ERR_UNSUPPORTED, "a U row mask needs R <= 64");
  // the roots-and-windows path (no sort of the whole tensor) unless the
  // sorting path is asked for or the shapes are outside what it supports
  if (!masked && ctx->ttm_method != 1) {
    bool handled = false;
    if ((rc = ttm_roots_run(ctx, x, I, J, K, R, U, ctx->ttm_method == 2, nfib_out, &handled))) return rc;
    if (handled) return SPWS_OK;
    SPWS_REQUIRE(ctx->ttm_method != 2, SPWS_ERR_UNSUPPORTED,
                 "the roots-and-windows TTM needs 1 <= R <= 64, at most 4,096 column windows of 1024 / R' "
                 "columns (R' = R rounded up to 16, 32 or 64), J < 2^23 and K times the window below 2^32");
  }
  // with a mask, root I is the key of the nonzeros that take no part
  const int bi = bits_of(masked ? (int64_t)I + 1 : (I > 1 ? I : 2)), bj = bits_of(J > 1 ? J : 2);
  SPWS_REQUIRE(bi + bj <= 63, SPWS_ERR_UNSUPPORTED, "tensor dimensions exceed the 64-bit fiber key");
  SPWS_REQUIRE(x.nnz < ((int64_t)1 << 30), SPWS_ERR_UNSUPPORTED, "TTM supports fewer than 2^30 nonzeros");
  hipStream_t s = ctx->stream;
  memset(&ctx->stats, 0, sizeof(ctx->stats));
  const size_t nz = (size_t)(x.nnz > 0 ? x.nnz : 1);
  const int bk_all = bits_of(K > 1 ? K : 2);
  const bool direct = bi + bj + bk_all <= 64;
  SPWS_REQUIRE(!masked || direct, SPWS_ERR_UNSUPPORTED,
               "a U row mask needs the root, leaf and contracted coordinates within 64 bits");
  // hash path: a table of 2 * nnz (power of two) slots
  uint64_t T = 1024;
  while (!direct && T < 2 * (uint64_t)nz) T <<= 1;
  const size_t nflag = T + 1;
  if ((rc = ctx->keys[0].ensure(nz * 8)) || (rc = ctx->keys[1].ensure(nz * 8)) || (rc = ctx->vals[0].ensure(nz * 8)) ||
      (rc = ctx->vals[1].ensure(nz * 8)))
    return rc;
  if (!direct && ((rc = ctx->row_nnz.ensure(nflag * 4 * 2)) || (rc = ctx->wide_tab.ensure(T * 8)) ||
                  (rc = ctx->slot_crd.ensure(nz * 4))))
    return rc;
  unsigned long long* table = ctx->wide_tab.as<unsigned long long>();
  int32_t* leaf_slot = ctx->slot_crd.as<int32_t>();
  int32_t* flag = ctx->row_nnz.as<int32_t>();
  int32_t* off = flag + nflag;
  int32_t* hm = ctx->host_meta.as<int32_t>();
  int64_t F = 0;
  if (x.nnz > 0 && direct) {
    // one sort of the nonzeros on (i, j, k)
    const int bk = bk_all;
    // the sort covers (i, j) only: within an i slice the CSF order already
    // has each (i, j)'s nonzeros in increasing k, and the sort is stable
    int in = 0;  // which of the two buffers holds the sorted nonzeros
    unsigned long long* dropped = nullptr;
    if (masked) {
      const unsigned g = (unsigned)std::min<int64_t>(div_up(x.nnz, 256), 65536);
      int32_t *leaf_fiber, *fiber_root;
      if ((rc = csf_owners(ctx, x, &leaf_fiber, &fiber_root))) return rc;
      if ((rc = ctx->obuf[6].ensure(256))) return rc;
      dropped = ctx->obuf[6].as<unsigned long long>();
      SPWS_HIP(hipMemsetAsync(dropped, 0, 8, s));
      SPWS_LAUNCH(ctx, "ttm_keys", k_ttm_direct_keys, dim3(g), dim3(256), 0, x.nnz, leaf_fiber, fiber_root,
                  x.l1_crd, x.l2_crd, x.l3_crd, bj, bk, ctx->keys[0].as<uint64_t>(), umask, (uint64_t)I, dropped);
      bool alt = false;
      if ((rc = radix_sort_pairs<uint64_t>(ctx, ctx->keys[0].as<uint64_t>(), ctx->vals[0].as<double>(),
                                           ctx->keys[1].as<uint64_t>(), ctx->vals[1].as<double>(), x.nnz, bk,
                                           bi + bj + bk, &alt, x.vals)))
        return rc;
      in = alt ? 1 : 0;
    } else if ((rc = csf_sort<false>(ctx, x, bj, bk, bk, bi + bj + bk, &in))) {
      return rc;
    }
    const uint64_t* nkeys = ctx->keys[in].as<uint64_t>();
    const double* nvals = ctx->vals[in].as<double>();
    // the nonzeros that take part come first after the sort
    int64_t kept = x.nnz;
    if (masked) {
      int64_t* hd = ctx->host_meta.as<int64_t>() + 1;
      SPWS_HIP(hipMemcpyAsync(hd, dropped, 8, hipMemcpyDeviceToHost, s));
      SPWS_HIP(hipStreamSynchronize(s));
      kept = x.nnz - *hd;
    }
    int segl;
    if ((rc = ttm_seg_offsets(ctx, kept, nkeys, bk, &segl))) return rc;
    SPWS_HIP(hipMemcpyAsync(hm, ctx->obuf[5].as<int32_t>() + div_up(kept, (int64_t)1 << segl), 4,
                            hipMemcpyDeviceToHost, s));
    SPWS_HIP(hipStreamSynchronize(s));
    F = *hm;
    if ((rc = ctx->out_crd.ensure((size_t)(F > 0 ? F : 1) * 4 * 2)) ||
        (rc = ctx->out_val.ensure((size_t)(F > 0 ? F : 1) * R * 8)))
      return rc;
    int32_t* out_i = ctx->out_crd.as<int32_t>();
    unsigned long long* fmask = nullptr;
    if (masked) {
      if ((rc = ctx->obuf[6].ensure(256 + (size_t)F * 8))) return rc;
      fmask = reinterpret_cast<unsigned long long*>(ctx->obuf[6].as<char>() + 256);
      if (F > 0) SPWS_HIP(hipMemsetAsync(fmask, 0, (size_t)F * 8, s));
    }
    if (kept > 0 && (rc = ttm_accumulate(ctx, kept, segl, R, bj, bk, nkeys, nvals, U, ctx->out_val.as<double>(), out_i,
                                         out_i + F, umask, fmask)))
      return rc;
    ctx->stats.products = kept * (int64_t)R;
  } else if (x.nnz > 0) {
    int32_t *leaf_fiber, *fiber_root;
    if ((rc = csf_owners(ctx, x, &leaf_fiber, &fiber_root))) return rc;
    SPWS_HIP(hipMemsetAsync(table, 0xff, T * 8, s));
    const unsigned g = (unsigned)std::min<int64_t>(div_up(x.nnz, 256), 65536);
    SPWS_LAUNCH(ctx, "ttm_insert", k_ttm_insert, dim3(g), dim3(256), 0, x.nnz, leaf_fiber, fiber_root, x.l1_crd,
                x.l3_crd, bj, table, (uint64_t)(T - 1), leaf_slot);
    const unsigned gt = (unsigned)std::min<int64_t>(div_up((int64_t)T, 256), 65536);
    SPWS_LAUNCH(ctx, "ttm_occupied", k_ttm_occupied, dim3(gt), dim3(256), 0, (int64_t)T, table, flag);
    if ((rc = exclusive_scan<int32_t, int32_t>(ctx, flag, off, (int64_t)T))) return rc;
    SPWS_HIP(hipMemcpyAsync(hm, off + T, 4, hipMemcpyDeviceToHost, s));
    SPWS_HIP(hipStreamSynchronize(s));
    F = *hm;
    uint64_t* keys = ctx->keys[0].as<uint64_t>();
    double* pay = ctx->vals[0].as<double>();
    SPWS_LAUNCH(ctx, "ttm_collect", k_ttm_collect, dim3(gt), dim3(256), 0, (int64_t)T, table, off, keys, pay);
    bool in_alt = false;
    if ((rc = radix_sort_pairs<uint64_t>(ctx, keys, pay, ctx->keys[1].as<uint64_t>(), ctx->vals[1].as<double>(), F, 0,
                                         bi + bj, &in_alt)))
      return rc;
    if (in_alt) {
      keys = ctx->keys[1].as<uint64_t>();
      pay = ctx->vals[1].as<double>();
    }
    // rank_of_slot reuses the flag array (T entries)
    int32_t* rank_of_slot = flag;
    if ((rc = ctx->out_crd.ensure((size_t)(F > 0 ? F : 1) * 4 * 2)) ||
        (rc = ctx->out_val.ensure((size_t)(F > 0 ? F : 1) * R * 8)))
      return rc;
    int32_t* out_i = ctx->out_crd.as<int32_t>();
    int32_t* out_j = out_i + F;
    const unsigned gf = (unsigned)std::min<int64_t>(div_up(F, 256), 65536);
    SPWS_LAUNCH(ctx, "ttm_rank", k_ttm_rank, dim3(gf), dim3(256), 0, F, keys, pay, bj, rank_of_slot, out_i, out_j);
    double* Y = ctx->out_val.as<double>();
    // group each fiber's nonzeros (stable sort on the fiber rank), then one
    // pass of in-order sums per fiber
    const int bq = bits_of(F > 1 ? F : 2);
    const int bk = bits_of(K > 1 ? K : 2);
    SPWS_REQUIRE(bq + bk <= 64, SPWS_ERR_UNSUPPORTED, "fiber count and K exceed the 64-bit sort key");
    uint64_t* nkeys = ctx->keys[0].as<uint64_t>();
    double* nvals = ctx->vals[0].as<double>();
    SPWS_LAUNCH(ctx, "ttm_keys", k_ttm_keys, dim3(g), dim3(256), 0, x.nnz, leaf_fiber, x.l2_crd, x.vals, leaf_slot,
                rank_of_slot, bk, nkeys, nvals);
    bool alt2 = false;
    if ((rc = radix_sort_pairs<uint64_t>(ctx, nkeys, nvals, ctx->keys[1].as<uint64_t>(), ctx->vals[1].as<double>(),
                                         x.nnz, bk, bk + bq, &alt2)))
      return rc;
    if (alt2) {
      nkeys = ctx->keys[1].as<uint64_t>();
      nvals = ctx->vals[1].as<double>();
    }
    int segl;
    if ((rc = ttm_seg_offsets(ctx, x.nnz, nkeys, bk, &segl)) ||
        (rc = ttm_accumulate(ctx, x.nnz, segl, R, bj, bk, nkeys, nvals, U, Y, nullptr, nullptr, nullptr, nullptr)))
      return rc;
    ctx->stats.products = x.nnz * (int64_t)R;
  } else {
    if ((rc = ctx->out_crd.ensure(8)) || (rc = ctx->out_val.ensure(8))) return rc;
  }
  SPWS_HIP(hipStreamSynchronize(s));
  *nfib_out = F;
  ctx->stats.nnz = F * R;
  return SPWS_OK;
}

}  // namespace spws

using namespace spws;

extern "C" {

int spws_ctx_set_ttm_method(spws_ctx* ctx, int32_t method) {
  SPWS_REQUIRE(ctx != nullptr, SPWS_ERR_INVALID, "null context");
  SPWS_REQUIRE(method >= 0 && method <= 2, SPWS_ERR_INVALID, "TTM method %d is not 0, 1 or 2", method);
  ctx->ttm_method = method;
  return SPWS_OK;
}

int spws_mttkrp(spws_ctx* ctx, int32_t I, int32_t J, int32_t K, int32_t R, int32_t nroots, const int32_t* l1_crd,
                const int32_t* l2_pos, const int32_t* l2_crd, int32_t nfibers, const int32_t* l3_pos,
                const int32_t* l3_crd, const double* vals, int64_t nnz, const double* Bf, const double* Cf,
                int32_t* nrows, int32_t** rows, double** M) {
  return spws_mttkrp_masked(ctx, I, J, K, R, nroots, l1_crd, l2_pos, l2_crd, nfibers, l3_pos, l3_crd, vals, nnz, Bf,
                            Cf, nullptr, nullptr, nrows, rows, nullptr, M);
}

int spws_mttkrp_masked(spws_ctx* ctx, int32_t I, int32_t J, int32_t K, int32_t R, int32_t nroots,
                       const int32_t* l1_crd, const int32_t* l2_pos, const int32_t* l2_crd, int32_t nfibers,
                       const int32_t* l3_pos, const int32_t* l3_crd, const double* vals, int64_t nnz, const double* Bf,
                       const double* Cf, const uint64_t* Bmask, const uint64_t* Cmask, int32_t* nrows,
                       int32_t** rows, uint64_t** row_mask, double** M) {
  SPWS_REQUIRE(nnz >= 0 && nroots >= 0 && nfibers >= 0, SPWS_ERR_INVALID, "negative size");
  SPWS_REQUIRE(nnz == 0 || (l1_crd && l2_pos && l2_crd && l3_pos && l3_crd && vals && Bf && Cf), SPWS_ERR_INVALID,
               "null pointer argument");
  SPWS_REQUIRE(nnz < ((int64_t)1 << 31), SPWS_ERR_UNSUPPORTED, "MTTKRP supports fewer than 2^31 nonzeros");
  Csf3 x{nroots, l1_crd, l2_pos, l2_crd, nfibers, l3_pos, l3_crd, vals, nnz};
  int32_t nr = 0;
  int rc = mttkrp_run(ctx, x, I, J, K, R, Bf, Cf, Bmask, Cmask, &nr);
  if (rc) return rc;
  if (nrows) *nrows = nr;
  if (rows) *rows = ctx->out_crd.as<int32_t>();
  if (row_mask) *row_mask = Bmask ? ctx->obuf[7].as<uint64_t>() : nullptr;
  if (M) *M = ctx->out_val.as<double>();
  return SPWS_OK;
}

int spws_ttm(spws_ctx* ctx, int32_t I, int32_t J, int32_t K, int32_t R, int32_t nroots, const int32_t* l1_crd,
             const int32_t* l2_pos, const int32_t* l2_crd, int32_t nfibers, const int32_t* l3_pos,
             const int32_t* l3_crd, const double* vals, int64_t nnz, const double* U, int64_t* nfib,
             int32_t** fib_i, int32_t** fib_j, double** Y) {
  return spws_ttm_masked(ctx, I, J, K, R, nroots, l1_crd, l2_pos, l2_crd, nfibers, l3_pos, l3_crd, vals, nnz, U,
                         nullptr, nfib, fib_i, fib_j, nullptr, Y);
}

int spws_ttm_masked(spws_ctx* ctx, int32_t I, int32_t J, int32_t K, int32_t R, int32_t nroots,
                    const int32_t* l1_crd, const int32_t* l2_pos, const int32_t* l2_crd, int32_t nfibers,
                    const int32_t* l3_pos, const int32_t* l3_crd, const double* vals, int64_t nnz, const double* U,
                    const uint64_t* Umask, int64_t* nfib, int32_t** fib_i, int32_t** fib_j, uint64_t** fib_mask,
                    double** Y) {
  SPWS_REQUIRE(nnz >= 0 && nroots >= 0 && nfibers >= 0, SPWS_ERR_INVALID, "negative size");
  SPWS_REQUIRE(nnz == 0 || (l1_crd && l2_pos && l2_crd && l3_pos && l3_crd && vals && U), SPWS_ERR_INVALID,
               "null pointer argument");
  Csf3 x{nroots, l1_crd, l2_pos, l2_crd, nfibers, l3_pos, l3_crd, vals, nnz};
  int64_t F = 0;
  int rc = ttm_run(ctx, x, I, J, K, R, U, Umask, &F);
  if (rc) return rc;
  if (nfib) *nfib = F;
  if (fib_i) *fib_i = ctx->out_crd.as<int32_t>();
  if (fib_j) *fib_j = ctx->out_crd.as<int32_t>() + F;
  if (fib_mask) *fib_mask = Umask ? reinterpret_cast<uint64_t*>(ctx->obuf[6].as<char>() + 256) : nullptr;
  if (Y) *Y = ctx->out_val.as<double>();
  return SPWS_OK;
}

}  // extern "C"
