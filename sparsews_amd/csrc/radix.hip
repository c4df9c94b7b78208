// The sort of (key, value) arrays (radix.hpp), instantiated once, and the tile
// offsets that every sort shares.
#include "radix.hpp"

namespace spws {

// hist's rows [c per, (c + 1) per) in place to their exclusive prefixes, their
// sum to row c of chunk; a digit per thread.
static __global__ __launch_bounds__(kSortBlock) void k_radix_chunks(int32_t* __restrict__ hist, int64_t ntiles,
                                                                    int64_t per, int nb,
                                                                    int32_t* __restrict__ chunk) {
  const int d = blockIdx.y * kSortBlock + threadIdx.x;
  if (d >= nb) return;
  const int64_t t0 = (int64_t)blockIdx.x * per;
  const int64_t t1 = t0 + per < ntiles ? t0 + per : ntiles;
  int32_t run = 0;
  for (int64_t t = t0; t < t1; t += kSortChunk) {
    int32_t c[kSortChunk];
#pragma unroll
    for (int q = 0; q < kSortChunk; ++q) c[q] = t + q < t1 ? hist[(t + q) * nb + d] : 0;
#pragma unroll
    for (int q = 0; q < kSortChunk; ++q) {
      if (t + q < t1) hist[(t + q) * nb + d] = run;
      run += c[q];
    }
  }
  chunk[(int64_t)blockIdx.x * nb + d] = run;
}

// The chunks' rows to their exclusive prefixes, the digits' totals to row n:
// 64 digits per workgroup, the rows split over its wavefronts.
constexpr int kSortDigitsBlock = 1024;
static __global__ __launch_bounds__(kSortDigitsBlock) void k_radix_digits(int32_t* __restrict__ chunk, int64_t n,
                                                                          int nb) {
  constexpr int kWaves = kSortDigitsBlock / kWave;
  __shared__ int32_t part[kWaves][kWave];
  const int lane = lane_id();
  const int w = threadIdx.x / kWave;
  const int d = blockIdx.x * kWave + lane;
  const int64_t per = (n + kWaves - 1) / kWaves;
  const int64_t c0 = w * per < n ? w * per : n;
  const int64_t c1 = c0 + per < n ? c0 + per : n;
  int32_t sum = 0;
  if (d < nb) {
#pragma unroll 8
    for (int64_t c = c0; c < c1; ++c) sum += chunk[c * nb + d];
  }
  part[w][lane] = sum;
  __syncthreads();
  int32_t run = 0, all = 0;
#pragma unroll
  for (int q = 0; q < kWaves; ++q) {
    const int32_t v = part[q][lane];
    run += q < w ? v : 0;
    all += v;
  }
  if (d >= nb) return;
#pragma unroll 8
  for (int64_t c = c0; c < c1; ++c) {
    const int32_t v = chunk[c * nb + d];
    chunk[c * nb + d] = run;
    run += v;
  }
  if (w == 0) chunk[n * nb + d] = all;
}

int radix_offsets(spws_ctx* ctx, int32_t* hist, int64_t ntiles, int nb, int32_t* chunk) {
  const int64_t per = radix_chunk_tiles(ntiles), chunks = div_up(ntiles, per);
  SPWS_LAUNCH(ctx, "radix_chunks", k_radix_chunks, dim3((unsigned)chunks, (unsigned)div_up(nb, kSortBlock)),
              dim3(kSortBlock), 0, hist, ntiles, per, nb, chunk);
  if (chunks > 1)
    SPWS_LAUNCH(ctx, "radix_digits", k_radix_digits, dim3((unsigned)div_up(nb, kWave)), dim3(kSortDigitsBlock), 0,
                chunk, chunks, nb);
  return SPWS_OK;
}

template <class K>
int radix_sort_pairs(spws_ctx* ctx, K* keys, double* vals, K* keys_alt, double* vals_alt, int64_t n, int begin_bit,
                     int end_bit, bool* in_alt, const double* vals_first) {
  *in_alt = false;
  if (n <= 0) return SPWS_OK;
  if (n <= 1 || end_bit <= begin_bit) {
    if (vals_first) SPWS_HIP(hipMemcpyAsync(vals, vals_first, (size_t)n * 8, hipMemcpyDeviceToDevice, ctx->stream));
    return SPWS_OK;
  }
  SPWS_REQUIRE(n < ((int64_t)1 << 31), SPWS_ERR_UNSUPPORTED, "radix sort of %lld keys exceeds int32 offsets",
               (long long)n);
  // the first pass writes the _alt buffers
  K* const kb[2] = {keys_alt, keys};
  double* const vb[2] = {vals_alt, vals};
  const int last = (radix_passes(end_bit - begin_bit) - 1) & 1;
  *in_alt = last == 0;
  return radix_sort_from<K>(ctx, PairSource<K>{keys, vals_first ? vals_first : vals}, kb, vb,
                            PairSink<K>{kb[last], vb[last]}, n, begin_bit, end_bit);
}

template int radix_sort_pairs<uint32_t>(spws_ctx*, uint32_t*, double*, uint32_t*, double*, int64_t, int, int, bool*,
                                        const double*);
template int radix_sort_pairs<uint64_t>(spws_ctx*, uint64_t*, double*, uint64_t*, double*, int64_t, int, int, bool*,
                                        const double*);

}  // namespace spws
