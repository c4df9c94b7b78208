// The sort of (key, value) arrays (radix.hpp), instantiated once.
#include "radix.hpp"

namespace spws {

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
