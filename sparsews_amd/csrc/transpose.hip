// CSR transpose on the device, the second half of the reference's non-fused
// transposed product (benchmark/CSC_CSR_T/nonfuse/CSC_CSR_T_hash.h:352-400,
// transpose(A, B) with A = B^T): there the entries of each column are
// counted, the counts prefixed into the output row pointers, and the input
// rows scattered in row order, so every output row lists its columns (the
// input rows) in increasing order.
//
// Here each entry is a key (column << 32 | row) carrying its value; a stable
// LSD radix sort on the column bits alone keeps the row order of equal columns
// (the input is row-major).  The sort's first pass makes the keys from the CSR
// (CsrSource) and its last one writes the output arrays (TransposeSink), so
// the keys go through memory once less at either end; the columns are kept
// beside them, and each output row pointer is a binary search in the sorted
// columns.  Pure data movement: the output is bit-identical to the
// reference's.  200k x 200k, 6.4M entries: 274 us with keys made and taken
// apart by passes of their own and counted columns, 189 us now (two passes,
// 2.9 TB/s in the scatters).
#include <mutex>
#include <utility>

#include "radix.hpp"

namespace spws {
namespace {

// bits that hold every column index below n
int column_bits(int32_t n) {
  int bits = 1;
  while (bits < 31 && ((int64_t)1 << bits) < (int64_t)n) ++bits;
  return bits;
}

// CSR entries as the sort's first pass reads them (row pointers int32, or
// int64 as the outer product returns them; nnz stays below 2^31 either way)
template <typename PosT>
struct CsrSource {
  static constexpr bool kOwners = true, kOwnedDigits = false;
  const PosT* __restrict__ pos;
  const int32_t* __restrict__ crd;
  const double* __restrict__ vals;
  int32_t m;
  using Raw = uint32_t;
  __device__ uint32_t raw(int64_t e) const { return (uint32_t)crd[e]; }
  __device__ double val(int64_t e) const { return vals[e]; }
  __device__ uint64_t digit_bits(uint32_t col) const { return (uint64_t)col << 32; }
  __device__ void owners(int64_t base, int64_t end, uint32_t* marks, int32_t (&own)[kSortItems]) const {
    tile_owners<kSortBlock, kSortItems>(pos, m, base, end, marks, own);
  }
  __device__ uint64_t key(uint32_t col, int32_t row) const { return ((uint64_t)col << 32) | (uint32_t)row; }
};

// where the last pass writes: the transpose's column indices (the input
// rows) and values, and the sorted columns
struct TransposeSink {
  uint32_t* __restrict__ cols;
  int32_t* __restrict__ out_crd;
  double* __restrict__ out_vals;
  __device__ void key(int64_t at, uint64_t k) const {
    cols[at] = (uint32_t)(k >> 32);
    out_crd[at] = (int32_t)(uint32_t)k;
  }
  __device__ void val(int64_t at, double v) const { out_vals[at] = v; }
};

// out_pos[c] = the first of the nnz sorted columns that is at least c, c <= n
__global__ __launch_bounds__(256) void k_tr_pos(int32_t n, int32_t nnz, const uint32_t* __restrict__ cols,
                                                int32_t* __restrict__ out_pos) {
  for (int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; c <= n; c += (int64_t)gridDim.x * blockDim.x) {
    int32_t lo = 0, hi = nnz;
    while (lo < hi) {
      const int32_t mid = lo + (hi - lo) / 2;
      if ((int64_t)cols[mid] < c) lo = mid + 1; else hi = mid;
    }
    out_pos[c] = lo;
  }
}

static bool overlap(const void* a, size_t an, const void* b, size_t bn) {
  const uintptr_t x = reinterpret_cast<uintptr_t>(a), y = reinterpret_cast<uintptr_t>(b);
  return x < y + bn && y < x + an;
}

// The transpose on a context: its workspaces are the context's buffers
// (tr_keys, tr_vals, and the radix scratch).  Outputs may lie in the inputs'
// memory.
template <typename PosT>
static int transpose_run(spws_ctx* ctx, int32_t m, int32_t n, int64_t nnz, const PosT* pos, const int32_t* crd,
                         const double* vals, int32_t* out_pos, int32_t* out_crd, double* out_vals) {
  int rc;
  const size_t nn = (size_t)(nnz > 0 ? nnz : 1);
  if ((rc = ctx->tr_keys.ensure(2 * nn * 8)) || (rc = ctx->tr_vals.ensure(2 * nn * 8))) return rc;
  uint64_t* const keys[2] = {ctx->tr_keys.as<uint64_t>(), ctx->tr_keys.as<uint64_t>() + nn};
  double* const kv[2] = {ctx->tr_vals.as<double>(), ctx->tr_vals.as<double>() + nn};
  int bits = column_bits(n);
  // A single pass writes the outputs while other workgroups still read the
  // inputs.  Where they share memory the columns are sorted on further bits,
  // all zero, in two passes: only the first reads the inputs.
  if (radix_passes(bits) == 1) {
    bool shared = false;
    for (const auto& [out, on] : {std::pair<const void*, size_t>{out_crd, nn * 4}, {out_vals, nn * 8}})
      shared = shared || overlap(out, on, pos, ((size_t)m + 1) * sizeof(PosT)) || overlap(out, on, crd, nn * 4) ||
               overlap(out, on, vals, nn * 8);
    if (shared) bits = kSortDigitMax + 1;
  }
  // the sorted columns take the key buffer that the last pass does not read
  uint32_t* const cols = reinterpret_cast<uint32_t*>(keys[(radix_passes(bits) - 1) & 1]);
  const bool any = m > 0 && nnz > 0;
  if (any && (rc = radix_sort_from<uint64_t>(ctx, CsrSource<PosT>{pos, crd, vals, m}, keys, kv,
                                             TransposeSink{cols, out_crd, out_vals}, nnz, 32, 32 + bits)))
    return rc;
  SPWS_LAUNCH(ctx, "tr_pos", k_tr_pos, dim3((unsigned)std::min<int64_t>(div_up((int64_t)n + 1, 256), 65536)),
              dim3(256), 0, n, any ? (int32_t)nnz : 0, (const uint32_t*)cols, out_pos);
  return SPWS_OK;
}

static int check_args(int32_t m, int32_t n, int64_t nnz, const void* pos, const int32_t* crd, const double* vals,
                      const int32_t* out_pos, const int32_t* out_crd, const double* out_vals) {
  SPWS_REQUIRE(m >= 0 && n >= 0 && nnz >= 0, SPWS_ERR_INVALID, "negative dimension or nnz");
  SPWS_REQUIRE(nnz <= INT32_MAX, SPWS_ERR_UNSUPPORTED, "nnz = %lld exceeds the int32 index range", (long long)nnz);
  SPWS_REQUIRE(pos && out_pos && (nnz == 0 || (crd && vals && out_crd && out_vals)), SPWS_ERR_INVALID,
               "null pointer argument");
  return SPWS_OK;
}

// ------------------------------------------------ no-allocation entry point
//
// spws_csr_transpose_dev_noalloc runs transpose_run on a context that lives
// on the host stack and whose workspaces are fixed views into `scratch`, a
// file-scope device array: nothing is allocated on the host or the device.
// Each GPU holds its own copy of the array (at its own address) for the life
// of the process; its address on a device comes from hipGetSymbolAddress,
// taken once per device with that device current and cached here.  The
// array's name is only a host-side handle: the kernels get the looked-up
// address.  Calls that overlap on one GPU share the array and race.

constexpr size_t kNoAllocScratchBytes = (size_t)48 << 20;
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

constexpr int kMaxDevices = 64;
static std::mutex g_scratch_mu;
static void* g_scratch_ptr[kMaxDevices];

// The scratch array's address on `device`, which must be current.
static int scratch_address(int device, unsigned char** out) {
  SPWS_REQUIRE(device >= 0 && device < kMaxDevices, SPWS_ERR_UNSUPPORTED, "device %d beyond the scratch table",
               device);
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[device]) {
    void* p = nullptr;
    SPWS_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    g_scratch_ptr[device] = p;
  }
  *out = static_cast<unsigned char*>(g_scratch_ptr[device]);
  return SPWS_OK;
}

static size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }

// Bytes of each workspace the transpose of nnz entries uses.
struct TransposeScratch {
  size_t keys, vals, hist, total;
  explicit TransposeScratch(int64_t nnz) {
    const size_t nn = (size_t)(nnz > 0 ? nnz : 1);
    keys = align256(2 * nn * 8);
    vals = align256(2 * nn * 8);
    hist = align256(radix_hist_entries((int64_t)nn) * 4);
    total = keys + vals + hist;
  }
};

}  // namespace

int csr_transpose_run(spws_ctx* ctx, int32_t m, int32_t n, int64_t nnz, const int32_t* pos, const int32_t* crd,
                      const double* vals, int32_t* out_pos, int32_t* out_crd, double* out_vals) {
  return transpose_run(ctx, m, n, nnz, pos, crd, vals, out_pos, out_crd, out_vals);
}

int noalloc_scratch_init(int device) {
  unsigned char* p;
  return scratch_address(device, &p);
}

}  // namespace spws

using namespace spws;

extern "C" int spws_csr_transpose_dev(spws_ctx* ctx, int32_t m, int32_t n, int64_t nnz, const int32_t* pos,
                                      const int32_t* crd, const double* vals, int32_t* out_pos, int32_t* out_crd,
                                      double* out_vals) {
  int rc = ctx_activate(ctx);
  if (rc) return rc;
  if ((rc = check_args(m, n, nnz, pos, crd, vals, out_pos, out_crd, out_vals))) return rc;
  return transpose_run(ctx, m, n, nnz, pos, crd, vals, out_pos, out_crd, out_vals);
}

extern "C" int spws_csr64_transpose_dev(spws_ctx* ctx, int32_t m, int32_t n, int64_t nnz, const int64_t* pos,
                                        const int32_t* crd, const double* vals, int32_t* out_pos, int32_t* out_crd,
                                        double* out_vals) {
  int rc = ctx_activate(ctx);
  if (rc) return rc;
  if ((rc = check_args(m, n, nnz, pos, crd, vals, out_pos, out_crd, out_vals))) return rc;
  return transpose_run(ctx, m, n, nnz, pos, crd, vals, out_pos, out_crd, out_vals);
}

extern "C" int spws_csr_transpose_dev_noalloc(void* stream, int32_t m, int32_t n, int64_t nnz, const int32_t* pos,
                                              const int32_t* crd, const double* vals, int32_t* out_pos,
                                              int32_t* out_crd, double* out_vals) {
  int rc = check_args(m, n, nnz, pos, crd, vals, out_pos, out_crd, out_vals);
  if (rc) return rc;
  const TransposeScratch need(nnz);
  SPWS_REQUIRE(need.total <= kNoAllocScratchBytes, SPWS_ERR_UNSUPPORTED,
               "the no-allocation transpose of %lld entries needs %zu bytes of scratch; the fixed scratch holds %zu "
               "(about 33 bytes per entry)",
               (long long)nnz, need.total, kNoAllocScratchBytes);
  int device = 0;
  SPWS_HIP(hipGetDevice(&device));
  unsigned char* base;
  if ((rc = scratch_address(device, &base))) return rc;
  spws_ctx local;  // host stack: stream and fixed workspace views only
  local.device = device;
  local.stream = static_cast<hipStream_t>(stream);
  size_t off = 0;
  local.tr_keys.borrow(base + off, need.keys);
  off += need.keys;
  local.tr_vals.borrow(base + off, need.vals);
  off += need.vals;
  local.radix_hist.borrow(base + off, need.hist);
  return transpose_run(&local, m, n, nnz, pos, crd, vals, out_pos, out_crd, out_vals);
}
