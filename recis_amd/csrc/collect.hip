// Rows of several strided arrays laid end to end in one dense array for gfx950: what the backward of a
// coalesced lookup does with the gradients of its outputs.
//
// A model that concatenates its features hands every one of them a column slice of one wide gradient: rows
// of 64 bytes, 2.5 KB apart for 39 features of 16 floats. Copied a part at a time, every 128-byte line of
// the wide gradient is fetched twice, for two parts that come to it at different times. With parts of equal
// length a workgroup therefore takes a few consecutive rows of ALL parts: between its waves it reads whole rows of the
// wide gradient, each line once from memory, and writes kSamples rows next to each other per part.
// Bound: one read and one write of every byte. 39 parts of 65536 rows of 64 bytes (327 MB moved): 66 us
// (4.9 TB/s; neighbouring lane groups on neighbouring parts instead of neighbouring rows: 79), a part at a time 89 - 91 us.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "common.cuh"

namespace recis_hip {
namespace {

constexpr int kParts = 64;      // of one launch (the table travels as a kernel argument)
constexpr int kSamples = 16;    // rows of every part a workgroup takes (few parts: more)
constexpr int kFly = 4;  // rows of a lane group in flight

struct CollectArgs {
  int32_t n;                  // rows of all parts
  int32_t rows_each;          // rows of every part when they are alike, else 0
  int32_t per_block;          // rows of a workgroup: a multiple of n_parts when the parts are alike
  int row_bytes, lpr_log2, n_parts;
  const void* base[kParts];   // NULL: a part of zeros
  int64_t stride[kParts];     // bytes
  int32_t first[kParts + 1];  // INT32_MAX from n_parts on
};

__device__ __align__(256) const unsigned char g_collect_zero_row[8192 * 4] = {};

// W: what a lane moves at a time. The arguments come first, so the table of parts is read where the kernel's
// arguments lie in memory, a lane per entry (indexing the by-value argument would copy it to scratch).
template <typename W>
__global__ void __launch_bounds__(kBlock, 8)
collect_rows_kernel(CollectArgs a, W* __restrict__ out) {
  __shared__ const char* s_base[kParts];
  __shared__ int64_t s_stride[kParts];
  __shared__ int32_t s_first[kParts + 1];
  {
    const CollectArgs* in_memory =
        reinterpret_cast<const CollectArgs*>(reinterpret_cast<uintptr_t>(__builtin_amdgcn_kernarg_segment_ptr()));
    const int k = threadIdx.x;
    if (k <= kParts) {
      s_first[k] = in_memory->first[k];
      if (k < kParts) {
        const char* base = static_cast<const char*>(in_memory->base[k]);
        s_base[k] = base ? base : reinterpret_cast<const char*>(g_collect_zero_row);
        s_stride[k] = base ? in_memory->stride[k] : 0;
      }
    }
    __syncthreads();
  }
  const int cl = threadIdx.x & ((1 << a.lpr_log2) - 1);
  const int g = threadIdx.x >> a.lpr_log2, groups = kBlock >> a.lpr_log2;
  const int packs = a.row_bytes / static_cast<int>(sizeof(W));
  const int32_t lo = static_cast<int32_t>(blockIdx.x) * a.per_block, n_here = min(a.per_block, a.n - lo);
  const int32_t sample0 = lo / a.n_parts, samples = max(1, n_here / a.n_parts);  // alike: rows sample0 .. of all parts
  for (int32_t t0 = g; t0 < n_here; t0 += kFly * groups) {
    const char* row[kFly];
    int32_t to[kFly];
#pragma unroll
    for (int x = 0; x < kFly; ++x) {
      const int32_t t = min(t0 + x * groups, n_here - 1);
      int32_t p = 0, r;
      if (a.rows_each > 0) {  // (uniform)
        p = t / samples;  // consecutive rows of one part side by side: whole lines written
        r = sample0 + t - p * samples;
        to[x] = p * a.rows_each + r;
      } else {
        to[x] = lo + t;
        for (int32_t hi = a.n_parts; hi - p > 1;) {
          const int32_t mid = (p + hi) >> 1;
          if (s_first[mid] <= to[x])
            p = mid;
          else
            hi = mid;
        }
        r = to[x] - s_first[p];
      }
      row[x] = s_base[p] + r * s_stride[p];
    }
    for (int c = cl; c < packs; c += 1 << a.lpr_log2) {
      W v[kFly];
#pragma unroll
      for (int x = 0; x < kFly; ++x) v[x] = reinterpret_cast<const W*>(row[x])[c];
#pragma unroll
      for (int x = 0; x < kFly; ++x)
        if (t0 + x * groups < n_here) out[static_cast<int64_t>(to[x]) * packs + c] = v[x];
    }
  }
}

}  // namespace
}  // namespace recis_hip

using namespace recis_hip;

extern "C" int recis_collect_rows(const void* const* part_rows, const int64_t* part_stride_bytes,
                                  const int64_t* part_counts, int64_t n_parts, int64_t row_bytes, int elem_bytes,
                                  void* out, void* stream_) {
  hipStream_t stream = static_cast<hipStream_t>(stream_);
  RECIS_REQUIRE(n_parts >= 0 && ((part_rows && part_stride_bytes && part_counts) || n_parts == 0), "bad part list");
  RECIS_REQUIRE(elem_bytes == 2 || elem_bytes == 4, "elements of %d bytes", elem_bytes);
  RECIS_REQUIRE(row_bytes >= elem_bytes && row_bytes % elem_bytes == 0 && row_bytes <= 8192 * 4, "rows of %lld bytes",
                (long long)row_bytes);
  int64_t rows = 0;
  for (int64_t f = 0; f < n_parts; ++f) {
    RECIS_REQUIRE(part_counts[f] >= 0 && part_stride_bytes[f] >= 0 && part_stride_bytes[f] % elem_bytes == 0 &&
                      reinterpret_cast<uintptr_t>(part_rows[f]) % elem_bytes == 0,
                  "part %lld: bad rows", (long long)f);
    rows += part_counts[f];
  }
  RECIS_REQUIRE(rows < INT32_MAX, "too many rows");
  if (rows == 0) return RECIS_OK;
  RECIS_REQUIRE(out != nullptr && reinterpret_cast<uintptr_t>(out) % elem_bytes == 0, "bad out");
  CollectArgs a{};
  a.row_bytes = static_cast<int>(row_bytes);
  char* dst = static_cast<char*>(out);
  for (int64_t f0 = 0; f0 < n_parts; f0 += kParts) {
    a.n_parts = static_cast<int>(std::min<int64_t>(kParts, n_parts - f0));
    uintptr_t align = reinterpret_cast<uintptr_t>(dst);
    int32_t first = 0;
    bool alike = true;
    for (int k = 0; k < kParts; ++k) {
      const bool used = k < a.n_parts;
      a.base[k] = used ? part_rows[f0 + k] : nullptr;
      a.stride[k] = used ? part_stride_bytes[f0 + k] : 0;
      a.first[k] = used ? first : INT32_MAX;
      if (!used) continue;
      align |= reinterpret_cast<uintptr_t>(a.base[k]) | static_cast<uintptr_t>(a.stride[k]);
      alike = alike && part_counts[f0 + k] == part_counts[f0];
      first += static_cast<int32_t>(part_counts[f0 + k]);
    }
    a.first[kParts] = INT32_MAX;
    a.n = first;
    a.rows_each = alike ? static_cast<int32_t>(part_counts[f0]) : 0;
    if (first == 0) continue;
    const int vb = pick_vec_bytes(row_bytes, align);
    a.lpr_log2 = std::min(6, ilog2_ceil(row_bytes / vb));
    // rows of a workgroup: about 512 workgroups for a small call, else kSamples rows of every part, or more where these are
    // fewer than its lane groups have in flight (65536 rows of 64 bytes of 4 parts, 16 of each: 8.4 us,
    // 64: 5.8; at::cat 6.3 - 8.1)
    const int32_t round = kFly * (kBlock >> a.lpr_log2);
    if (alike)
      a.per_block = a.n_parts * std::max(1, std::min(std::max(kSamples, round / a.n_parts), a.rows_each / 512));
    else
      a.per_block = round;
    const dim3 grid(static_cast<uint32_t>((a.n + a.per_block - 1) / a.per_block)), block(kBlock);
    RECIS_TIME_KERNEL("collect_rows_kernel", stream) {
      switch (vb) {
        case 16: collect_rows_kernel<uint4><<<grid, block, 0, stream>>>(a, reinterpret_cast<uint4*>(dst)); break;
        case 8: collect_rows_kernel<uint2><<<grid, block, 0, stream>>>(a, reinterpret_cast<uint2*>(dst)); break;
        case 4: collect_rows_kernel<uint32_t><<<grid, block, 0, stream>>>(a, reinterpret_cast<uint32_t*>(dst)); break;
        default: collect_rows_kernel<uint16_t><<<grid, block, 0, stream>>>(a, reinterpret_cast<uint16_t*>(dst)); break;
      }
      RECIS_LAUNCH_CHECK();
    }
    dst += static_cast<int64_t>(first) * row_bytes;
  }
  return RECIS_OK;
}
