// EmbeddingBlocks row movement for gfx950: gather / insert / filter over a slot
// stored as a list of equally sized blocks.
//
// Stands in for the device branches of csrc/ops/block_ops.cc:262-397
// (kernels: csrc/ops/block_ops_kernel.cu:16-392). Differences in design:
//   * the block pointer table is a device array owned by the caller and reused
//     across calls (the reference rebuilds and uploads it on every launch and
//     synchronises the stream afterwards, block_ops_kernel.cu:100-116,263-266)
//   * rows are moved as raw bytes with 16-byte vectors, a power-of-two group of
//     lanes per row, so one instantiation serves every element type
//   * a row index outside the table raises a soft error instead of faulting
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "common.cuh"

namespace recis_hip {
namespace {

template <int VB>
struct alignas(VB) Bytes {
  unsigned char b[VB];
};

struct BlockArgs {
  const int64_t* ids;
  char* const* blocks;
  int64_t n_blocks;
  int64_t block_size;
  int64_t n;
  int row_bytes;
  int64_t pitch_bytes;  // from one row of a block to the next (row_bytes when the rows are dense)
  int lpr_log2;
  int* err;
};

// row index -> address of the row; NULL (and a soft error) when out of range
__device__ __forceinline__ char* row_address(const BlockArgs& a, int64_t idx) {
  if (idx < 0) return nullptr;
  int64_t b, r;
  if (a.n_blocks == 1) {
    b = 0;
    r = idx;
    if (idx >= a.block_size) return nullptr;
  } else if ((static_cast<uint64_t>(idx) | static_cast<uint64_t>(a.block_size)) >> 32) {
    b = idx / a.block_size;
    r = idx - b * a.block_size;
  } else {
    const uint32_t bs = static_cast<uint32_t>(a.block_size);
    const uint32_t q = static_cast<uint32_t>(idx) / bs;
    b = q;
    r = static_cast<uint32_t>(idx) - q * bs;
  }
  if (b >= a.n_blocks) return nullptr;
  return a.blocks[b] + r * a.pitch_bytes;
}

template <int VB>
__global__ void __launch_bounds__(kBlock)
block_gather_kernel(BlockArgs a, int64_t default_key, int readonly, char* __restrict__ out) {
  const int rows_per_block = kBlock >> a.lpr_log2;
  const int64_t i = static_cast<int64_t>(blockIdx.x) * rows_per_block + (threadIdx.x >> a.lpr_log2);
  if (i >= a.n) return;
  const int cl = threadIdx.x & ((1 << a.lpr_log2) - 1);
  const int64_t idx = a.ids[i];
  const char* src = nullptr;
  if (!(readonly && idx == default_key)) {
    src = row_address(a, idx);
    if (!src) raise_device_error(a.err, RECIS_DEVERR_INDEX_RANGE);
  }
  char* dst = out + i * static_cast<int64_t>(a.row_bytes);
  for (int c = cl * VB; c < a.row_bytes; c += VB << a.lpr_log2) {
    Bytes<VB> v;
    if (src) {
      v = *reinterpret_cast<const Bytes<VB>*>(src + c);
    } else {
#pragma unroll
      for (int k = 0; k < VB; ++k) v.b[k] = 0;
    }
    *reinterpret_cast<Bytes<VB>*>(dst + c) = v;
  }
}

template <int VB>
__global__ void __launch_bounds__(kBlock)
block_insert_kernel(BlockArgs a, const char* __restrict__ emb, int broadcast,
                    const uint8_t* __restrict__ mask) {
  const int rows_per_block = kBlock >> a.lpr_log2;
  const int64_t i = static_cast<int64_t>(blockIdx.x) * rows_per_block + (threadIdx.x >> a.lpr_log2);
  if (i >= a.n) return;
  if (mask && !mask[i]) return;
  const int cl = threadIdx.x & ((1 << a.lpr_log2) - 1);
  char* dst = row_address(a, a.ids[i]);
  if (!dst) {
    raise_device_error(a.err, RECIS_DEVERR_INDEX_RANGE);
    return;
  }
  const char* src = emb + (broadcast ? 0 : i * static_cast<int64_t>(a.row_bytes));
  for (int c = cl * VB; c < a.row_bytes; c += VB << a.lpr_log2)
    *reinterpret_cast<Bytes<VB>*>(dst + c) = *reinterpret_cast<const Bytes<VB>*>(src + c);
}

// Rows of several slots set to one element each: what a constant initialiser gives the rows that an eviction frees. The
// element travels as an argument (16 bytes of it, repeated), so nothing is materialised or read but the row numbers, and one launch does
// all slots (grid.y). Bound: one random write request per 128 bytes of row. (A tensor of initial values filled and scattered per slot, six
// launches for three slots of 32 floats: 70 us for 178 k rows, now 27.)
struct FillSlot {
  char* const* blocks;
  int64_t n_blocks, block_size, pitch_bytes;
  int row_bytes, vb, lpr_log2;
  uint32_t element[4];
};
struct FillRowsArgs {
  const int64_t* ids;
  int64_t n;
  int* err;
  FillSlot slot[RECIS_FILL_ROWS_MAX_SLOTS];
};
template <int VB>
__device__ __forceinline__ void fill_row(char* dst, int row_bytes, int cl, int lpr_log2, const uint32_t* element) {
  Bytes<VB> v;
  __builtin_memcpy(&v, element, VB);
  for (int c = cl * VB; c < row_bytes; c += VB << lpr_log2) *reinterpret_cast<Bytes<VB>*>(dst + c) = v;
}
__global__ void __launch_bounds__(kBlock)
block_fill_rows_kernel(FillRowsArgs f) {
  const FillSlot& s = f.slot[blockIdx.y];  // uniform
  BlockArgs a;
  a.blocks = s.blocks;
  a.n_blocks = s.n_blocks;
  a.block_size = s.block_size;
  a.pitch_bytes = s.pitch_bytes;
  const int rows_per_block = kBlock >> s.lpr_log2;
  const int cl = threadIdx.x & ((1 << s.lpr_log2) - 1);
  const uint32_t element[4] = {s.element[0], s.element[1], s.element[2], s.element[3]};
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * rows_per_block + (threadIdx.x >> s.lpr_log2); i < f.n;
       i += static_cast<int64_t>(gridDim.x) * rows_per_block) {
    char* dst = row_address(a, f.ids[i]);
    if (!dst) {
      raise_device_error(f.err, RECIS_DEVERR_INDEX_RANGE);
      continue;
    }
    switch (s.vb) {  // uniform
      case 16: fill_row<16>(dst, s.row_bytes, cl, s.lpr_log2, element); break;
      case 8: fill_row<8>(dst, s.row_bytes, cl, s.lpr_log2, element); break;
      case 4: fill_row<4>(dst, s.row_bytes, cl, s.lpr_log2, element); break;
      case 2: fill_row<2>(dst, s.row_bytes, cl, s.lpr_log2, element); break;
      default: fill_row<1>(dst, s.row_bytes, cl, s.lpr_log2, element); break;
    }
  }
}

// flat table gather: out[i] = emb[ids[i]]
template <int VB>
__global__ void __launch_bounds__(kBlock)
gather_kernel(const void* __restrict__ ids, int ids64, const char* __restrict__ emb, int64_t rows,
              char* __restrict__ out, int64_t n, int row_bytes, int lpr_log2, int* err) {
  const int rows_per_block = kBlock >> lpr_log2;
  const int64_t i = static_cast<int64_t>(blockIdx.x) * rows_per_block + (threadIdx.x >> lpr_log2);
  if (i >= n) return;
  const int cl = threadIdx.x & ((1 << lpr_log2) - 1);
  const int64_t idx = load_index(ids, ids64, i);
  const bool ok = static_cast<uint64_t>(idx) < static_cast<uint64_t>(rows);
  if (!ok) raise_device_error(err, RECIS_DEVERR_INDEX_RANGE);
  const char* src = emb + idx * static_cast<int64_t>(row_bytes);
  char* dst = out + i * static_cast<int64_t>(row_bytes);
  for (int c = cl * VB; c < row_bytes; c += VB << lpr_log2) {
    Bytes<VB> v;
    if (ok) {
      v = *reinterpret_cast<const Bytes<VB>*>(src + c);
    } else {
#pragma unroll
      for (int k = 0; k < VB; ++k) v.b[k] = 0;
    }
    *reinterpret_cast<Bytes<VB>*>(dst + c) = v;
  }
}

__global__ void __launch_bounds__(kBlock)
block_filter_kernel(BlockArgs a, int64_t threshold, int slot64, uint8_t* __restrict__ mask_out) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
  if (i >= a.n) return;
  const char* p = row_address(a, a.ids[i]);
  if (!p) {
    raise_device_error(a.err, RECIS_DEVERR_INDEX_RANGE);
    mask_out[i] = 0;
    return;
  }
  const int64_t v = slot64 ? *reinterpret_cast<const int64_t*>(p)
                           : static_cast<int64_t>(*reinterpret_cast<const int32_t*>(p));
  mask_out[i] = v < threshold;
}

template <typename F>
int dispatch_vb(int vb, F&& f) {
  switch (vb) {
    case 16: return f(std::integral_constant<int, 16>{});
    case 8: return f(std::integral_constant<int, 8>{});
    case 4: return f(std::integral_constant<int, 4>{});
    case 2: return f(std::integral_constant<int, 2>{});
    case 1: return f(std::integral_constant<int, 1>{});
    default: return fail(RECIS_ERR_ARG, "bad vector bytes %d", vb);
  }
}

int fill_args(BlockArgs& a, const int64_t* ids, void* const* blocks_dev, int64_t n_blocks,
              int64_t block_size, int64_t row_pitch_bytes, int64_t n, int64_t row_bytes, int vb) {
  RECIS_REQUIRE(n >= 0, "n must be >= 0");
  RECIS_REQUIRE(n_blocks >= 1 && block_size >= 1, "need at least one block (n_blocks=%lld block_size=%lld)",
                (long long)n_blocks, (long long)block_size);
  RECIS_REQUIRE(row_bytes >= 1 && row_bytes <= (1 << 22), "row_bytes out of range: %lld", (long long)row_bytes);
  RECIS_REQUIRE(ids != nullptr && blocks_dev != nullptr, "ids / blocks must not be NULL");
  a.ids = ids;
  a.blocks = reinterpret_cast<char* const*>(blocks_dev);
  a.n_blocks = n_blocks;
  a.block_size = block_size;
  a.n = n;
  a.row_bytes = static_cast<int>(row_bytes);
  a.pitch_bytes = row_pitch_bytes > 0 ? row_pitch_bytes : row_bytes;
  RECIS_REQUIRE(a.pitch_bytes >= row_bytes && a.pitch_bytes % vb == 0,
                "row pitch %lld does not fit rows of %lld bytes moved %d bytes at a time", (long long)a.pitch_bytes,
                (long long)row_bytes, vb);
  a.lpr_log2 = std::min(6, ilog2_ceil((row_bytes + vb - 1) / vb));
  a.err = device_error_word(current_device());
  RECIS_REQUIRE(a.err != nullptr, "could not reach the device error word");
  return RECIS_OK;
}

}  // namespace
}  // namespace recis_hip

using namespace recis_hip;

extern "C" {

int recis_gather(const void* ids, int ids_is64, const void* emb, int64_t rows, void* out, int64_t n,
                 int64_t row_bytes, void* stream_) {
  hipStream_t stream = static_cast<hipStream_t>(stream_);
  RECIS_REQUIRE(n >= 0 && rows >= 0, "negative size");
  if (n == 0) return RECIS_OK;
  RECIS_REQUIRE(ids && emb && out, "NULL argument");
  RECIS_REQUIRE(row_bytes >= 1 && row_bytes <= (1 << 22), "row_bytes out of range: %lld", (long long)row_bytes);
  const int vb = pick_vec_bytes(row_bytes, reinterpret_cast<uintptr_t>(emb) | reinterpret_cast<uintptr_t>(out));
  const int lpr_log2 = std::min(6, ilog2_ceil((row_bytes + vb - 1) / vb));
  int* err = device_error_word(current_device());
  RECIS_REQUIRE(err != nullptr, "could not reach the device error word");
  const int rows_per_block = kBlock >> lpr_log2;
  const int64_t grid = (n + rows_per_block - 1) / rows_per_block;
  return dispatch_vb(vb, [&](auto tag) {
    constexpr int VB = decltype(tag)::value;
    RECIS_TIME_KERNEL("gather_kernel", stream)
    gather_kernel<VB><<<dim3(grid), dim3(kBlock), 0, stream>>>(
        ids, ids_is64, static_cast<const char*>(emb), rows, static_cast<char*>(out), n,
        static_cast<int>(row_bytes), lpr_log2, err);
    RECIS_LAUNCH_CHECK();
    return RECIS_OK;
  });
}

int recis_block_gather(const int64_t* ids, void* const* blocks_dev, int64_t n_blocks,
                       int64_t block_size, int64_t row_pitch_bytes, int64_t default_key, int readonly, void* out,
                       int64_t n, int64_t row_bytes, void* stream_) {
  hipStream_t stream = static_cast<hipStream_t>(stream_);
  if (n == 0) return RECIS_OK;
  RECIS_REQUIRE(out != nullptr, "out must not be NULL");
  const int vb = pick_vec_bytes(row_bytes, reinterpret_cast<uintptr_t>(out) | static_cast<uintptr_t>(row_pitch_bytes));
  BlockArgs a;
  if (int rc = fill_args(a, ids, blocks_dev, n_blocks, block_size, row_pitch_bytes, n, row_bytes, vb)) return rc;
  const int rows_per_block = kBlock >> a.lpr_log2;
  const int64_t grid = (n + rows_per_block - 1) / rows_per_block;
  return dispatch_vb(vb, [&](auto tag) {
    constexpr int VB = decltype(tag)::value;
    RECIS_TIME_KERNEL("block_gather_kernel", stream)
    block_gather_kernel<VB><<<dim3(grid), dim3(kBlock), 0, stream>>>(a, default_key, readonly,
                                                                    static_cast<char*>(out));
    RECIS_LAUNCH_CHECK();
    return RECIS_OK;
  });
}

int recis_block_insert(const int64_t* ids, const void* emb, int broadcast, const uint8_t* mask,
                       void* const* blocks_dev, int64_t n_blocks, int64_t block_size, int64_t row_pitch_bytes,
                       int64_t n, int64_t row_bytes, void* stream_) {
  hipStream_t stream = static_cast<hipStream_t>(stream_);
  if (n == 0) return RECIS_OK;
  RECIS_REQUIRE(emb != nullptr, "emb must not be NULL");
  const int vb = pick_vec_bytes(row_bytes, reinterpret_cast<uintptr_t>(emb) | static_cast<uintptr_t>(row_pitch_bytes));
  BlockArgs a;
  if (int rc = fill_args(a, ids, blocks_dev, n_blocks, block_size, row_pitch_bytes, n, row_bytes, vb)) return rc;
  const int rows_per_block = kBlock >> a.lpr_log2;
  const int64_t grid = (n + rows_per_block - 1) / rows_per_block;
  return dispatch_vb(vb, [&](auto tag) {
    constexpr int VB = decltype(tag)::value;
    block_insert_kernel<VB><<<dim3(grid), dim3(kBlock), 0, stream>>>(a, static_cast<const char*>(emb),
                                                                    broadcast, mask);
    RECIS_LAUNCH_CHECK();
    return RECIS_OK;
  });
}

int recis_block_fill_rows(const int64_t* ids, int64_t n, const recis_fill_slot* slots, int64_t n_slots, void* stream_) {
  hipStream_t stream = static_cast<hipStream_t>(stream_);
  RECIS_REQUIRE(n >= 0 && n_slots >= 0 && n_slots <= RECIS_FILL_ROWS_MAX_SLOTS, "bad sizes");
  if (n == 0 || n_slots == 0) return RECIS_OK;
  RECIS_REQUIRE(slots != nullptr, "slots must not be NULL");
  FillRowsArgs f{};
  f.ids = ids;
  f.n = n;
  f.err = device_error_word(current_device());
  int64_t grid = 1;
  for (int64_t k = 0; k < n_slots; ++k) {
    const recis_fill_slot& in = slots[k];
    RECIS_REQUIRE((in.elem_bytes == 1 || in.elem_bytes == 2 || in.elem_bytes == 4 || in.elem_bytes == 8) &&
                      in.row_bytes % in.elem_bytes == 0 && in.row_pitch_bytes % in.elem_bytes == 0,
                  "slot %lld: rows of %lld bytes of elements of %d", (long long)k, (long long)in.row_bytes, in.elem_bytes);
    const int vb = pick_vec_bytes(in.row_bytes, static_cast<uintptr_t>(in.row_pitch_bytes));
    BlockArgs a;
    if (int rc = fill_args(a, ids, in.blocks_dev, in.n_blocks, in.block_size, in.row_pitch_bytes, n, in.row_bytes, vb)) return rc;
    FillSlot& out = f.slot[k];
    out.blocks = a.blocks;
    out.n_blocks = a.n_blocks;
    out.block_size = a.block_size;
    out.pitch_bytes = a.pitch_bytes;
    out.row_bytes = a.row_bytes;
    out.vb = vb;
    out.lpr_log2 = a.lpr_log2;
    for (int b = 0; b < 16; b += in.elem_bytes) __builtin_memcpy(reinterpret_cast<char*>(out.element) + b, in.element, in.elem_bytes);
    const int64_t rows_per_block = kBlock >> a.lpr_log2;
    grid = std::max(grid, std::min<int64_t>((n + rows_per_block - 1) / rows_per_block, 256 * 32));
  }
  RECIS_TIME_KERNEL("block_fill_rows_kernel", stream)
  block_fill_rows_kernel<<<dim3(static_cast<unsigned>(grid), static_cast<unsigned>(n_slots)), dim3(kBlock), 0, stream>>>(f);
  RECIS_LAUNCH_CHECK();
  return RECIS_OK;
}

int recis_block_filter(const int64_t* ids, void* const* blocks_dev, int64_t n_blocks,
                       int64_t block_size, int64_t threshold, int slot_is64, uint8_t* mask_out,
                       int64_t n, void* stream_) {
  hipStream_t stream = static_cast<hipStream_t>(stream_);
  if (n == 0) return RECIS_OK;
  RECIS_REQUIRE(mask_out != nullptr, "mask_out must not be NULL");
  BlockArgs a;
  if (int rc = fill_args(a, ids, blocks_dev, n_blocks, block_size, 0, n, slot_is64 ? 8 : 4, slot_is64 ? 8 : 4))
    return rc;
  block_filter_kernel<<<dim3((n + kBlock - 1) / kBlock), dim3(kBlock), 0, stream>>>(a, threshold, slot_is64,
                                                                                   mask_out);
  RECIS_LAUNCH_CHECK();
  return RECIS_OK;
}

}  // extern "C"
