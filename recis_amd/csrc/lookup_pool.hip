// Read-only lookup and pooling in one pass for gfx950: out[s] = sum over the ids of segment s of
// w * row(id), straight from the ids to the pooled rows, for several features of one table at once.
//
// What the evaluation / serving forward of the reference does with ids_encode + ids_partition +
// IdMap::Lookup(readonly) + block_gather + segment_reduce (csrc/embedding/hashtable.cc:153-165,
// recis/nn/modules/embedding_engine.py:607-675). A training lookup dedups its batch because the
// backward needs the occurrences of every id side by side and because a key may be inserted only
// once. A read-only lookup needs neither: an id that occurs ten times finds its slot of the map and
// its row in the L2 nine times, which costs less than the five passes of the batch plan. So there is
// no plan here, no copy of the looked-up rows, one launch, and nothing that the host has to wait for.
//
// Bound: random requests to memory (one 16-byte slot and one row per distinct id) for large
// batches, the chain id -> slot -> row -> store (three round trips) for a request of a few hundred samples.
// Measured with 26 id columns and 4 ragged features (0..20 ids) of rows of 16 floats: batch 256 in 6.7 us where the plan,
// the look-up of its unique ids and the pooling took 63 us; batch 16384 (1.1 M ids) in 32 us instead of 145; one row
// per lookup of 0.5 M Zipf ids over rows of 32 floats (half a million rows of 128 bytes written) 27 us instead of 107.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "common.cuh"
#include "idmap_internal.cuh"

namespace recis_hip {
namespace {

constexpr int kPoolJobs = 64;    // features of one launch (the table travels as a kernel argument)
constexpr int kPoolRows = 1024;  // ids of a workgroup whose rows are known at a time (LDS)
constexpr int kMaxSegs = 256;    // segments of a workgroup
// Workgroups from which on the chip is full and a workgroup may take more than one segment per team.
constexpr int64_t kGridFull = 1024;

struct PoolJob {
  const int64_t* ids;
  const void* offs;  // [n_seg + 1] int32 / int64, or NULL: every segment holds `width` ids
  const void* weight;
  int32_t n_ids, n_seg;
  int32_t first_tile, out_row0;
  int32_t width;
  uint32_t flags;  // bits 0-11 table id, 12 offsets are int64, 13-14 weight dtype, 16-18 row groups (log2), 20-23 segments per team (log2)
};
struct PoolJobs {
  int n_jobs;
  PoolJob job[kPoolJobs];
};
struct PoolArgs {
  const Slot* table;
  uint64_t mask;
  const void* const* blocks;
  int64_t n_blocks, block_rows, pitch;  // pitch in elements
  int64_t id_mask;                      // of the id's own bits; ~0 = ids are taken as they are
  int D, lpr_log2, mode;                // RECIS_SUM, RECIS_MEAN or RECIS_LOOKUP_WEIGHT_MEAN
  int* err;
  int* report;  // pinned: this call has no count for the error bits to travel with
};

__device__ __forceinline__ void raise_and_report(const PoolArgs& a, int bit) {
  raise_device_error(a.err, bit);
  report_device_errors(a.report);
}

// A row of zeros (D <= 8192 of at most 4 bytes): what an id without a row reads, so that the loads of
// a round need no branch around each.
__device__ __align__(256) const unsigned char g_pool_zero_row[8192 * 4] = {};

// Row of `key` in the map, or -1. `hint` is the key's home slot as it was read.
__device__ __forceinline__ int64_t find_row(const Slot* __restrict__ table, uint64_t mask, int64_t key, uint64_t home,
                                            longlong2 hint) {
  uint64_t p = home;
  for (uint64_t probes = 0;;) {
    if (hint.x == key) return hint.y;
    if (hint.x == kEmpty || ++probes > mask) return -1;
    p = (p + 1) & mask;
    hint = *reinterpret_cast<const longlong2*>(&table[p]);
  }
}

template <typename T>
__device__ __forceinline__ uint64_t address_of_row(const PoolArgs& a, int64_t row) {
  if (row < 0) return 0;
  int64_t b = 0, r = row;
  if (a.n_blocks != 1) {
    if ((static_cast<uint64_t>(row) | static_cast<uint64_t>(a.block_rows)) >> 32) {
      b = row / a.block_rows;
    } else {
      b = static_cast<uint32_t>(row) / static_cast<uint32_t>(a.block_rows);
    }
    r = row - b * a.block_rows;
  }
  if (b >= a.n_blocks || r >= a.block_rows) {
    raise_and_report(a, RECIS_DEVERR_INDEX_RANGE);
    return 0;
  }
  return reinterpret_cast<uint64_t>(static_cast<const T*>(a.blocks[b]) + r * a.pitch);
}

// The weight in the precision of the rows, as a caller that casts its weights to the table's type has it.
template <typename T>
__device__ __forceinline__ float weight_at(const void* w, int dt, int64_t i) {
  float x;
  if (dt == RECIS_F32)
    x = static_cast<const float*>(w)[i];
  else if (dt == RECIS_BF16)
    x = to_float(static_cast<const bf16_t*>(w)[i]);
  else
    x = to_float(static_cast<const f16_t*>(w)[i]);
  return to_float(from_float<T>(x));
}

// A workgroup takes a tile of consecutive segments of one feature: its threads look up the ids of
// the tile, up to four each at a time, and leave the addresses of the rows in LDS; then teams of lanes
// (2^lpr lanes per row, 2^rg row groups per segment) sum the rows of their segments, several row
// loads in flight per lane, and store each pooled row once. Looking an id up by one lane instead of
// by the whole lane group that reads its row keeps 256 probes of the map in flight per workgroup.
// (Six waves a SIMD: four rows and four probes in flight are 80 registers; held to 64 they spill, 36.6 us instead of 32.2 for
// 1.1 M ids of rows of 64 bytes.)
template <typename T, int VEC>
__global__ void __launch_bounds__(kBlock, 6)
lookup_pool_kernel(PoolJobs J, PoolArgs a, T* __restrict__ out) {
  __shared__ uint64_t s_row[kPoolRows];
  __shared__ float s_w[kPoolRows];
  __shared__ int32_t s_off[kMaxSegs + 1];
  __shared__ int s_bad;
  const int tid = threadIdx.x;
  const int tile = static_cast<int>(blockIdx.x);
  int j = 0;
  for (int hi = J.n_jobs; hi - j > 1;) {  // uniform: scalar loads
    const int mid = (j + hi) >> 1;
    if (J.job[mid].first_tile <= tile)
      j = mid;
    else
      hi = mid;
  }
  const PoolJob& job = J.job[j];
  const int64_t* __restrict__ ids = job.ids;
  const void* weight = job.weight;
  const int32_t n_ids = job.n_ids, n_seg = job.n_seg, width = job.width;
  const uint32_t flags = job.flags;
  const int64_t tag = a.id_mask == ~int64_t(0) ? 0 : static_cast<int64_t>(static_cast<uint64_t>(flags & 4095u) << 52);
  const int off64 = (flags >> 12) & 1, wdt = (flags >> 13) & 3;
  const int rg_log2 = (flags >> 16) & 7, spt_log2 = (flags >> 20) & 15;
  const int team_log2 = a.lpr_log2 + rg_log2;
  const int teams = kBlock >> team_log2;
  const int32_t seg0 = (tile - job.first_tile) * (teams << spt_log2);
  const int n_here = min(teams << spt_log2, n_seg - seg0);
  const void* offs = job.offs;

  if (tid == 0) {
    s_bad = 0;
    // what earlier kernels of the device found
    if (tile == 0 && __hip_atomic_load(a.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) report_device_errors(a.report);
  }
  if (offs == nullptr) {
    for (int i = tid; i <= n_here; i += kBlock) s_off[i] = (seg0 + i) * width;
    __syncthreads();
  } else {
    for (int i = tid; i <= n_here; i += kBlock) {
      const int64_t o = load_index(offs, off64, seg0 + i);
      // past either end of the ids: told apart below (a segment is bad unless 0 <= start <= end <= n_ids)
      s_off[i] = static_cast<int32_t>(o < 0 ? -1 : (o > n_ids ? int64_t(INT32_MAX) : o));
    }
    __syncthreads();
    bool bad = false;
    for (int i = tid; i < n_here; i += kBlock) bad |= s_off[i] < 0 || s_off[i + 1] > n_ids || s_off[i + 1] < s_off[i];
    if (bad) s_bad = 1;
    __syncthreads();
    if (s_bad) {  // uniform; the tile's rows come out as zeros
      if (tid == 0) raise_and_report(a, RECIS_DEVERR_OFFSETS);
      for (int i = tid; i <= n_here; i += kBlock) s_off[i] = 0;
      __syncthreads();
    }
  }

  // rows of the n ids from id `from` of the feature on into LDS (at most kPoolRows: places in LDS cannot overflow, as numbers of
  // ids up to 2^31 may)
  auto look_up_by = [&](auto probes, int32_t from, int n) {
    constexpr int kProbes = decltype(probes)::value;  // of a thread in flight
    const int64_t* __restrict__ id = ids + from;
    for (int q0 = tid; q0 < n; q0 += kProbes * kBlock) {
      int64_t key[kProbes];
      longlong2 hint[kProbes];
#pragma unroll
      for (int x = 0; x < kProbes; ++x) key[x] = q0 + x * kBlock < n ? (id[q0 + x * kBlock] & a.id_mask) | tag : kEmpty;
#pragma unroll
      for (int x = 0; x < kProbes; ++x)  // (a reserved key has a home slot too: no branch around the load)
        hint[x] = *reinterpret_cast<const longlong2*>(&a.table[home_slot(key[x], a.mask)]);
      uint32_t further = 0;  // probes that the home slot does not end
#pragma unroll
      for (int x = 0; x < kProbes; ++x) {
        const bool reserved = key[x] == kEmpty || key[x] == kTomb, found = hint[x].x == key[x] && !reserved;
        further |= !found && !reserved && hint[x].x != kEmpty ? 1u << x : 0u;
        if (q0 + x * kBlock < n) s_row[q0 + x * kBlock] = static_cast<uint64_t>(found ? hint[x].y : -1);
      }
#pragma unroll 1
      for (int x = 0; x < kProbes; ++x) {  // (one body: four of them spill)
        const int q = q0 + x * kBlock;
        if (q >= n) break;
        int64_t row = static_cast<int64_t>(s_row[q]);
        if ((further >> x) & 1u) {
          const int64_t k = (id[q] & a.id_mask) | tag;
          const uint64_t home = home_slot(k, a.mask);
          row = find_row(a.table, a.mask, k, home, *reinterpret_cast<const longlong2*>(&a.table[home]));
        }
        s_row[q] = address_of_row<T>(a, row);
        if (weight) s_w[q] = weight_at<T>(weight, wdt, static_cast<int64_t>(from) + q);
      }
    }
  };
  auto look_up = [&](int32_t from, int n) {
    if (n <= kBlock)  // uniform
      look_up_by(std::integral_constant<int, 1>{}, from, n);
    else
      look_up_by(std::integral_constant<int, 4>{}, from, n);
  };
  const int lane_t = tid & ((1 << team_log2) - 1);
  const int team = tid >> team_log2;
  const int rg = lane_t >> a.lpr_log2, step = 1 << rg_log2;
  const int cl = lane_t & ((1 << a.lpr_log2) - 1);
  const int D = a.D;
  const T* const zero_row = reinterpret_cast<const T*>(g_pool_zero_row);
  auto row_of = [&](int q) -> const T* {
    const uint64_t at = s_row[q];
    return at ? reinterpret_cast<const T*>(at) : zero_row;
  };
  // acc += the rows first, first + step, ... < last of the LDS list, columns c0 ..
  auto add_rows = [&](int first, int last, int c0, float (&acc)[VEC]) {
    constexpr int kFly = 4;
    for (int q = first; q < last; q += kFly * step) {  // past the end: the row of zeros, so that a short list is one round trip too
      Pack<T, VEC> v[kFly];  // (converted as they are added: in flight they cost the registers of their own type)
#pragma unroll
      for (int k = 0; k < kFly; ++k)
        v[k] = *reinterpret_cast<const Pack<T, VEC>*>((q + k * step < last ? row_of(q + k * step) : zero_row) + c0);
      __builtin_amdgcn_sched_barrier(0);  // all loads first
#pragma unroll
      for (int k = 0; k < kFly; ++k) {
        const float w = weight ? (q + k * step < last ? s_w[q + k * step] : 0.f) : 1.0f;
#pragma unroll
        for (int x = 0; x < VEC; ++x) acc[x] = fmaf(to_float(v[k].v[x]), w, acc[x]);
      }
    }
  };
  auto weight_sum = [&](int first, int last) {
    float sum = 0.f;
    for (int q = first; q < last; q += step) sum += weight ? s_w[q] : 1.0f;
    return sum;
  };
  // the row groups of the team meet; every lane of the team calls
  auto fold = [&](float x) {
    for (int off = 1 << a.lpr_log2; off < (1 << team_log2); off <<= 1) x += __shfl_xor(x, off, kWave);
    return x;
  };
  auto finish = [&](int s, int c0, float (&acc)[VEC], int32_t len, float w_sum) {
    float scale = 1.0f;
    if (a.mode == RECIS_MEAN) {
      if (len > 0) scale = 1.0f / static_cast<float>(len);
    } else if (a.mode == RECIS_LOOKUP_WEIGHT_MEAN) {
      if (len > 0) scale = 1.0f / w_sum;
    }
#pragma unroll
    for (int x = 0; x < VEC; ++x) acc[x] *= scale;
    store_pack<T, VEC>(out + (static_cast<int64_t>(job.out_row0) + seg0 + s) * D + c0, acc);
  };

  const int32_t lo = s_off[0], hi = s_off[n_here];
  if (hi - lo <= kPoolRows) {  // the usual tile: one look-up for all of it
    look_up(lo, hi - lo);
    __syncthreads();
    if (offs == nullptr && width == 1 && !weight) {  // a dense column: its rows, four in flight per lane
      for (int c0 = cl * VEC; c0 < D; c0 += VEC << a.lpr_log2) {
        for (int s = team; s < n_here; s += 4 * teams) {
          float v[4][VEC];
#pragma unroll
          for (int k = 0; k < 4; ++k)
            load_pack<T, VEC>(s + k * teams < n_here ? row_of(s + k * teams) + c0 : zero_row, v[k]);
#pragma unroll
          for (int k = 0; k < 4; ++k)
            if (s + k * teams < n_here)
              store_pack<T, VEC>(out + (static_cast<int64_t>(job.out_row0) + seg0 + s + k * teams) * D + c0, v[k]);
        }
      }
      return;
    }
    for (int s = team; s < n_here; s += teams) {
      const int first = s_off[s] - lo, last = s_off[s + 1] - lo;
      const float w_sum = a.mode == RECIS_LOOKUP_WEIGHT_MEAN ? fold(weight_sum(first + rg, last)) : 0.f;
      for (int cb = 0; cb < D; cb += VEC << a.lpr_log2) {
        const int c0 = cb + cl * VEC;
        float acc[VEC];
#pragma unroll
        for (int x = 0; x < VEC; ++x) acc[x] = 0.f;
        if (c0 < D) add_rows(first + rg, last, c0, acc);
#pragma unroll
        for (int x = 0; x < VEC; ++x) acc[x] = fold(acc[x]);
        if (rg == 0 && c0 < D) finish(s, c0, acc, last - first, w_sum);
      }
    }
    return;
  }
  // more ids than LDS takes: the segments `teams` at a time, their ids in rounds, the sums kept over
  // the rounds (a row of more than 64 packs takes the rounds once per stretch of its columns)
  for (int s0 = 0; s0 < n_here; s0 += teams) {
    const int s = s0 + team;
    const bool mine = s < n_here;
    const int32_t first = mine ? s_off[s] : 0, last = mine ? s_off[s + 1] : 0;
    const int32_t b_lo = s_off[s0], b_hi = s_off[min(n_here, s0 + teams)];
    for (int cb = 0; cb < D; cb += VEC << a.lpr_log2) {  // uniform
      const int c0 = cb + cl * VEC;
      float acc[VEC], w_sum = 0.f;
#pragma unroll
      for (int x = 0; x < VEC; ++x) acc[x] = 0.f;
      for (int32_t base = b_lo; base < b_hi; base = b_hi - base > kPoolRows ? base + kPoolRows : b_hi) {
        const int n = min(b_hi - base, kPoolRows);
        __syncthreads();  // the previous round has been read
        look_up(base, n);
        __syncthreads();
        // the row group's rows of this round, counted from `base`
        const uint32_t behind = base > first ? (static_cast<uint32_t>(base - first) + step - 1 - rg) >> rg_log2 : 0;
        const int from = static_cast<int>(static_cast<uint32_t>(first - base) + rg + (behind << rg_log2));
        const int to = min(last - base, n);
        if (mine && from < to) {
          if (c0 < D) add_rows(from, to, c0, acc);
          if (a.mode == RECIS_LOOKUP_WEIGHT_MEAN) w_sum += weight_sum(from, to);
        }
      }
#pragma unroll
      for (int x = 0; x < VEC; ++x) acc[x] = fold(acc[x]);
      w_sum = fold(w_sum);
      if (mine && rg == 0 && c0 < D) finish(s, c0, acc, last - first, w_sum);
    }
  }
}

template <typename F>
int dispatch_pool_vec(int vec, F&& f) {
  switch (vec) {
    case 8: return f(std::integral_constant<int, 8>{});
    case 4: return f(std::integral_constant<int, 4>{});
    case 2: return f(std::integral_constant<int, 2>{});
    default: return f(std::integral_constant<int, 1>{});
  }
}

}  // namespace
}  // namespace recis_hip

using namespace recis_hip;

extern "C" int recis_lookup_pool_readonly(recis_idmap* map, const recis_lookup_job* jobs, int64_t n_jobs, int tagged,
                                          const void* const* emb_blocks_dev, int64_t n_blocks, int64_t block_rows,
                                          int64_t row_pitch_bytes, int row_dtype, void* out, int64_t D, int mode,
                                          void* stream_) {
  hipStream_t stream = static_cast<hipStream_t>(stream_);
  RECIS_REQUIRE(map != nullptr, "id map is NULL");
  RECIS_REQUIRE(n_jobs >= 0 && (jobs || n_jobs == 0), "bad job list");
  RECIS_REQUIRE(mode == RECIS_SUM || mode == RECIS_MEAN || mode == RECIS_LOOKUP_WEIGHT_MEAN, "invalid mode %d", mode);
  RECIS_REQUIRE(D >= 1 && D <= 8192, "embedding dim %lld out of range", (long long)D);
  const int size = dtype_size(row_dtype);
  RECIS_REQUIRE(size, "invalid row dtype %d", row_dtype);
  RECIS_REQUIRE(n_blocks >= 0 && block_rows > 0 && (emb_blocks_dev || n_blocks == 0), "bad block list");
  int64_t segs = 0;
  for (int64_t k = 0; k < n_jobs; ++k) {
    const recis_lookup_job& q = jobs[k];
    RECIS_REQUIRE(q.n_ids >= 0 && q.n_seg >= 0 && q.n_ids < INT32_MAX && q.n_seg < INT32_MAX - kMaxSegs, "feature %lld: bad size",
                  (long long)k);
    RECIS_REQUIRE(q.ids || q.n_ids == 0, "feature %lld: ids must not be NULL", (long long)k);
    RECIS_REQUIRE(q.offsets || (q.width >= 0 && q.width * q.n_seg == q.n_ids),
                  "feature %lld: %lld ids are not %lld segments of %lld", (long long)k, (long long)q.n_ids, (long long)q.n_seg,
                  (long long)q.width);
    RECIS_REQUIRE(q.weight == nullptr || dtype_size(q.weight_dtype), "feature %lld: invalid weight dtype", (long long)k);
    RECIS_REQUIRE(!tagged || (q.table_id >= 0 && q.table_id < 4096), "table id %lld out of 12 bits", (long long)q.table_id);
    segs += q.n_seg;
  }
  RECIS_REQUIRE(segs < INT32_MAX, "too many segments");
  if (segs == 0) return RECIS_OK;
  RECIS_REQUIRE(out != nullptr, "out must not be NULL");
  PoolArgs a{};
  a.table = map->table;
  a.mask = static_cast<uint64_t>(map->capacity - 1);
  a.blocks = emb_blocks_dev;
  a.n_blocks = n_blocks;
  a.block_rows = block_rows;
  a.id_mask = tagged ? (int64_t(1) << 52) - 1 : ~int64_t(0);
  a.D = static_cast<int>(D);
  a.mode = mode;
  const int dev = current_device();
  a.err = device_error_word(dev);
  a.report = error_report_word(dev);
  RECIS_REQUIRE(a.err != nullptr && a.report != nullptr, "could not reach the device error word");
  // blocks are 16-byte aligned by contract
  const int vec_bytes = pick_vec_bytes(D * size, reinterpret_cast<uintptr_t>(out));
  a.pitch = D;
  if (row_pitch_bytes) {
    RECIS_REQUIRE(row_pitch_bytes >= D * size && row_pitch_bytes % size == 0 && row_pitch_bytes % vec_bytes == 0,
                  "row pitch of %lld bytes does not fit rows of %lld elements", (long long)row_pitch_bytes, (long long)D);
    a.pitch = row_pitch_bytes / size;
  }
  const RowGeom g = make_row_geom(D, size, vec_bytes);
  a.lpr_log2 = g.lpr_log2;

  // One segment per team while that leaves compute units idle; with the chip full, two or four (a tile
  // of a dense column is then 256 ids, a probe per thread), as far as the ids of a tile fit in LDS.
  int64_t tiles_at_one = 0;
  auto groups_of = [&](const recis_lookup_job& q) {  // row groups (log2) per segment, as the pooling kernels choose them
    const int64_t avg = q.n_seg > 0 ? q.n_ids / q.n_seg : 1;
    int r = 0;
    while ((int64_t(2) << r) <= avg / 2 && r + g.lpr_log2 < 6) ++r;
    return r;
  };
  for (int64_t k = 0; k < n_jobs; ++k) {
    const int teams = kBlock >> (g.lpr_log2 + groups_of(jobs[k]));
    tiles_at_one += (jobs[k].n_seg + teams - 1) / teams;
  }
  PoolJobs J;
  J.n_jobs = 0;
  int64_t tiles = 0;
  auto launch = [&]() -> int {
    if (tiles == 0) return RECIS_OK;
    RECIS_TIME_KERNEL("lookup_pool_kernel", stream) {
      const int rc = dispatch_pool_vec(g.vec, [&](auto vtag) {
        constexpr int VEC = decltype(vtag)::value;
        const dim3 grid(static_cast<uint32_t>(tiles)), block(kBlock);
        if (row_dtype == RECIS_F32) {
          if constexpr (VEC <= 4) lookup_pool_kernel<float, VEC><<<grid, block, 0, stream>>>(J, a, static_cast<float*>(out));
        } else if (row_dtype == RECIS_BF16) {
          lookup_pool_kernel<bf16_t, VEC><<<grid, block, 0, stream>>>(J, a, static_cast<bf16_t*>(out));
        } else {
          lookup_pool_kernel<f16_t, VEC><<<grid, block, 0, stream>>>(J, a, static_cast<f16_t*>(out));
        }
        RECIS_LAUNCH_CHECK();
        return static_cast<int>(RECIS_OK);
      });
      if (rc) return rc;
    }
    J.n_jobs = 0;
    tiles = 0;
    return RECIS_OK;
  };
  // Features of several ids per segment first: workgroups start in the order of their index, and what starts last should be
  // short.
  auto add = [&](const recis_lookup_job& q, int64_t row0) -> int {
    const int rg = groups_of(q);
    const int teams = kBlock >> (g.lpr_log2 + rg);
    const int64_t avg = (q.n_ids + q.n_seg - 1) / q.n_seg;
    int spt = 0;
    while (spt < 2 && (tiles_at_one >> (spt + 1)) >= kGridFull && (teams << (spt + 1)) <= kMaxSegs &&
           (teams << (spt + 1)) * avg <= 3 * kPoolRows / 4)
      ++spt;
    PoolJob& p = J.job[J.n_jobs++];
    p.ids = q.ids;
    p.offs = q.offsets;
    p.weight = q.weight;
    p.n_ids = static_cast<int32_t>(q.n_ids);
    p.n_seg = static_cast<int32_t>(q.n_seg);
    p.first_tile = static_cast<int32_t>(tiles);
    p.out_row0 = static_cast<int32_t>(row0);
    p.width = static_cast<int32_t>(q.width);
    p.flags = (tagged ? static_cast<uint32_t>(q.table_id) : 0u) | (q.off_is64 ? 1u << 12 : 0u) |
              (q.weight ? static_cast<uint32_t>(q.weight_dtype) << 13 : 0u) | (static_cast<uint32_t>(rg) << 16) |
              (static_cast<uint32_t>(spt) << 20);
    tiles += (q.n_seg + (teams << spt) - 1) / (teams << spt);
    if (J.n_jobs == kPoolJobs) {
      if (int rc = launch()) return rc;
    }
    return RECIS_OK;
  };
  for (const bool several : {true, false}) {
    int64_t row0 = 0;
    for (int64_t k = 0; k < n_jobs; row0 += jobs[k++].n_seg) {
      if (jobs[k].n_seg == 0 || (jobs[k].n_ids > jobs[k].n_seg) != several) continue;
      if (int rc = add(jobs[k], row0)) return rc;
    }
  }
  return launch();
}
