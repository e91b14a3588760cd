// Key-range splitting of the prefill attention kernels (FP32 and BF16).
//
// A 128-query tile of a causal or image-prefixed prefill sees between 128 and
// the whole context's keys, so one workgroup per tile leaves the chip idle
// while the last (longest) tiles finish. Each tile's visible keys are split
// into equal work items (about `target_items` items per call, of about
// kMinChunkKeys keys or more; of kSmallChunkKeys or more in small grids); an item
// runs the tile's online softmax over its keys only and, when its tile is split, stores the unnormalized state (max, denominator,
// output) per query row. merge_kernel combines the parts of a row in part
// order — M = max of the maxima, den = sum den_p exp(m_p - M),
// o = sum o_p exp(m_p - M) — and applies the final step of
// prefill64.rs:468-479: lse = M + ln(den), out = (o / den) / (1 + exp(sink - lse)).
// A static-softmax part has no shift and stores max 0 (weights exp(0) = 1).
#pragma once

#include "focr_internal.hpp"

namespace focr {
namespace split {

constexpr int kQueries = 128;   // query rows per tile
constexpr int kMaxTiles = 256;  // plan table size: 32,768 query rows per launch
// Target work items per call. The FP32 kernel's items are long (about 3 per
// workgroup slot balance the tail); the BF16 kernel's are about five times
// shorter, so fewer, larger parts (less partial-state traffic and merge
// work) measure faster there. The FP16-pair kernel's items are about half
// as long as the FP32 kernel's; 2,048 to 4,096 items measured within noise
// of each other at 6,544 and 16,320 rows (1,536: 5-15 % slower).
constexpr long long kSplitItemsF32 = 3072;
constexpr long long kSplitItemsBf16 = 1536;
constexpr long long kSplitItemsPair = 3072;
constexpr long long kMinChunkKeys = 1024;
// With at most one workgroup per compute unit (tiles x heads), the FP32 and
// FP16-pair kernels are bound by the chain of one workgroup's key tiles (1.2 us
// per 32 keys with one wave per SIMD in the FP16-pair kernel, 2.4 us in the FP32
// one): such calls take parts of about 192 keys or more, about two workgroups per
// compute unit, where that is estimated to be faster than the plan above it.
// The estimate, in keys: the longest item, times the items a compute unit holds
// and how far they run beside each other, plus the merge. Two workgroups of the
// FP16-pair kernel overlap fully; those of the FP32 kernel, bound by the matrix
// cores, hardly, and run in whole rounds. The constants are fitted to 1,790
// measured plans of 1 to 256 heads and 9 to 16,900 visible keys: the rule loses
// at most 5 % (FP16 pairs; 3 % with 16 heads) and 8 % (FP32) against either plan,
// 0.1 % on average.
// us per call, without / with the small parts. FP16 pairs, 16 heads, 0.6 of the
// rows an image: 225 rows 27.5 / 25.2, 400 34.1 / 30.0, 1,000 63 / 42, 1,501 66 /
// 55; 64 heads, 314 rows 37.0 and 37.5 (not split). FP32, 16 heads: 512 rows 47 /
// 25, 1,024 91 / 57, 2,000 rows of 1,600 image 158 and 180 (not split); 128 heads,
// 256 rows 30 and 36 (not split). The BF16 kernel's tiles are too short for
// it: 1,000 rows 26.7 -> 25.0, 400 rows 15.2 -> 15.6.
constexpr int kComputeUnits = 256;
constexpr long long kSmallItems = 512, kSmallChunkKeys = 192;
struct SmallGrid {
  double share;        // of an item's time that each one on a shared compute unit takes
  bool rounds;         // items count in whole rounds of one per compute unit
  double merge, slot;  // the merge as such, and per partial state and head
};
constexpr SmallGrid kSmallPair = {0.5, false, 40.0, 0.3};
constexpr SmallGrid kSmallF32 = {0.85, true, 60.0, 0.05};

// Work plan (computed on the host, passed by value): query tiles in dispatch
// order i (tile tiles - 1 - i: the latest, longest tiles first), each split
// into parts of equal size.
struct Plan {
  int first[kMaxTiles + 1];  // first work item of the i-th tile; first[tiles] = items
  int slot[kMaxTiles];       // first partial slot of the i-th tile if it is split
  int keys[kMaxTiles];       // keys per part of the i-th tile
};

struct Args {
  const float *sinks;
  float *out;
  float *part;  // [slot][head][128 rows][64] outputs, then [slot][head][128][2] (max, den)
  int query_len, n_heads, tiles, slots;
  int merge_end;  // rows at or past it are written by another kernel
};

// Keys [0, end) that query tile `tile` sees (tile_span, prefill64/span.rs:9-20).
__host__ __device__ inline int tile_visible_end(int tile, int query_len, int query_offset, int image_start,
                                                int image_end) {
  const int first_query = tile * kQueries;
  const int queries = query_len - first_query < kQueries ? query_len - first_query : kQueries;
  const int first_abs = query_offset + first_query, last_abs = first_abs + queries - 1;
  const bool intersects = first_abs < image_end && last_abs >= image_start;
  return intersects ? (last_abs + 1 > image_end ? last_abs + 1 : image_end) : last_abs + 1;
}

// Keys per part of a tile of `end` visible keys cut into parts of at most
// `chunk` keys, as equal as multiples of `align` allow.
inline int part_keys(int end, long long chunk, int align) {
  const int parts = static_cast<int>((end + chunk - 1) / chunk);
  return ((end + parts - 1) / parts + align - 1) / align * align;
}

// The items of tiles of vis[] keys cut into parts of at most `chunk`.
struct Cut {
  long long items = 0, slots = 0;
  int part = 0, whole = 0;  // the longest part of a split tile, the longest unsplit tile
};
inline Cut cut_of(const int *vis, int tiles, long long chunk, int align) {
  Cut c;
  for (int t = 0; t < tiles; t++) {
    const int per = part_keys(vis[t], chunk, align), parts = (vis[t] + per - 1) / per;
    int &longest = parts > 1 ? c.part : c.whole;
    const int keys = parts > 1 ? per : vis[t];
    longest = keys > longest ? keys : longest;
    c.items += parts;
    c.slots += parts > 1 ? parts : 0;
  }
  return c;
}
inline double estimate(const Cut &c, int n_heads, const SmallGrid &g) {
  const long long items = c.items * n_heads;
  const double full = g.rounds ? static_cast<double>((items + kComputeUnits - 1) / kComputeUnits)
                               : static_cast<double>(items) / kComputeUnits;
  const double share = items <= kComputeUnits || full * g.share < 1.0 ? 1.0 : full * g.share;
  return (c.part > c.whole ? c.part : c.whole) * share + (c.slots > 0 ? g.merge + g.slot * c.slots * n_heads : 0.0);
}

// Builds the plan for `tiles` (<= kMaxTiles) tiles; part sizes are multiples
// of `align` keys. `small` (optional): the small-grid parts may be taken.
// Returns the number of work items; *slots = partial slots.
inline int make_plan(Plan &plan, int tiles, int query_len, int query_offset, int image_start, int image_end,
                     int n_heads, int align, long long target_items, const SmallGrid *small, int *slots_out) {
  long long total = 0;
  int vis[kMaxTiles], most = 0;
  for (int t = 0; t < tiles; t++) {
    vis[t] = tile_visible_end(t, query_len, query_offset, image_start, image_end);
    total += vis[t];
    most = vis[t] > most ? vis[t] : most;
  }
  const long long want = total * static_cast<long long>(n_heads) / target_items;
  long long chunk = ((want > kMinChunkKeys ? want : kMinChunkKeys) + align - 1) / align * align;
  // Tiles of nearly equal cost (an all-image or short prefill) balance by
  // themselves: splitting them would only add the merge traffic.
  if (5LL * most <= 6LL * total / (tiles > 0 ? tiles : 1)) chunk = most;
  if (small && static_cast<long long>(tiles) * n_heads <= kComputeUnits) {
    const long long few = total * static_cast<long long>(n_heads) / kSmallItems;
    long long fine = ((few > kSmallChunkKeys ? few : kSmallChunkKeys) + align - 1) / align * align;
    fine = fine < chunk ? fine : chunk;
    Cut c = cut_of(vis, tiles, fine, align);
    // An unsplit tile longer than the parts would be the longest item: it is
    // cut too (256 rows of 153 image, 28.7 -> 25.4 us).
    if (c.part > 0 && c.whole > c.part) {
      fine = c.part;
      c = cut_of(vis, tiles, fine, align);
    }
    if (estimate(c, n_heads, *small) < estimate(cut_of(vis, tiles, chunk, align), n_heads, *small)) chunk = fine;
  }
  int items = 0, slots = 0;
  for (int i = 0; i < tiles; i++) {
    const int end = vis[tiles - 1 - i];
    const int per = part_keys(end, chunk, align);
    const int parts = (end + per - 1) / per;  // every part starts before `end`
    plan.first[i] = items;
    plan.slot[i] = parts > 1 ? slots : -1;
    plan.keys[i] = per;
    items += parts;
    slots += parts > 1 ? parts : 0;
  }
  plan.first[tiles] = items;
  *slots_out = slots;
  return items;
}

// This workgroup's work item: plan order and part.
struct Item {
  int order, part, parts, key_begin, keys;
};
__device__ inline Item find_item(const Plan &plan, int tiles, int item) {
  int lo = 0, hi = tiles - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (plan.first[mid] <= item) lo = mid; else hi = mid - 1;
  }
  Item it;
  it.order = lo;
  it.part = item - plan.first[lo];
  it.parts = plan.first[lo + 1] - plan.first[lo];
  it.keys = plan.keys[lo];
  it.key_begin = it.part * it.keys;
  return it;
}

// Where part `it` of head `head` stores row `row_in_tile`'s state.
__device__ inline float *part_out(const Args &a, const Plan &plan, const Item &it, int head, int row_in_tile) {
  const size_t slot = static_cast<size_t>(plan.slot[it.order] + it.part) * a.n_heads + head;
  return a.part + (slot * kQueries + row_in_tile) * 64;
}
__device__ inline float2 *part_md(const Args &a, const Plan &plan, const Item &it, int head, int row_in_tile) {
  const size_t slot = static_cast<size_t>(plan.slot[it.order] + it.part) * a.n_heads + head;
  return reinterpret_cast<float2 *>(a.part + static_cast<size_t>(a.slots) * a.n_heads * kQueries * 64) +
         slot * kQueries + row_in_tile;
}

// Grid (tiles, heads, kMergeSplit): a workgroup merges kQueries /
// kMergeSplit rows of one tile and head (unsplit tiles exit), eight threads
// per row, each 8 of the 64 dims. The parts' maxima are read first, then
// their outputs kMergeBatch parts at a time (all loads of a batch in flight
// together), added in part order.
constexpr int kMergeSplit = 4;
constexpr int kMergeBatch = 4;
static __global__ __launch_bounds__(256) void merge_kernel(Args a, Plan plan) {
  const int order = blockIdx.x, head = blockIdx.y;
  const int parts = plan.first[order + 1] - plan.first[order];
  if (parts <= 1) return;
  const int row_in_tile = blockIdx.z * (kQueries / kMergeSplit) + (threadIdx.x >> 3), slice = threadIdx.x & 7;
  const int row = (a.tiles - 1 - order) * kQueries + row_in_tile;
  if (row >= a.merge_end) return;
  const float2 *md = reinterpret_cast<const float2 *>(a.part + static_cast<size_t>(a.slots) * a.n_heads * kQueries * 64);
  const size_t slot0 = static_cast<size_t>(plan.slot[order]) * a.n_heads + head;
  const size_t pstride = static_cast<size_t>(a.n_heads);  // slots between consecutive parts of a tile and head
  const float ninf = -__builtin_inff();
  float big = ninf;
  for (int p0 = 0; p0 < parts; p0 += kMergeBatch) {
    float2 m[kMergeBatch];
#pragma unroll
    for (int j = 0; j < kMergeBatch; j++) {
      const int p = p0 + j < parts ? p0 + j : parts - 1;
      m[j] = md[(slot0 + p * pstride) * kQueries + row_in_tile];
    }
#pragma unroll
    for (int j = 0; j < kMergeBatch; j++)
      if (p0 + j < parts) big = __builtin_fmaxf(big, m[j].x);
  }
  float den = 0.0f;
  float4 o[2] = {make_float4(0.f, 0.f, 0.f, 0.f), make_float4(0.f, 0.f, 0.f, 0.f)};
  for (int p0 = 0; p0 < parts; p0 += kMergeBatch) {
    float2 m[kMergeBatch];
    float4 v[kMergeBatch][2];
#pragma unroll
    for (int j = 0; j < kMergeBatch; j++) {
      const int p = p0 + j < parts ? p0 + j : parts - 1;
      const size_t slot = slot0 + p * pstride;
      m[j] = md[slot * kQueries + row_in_tile];
      const float4 *src = reinterpret_cast<const float4 *>(a.part + (slot * kQueries + row_in_tile) * 64 + 8 * slice);
      v[j][0] = src[0];
      v[j][1] = src[1];
    }
#pragma unroll
    for (int j = 0; j < kMergeBatch; j++) {
      if (p0 + j >= parts) break;
      const float f = m[j].x == ninf ? 0.0f : expf_acc(m[j].x - big);
      den = den + m[j].y * f;
#pragma unroll
      for (int i = 0; i < 2; i++)
        o[i] = make_float4(fmaf_(v[j][i].x, f, o[i].x), fmaf_(v[j][i].y, f, o[i].y), fmaf_(v[j][i].z, f, o[i].z),
                           fmaf_(v[j][i].w, f, o[i].w));
    }
  }
  const float lse = big + logf_acc(den);
  const float sink_scale = __fdiv_rn(1.0f, 1.0f + expf_acc(a.sinks[head] - lse));
  float4 *dst = reinterpret_cast<float4 *>(a.out + (static_cast<size_t>(row) * a.n_heads + head) * 64 + 8 * slice);
#pragma unroll
  for (int i = 0; i < 2; i++)
    dst[i] = make_float4(__fmul_rn(__fdiv_rn(o[i].x, den), sink_scale), __fmul_rn(__fdiv_rn(o[i].y, den), sink_scale),
                         __fmul_rn(__fdiv_rn(o[i].z, den), sink_scale), __fmul_rn(__fdiv_rn(o[i].w, den), sink_scale));
}

}  // namespace split
}  // namespace focr
