// Block mask -> compacted active-tile list (CSR over query tiles, CSC over key tiles).
//
// Refinement rule (one block -> rate x rate tiles): EMPTY stays empty, FULL becomes all full,
// CAUSAL becomes causal on the sub-diagonal, full below it and empty above it.  Tiles are
// emitted row-major (query tile outer, key tile inner).
#include <algorithm>
#include <atomic>
#include <numeric>
#include <type_traits>
#include <vector>
#include "ua_common.h"

// Scratch of the entry point that allocates nothing (ua_tilelist_build_device_noalloc): the
// per-row and per-column tile counts that the device builder otherwise keeps in the caller's
// `work` argument.  Every GPU the library runs on holds its own copy (256 KiB) until the process
// ends; calls on one GPU share it, so two such calls must not overlap.
static __device__ __align__(256) int32_t scratch[UA_NOALLOC_MAX_LINES + 8];

namespace ua {

// type of tile (qt, kt): 0 empty, 1 full, 2 causal
inline int tile_type(const uint8_t* mask, int nkb, int rate, int qt, int kt) {
  const int t = mask[(int64_t)(qt / rate) * nkb + kt / rate];
  if (t != 2) return t == 1 ? 1 : 0;
  const int a = qt % rate, b = kt % rate;
  return a == b ? 2 : (a > b ? 1 : 0);
}

// Launch order: does line a (a row of the CSR, or a column of the CSC) come before line b?
//  1. Lines much longer than average (len * n > 2 * nnz) first, so that they cannot end up as
//     the tail of the launch; among them the longer block lines first (see 3), then as in 4.
//  2. The rest by their anchor index, ascending.  The anchor is the first index of the list, or
//     the last one when `from_end`: lines that share it walk common tiles (the rows of a causal
//     mask share their oldest keys, its columns their latest queries).
//  3. Among those, the lines of longer block lines first (the length of a tile's block line =
//     the list length of that block's longest tile: sub-tile rate-1 of a row block, sub-tile 0 of
//     a column block): the short lists end the group, and a list that leaves the common part
//     early does not run ahead of the lists that still walk it.
//  4. Then lexicographic order of the index lists read from the anchor, a list that is a prefix
//     (from_end: a suffix) of another sorting after it; ties by line number.  Lines that walk the
//     same K/V (or Q/dO) tiles thus sit next to each other in the launch and share them in L2.
inline bool very_long(const int32_t* ptr, int n, int a) {
  return (int64_t)(ptr[a + 1] - ptr[a]) * n > 2 * (int64_t)ptr[n];
}
inline bool row_precedes(const int32_t* ptr, const int32_t* idx, int n, int rate, int longest_sub,
                                                      bool from_end, int a, int b) {
  const int pa = ptr[a], pb = ptr[b];
  const int la = ptr[a + 1] - pa, lb = ptr[b + 1] - pb;
  const bool va = very_long(ptr, n, a), vb = very_long(ptr, n, b);
  if (va != vb) return va;
  if (la > 0 && lb > 0) {
    // element t of a list, counted from its anchor
    const int sa = from_end ? pa + la - 1 : pa, sb = from_end ? pb + lb - 1 : pb, step = from_end ? -1 : 1;
    const int fa = idx[sa], fb = idx[sb];
    const int ra = a / rate * rate + longest_sub, rb = b / rate * rate + longest_sub;
    const int ba = ptr[ra + 1] - ptr[ra], bb = ptr[rb + 1] - ptr[rb];
    if (va) {                       // rule 1: block-line length decides before the anchor
      if (ba != bb) return ba > bb;
      if (fa != fb) return fa < fb;
    } else {
      if (fa != fb) return fa < fb;
      if (ba != bb) return ba > bb;
    }
    const int m = la < lb ? la : lb;
    for (int t = 1; t < m; ++t) {
      const int ca = idx[sa + t * step], cb = idx[sb + t * step];
      if (ca != cb) return ca < cb;
    }
  }
  if (la != lb) return la > lb;
  return a < b;
}
// Which end anchors the order of one side: the one with FEWER distinct values over the lines that
// rule 2 applies to (more lines share it); the start on a tie.
inline bool anchor_from_end(const int32_t* ptr, const int32_t* idx, int n) {
  std::vector<int32_t> first, last;
  for (int i = 0; i < n; ++i)
    if (ptr[i + 1] > ptr[i] && !very_long(ptr, n, i)) { first.push_back(idx[ptr[i]]); last.push_back(idx[ptr[i + 1] - 1]); }
  auto distinct = [](std::vector<int32_t>& v) { std::sort(v.begin(), v.end()); return std::unique(v.begin(), v.end()) - v.begin(); };
  return distinct(last) < distinct(first);
}

static int check_mask(const uint8_t* mask, int nqb, int nkb, int rate) {
  if (!mask) return UA_ERR_NULL;
  if (nqb <= 0 || nkb <= 0 || rate <= 0) return UA_ERR_SHAPE;
  if ((int64_t)nqb * rate > (1 << 24) || (int64_t)nkb * rate > (1 << 24)) return UA_ERR_SHAPE;
  for (int64_t i = 0; i < (int64_t)nqb * nkb; ++i)
    if (mask[i] > 2) return UA_ERR_MASK;
  return UA_OK;
}

// ---- device variant -----------------------------------------------------------------------
// Three launches: count, fill, order.  At the benchmark's 256 x 256 blocks every one of them is a chain of a few
// dependent loads, so what counts is how many launches there are and how long the longest chain is; eleven
// launches (init, check, count, two scans, fill, three for the anchors, order) took 61 us a pass, these three 16.
//
// One wavefront per query tile (a "row" of the list) and per key tile (a "column"); lanes
// stride over the blocks of that row or column of the block mask.  Number of active tiles
// that block (qb, kb) gives to query tile qt = qb*rate + a: FULL rate, CAUSAL a + 1 (key
// sub-tiles 0..a); to key tile kt = kb*rate + b: FULL rate, CAUSAL rate - b (query sub-tiles
// b..rate-1).
constexpr int kWavesPerGroup = 4;

struct Line {          // one row or one column of the tile grid, as seen by its wavefront
  bool is_row;
  int id;              // tile index of the row or column
  int n_blocks;        // blocks along it
  int sub;             // id % rate
  int64_t base, step;  // block (i) of the line sits at mask[base + i*step]
};
inline int line_groups(int n) { return (n + kWavesPerGroup - 1) / kWavesPerGroup; }
// The first workgroups take the rows, the others the columns: a workgroup's lines belong to one side.
__device__ __forceinline__ bool line_of_wave(int nqb, int nkb, int rate, Line& ln) {
  const int nqt = nqb * rate, nkt = nkb * rate;
  const int groups_q = (nqt + kWavesPerGroup - 1) / kWavesPerGroup;
  ln.is_row = (int)blockIdx.x < groups_q;
  ln.id = (blockIdx.x - (ln.is_row ? 0 : groups_q)) * kWavesPerGroup + (threadIdx.x >> 6);
  ln.n_blocks = ln.is_row ? nkb : nqb;
  ln.sub = ln.id % rate;
  ln.base = ln.is_row ? (int64_t)(ln.id / rate) * nkb : ln.id / rate;
  ln.step = ln.is_row ? 1 : nkb;
  return ln.id < (ln.is_row ? nqt : nkt);
}
// Tiles that a CAUSAL block gives to the line; all of them give the same number, so sums over lanes are bit counts.
__device__ __forceinline__ int causal_tiles(const Line& ln, int rate) { return ln.is_row ? ln.sub + 1 : rate - ln.sub; }
// Types of 64 * kAhead blocks of the line, block i0 + 64 * u + lane in type[u], 0 beyond its end; all loads in flight at once.
constexpr int kAhead = 4;
__device__ __forceinline__ void load_types(const uint8_t* mask, const Line& ln, int i0, int (&type)[kAhead]) {
#pragma unroll
  for (int u = 0; u < kAhead; ++u) {
    const int i = i0 + 64 * u + (threadIdx.x & 63);
    type[u] = i < ln.n_blocks ? mask[ln.base + i * ln.step] : 0;
  }
}
// Sum over the wavefront by DPP additions (rows of 16, then across them; the total arrives in lane 63): through
// LDS, as shuffles go, each of the six steps takes 60 ns.
template <int kCtrl, int kRows>
__device__ __forceinline__ int dpp_add(int v) { return v + __builtin_amdgcn_update_dpp(0, v, kCtrl, kRows, 0xf, false); }
__device__ __forceinline__ int wave_sum(int v) {
  v = dpp_add<0x111, 0xf>(v);      // row_shr 1, 2, 4, 8
  v = dpp_add<0x112, 0xf>(v);
  v = dpp_add<0x114, 0xf>(v);
  v = dpp_add<0x118, 0xf>(v);
  v = dpp_add<0x142, 0xa>(v);      // row_bcast 15 into rows 1 and 3
  v = dpp_add<0x143, 0xc>(v);      // row_bcast 31 into rows 2 and 3
  return __builtin_amdgcn_readlane(v, 63);
}

// count: tiles per line.  The builder treats mask entries that are not a Block_Type (> 2) as EMPTY; how many
// there are is left in q_order (one entry per row, still free here) and added up by the fill kernel, so that
// the caller can detect them after the stream has been synchronised (the host builder returns UA_ERR_MASK).
__global__ __launch_bounds__(64 * kWavesPerGroup) void tl_count_kernel(const uint8_t* mask, int nqb, int nkb, int rate,
                                                                        int32_t* qcnt, int32_t* kcnt, int32_t* row_invalid) {
  Line ln;
  if (!line_of_wave(nqb, nkb, rate, ln)) return;
  const int lane = threadIdx.x & 63;
  int n = 0, bad = 0;
  for (int i0 = 0; i0 < ln.n_blocks; i0 += 64 * kAhead) {
    int type[kAhead];
    load_types(mask, ln, i0, type);
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      n += rate * __popcll(__ballot(type[u] == 1)) + causal_tiles(ln, rate) * __popcll(__ballot(type[u] == 2));
      bad += __popcll(__ballot(type[u] > 2));
    }
  }
  if (lane != 0) return;
  (ln.is_row ? qcnt : kcnt)[ln.id] = n;
  if (ln.is_row) row_invalid[ln.id] = ln.sub == 0 ? bad : 0;
}

typedef __attribute__((ext_vector_type(4), aligned(4))) int32_t i32x4_any;       // at any element of a list
typedef __attribute__((aligned(1))) uint32_t u32_any;
// The tiles that 64 blocks of a line, of which `full` and `causal` tell the types, give it, from slot e on; returns the slot behind
// them.  An exclusive scan of the per-block tile counts gives every lane the slot where its block's tiles go, in ascending order.
__device__ __forceinline__ int fill_blocks(bool is_row, int sub, int rate, int i0, uint64_t full, uint64_t causal, int e, int32_t* idx, uint8_t* flg) {
  if (!(full | causal)) return e;
  const int lane = threadIdx.x & 63, n_causal = is_row ? sub + 1 : rate - sub, i = i0 + lane;
  const uint64_t below = (1ull << lane) - 1;
  const int ty = (full >> lane & 1) ? 1 : ((causal >> lane & 1) ? 2 : 0);
  const int c = ty == 1 ? rate : (ty == 2 ? n_causal : 0);
  int at = e + rate * __popcll(full & below) + n_causal * __popcll(causal & below);
  // sub-tiles along the line: a row takes key sub-tiles 0..sub of a causal block (the last one
  // causal), a column takes query sub-tiles sub..rate-1 (the first one causal)
  const int first = (ty == 2 && !is_row) ? sub : 0;
  // four tiles and their flags per store
  int t = 0;
  for (; t + 4 <= c; t += 4, at += 4) {
    const int s = i * rate + first + t, mark = sub - first - t;           // the causal one among them, if 0..3
    *reinterpret_cast<i32x4_any*>(idx + at) = i32x4_any{s, s + 1, s + 2, s + 3};
    *reinterpret_cast<u32_any*>(flg + at) = ty == 2 && (unsigned)mark < 4 ? 1u << (8 * mark) : 0;
  }
  for (; t < c; ++t, ++at) {
    idx[at] = i * rate + first + t;
    flg[at] = ty == 2 && first + t == sub;
  }
  return e + rate * __popcll(full) + n_causal * __popcll(causal);
}
// fill: a workgroup first adds up the counts of its side (those before its lines give its place in the list,
// all of them the list's length), then each wavefront walks its line 64 blocks at a time.
__global__ __launch_bounds__(64 * kWavesPerGroup) void tl_fill_kernel(const uint8_t* mask, int nqb, int nkb, int rate,
                                                                       const int32_t* qcnt, const int32_t* kcnt, int32_t* row_ptr, int32_t* col_idx, uint8_t* flag,
                                                                       int32_t* col_ptr, int32_t* row_idx, uint8_t* cflag,
                                                                       const int32_t* row_invalid, int32_t* n_invalid) {
  __shared__ int32_t part[kWavesPerGroup][3];
  Line ln;
  const bool live = line_of_wave(nqb, nkb, rate, ln);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int n = (ln.is_row ? nqb : nkb) * rate, first_line = ln.id - wave;
  const int32_t* cnt = ln.is_row ? qcnt : kcnt;
  int type[kAhead];                   // the first blocks are on their way while the counts are added up
  if (live) load_types(mask, ln, 0, type);
  int before = 0, all = 0, bad = 0;
  for (int i0 = threadIdx.x; i0 < n; i0 += 64 * kWavesPerGroup * kAhead) {
    int c[kAhead];
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      const int i = i0 + 64 * kWavesPerGroup * u;
      c[u] = i < n ? cnt[i] : 0;
    }
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      all += c[u];
      if (i0 + 64 * kWavesPerGroup * u < first_line) before += c[u];
    }
  }
  if (blockIdx.x == 0)
    for (int i = threadIdx.x; i < n; i += 64 * kWavesPerGroup) bad += row_invalid[i];
  int own = 0;                        // lines of the workgroup before this wavefront's
  for (int w = 0; w < wave; ++w) own += first_line + w < n ? cnt[first_line + w] : 0;
  before = wave_sum(before); all = wave_sum(all);
  if (blockIdx.x == 0) bad = wave_sum(bad);
  if (lane == 0) { part[wave][0] = before; part[wave][1] = all; part[wave][2] = bad; }
  __syncthreads();
  before = all = bad = 0;
#pragma unroll
  for (int w = 0; w < kWavesPerGroup; ++w) { before += part[w][0]; all += part[w][1]; bad += part[w][2]; }
  if (blockIdx.x == 0 && threadIdx.x == 0) *n_invalid = bad;
  if (!live) return;
  int e = before + own;
  int32_t* ptr = ln.is_row ? row_ptr : col_ptr;
  if (lane == 0) {
    ptr[ln.id] = e;
    if (ln.id == n - 1) ptr[n] = all;
  }
  int32_t* idx = ln.is_row ? col_idx : row_idx;
  uint8_t* flg = ln.is_row ? flag : cflag;
  for (int i0 = 0; i0 < ln.n_blocks; i0 += 64 * kAhead) {
    if (i0 > 0) load_types(mask, ln, i0, type);
#pragma unroll
    for (int u = 0; u < kAhead; ++u)
      e = fill_blocks(ln.is_row, ln.sub, rate, i0 + 64 * u, __ballot(type[u] == 1), __ballot(type[u] == 2), e, idx, flg);
  }
}

// order: rank of a line = number of lines that precede it by row_precedes.  A workgroup ranks kOrderLines lines:
// every thread packs what decides first about one other line (very long, anchor, block-line length) into one 64-bit key
// and compares it with those of all kOrderLines; counts are ballots.  Pairs with equal keys are queued: lines of one block are decided by what refinement
// makes of their common row of the mask, for the others 16 lanes compare 64 indices of both lists at once.  One line per workgroup and a thread per pair, list comparison included: 32 us for
// 2 x 1024 lines, most of it the four rows of a block walking their common list one index at a time.
constexpr int kOrderThreads = 1024, kOrderLines = 8, kSeen = 8192;
__global__ __launch_bounds__(kOrderThreads) void tl_order_kernel(const int32_t* qptr, const int32_t* qidx, int nq, int32_t* q_order,
                                                                 const int32_t* kptr, const int32_t* kidx, int nk, int32_t* k_order, int rate) {
  struct ListOf { int32_t at, len, first; };
  __shared__ uint64_t own_key[kOrderLines];
  __shared__ ListOf own[kOrderLines], other[kOrderThreads];
  __shared__ int32_t rank[kOrderLines], n_first, n_last, n_queued;
  __shared__ uint32_t seen_first[kSeen / 4], seen_last[kSeen / 4];             // a byte per value
  __shared__ uint32_t queue[kOrderThreads * kOrderLines];          // pairs of one round: line | slot << 28
  const int groups_q = (nq + kOrderLines - 1) / kOrderLines;
  const bool rows = (int)blockIdx.x < groups_q;
  const int32_t *ptr = rows ? qptr : kptr, *idx = rows ? qidx : kidx;
  const int n = rows ? nq : nk, n_marks = rows ? nk : nq, longest_sub = rows ? rate - 1 : 0;
  const int line0 = (blockIdx.x - (rows ? 0 : groups_q)) * kOrderLines, n_own = min(kOrderLines, n - line0);
  const int tid = threadIdx.x, lane = tid & 63;
  if (tid < kOrderLines) rank[tid] = 0;
  if (tid == 0) n_first = n_last = n_queued = 0;
  // Both ends of the list are read, so that everything the first round needs is on its way before the first barrier.
  struct Raw { int32_t at, len, first, last, block_len; };
  auto raw_of = [&](int i) {
    const int p = ptr[i], len = ptr[i + 1] - p, r = i / rate * rate + longest_sub;
    return Raw{p, len, len ? idx[p] : 0, len ? idx[p + len - 1] : 0, ptr[r + 1] - ptr[r]};
  };
  const int64_t twice_all = 2 * (int64_t)ptr[n];
  Raw mine{}, own_raw{};
  if (tid < n) mine = raw_of(tid);
  if (tid < n_own) own_raw = raw_of(line0 + tid);
  // Which end anchors the lists: the one with fewer distinct values over the lines that are neither empty nor very
  // long, counted kSeen values at a time.  (Marking them in memory, in the fill kernel, cost 5 us: lines share
  // their anchors, and atomics of many XCDs on one word are served one by one.)
  auto very_long = [&](int len) { return (int64_t)len * n > twice_all; };
  for (int v0 = 0; v0 < n_marks; v0 += kSeen) {
    const int words = (min(n_marks - v0, kSeen) + 3) / 4;
    for (int i = tid; i < words; i += kOrderThreads) seen_first[i] = seen_last[i] = 0;
    __syncthreads();
    for (int i = tid; i < n; i += kOrderThreads) {
      const Raw r = i == tid ? mine : raw_of(i);
      const uint32_t f = r.first - v0, l = r.last - v0;
      if (r.len == 0 || very_long(r.len)) continue;
      if (f < kSeen) reinterpret_cast<uint8_t*>(seen_first)[f] = 1;
      if (l < kSeen) reinterpret_cast<uint8_t*>(seen_last)[l] = 1;
    }
    __syncthreads();
    int f = 0, l = 0;
    for (int i = tid; i < words; i += kOrderThreads) { f += __popc(seen_first[i]); l += __popc(seen_last[i]); }
    f = wave_sum(f); l = wave_sum(l);
    if (lane == 0 && (f | l)) { atomicAdd(&n_first, f); atomicAdd(&n_last, l); }
    __syncthreads();
  }
  const bool from_end = n_last < n_first;
  // very long lines first, among them by block-line length before the anchor; empty ones last, by number
  auto key_of = [&](const Raw& r, int i) {
    const uint64_t anchor = from_end ? r.last : r.first, shorter = (1 << 30) - 1 - r.block_len;
    if (r.len == 0) return 1ull << 63 | (uint64_t)i;
    return very_long(r.len) ? shorter << 30 | anchor : 1ull << 62 | anchor << 30 | shorter;
  };
  if (tid < kOrderLines) {
    own_key[tid] = tid < n_own ? key_of(own_raw, line0 + tid) : 0;            // no line has a smaller key than 0, nor that one
    own[tid] = {own_raw.at, own_raw.len, own_raw.first};
  }
  __syncthreads();
  int before[kOrderLines] = {};        // of this wavefront's lines, how many come first
  for (int j0 = 0; j0 < n; j0 += kOrderThreads) {
    const int j = j0 + tid;
    if (j0 > 0 && j < n) mine = raw_of(j);
    const uint64_t key = j < n ? key_of(mine, j) : ~0ull;
    other[tid] = {mine.at, mine.len, mine.first};
#pragma unroll
    for (int s = 0; s < kOrderLines; ++s) {
      const uint64_t b = own_key[s];
      before[s] += __popcll(__ballot(key < b));
      if (__any(key == b)) {
        if (key == b && j < n && j != line0 + s) queue[atomicAdd(&n_queued, 1)] = (uint32_t)j | (uint32_t)s << 28;
      }
    }
    __syncthreads();
    const int queued = n_queued;
    for (int e0 = (tid >> 6) * 4; e0 < queued; e0 += kOrderThreads / 16) {
      const int quarter = lane >> 4, sub = lane & 15;
      const bool live = e0 + quarter < queued;
      const uint32_t pair = queue[live ? e0 + quarter : e0];
      const int ja = pair & 0xfffffff, slot = pair >> 28;
      const ListOf a = other[ja - j0], b = own[slot];
      const int m = min(a.len, b.len), step = from_end ? -1 : 1;
      const int sa = from_end ? a.at + a.len - 1 : a.at, sb = from_end ? b.at + b.len - 1 : b.at;
      const int d = ja - (line0 + slot), d_len = a.len - b.len;
      bool less = d_len != 0 ? d_len > 0 : d < 0;                  // one list ends inside the other, or they are equal
      bool open = live;
      // Lines of one block: their lists differ only where the block's line of the mask is CAUSAL, and by the number of
      // such blocks in length (the same lists if there is none).
      if (ja / rate == (line0 + slot) / rate) {
        if (d_len == 0)                 open = false;
        else if (rows)                { open = false; less = from_end ? d < 0 : d > 0; }      // keys 0..sub of the block: the longer list goes on in it
        else if (!from_end)           { open = false; less = d < 0; }                         // queries sub..: the smaller sub's come first
        else if (a.first == b.first)  { open = false; less = d > 0; }                         // read backwards, the larger sub leaves the block first
        else if (abs(d_len) == abs(d)){ open = false; less = d < 0; }                         // and, this being the only one, ends there
      }
      for (int t0 = 1; __any(open && t0 < m); t0 += 64) {
        int ca[4] = {}, cb[4] = {};
        open &= t0 < m;
        if (open) {
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const int t = min(t0 + 16 * u + sub, m - 1);
            ca[u] = idx[sa + t * step];
            cb[u] = idx[sb + t * step];
          }
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const uint32_t differ = (uint32_t)(__ballot(ca[u] != cb[u]) >> (16 * quarter)) & 0xffff;
          const uint32_t smaller = (uint32_t)(__ballot(ca[u] < cb[u]) >> (16 * quarter));
          if (open && differ) {
            less = (smaller >> (__ffs(differ) - 1)) & 1;
            open = false;
          }
        }
      }
      if (sub == 0 && live && less) atomicAdd(&rank[slot], 1);
    }
    __syncthreads();
    if (tid == 0) n_queued = 0;
    __syncthreads();
  }
  int add = 0;
#pragma unroll
  for (int s = 0; s < kOrderLines; ++s) add = lane == s ? before[s] : add;
  if (lane < n_own && add) atomicAdd(&rank[lane], add);
  __syncthreads();
  if (tid < n_own) (rows ? q_order : k_order)[rank[tid]] = line0 + tid;
}

// ---- the same in two launches, for masks of up to kScanBlocks blocks a side and a caller that has scratch for them ---------------
// The lists' places, ends and order all follow from the block lines.  The first launch leaves each of them as bits (FULL blocks,
// CAUSAL blocks) and as what is asked of it most; the second reads that, fills the lists and ranks them, in workgroups of their own
// that do not wait for each other.  In three launches the ranks wait for the lists, and lines with equal keys are told apart by
// walking both.  Two dependent launches that do nothing take 5 us.  A pass of 256 x 256 blocks of 512: strided 15.8 -> 10.5 us, causal 17.0 ->
// 10.8, global+local, whose rows all begin with the same blocks, 67.8 -> 10.3; 8 x 8 blocks of 128: 11.3 -> 8.7.
constexpr int kScanBlocks = 256, kScanWords = kScanBlocks / 64, kListThreads = 256;
struct BlockLine {
  uint64_t full[kScanWords], causal[kScanWords];
};
struct BlockStat {
  uint16_t n, n_causal;                    // blocks that are not EMPTY, CAUSAL ones
  uint8_t first, last;                     // of those that are not EMPTY
  uint8_t ends;                            // bit 0: the first is CAUSAL, 1: the last is, 2: the line holds an entry that is no Block_Type
  uint8_t unused;
};
static_assert(sizeof(BlockLine) == 64 && sizeof(BlockStat) == 8, "read 16 and 8 bytes at a time");
struct ListSide {
  BlockLine* lines;
  BlockStat* stats;
  int32_t *ptr, *idx, *order;
  uint8_t* flag;
  int n_blocks, n_other;                   // block lines, blocks along each
};
// Tiles of line `sub` of a block line, and of all of its lines.
__device__ __forceinline__ int line_tiles(const BlockStat& b, bool rows, int sub, int rate) {
  return rate * (b.n - b.n_causal) + b.n_causal * (rows ? sub + 1 : rate - sub);
}
__device__ __forceinline__ int block_tiles(const BlockStat& b, int rate) { return rate * rate * (b.n - b.n_causal) + b.n_causal * (rate * (rate + 1) / 2); }

__global__ __launch_bounds__(64 * kWavesPerGroup) void tl_scan_kernel(const uint8_t* mask, int nqb, int nkb, ListSide q, ListSide k) {
  Line ln;
  if (!line_of_wave(nqb, nkb, 1, ln)) return;
  static_assert(kAhead == kScanWords, "a line's blocks are loaded in one go");
  int type[kAhead];
  load_types(mask, ln, 0, type);
  BlockLine bits;
  BlockStat st = {};
#pragma unroll
  for (int u = 0; u < kAhead; ++u) {
    const uint64_t full = __ballot(type[u] == 1), causal = __ballot(type[u] == 2), any = full | causal;
    bits.full[u] = full; bits.causal[u] = causal;
    if (__any(type[u] > 2)) st.ends |= 4;
    if (!any) continue;
    const int lo = __builtin_ctzll(any), hi = 63 - __builtin_clzll(any);
    if (st.n == 0) { st.first = 64 * u + lo; st.ends |= (uint8_t)(causal >> lo & 1); }
    st.last = 64 * u + hi;
    st.ends = (st.ends & 5) | (uint8_t)(causal >> hi & 1) << 1;
    st.n += __popcll(any);
    st.n_causal += __popcll(causal);
  }
  if ((threadIdx.x & 63) != 0) return;
  const ListSide& s = ln.is_row ? q : k;
  s.lines[ln.id] = bits;
  s.stats[ln.id] = st;
}

// One wavefront fills one line: its place is what the block lines before it hold.
__device__ __forceinline__ void fill_line(const ListSide& s, bool rows, int rate, int id) {
  const int lane = threadIdx.x & 63, own = id / rate, sub = id % rate;
  BlockStat x[kScanWords];
#pragma unroll
  for (int u = 0; u < kScanWords; ++u) x[u] = 64 * u + lane < own ? s.stats[64 * u + lane] : BlockStat{};
  const BlockStat me = s.stats[own];
  const BlockLine bits = s.lines[own];
  int e = 0;
#pragma unroll
  for (int u = 0; u < kScanWords; ++u) e += block_tiles(x[u], rate);
  e = wave_sum(e) + sub * rate * (me.n - me.n_causal) + me.n_causal * (rows ? sub * (sub + 1) / 2 : sub * rate - sub * (sub - 1) / 2);
  if (lane == 0) {
    s.ptr[id] = e;
    if (id == s.n_blocks * rate - 1) s.ptr[id + 1] = e + line_tiles(me, rows, sub, rate);
  }
#pragma unroll
  for (int u = 0; u < kScanWords; ++u) e = fill_blocks(rows, sub, rate, 64 * u, bits.full[u], bits.causal[u], e, s.idx, s.flag);
}

// Where two block lines part, read from the anchor (distance 0 = that end of the line, kNever = nowhere): the first block that
// only one of them holds, the first that is FULL in a and CAUSAL in b, the other way round, and CAUSAL in both.
constexpr int kNever = 512;
struct Parting {
  int one, full_causal, causal_full, both_causal;
  bool one_is_a;
};
__device__ __forceinline__ Parting part_lines(const BlockLine& a, const BlockLine& b, bool from_end) {
  int d[4] = {kNever, kNever, kNever, kNever};
  uint32_t one_is_a = 0;
  auto words = [](const uint64_t (&x)[kScanWords], int w) { return (uint32_t)(x[w >> 1] >> (32 * (w & 1))); };
  auto part = [&](auto towards_end) {
    constexpr bool kEnd = decltype(towards_end)::value;
#pragma unroll
    for (int v = 0; v < 2 * kScanWords; ++v) {             // from the far end: the last one found is the first one met
      const int w = kEnd ? v : 2 * kScanWords - 1 - v, base = 32 * (2 * kScanWords - 1 - v);
      const uint32_t fa = words(a.full, w), ca = words(a.causal, w), fb = words(b.full, w), cb = words(b.causal, w);
      const uint32_t m[4] = {(fa | ca) ^ (fb | cb), fa & cb, ca & fb, ca & cb};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int at = kEnd ? __builtin_clz(m[i] | 1) : __builtin_ctz(m[i] | 1u << 31);
        d[i] = m[i] ? base + at : d[i];
        if (i == 0) one_is_a = m[0] ? (fa | ca) >> (kEnd ? 31 - at : at) & 1 : one_is_a;
      }
    }
  };
  if (from_end) part(std::true_type{}); else part(std::false_type{});
  return {d[0], d[1], d[2], d[3], one_is_a != 0};
}

// Rank of kRankLines lines among all of their side, in the order of row_precedes.  Thread t has block line t: what decides first about
// each of its lines (very long, anchor, block-line length) is packed into one key and compared with those of the workgroup's
// lines, and where keys are equal the block lines' bits tell which list goes on how.
// (Keys of 32 bits, counts added up per thread, no branch in part_lines: with 64-bit keys, a ballot per comparison and a branch around every
// word that has nothing to tell, comparing took 6 of 11 us.)
constexpr int kRankLines = 4;          // lines of a workgroup
constexpr int kSubs = 4;               // lines of its block that a thread compares at a time
constexpr int kScanRate = 64;          // an index and a block line's length have 15 bits each in a key
__device__ __forceinline__ void rank_lines(const ListSide& s, bool rows, int rate, int line0) {
  __shared__ BlockLine own_bits[kRankLines];
  __shared__ BlockStat own_stat[kRankLines];
  __shared__ int32_t rank[kRankLines], sums[3][kListThreads / 64];
  __shared__ uint32_t seen_first[kScanBlocks * kScanRate / 4], seen_last[kScanBlocks * kScanRate / 4];             // a byte per tile
  static_assert(kListThreads == kScanBlocks, "a thread has one block line");
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, n = s.n_blocks * rate, n_own = min(kRankLines, n - line0), n_words = (s.n_other * rate + 3) / 4;
  const int own0 = line0 / rate;                             // block line of the first of the workgroup's lines
  const bool held = tid < s.n_blocks;
  BlockStat st = {};
  BlockLine bits = {};
  if (held) { st = s.stats[tid]; bits = s.lines[tid]; }
  if (tid < kRankLines) rank[tid] = 0;
  for (int i = tid; i < n_words; i += kListThreads) seen_first[i] = seen_last[i] = 0;
  if (tid >= own0 && tid < own0 + kRankLines) { own_bits[tid - own0] = bits; own_stat[tid - own0] = st; }
  const int tiles = wave_sum(block_tiles(st, rate));
  if (lane == 0) sums[0][wave] = tiles;
  __syncthreads();
  auto total = [&](int which) {
    int x = 0;
#pragma unroll
    for (int w = 0; w < kListThreads / 64; ++w) x += sums[which][w];
    return x;
  };
  const int64_t twice_all = 2 * (int64_t)total(0);
  auto very_long = [&](int len) { return (int64_t)len * n > twice_all; };
  auto first_tile = [&](const BlockStat& x, int sub) { return x.first * rate + (!rows && (x.ends & 1) ? sub : 0); };
  auto last_tile = [&](const BlockStat& x, int sub) { return x.last * rate + (rows && (x.ends & 2) ? sub : rate - 1); };
  // Which end anchors the lists: the one with fewer distinct values over the lines that are neither empty nor very long.
  if (st.n > 0)
    for (int sub = 0; sub < rate; ++sub)
      if (!very_long(line_tiles(st, rows, sub, rate))) {
        reinterpret_cast<uint8_t*>(seen_first)[first_tile(st, sub)] = 1;
        reinterpret_cast<uint8_t*>(seen_last)[last_tile(st, sub)] = 1;
      }
  __syncthreads();
  int n_first = 0, n_last = 0;
  for (int i = tid; i < n_words; i += kListThreads) { n_first += __popc(seen_first[i]); n_last += __popc(seen_last[i]); }
  n_first = wave_sum(n_first); n_last = wave_sum(n_last);
  if (lane == 0) { sums[1][wave] = n_first; sums[2][wave] = n_last; }
  __syncthreads();
  const bool from_end = total(2) < total(1);
  // very long lines first, among them by block-line length before the anchor; empty ones last, by number
  auto key_of = [&](const BlockStat& x, int sub, int line) {
    const int len = line_tiles(x, rows, sub, rate);
    const uint32_t anchor = from_end ? last_tile(x, sub) : first_tile(x, sub), shorter = (1 << 15) - 1 - rate * x.n;
    if (len == 0) return 1u << 31 | (uint32_t)line;
    return very_long(len) ? shorter << 15 | anchor : 1u << 30 | anchor << 15 | shorter;
  };
  // lane t: line t of the workgroup
  const int own_line = line0 + min(lane, n_own - 1), own_block = own_line / rate, own_sub = own_line - own_block * rate;
  const uint32_t own_key = key_of(own_stat[own_block - own0], own_sub, own_line);
  int before = 0;                      // lane t: how many of this wavefront's lines come before line t
  if (wave == 0 && lane < n_own) {
    // Lines of one block: their lists differ only where the block's line of the mask is CAUSAL, and by the number of such blocks in
    // length (the same lists if there is none).  The smaller sub's comes first, or else the larger's: rows hold keys 0..sub of a CAUSAL
    // block, so read forwards the longer list goes on in it, and read backwards the smaller sub's index there is smaller; columns hold
    // queries sub.., so read forwards the smaller sub's index is smaller, and read backwards the larger sub leaves the last such block
    // first, unless the list's first block is the only one, where it ends.
    const BlockStat x = own_stat[own_block - own0];
    const bool larger_first = x.n_causal > 0 && (rows ? !from_end : from_end && !((x.ends & 1) && x.n_causal == 1));
    for (int sub = 0; sub < rate; ++sub) {
      const uint32_t key = key_of(x, sub, own_block * rate + sub);
      before += key < own_key || (key == own_key && (larger_first ? sub > own_sub : sub < own_sub));
    }
  }
  for (int sub0 = 0; sub0 < rate; sub0 += kSubs) {
    uint32_t key[kSubs];
#pragma unroll
    for (int u = 0; u < kSubs; ++u) key[u] = held && sub0 + u < rate ? key_of(st, sub0 + u, tid * rate + sub0 + u) : ~0u;
    int count[kRankLines];             // of this thread's lines, how many come before line t by their keys
    uint32_t ask = 0;                  // lines whose key a line of another block has
#pragma unroll
    for (int t = 0; t < kRankLines; ++t) {
      const uint32_t key_b = __builtin_amdgcn_readlane(own_key, t);
      const bool other = tid != __builtin_amdgcn_readlane(own_block, t);
      uint32_t apart = ~0u;
      count[t] = 0;
#pragma unroll
      for (int u = 0; u < kSubs; ++u) {
        count[t] += key[u] < key_b;
        apart = min(apart, key[u] ^ key_b);
      }
      count[t] = other ? count[t] : 0;
      ask |= __any(apart == 0 && other) ? 1u << t : 0;
    }
    for (ask &= (1u << n_own) - 1; ask;) {
      // all lines of one block: how this thread's block line and that one part
      const int t0 = __builtin_ctz(ask), block_b = __builtin_amdgcn_readlane(own_block, t0), first_b = own_stat[block_b - own0].first;
      const Parting p = part_lines(bits, own_bits[block_b - own0], from_end);
      // Does line a come first, that holds more (`a_more`) tiles of the block `at` where they part?  Read forwards, the tile that only one of
      // them holds comes next in its list.  Read backwards, the one with more tiles there holds the larger index, and comes first only
      // if the other's list has ended.  Equal lists: by number.
      auto comes_first = [&](int at, bool a_more) {
        const bool ended = (a_more ? first_b : (int)st.first) >= kScanBlocks - 1 - at && (at == p.one || !rows);
        return at == kNever ? tid < block_b : (!from_end || ended ? a_more : !a_more);
      };
      const bool plain = comes_first(p.one, p.one_is_a);
#pragma unroll
      for (int t = 0; t < kRankLines; ++t) {
        if (!(ask >> t & 1) || __builtin_amdgcn_readlane(own_block, t) != block_b) continue;
        ask &= ~(1u << t);
        const uint32_t key_b = __builtin_amdgcn_readlane(own_key, t);
        const int sub_b = __builtin_amdgcn_readlane(own_sub, t), causal_b = rows ? sub_b + 1 : rate - sub_b;
        const int fc = causal_b < rate ? p.full_causal : kNever;
#pragma unroll
        for (int u = 0; u < kSubs; ++u) {
          const int causal_a = rows ? sub0 + u + 1 : rate - sub0 - u;
          const int cf = causal_a < rate ? p.causal_full : kNever, cc = causal_a != causal_b ? p.both_causal : kNever, at = min(fc, min(cf, cc));
          const bool comes = at < p.one ? comes_first(at, at == fc || (at == cc && causal_a > causal_b)) : plain;
          count[t] += key[u] == key_b && tid != block_b && comes;
        }
      }
    }
    static_assert(kRankLines == 4 && kSubs * 64 < 65536, "two lines' counts in one sum");
    const int sum01 = wave_sum(count[0] | count[1] << 16), sum23 = wave_sum(count[2] | count[3] << 16);
    const int sum = lane & 2 ? sum23 : sum01;
    before += lane < kRankLines ? (lane & 1 ? sum >> 16 : sum & 0xffff) : 0;
  }
  if (lane < n_own && before) atomicAdd(&rank[lane], before);
  __syncthreads();
  if (tid < n_own) s.order[rank[tid]] = line0 + tid;
}

// Workgroups: ranks of the rows and of the columns, lines of both, and one that counts the invalid entries of the rows that hold some.
__global__ __launch_bounds__(kListThreads) void tl_lists_kernel(const uint8_t* mask, int rate, ListSide q, ListSide k, int32_t* n_invalid) {
  constexpr int kWaves = kListThreads / 64;
  const int nq = q.n_blocks * rate, nk = k.n_blocks * rate, rank_q = (nq + kRankLines - 1) / kRankLines, rank_k = (nk + kRankLines - 1) / kRankLines;
  const int fill_q = (nq + kWaves - 1) / kWaves, fill_k = (nk + kWaves - 1) / kWaves;
  int g = blockIdx.x;
  if (g < rank_q + rank_k) {
    const bool rows = g < rank_q;
    rank_lines(rows ? q : k, rows, rate, (rows ? g : g - rank_q) * kRankLines);
    return;
  }
  g -= rank_q + rank_k;
  if (g < fill_q + fill_k) {
    const bool rows = g < fill_q;
    const int id = __builtin_amdgcn_readfirstlane((rows ? g : g - fill_q) * kWaves + (threadIdx.x >> 6));
    if (id < (rows ? nq : nk)) fill_line(rows ? q : k, rows, rate, id);
    return;
  }
  __shared__ int32_t bad;
  if (threadIdx.x == 0) bad = 0;
  __syncthreads();
  int here = 0;
  if ((int)threadIdx.x < q.n_blocks && (q.stats[threadIdx.x].ends & 4))
    for (int i = 0; i < q.n_other; ++i) here += mask[(int64_t)threadIdx.x * q.n_other + i] > 2;
  if (here) atomicAdd(&bad, here);
  __syncthreads();
  if (threadIdx.x == 0) *n_invalid = bad;
}

}  // namespace ua

extern "C" int ua_tilelist_size(const uint8_t* block_mask, int n_qblocks, int n_kblocks, int rate,
                                int64_t* n_qtiles, int64_t* n_ktiles, int64_t* nnz) {
  using namespace ua;
  if (!n_qtiles || !n_ktiles || !nnz) return UA_ERR_NULL;
  if (int rc = check_mask(block_mask, n_qblocks, n_kblocks, rate)) return rc;
  int64_t n = 0;
  for (int64_t i = 0; i < (int64_t)n_qblocks * n_kblocks; ++i) {
    const int t = block_mask[i];
    n += t == 1 ? (int64_t)rate * rate : (t == 2 ? (int64_t)rate * (rate + 1) / 2 : 0);
  }
  if (n > INT32_MAX) return UA_ERR_SHAPE;
  *n_qtiles = (int64_t)n_qblocks * rate;
  *n_ktiles = (int64_t)n_kblocks * rate;
  *nnz = n;
  return UA_OK;
}

extern "C" int ua_tilelist_build(const uint8_t* block_mask, int n_qblocks, int n_kblocks, int rate,
                                 int32_t* row_ptr, int32_t* col_idx, uint8_t* flag,
                                 int32_t* col_ptr, int32_t* row_idx, uint8_t* cflag,
                                 int32_t* q_order, int32_t* k_order) {
  using namespace ua;
  if (int rc = check_mask(block_mask, n_qblocks, n_kblocks, rate)) return rc;
  if (!row_ptr || !col_ptr || !q_order || !k_order) return UA_ERR_NULL;
  const int nqt = n_qblocks * rate, nkt = n_kblocks * rate;
  std::vector<int32_t> kcnt(nkt, 0);
  int64_t e = 0;
  for (int qt = 0; qt < nqt; ++qt) {
    row_ptr[qt] = (int32_t)e;
    for (int kb = 0; kb < n_kblocks; ++kb) {
      if (!block_mask[(int64_t)(qt / rate) * n_kblocks + kb]) continue;
      for (int kt = kb * rate; kt < (kb + 1) * rate; ++kt) {
        const int ty = tile_type(block_mask, n_kblocks, rate, qt, kt);
        if (!ty) continue;
        if (!col_idx || !flag) return UA_ERR_NULL;
        col_idx[e] = kt; flag[e] = ty == 2; ++e; ++kcnt[kt];
      }
    }
  }
  row_ptr[nqt] = (int32_t)e;
  col_ptr[0] = 0;
  for (int kt = 0; kt < nkt; ++kt) col_ptr[kt + 1] = col_ptr[kt] + kcnt[kt];
  if (e > 0 && (!row_idx || !cflag)) return UA_ERR_NULL;
  std::vector<int32_t> cur(col_ptr, col_ptr + nkt);
  for (int qt = 0; qt < nqt; ++qt)
    for (int32_t i = row_ptr[qt]; i < row_ptr[qt + 1]; ++i) {
      const int32_t pos = cur[col_idx[i]]++;
      row_idx[pos] = qt; cflag[pos] = flag[i];
    }
  std::iota(q_order, q_order + nqt, 0);
  const bool q_end = anchor_from_end(row_ptr, col_idx, nqt), k_end = anchor_from_end(col_ptr, row_idx, nkt);
  std::sort(q_order, q_order + nqt, [&](int32_t a, int32_t b) { return row_precedes(row_ptr, col_idx, nqt, rate, rate - 1, q_end, a, b); });
  std::iota(k_order, k_order + nkt, 0);
  std::sort(k_order, k_order + nkt, [&](int32_t a, int32_t b) { return row_precedes(col_ptr, row_idx, nkt, rate, 0, k_end, a, b); });
  return UA_OK;
}

namespace ua {

// Bytes of scratch that the two-launch build works in; 0: larger masks go through the lists.
static int64_t scan_bytes(int n_qblocks, int n_kblocks, int rate) {
  if (n_qblocks > kScanBlocks || n_kblocks > kScanBlocks || rate > kScanRate) return 0;
  return (int64_t)(n_qblocks + n_kblocks) * (sizeof(BlockLine) + sizeof(BlockStat));
}
static int build_device_impl(const uint8_t* block_mask, int n_qblocks, int n_kblocks, int rate,
                             int32_t* row_ptr, int32_t* col_idx, uint8_t* flag,
                             int32_t* col_ptr, int32_t* row_idx, uint8_t* cflag,
                             int32_t* q_order, int32_t* k_order, int32_t* work, int32_t* n_invalid, void* scratch, int64_t scratch_bytes, hipStream_t st) {
  const int nqt = n_qblocks * rate, nkt = n_kblocks * rate;
  const int64_t wanted = scan_bytes(n_qblocks, n_kblocks, rate);
  if (scratch && wanted > 0 && scratch_bytes >= wanted && aligned16(scratch)) {
    BlockLine* lines = static_cast<BlockLine*>(scratch);
    BlockStat* stats = reinterpret_cast<BlockStat*>(lines + n_qblocks + n_kblocks);
    const ListSide q = {lines, stats, row_ptr, col_idx, q_order, flag, n_qblocks, n_kblocks};
    const ListSide k = {lines + n_qblocks, stats + n_qblocks, col_ptr, row_idx, k_order, cflag, n_kblocks, n_qblocks};
    auto groups = [](int n, int per) { return (unsigned)((n + per - 1) / per); };
    hipLaunchKernelGGL(tl_scan_kernel, dim3(line_groups(n_qblocks) + line_groups(n_kblocks)), dim3(64 * kWavesPerGroup), 0, st, block_mask, n_qblocks, n_kblocks, q, k);
    hipLaunchKernelGGL(tl_lists_kernel, dim3(groups(nqt, kRankLines) + groups(nkt, kRankLines) + groups(nqt, kListThreads / 64) + groups(nkt, kListThreads / 64) + 1),
                       dim3(kListThreads), 0, st, block_mask, rate, q, k, n_invalid);
    return hipGetLastError() == hipSuccess ? UA_OK : UA_ERR_LAUNCH;
  }
  int32_t* qcnt = work;
  int32_t* kcnt = work + nqt + 1;
  const dim3 lines((unsigned)(line_groups(nqt) + line_groups(nkt))), group(64 * kWavesPerGroup);
  hipLaunchKernelGGL(tl_count_kernel, lines, group, 0, st, block_mask, n_qblocks, n_kblocks, rate, qcnt, kcnt, q_order);
  hipLaunchKernelGGL(tl_fill_kernel, lines, group, 0, st, block_mask, n_qblocks, n_kblocks, rate, (const int32_t*)qcnt, (const int32_t*)kcnt, row_ptr, col_idx, flag,
                     col_ptr, row_idx, cflag, (const int32_t*)q_order, n_invalid);
  hipLaunchKernelGGL(tl_order_kernel, dim3((unsigned)((nqt + kOrderLines - 1) / kOrderLines + (nkt + kOrderLines - 1) / kOrderLines)),
                     dim3(kOrderThreads), 0, st, (const int32_t*)row_ptr, (const int32_t*)col_idx, nqt, q_order,
                     (const int32_t*)col_ptr, (const int32_t*)row_idx, nkt, k_order, rate);
  return hipGetLastError() == hipSuccess ? UA_OK : UA_ERR_LAUNCH;
}

static int check_device_builder_args(const uint8_t* block_mask, int n_qblocks, int n_kblocks, int rate,
                                     const void* row_ptr, const void* col_idx, const void* flag, const void* col_ptr,
                                     const void* row_idx, const void* cflag, const void* q_order, const void* k_order) {
  if (!block_mask || !row_ptr || !col_idx || !flag || !col_ptr || !row_idx || !cflag || !q_order || !k_order)
    return UA_ERR_NULL;
  if (n_qblocks <= 0 || n_kblocks <= 0 || rate <= 0) return UA_ERR_SHAPE;
  if ((int64_t)n_qblocks * rate > (1 << 24) || (int64_t)n_kblocks * rate > (1 << 24)) return UA_ERR_SHAPE;
  return UA_OK;
}

}  // namespace ua

extern "C" int64_t ua_tilelist_scratch_bytes(int n_qblocks, int n_kblocks, int rate) {
  return n_qblocks > 0 && n_kblocks > 0 && rate > 0 ? ua::scan_bytes(n_qblocks, n_kblocks, rate) : 0;
}

extern "C" int ua_tilelist_build_device_scratch(const uint8_t* block_mask, int n_qblocks, int n_kblocks, int rate,
                                                int32_t* row_ptr, int32_t* col_idx, uint8_t* flag,
                                                int32_t* col_ptr, int32_t* row_idx, uint8_t* cflag,
                                                int32_t* q_order, int32_t* k_order, int32_t* work,
                                                void* scratch, int64_t scratch_bytes, void* stream) {
  using namespace ua;
  if (!work) return UA_ERR_NULL;
  if (int rc = check_device_builder_args(block_mask, n_qblocks, n_kblocks, rate, row_ptr, col_idx, flag, col_ptr,
                                         row_idx, cflag, q_order, k_order)) return rc;
  if (int rc = check_device()) return rc;
  const int nqt = n_qblocks * rate, nkt = n_kblocks * rate;
  return build_device_impl(block_mask, n_qblocks, n_kblocks, rate, row_ptr, col_idx, flag, col_ptr, row_idx, cflag,
                           q_order, k_order, work, work + nqt + nkt + 2, scratch, scratch_bytes, (hipStream_t)stream);
}

extern "C" int ua_tilelist_build_device(const uint8_t* block_mask, int n_qblocks, int n_kblocks, int rate,
                                        int32_t* row_ptr, int32_t* col_idx, uint8_t* flag,
                                        int32_t* col_ptr, int32_t* row_idx, uint8_t* cflag,
                                        int32_t* q_order, int32_t* k_order, int32_t* work, void* stream) {
  return ua_tilelist_build_device_scratch(block_mask, n_qblocks, n_kblocks, rate, row_ptr, col_idx, flag, col_ptr, row_idx, cflag, q_order, k_order, work,
                                          nullptr, 0, stream);
}

// The device address of `scratch`, looked up once per device with that device current.  In host
// code the array's name is only a handle for this lookup, never an address to pass on.
static int scratch_of_current_device(int32_t** out) {
  static std::atomic<int32_t*> ptrs[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return UA_ERR_DEVICE;
  int32_t* p = ptrs[dev].load(std::memory_order_acquire);
  if (!p) {
    void* sym = nullptr;
    if (hipGetSymbolAddress(&sym, HIP_SYMBOL(scratch)) != hipSuccess || !sym) return UA_ERR_DEVICE;
    p = static_cast<int32_t*>(sym);
    ptrs[dev].store(p, std::memory_order_release);
  }
  *out = p;
  return UA_OK;
}

// Everything the entry points resolve lazily per device, resolved now (outside any graph capture).
extern "C" int ua_init(void) {
  if (int rc = ua::check_device()) return rc;
  int32_t* p = nullptr;
  return scratch_of_current_device(&p);
}

extern "C" int ua_tilelist_build_device_noalloc(const uint8_t* block_mask, int n_qblocks, int n_kblocks, int rate,
                                                int32_t* row_ptr, int32_t* col_idx, uint8_t* flag,
                                                int32_t* col_ptr, int32_t* row_idx, uint8_t* cflag,
                                                int32_t* q_order, int32_t* k_order, int32_t* n_invalid, void* stream) {
  using namespace ua;
  if (int rc = check_device_builder_args(block_mask, n_qblocks, n_kblocks, rate, row_ptr, col_idx, flag, col_ptr,
                                         row_idx, cflag, q_order, k_order)) return rc;
  const int64_t lines = (int64_t)n_qblocks * rate + (int64_t)n_kblocks * rate;
  if (lines > UA_NOALLOC_MAX_LINES) return UA_ERR_TOO_LARGE;
  if (int rc = check_device()) return rc;
  int32_t* work = nullptr;
  if (int rc = scratch_of_current_device(&work)) return rc;
  // What is read is written before, and the invalid-entry count is stored, not accumulated: nothing in the scratch has to start at zero.
  // Masks that the two-launch build takes have at most 32768 lines, which leaves it its room behind them.
  static_assert(2 * kScanBlocks * kScanRate + 12 + 2 * kScanBlocks * (int)(sizeof(BlockLine) + sizeof(BlockStat)) / 4 <= UA_NOALLOC_MAX_LINES + 8, "fits the scratch");
  const int64_t room = (lines + 8 + 3) / 4 * 4;
  return build_device_impl(block_mask, n_qblocks, n_kblocks, rate, row_ptr, col_idx, flag, col_ptr, row_idx, cflag,
                           q_order, k_order, work, n_invalid ? n_invalid : work + lines + 2, work + room, (UA_NOALLOC_MAX_LINES + 8 - room) * 4, (hipStream_t)stream);
}
