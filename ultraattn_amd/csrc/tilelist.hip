// Block mask -> compacted active-tile list (CSR over query tiles, CSC over key tiles).
//
// Refinement rule (one block -> rate x rate tiles): EMPTY stays empty, FULL becomes all full,
// CAUSAL becomes causal on the sub-diagonal, full below it and empty above it.  Tiles are
// emitted row-major (query tile outer, key tile inner).
#include <algorithm>
#include <atomic>
#include <numeric>
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
// fill: a workgroup first adds up the counts of its side (those before its lines give its place in the list,
// all of them the list's length), then each wavefront walks its line 64 blocks at a time; an exclusive
// scan of the per-block tile counts gives every lane the slot where its block's tiles go, in ascending order.
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
  const int n_causal = causal_tiles(ln, rate);
  const uint64_t below = (1ull << lane) - 1;
  int32_t* idx = ln.is_row ? col_idx : row_idx;
  uint8_t* flg = ln.is_row ? flag : cflag;
  for (int i0 = 0; i0 < ln.n_blocks; i0 += 64 * kAhead) {
    if (i0 > 0) load_types(mask, ln, i0, type);
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      const int i = i0 + 64 * u + lane, ty = type[u];
      const uint64_t full = __ballot(ty == 1), causal = __ballot(ty == 2);
      if (!(full | causal)) continue;
      const int c = ty == 1 ? rate : (ty == 2 ? n_causal : 0);
      int at = e + rate * __popcll(full & below) + n_causal * __popcll(causal & below);
      // sub-tiles along the line: a row takes key sub-tiles 0..sub of a causal block (the last one
      // causal), a column takes query sub-tiles sub..rate-1 (the first one causal)
      const int first = (ty == 2 && !ln.is_row) ? ln.sub : 0;
      // four tiles and their flags per store
      int t = 0;
      for (; t + 4 <= c; t += 4, at += 4) {
        const int s = i * rate + first + t, mark = ln.sub - first - t;           // the causal one among them, if 0..3
        *reinterpret_cast<i32x4_any*>(idx + at) = i32x4_any{s, s + 1, s + 2, s + 3};
        *reinterpret_cast<u32_any*>(flg + at) = ty == 2 && (unsigned)mark < 4 ? 1u << (8 * mark) : 0;
      }
      for (; t < c; ++t, ++at) {
        idx[at] = i * rate + first + t;
        flg[at] = ty == 2 && first + t == ln.sub;
      }
      e += rate * __popcll(full) + n_causal * __popcll(causal);
    }
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

static int build_device_impl(const uint8_t* block_mask, int n_qblocks, int n_kblocks, int rate,
                             int32_t* row_ptr, int32_t* col_idx, uint8_t* flag,
                             int32_t* col_ptr, int32_t* row_idx, uint8_t* cflag,
                             int32_t* q_order, int32_t* k_order, int32_t* work, int32_t* n_invalid, hipStream_t st) {
  const int nqt = n_qblocks * rate, nkt = n_kblocks * rate;
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

extern "C" int ua_tilelist_build_device(const uint8_t* block_mask, int n_qblocks, int n_kblocks, int rate,
                                        int32_t* row_ptr, int32_t* col_idx, uint8_t* flag,
                                        int32_t* col_ptr, int32_t* row_idx, uint8_t* cflag,
                                        int32_t* q_order, int32_t* k_order, int32_t* work, void* stream) {
  using namespace ua;
  if (!work) return UA_ERR_NULL;
  if (int rc = check_device_builder_args(block_mask, n_qblocks, n_kblocks, rate, row_ptr, col_idx, flag, col_ptr,
                                         row_idx, cflag, q_order, k_order)) return rc;
  if (int rc = check_device()) return rc;
  const int nqt = n_qblocks * rate, nkt = n_kblocks * rate;
  return build_device_impl(block_mask, n_qblocks, n_kblocks, rate, row_ptr, col_idx, flag, col_ptr, row_idx, cflag,
                           q_order, k_order, work, work + nqt + nkt + 2, (hipStream_t)stream);
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
  // the counts are written before they are read and the invalid-entry count is stored, not
  // accumulated: nothing in the scratch has to start at zero
  return build_device_impl(block_mask, n_qblocks, n_kblocks, rate, row_ptr, col_idx, flag, col_ptr, row_idx, cflag,
                           q_order, k_order, work, n_invalid ? n_invalid : work + lines + 2, (hipStream_t)stream);
}
