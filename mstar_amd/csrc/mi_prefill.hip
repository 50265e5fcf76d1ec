// Ragged paged prefill (P3 + P7) for MI355X (gfx950).
//
// Replaces FlashInferPrefillWrapper.plan/run (mstar/utils/flashinfer_utils.py:162-269).
//
// plan:  one launch (prefill_plan_kernel): the token map (the per-new-token
//        (page, slot) of flashinfer_utils.py:211-256), the tiles of every
//        long-query request, costed and put as (kv-head, tile) units, or
//        pieces of them, into 8 per-XCD queues (pf_choose), and, for the
//        short-query requests (qo_len * group <= 16, e.g. the decode rows of
//        a mixed batch), a split-KV plan for the decode kernel in the same
//        workspace.
// run:   mi_prefill_short (decode kernel + merge for the short-query
//        requests) and mi_prefill_tiles (prefill_kernel, and the merge of
//        tiles that the plan has cut into key pieces); mi_prefill_run does
//        both in turn, with one launch for the two merges.
//
// prefill_kernel (persistent, one workgroup per CU): a unit is a tile of
// 256 (query token, q-head) rows of one request and kv-head -- GQA rows
// packed token-major, so K/V are read once per group of q-heads -- and each
// of the 8 wavefronts owns 2 groups of 16 rows.  Keys go in 32-key steps
// through a three-stage LDS ring filled from registers loaded two steps
// ahead (page ids staged in LDS, so no load waits on an index load); a
// tile's V^T fragments are read in the step that computes its scores and
// consumed by the next step's P.V MFMAs:
//   S^T[16 keys x 16 rows] = K . Q^T    (v_mfma_f32_16x16x32, K from LDS)
//   online softmax in fp32 (exp2 domain), causal mask aligned to the end of the KV
//   O^T[16 dims x 16 rows] += V^T . P^T (v_mfma_f32_16x16x32, V^T from the
//                                        transposing LDS read ds_read_b64_tr_b16)
// The two wavefronts of each SIMD run their softmax on opposite sides of
// their MFMA work (ping-pong), so vector and matrix work overlap.
// At head_dim 256, prefill_rs_kernel (mi_prefill_rs.h) runs the same units
// (128-row tiles), plan, queues, loader and LDS ring with the work split by
// role inside each wavefront pair: one computes the scores and the softmax
// of 32 rows, the other accumulates their P.V over all 256 dims.
// fp8 K/V are converted to the MFMA type when a tile is stored to LDS; the
// per-head scales multiply the scores and the output.
#include "mi_prefill_kernel.h"
#include "mi_prefill_rs.h"
#include "mi_merge.h"

namespace mi {
constexpr int kShortRows = kShortRowsMax;  // qo_len * group <= 16 -> decode kernel (8 on a paired plan)

// Workspace: header | per-XCD queue counters + finished-workgroup counter |
// tile list | tile cost prefix | unit order | decode split plan | (where room
// is left) piece list | split tile list | piece partials (lse, o).
// Header words: [kPfTiles] tiles, [kPfUnits] units (tiles x kv-heads, or
// pieces x kv-heads when tiles are split), [kPfPieces] pieces per kv-head (0:
// no tile is split), [kPfSplitTiles] split tiles, [kPfSlots] partials,
// [kPfCuts + x] first unit of XCD x's queue (x = 0..8, [16] = units).
struct PrefillLayout {
  int64_t hdr, ctr, tiles, tcum, order, split;
  int32_t max_tiles;
};

// What a split of tiles into key pieces needs, behind the decode split plan:
// as many partials as fit the workspace, up to kPfMaxParts (three rounds of
// one piece per CU; a split of more pieces never paid).  parts == 0: no room.
// Every table has its place whatever the workspace's size, so a run finds them
// also where it is given another size than the plan was.
constexpr int32_t kPfMaxParts = 768;
struct PfSplitLayout {
  int64_t pieces, split_tiles, lse, o, total;
  int32_t max_pieces, parts;
};

static PfSplitLayout pf_split_layout(int64_t base, int32_t max_tiles, int32_t nkv, int32_t head_dim, int64_t ws_avail) {
  PfSplitLayout P;
  const int64_t rows = pf_rows(head_dim), per_part = 4 * rows * head_dim;
  P.max_pieces = max_tiles + kPfMaxParts;
  P.pieces = mi_align_up(base, 256);
  P.split_tiles = mi_align_up(P.pieces + 16LL * P.max_pieces, 256);
  P.lse = mi_align_up(P.split_tiles + 16LL * kPfMaxParts, 256);
  P.o = mi_align_up(P.lse + 4 * rows * kPfMaxParts, 256);
  int64_t parts = kPfMaxParts;
  if (ws_avail >= 0 && ws_avail < P.o + parts * per_part) parts = ws_avail > P.o ? (ws_avail - P.o) / per_part : 0;
  P.parts = parts < 2 * nkv ? 0 : (int32_t)parts;
  P.total = P.parts ? P.o + P.parts * per_part : base;
  return P;
}

static PrefillLayout prefill_layout(int32_t batch, int32_t max_qo_tokens, int32_t group, int32_t nkv,
                                    int32_t head_dim) {
  const int tile_rows = pf_rows(head_dim);
  PrefillLayout L;
  const int64_t rows = (int64_t)max_qo_tokens * group;
  int64_t mt = (rows + tile_rows - 1) / tile_rows + batch;
  if (mt > (1 << 21)) mt = 1 << 21;
  L.max_tiles = (int32_t)mt;
  L.hdr = 0;
  L.ctr = 256;
  L.tiles = L.ctr + 9 * kCtrStride * 4;
  L.tcum = mi_align_up(L.tiles + 8LL * L.max_tiles, 256);
  L.order = mi_align_up(L.tcum + 4LL * (L.max_tiles + 1), 256);
  L.split = mi_align_up(L.order + 4LL * L.max_tiles * nkv, 256);
  return L;
}

// The split layout of a plan or run call: from its shapes, and how much of it there is room for.
static PfSplitLayout pf_split_of(const PrefillLayout& L, int32_t batch, int32_t group, int32_t nkv, int32_t head_dim,
                                 int64_t ws_bytes) {
  const bool pair = pair_heads(nullptr, batch, nkv, group, head_dim, true);
  const int64_t split = split_layout(batch, nkv, head_dim, ws_bytes < 0 ? -1 : ws_bytes - L.split, pair).total;
  return pf_split_layout(L.split + split, L.max_tiles, nkv, head_dim, ws_bytes);
}

// ------------------------------------------------------------ token map
struct TokenMapArgs {
  const int32_t* qo_indptr;
  const int32_t* kv_indptr;
  const int32_t* kv_indices;
  const int32_t* last_page_len;
  int32_t batch, page_size;
  int64_t* t2p;
  int64_t* t2c;
  int32_t map_len;
};

__device__ inline void token_map_body(const TokenMapArgs& m, int t) {
  const int32_t* qo_indptr = m.qo_indptr;
  const int32_t* kv_indptr = m.kv_indptr;
  const int32_t* kv_indices = m.kv_indices;
  const int32_t* last_page_len = m.last_page_len;
  const int batch = m.batch, page_size = m.page_size;
  int64_t* t2p = m.t2p;
  int64_t* t2c = m.t2c;
  if (t >= m.map_len) return;
  const int total = qo_indptr[batch];
  if (t >= total) {  // graph-mode tail (flashinfer_utils.py:251-253)
    t2p[t] = 0;
    t2c[t] = 0;
    return;
  }
  int lo = 0, hi = batch - 1;  // last request r with qo_indptr[r] <= t
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (qo_indptr[mid] <= t) lo = mid; else hi = mid - 1;
  }
  const int r = lo;
  const int qo_len = qo_indptr[r + 1] - qo_indptr[r];
  const int np = kv_indptr[r + 1] - kv_indptr[r];
  const int kv_len = (np - 1) * page_size + last_page_len[r];
  const int g = kv_len - qo_len + (t - qo_indptr[r]);  // absolute position of the new token
  if (g < 0 || g / page_size >= np) {  // inconsistent metadata: nothing to write
    t2p[t] = -1;
    t2c[t] = -1;
    return;
  }
  t2p[t] = kv_indices[kv_indptr[r] + g / page_size];
  t2c[t] = g % page_size;
}

// ------------------------------------------------------------ tile plan
// Tiles of tile_rows (token, q-head) rows, request by request, heaviest
// (latest rows, most keys under the causal mask) first within a request.
// A tile's cost is its number of 32-key steps.  Units (kv-head, tile) in
// head-major order are cut into 8 contiguous runs of equal cost, one queue
// per XCD, so each XCD's L2 serves few (request, head) KV streams and the
// XCDs finish together; within a queue the units are taken heaviest first
// (longest-processing-time order), so the kernel's tail holds short units.
__device__ int pf_tile_cost(int kv_len, int qo_len, int rows_total, int row0, int tile_rows, int group,
                            int causal) {
  const int last_row = min(row0 + tile_rows, rows_total) - 1;
  const int kv_end = causal ? min(kv_len, kv_len - qo_len + last_row / group + 1) : kv_len;
  return kv_end > 0 ? (kv_end + kPfKeys - 1) / kPfKeys : 0;
}

struct PfPlanArgs {
  const int32_t* qo_indptr;
  const int32_t* kv_indptr;
  const int32_t* last_page_len;
  int32_t batch, page_size, group, nkv, tile_rows, max_tiles, causal;
  int32_t short_rows;  // requests with qo_len * group <= short_rows are the decode plan's, not tiles
  int32_t* hdr;
  int2* tiles;
  int32_t* tcum;
  int32_t* order;
  int32_t* ctr;
  // splitting tiles into key pieces (max_parts 0: never)
  int32_t max_parts, workgroups;
  float unit_steps, part_steps, merge_steps, merge_part_steps;  // costs in key steps (pf_split_costs)
  int4* pieces;
  int4* split_tiles;
};

// What a unit costs beyond its key steps, in key steps of the kernel.
struct PfSplitCosts {
  float unit, part, merge, merge_part;
};
static PfSplitCosts pf_split_costs(int head_dim) {
  if (head_dim > 128) return {6.f, 3.f, 5.f, 0.03f};
  return {7.f, 5.5f, 5.5f, 0.03f};
}

// How a plan's tiles go to the queues: as units in head-major order cut into
// 8 runs of equal cost (kPfLocal: each XCD's L2 serves few K/V streams), or
// dealt to the queues heaviest first (kPfWhole), or cut into key pieces of at
// most `cap` steps and those dealt.
//
// A call with few tiles leaves most CUs idle unless they are cut (one
// 512-token chunk at 32 q / 4 kv heads is 64 units for 256 CUs: 109 us of
// prefill kernel uncut, 44 + 8 us of merge cut in four), and with two or three
// units per CU a queue of one request's long units ends long after the others
// (4 chunks of 512-2048 tokens, 32 q / 4 kv heads, fp8 cache: 437 us from the
// local queues, 320 us dealt).  Where the local queues are as even as a deal
// they stay: 8 x 2048 tokens at head_dim 256 1262 us local, 1286 us dealt.
// Each candidate is priced, one wavefront each, by the bounds that any schedule
// of units u_1 >= u_2 >= ... on m workgroups obeys: their mean load, and
// (k + 1) u_{km + 1} for each k (of the km + 1 longest, k + 1 share a
// workgroup).  Heaviest-first queues come close to the larger of the two.
// The bounds are taken over all workgroups, and for kPfLocal also over each
// queue's units on the queue's eighth of them.
constexpr int kPfLocal = 0, kPfWhole = 0x7fffffff;
constexpr int kPfCandidates = 8;
__device__ inline int pf_candidate_cap(int i, float share) {
  // in mean loads of a workgroup, and at least so many steps
  constexpr float kShare[kPfCandidates] = {0.f, 2.4f, 1.7f, 1.35f, 1.15f, 1.f, .75f, .5f};
  constexpr int kMin[kPfCandidates] = {0, 16, 8, 6, 4, 4, 4, 4};
  return i == 0 ? kPfWhole : max(kMin[i], (int)ceilf(share * kShare[i]));
}
// prefix(t): cost of the tiles before tile t (one kv-head).  One histogram of
// the units' costs per queue of kPfLocal serves all candidates, so the price
// of a plan hardly grows with its tiles.
template <typename Prefix>
__device__ inline int pf_choose(const PfPlanArgs& a, int n_tiles, int64_t ct, int mc, Prefix prefix, int* s_bin) {
  __shared__ float s_est[16];
  constexpr int kBins = 128, kPer = kBins / 64;
  const int tid = (int)threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int64_t total = ct * a.nkv, units = (int64_t)n_tiles * a.nkv;
  const float share = (float)total / a.workgroups;
  if (total == 0 || (units > 16LL * a.workgroups && mc < 0.1f * share)) return kPfLocal;  // many short units balance by themselves
  // bin i: costs up to top(i), exact below 128 steps
  const float width = mc < kBins ? 1.f : (float)(mc + 1) / kBins, inv_width = 1.f / width;
  auto top = [&](int i) { return mc < kBins ? (float)i : (i + 1) * width; };
  auto bin_of = [&](float c) { return min(kBins - 1, (int)(c * inv_width)); };
  for (int i = tid; i < 16 * kBins; i += 1024) s_bin[i] = 0;
  __syncthreads();
  const float per_queue = 8.f / (float)total, ctf = (float)ct;
  for (int h = 0; h < a.nkv; ++h)
    for (int t = tid; t < n_tiles; t += 1024) {
      const int p = prefix(t);
      const int x = min(7, (int)((h * ctf + p) * per_queue));
      atomicAdd(&s_bin[x * kBins + bin_of((float)(prefix(t + 1) - p))], 1);
    }
  __syncthreads();
  // wavefronts 0..7: queue w of kPfLocal; 8..15: the dealt candidates
  const bool local = w < 8;
  const int cap = local ? kPfWhole : pf_candidate_cap(w - 8, share);
  const float m = local ? max(1, a.workgroups / 8) : a.workgroups, inv_m = 1.f / m;
  int* hist = s_bin + w * kBins;  // of the pieces
  // (a bin's top is at least its units' costs: the piece counts are upper bounds)
  const int biggest = cap == kPfWhole ? 1 : (mc + cap - 1) / cap;
  int parts = 0;
  if (!local) {
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      const int b = 64 * k + lane;
      int cnt = 0;
#pragma unroll
      for (int x = 0; x < 8; ++x) cnt += s_bin[x * kBins + b];
      if (cnt > 0) {
        const int c = (int)ceilf(top(b));
        const int n = cap == kPfWhole ? 1 : max(1, (c + cap - 1) / cap);
        parts += n > 1 ? n * cnt : 0;
        atomicAdd(&hist[bin_of((float)((c + n - 1) / n))], n * cnt);
      }
    }
    parts = wave_sum(parts);
  }
  // lane l owns kPer bins from the top: ranks of its pieces by an exclusive scan
  int cnt[kPer], mine = 0;
#pragma unroll
  for (int k = 0; k < kPer; ++k) mine += cnt[k] = hist[kBins - 1 - kPer * lane - k];
  const int upto = wave_inclusive_sum(mine), pieces = __builtin_amdgcn_readlane(upto, 63);
  const float extra = a.unit_steps + (parts > 0 ? a.part_steps : 0.f);
  float est = (share * m + pieces * a.unit_steps + parts * a.part_steps) * inv_m;
  int rank = upto - mine;
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const float q = floorf((rank + cnt[k] - 0.5f) * inv_m);  // the last k with a (km + 1)-th longest piece in this bin
    if (cnt[k] > 0 && q * m >= rank) est = fmaxf(est, (q + 1.f) * (top(kBins - 1 - kPer * lane - k) + extra));
    rank += cnt[k];
  }
  est = bitcast<float>((uint32_t)wave_max(bitcast<int>(est)));  // non-negative floats order as ints
  if (parts > 0) est += a.merge_steps + a.merge_part_steps * parts;
  if (parts > a.max_parts || biggest > kPfMaxPieces || (cap != kPfWhole && parts == 0)) est = __builtin_inff();
  if (lane == 0) s_est[w] = est;
  __syncthreads();
  float e_local = 0.f;
#pragma unroll
  for (int k = 0; k < 8; ++k) e_local = fmaxf(e_local, s_est[k]);
  // dealing gives up some L2 locality and a cut needs a merge: each has to win by a margin
  int best = -1;
  float e_best = 0.97f * e_local;
#pragma unroll
  for (int k = 0; k < kPfCandidates; ++k)
    if (s_est[8 + k] < (best == 0 ? 0.97f : 1.f) * e_best) {
      best = k;
      e_best = s_est[8 + k];
    }
  return best < 0 ? kPfLocal : pf_candidate_cap(best, share);
}

// Lists the pieces of a cut and deals them to the queues.  Tile t's
// n = ceil(cost / cap) pieces share its key steps evenly; split tiles get n
// slots per kv-head and a merge entry.  The pieces of one kv-head are listed
// heaviest first (a counting sort), and entry i of queue x is a closed form of
// (i, x) (pf_dealt), so the queues themselves need no list.
// mine: the thread's tile, where there is one tile per thread.
template <typename Prefix>
__device__ inline void pf_deal(const PfPlanArgs& a, int n_tiles, int cap, int mc, Prefix prefix, bool one, int2 mine,
                               int* s_bin, int* smem) {
  const int tid = (int)threadIdx.x;
  auto pieces_of = [&](int c) { return cap == kPfWhole ? 1 : max(1, (c + cap - 1) / cap); };
  const int most = min(cap, mc);
  const float scale = most < 1024 ? 1.f : 1024.f / (float)(most + 1);
  auto key_of = [&](int steps) { return 1023 - min(1023, (int)(steps * scale)); };
  s_bin[tid] = 0;
  __syncthreads();
  // piece k of n covers steps [k c / n, (k + 1) c / n): c % n of them are one
  // step longer than c / n
  for (int t = tid; t < n_tiles; t += 1024) {
    const int c = prefix(t + 1) - prefix(t), n = pieces_of(c), q = n == 1 ? c : c / n, r = c - q * n;
    atomicAdd(&s_bin[key_of(q)], n - r);
    if (r > 0) atomicAdd(&s_bin[key_of(q + 1)], r);
  }
  __syncthreads();
  int np;
  const int first = block_exclusive_scan_1024(s_bin[tid], np, smem);
  s_bin[tid] = first;
  int carry_slots = 0, carry_split = 0;
  for (int t0 = 0; t0 < n_tiles; t0 += 1024) {
    const int t = t0 + tid;
    int n = 0, c = 0;
    if (t < n_tiles) {
      c = prefix(t + 1) - prefix(t);
      n = pieces_of(c);
    }
    // slots (at most kPfMaxParts) and split tiles in one scan
    int tot = 0;
    const int at = cap == kPfWhole ? 0 : block_exclusive_scan_1024(n > 1 ? n << 16 | 1 : 0, tot, smem);
    const int slot = a.nkv * (carry_slots + (at >> 16));
    if (cap == kPfWhole) __syncthreads();  // s_bin is complete
    if (t < n_tiles) {
      const int2 te = one ? mine : a.tiles[t];
      const int q = n == 1 ? c : c / n, r = c - q * n;
      int at_short = atomicAdd(&s_bin[key_of(q)], n - r), at_long = r > 0 ? atomicAdd(&s_bin[key_of(q + 1)], r) : 0;
      for (int k = 0, part = 0; k < n; ++k) {
        part += r;
        const bool longer = part >= n;
        if (longer) part -= n;
        a.pieces[longer ? at_long++ : at_short++] = make_int4(te.x, te.y, k | n << 16, slot);
      }
      if (n > 1) a.split_tiles[carry_split + (at & 0xffff)] = make_int4(te.x, te.y, n, slot);
    }
    carry_slots += tot >> 16;
    carry_split += tot & 0xffff;
  }
  if (tid < 64) {
    const int len = tid < 8 ? pf_dealt_len(np, a.nkv, tid) : 0;
    const int at = wave_inclusive_sum(len) - len;
    if (tid < 9) a.hdr[kPfCuts + tid] = at;
  }
  if (tid == 0) {
    a.hdr[kPfUnits] = np * a.nkv;
    a.hdr[kPfPieces] = np;
    a.hdr[kPfSplitTiles] = carry_split;
    a.hdr[kPfSlots] = a.nkv * carry_slots;
  }
}

// One 1024-thread workgroup.  Requests go in windows of 1024 (one per
// thread: tile count, exclusive scan); the window's tiles are then listed
// 1024 at a time, one per thread, each finding its request by a binary
// search over the window's scan in LDS, so no thread loops over a long
// request's tiles.
__device__ inline void prefill_plan_body(const PfPlanArgs& a) {
  __shared__ int smem[16];
  __shared__ int s_cut[9];
  __shared__ int s_first[1025];  // window-relative first tile of each request, [1024] = window total
  __shared__ int s_kvl[1024], s_qol[1024];
  __shared__ int s_bin[8 * 1024];
  __shared__ int s_cum[1025];  // cost prefix of the first 1024 tiles
  const int tid = (int)threadIdx.x;
  const int group = a.group, tile_rows = a.tile_rows, causal = a.causal, max_tiles = a.max_tiles;
  int carry = 0, carry_cost = 0, mc = 0;
  int2 mine = make_int2(0, 0);  // the thread's last tile
  for (int base = 0; base < a.batch; base += 1024) {
    const int b = base + tid;
    int n = 0;
    if (b < a.batch) {
      const int qo_len = a.qo_indptr[b + 1] - a.qo_indptr[b];
      const int rows = qo_len * group;
      n = rows > a.short_rows ? (rows + tile_rows - 1) / tile_rows : 0;
      s_qol[tid] = qo_len;
      s_kvl[tid] = (a.kv_indptr[b + 1] - a.kv_indptr[b] - 1) * a.page_size + a.last_page_len[b];
    }
    int total;
    s_first[tid] = block_exclusive_scan_1024(n, total, smem);
    if (tid == 0) s_first[1024] = total;
    __syncthreads();
    const int nreq = min(1024, a.batch - base);
    for (int j0 = 0; j0 < total; j0 += 1024) {
      const int j = j0 + tid;
      int cost = 0, r = 0, row0 = 0;
      // only listed tiles are priced: the prefix ends with the cost of the last of them
      const bool listed = j < total && carry + j < max_tiles;
      if (listed) {
        int lo = 0, hi = nreq - 1;  // last request whose first tile is <= j (it has tiles)
        while (lo < hi) {
          const int mid = (lo + hi + 1) >> 1;
          if (s_first[mid] <= j) lo = mid; else hi = mid - 1;
        }
        r = lo;
        const int nr = s_first[r + 1] - s_first[r];
        row0 = (nr - 1 - (j - s_first[r])) * tile_rows;
        cost = pf_tile_cost(s_kvl[r], s_qol[r], s_qol[r] * group, row0, tile_rows, group, causal);
      }
      int tot_cost;
      const int cum = block_exclusive_scan_1024(cost, tot_cost, smem);
      if (listed) {
        mine = make_int2(base + r, row0);
        a.tiles[carry + j] = mine;
        a.tcum[carry + j] = carry_cost + cum;
        if (carry + j < 1024) s_cum[carry + j] = carry_cost + cum;
        mc = max(mc, cost);
      }
      carry_cost += tot_cost;
    }
    carry += total;
    __syncthreads();  // s_first / s_kvl / s_qol are rewritten by the next window
  }
  const int listed = min(carry, max_tiles);
  if (tid == 0) {
    a.tcum[listed] = carry_cost;
    if (listed <= 1024) s_cum[listed] = carry_cost;
  }
  __threadfence_block();
  __syncthreads();
  const int64_t ct = carry_cost;
  const int64_t total = ct * a.nkv;
  const int n_tiles = listed;
  if (tid < 9) a.ctr[tid * kCtrStride] = 0;  // queues of the first run
  if (tid == 0) {
    a.hdr[kPfTiles] = n_tiles;
    a.hdr[kPfPieces] = 0;
    a.hdr[kPfSplitTiles] = 0;
    a.hdr[kPfSlots] = 0;
  }
  const int32_t* tcum = a.tcum;
  auto prefix = [&](int t) { return n_tiles <= 1024 ? s_cum[t] : tcum[t]; };
  if (a.max_parts > 0) {
    mc = block_max_1024(mc, smem);
    const int cap = pf_choose(a, n_tiles, ct, mc, prefix, s_bin);
    if (cap != kPfLocal) {
      pf_deal(a, n_tiles, cap, mc, prefix, a.batch <= 1024 && n_tiles <= 1024, mine, s_bin, smem);
      return;
    }
  }
  const int units = n_tiles * a.nkv;
  if (tid == 0) a.hdr[kPfUnits] = units;
  // Queue cuts: queue x starts at the first unit whose cost prefix
  // h*ct + prefix(t) (unit u = h*n_tiles + t) reaches ceil(x * total / 8).
  // The prefix never decreases, so that unit is the one u with
  // prefix(u-1) < target <= prefix(u); every thread tests its units.
  if (tid <= 8) s_cut[tid] = tid == 0 ? 0 : units;
  __syncthreads();
  if (total > 0) {
    for (int h = 0; h < a.nkv; ++h)
      for (int t = tid; t < n_tiles; t += 1024) {
        if (h + t == 0) continue;
        const int64_t pu = h * ct + prefix(t), pp = t > 0 ? h * ct + prefix(t - 1) : (h - 1) * ct + prefix(n_tiles - 1);
#pragma unroll
        for (int x = 1; x < 8; ++x) {
          const int64_t target = (x * total + 7) >> 3;
          if (pp < target && target <= pu) s_cut[x] = h * n_tiles + t;
        }
      }
  }
  __syncthreads();
  if (tid <= 8) a.hdr[kPfCuts + tid] = s_cut[tid];
  // Within each queue, units go heaviest first: one counting sort over
  // (queue, 1023 - min(cost, 1023)) keys in LDS.  Queues are contiguous unit
  // ranges, so the sorted positions of queue x start at its first unit.
  for (int i = tid; i < 8 * 1024; i += 1024) s_bin[i] = 0;
  int cut[8];
#pragma unroll
  for (int k = 1; k < 8; ++k) cut[k] = uniform(s_cut[k]);
  __syncthreads();
  auto key_of = [&](int h, int t) {
    const int u = h * n_tiles + t;
    int x = 0;
#pragma unroll
    for (int k = 1; k < 8; ++k) x += u >= cut[k];
    return x * 1024 + 1023 - min(prefix(t + 1) - prefix(t), 1023);
  };
  for (int h = 0; h < a.nkv; ++h)
    for (int t = tid; t < n_tiles; t += 1024) atomicAdd(&s_bin[key_of(h, t)], 1);
  __syncthreads();
  {
    int loc[8], sum = 0;  // thread t owns bins [8t, 8t + 8)
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      loc[k] = sum;
      sum += s_bin[8 * tid + k];
    }
    int tot;
    const int base = block_exclusive_scan_1024(sum, tot, smem);
#pragma unroll
    for (int k = 0; k < 8; ++k) s_bin[8 * tid + k] = base + loc[k];
  }
  __syncthreads();
  for (int h = 0; h < a.nkv; ++h)
    for (int t = tid; t < n_tiles; t += 1024) a.order[atomicAdd(&s_bin[key_of(h, t)], 1)] = h * n_tiles + t;
}

// The whole plan in one launch: workgroup 0 lists and orders the MFMA tiles,
// workgroup 1 builds the split-KV plan of the short-query requests, the
// others write the token map (1024 tokens each).  None reads another's output.
__global__ __launch_bounds__(1024) void prefill_plan_kernel(PfPlanArgs a, PlanParams d, TokenMapArgs m) {
  if (blockIdx.x == 0) {
    prefill_plan_body(a);
  } else if (blockIdx.x == 1) {
    decode_plan_body(d);
  } else {
    token_map_body(m, ((int)blockIdx.x - 2) * 1024 + (int)threadIdx.x);
  }
}

// One workgroup's part of the plan, from index arrays of its own.
__device__ inline void plan_part(PfPlanArgs& a, PlanParams& d, TokenMapArgs& m, const int32_t* qo, const int32_t* kvp,
                                 const int32_t* idx, const int32_t* last) {
  if (blockIdx.x == 0) {
    a.qo_indptr = qo;
    a.kv_indptr = kvp;
    a.last_page_len = last;
    prefill_plan_body(a);
  } else if (blockIdx.x == 1) {
    d.qo_indptr = qo;
    d.kv_indptr = kvp;
    d.kv_indices = idx;
    d.last_page_len = last;
    decode_plan_body(d);
  } else {
    m.qo_indptr = qo;
    m.kv_indptr = kvp;
    m.kv_indices = idx;
    m.last_page_len = last;
    token_map_body(m, ((int)blockIdx.x - 2) * 1024 + (int)threadIdx.x);
  }
}

// The index arrays in the argument: every workgroup plans from its own copy in
// LDS, workgroup 0 also writes the device arrays.
__global__ __launch_bounds__(1024) void prefill_plan_host_kernel(PfPlanArgs a, PlanParams d, TokenMapArgs m, HostIndices h) {
  __shared__ int32_t s_idx[MI_PLAN_HOST_ARGS];
  host_indices_copy(h, s_idx, blockIdx.x == 0);
  plan_part(a, d, m, s_idx, s_idx + h.end[0], s_idx + h.end[1], s_idx + h.end[2]);
}

// The index arrays in pinned host memory, for plans that the argument cannot
// hold: every workgroup that plans reads the per-request ones over the bus into
// LDS, workgroup 0 also writes their device copies, the token map reads the
// pages of its tokens over the bus, and the last workgroups copy the page list.
// The staged copy (a copy on a side stream, events, and in graph mode four
// device copies) took the host 65 us a plan: 6 chunks and 17 decodes of up to
// 5.7k tokens, a layer launched eagerly, 205 -> 139 us a pass; 4 chunks over up
// to 8k cached tokens with an fp8 cache, bound by their tiles, 322 -> 317.  This kernel
// 12.4 us on the former (bus reads in a chain of two).
struct PfPinned {
  const int32_t* src;  // [qo_indptr | kv_indptr | last_page_len | kv_indices]
  int32_t num_indices, copy_blocks;
  int32_t *qo_indptr, *kv_indptr, *last_page_len, *kv_indices;
};
__global__ __launch_bounds__(1024) void prefill_plan_pinned_kernel(PfPlanArgs a, PlanParams d, TokenMapArgs m, PfPinned h) {
  __shared__ int32_t s_idx[3 * MI_PLAN_PINNED_BATCH + 2];
  const int b = a.batch, per_request = 3 * b + 2;
  const int32_t* idx = h.src + per_request;
  const int copy = (int)blockIdx.x - ((int)gridDim.x - h.copy_blocks);
  if (copy >= 0) {
    for (int i = copy * 1024 + (int)threadIdx.x; i < h.num_indices; i += h.copy_blocks * 1024) h.kv_indices[i] = idx[i];
    return;
  }
  for (int i = (int)threadIdx.x; i < per_request; i += 1024) {
    const int32_t v = h.src[i];
    s_idx[i] = v;
    if (blockIdx.x == 0) {
      if (i <= b) h.qo_indptr[i] = v;
      else if (i <= 2 * b + 1) h.kv_indptr[i - b - 1] = v;
      else h.last_page_len[i - 2 * b - 2] = v;
    }
  }
  __syncthreads();
  plan_part(a, d, m, s_idx, s_idx + b + 1, idx, s_idx + 2 * b + 2);
}

template <typename MT, bool FP8>
static int launch_prefill(const PrefillParams& pp, int head_dim, int grid, hipStream_t stream) {
  switch (head_dim) {
    case 64: hipLaunchKernelGGL((prefill_kernel<MT, FP8, 64>), dim3(grid), dim3(64 * pf_waves(64)), 0, stream, pp); break;
    case 128: return prefill_d128_launch(pp, MT::kDtype == MI_F16, FP8, grid, stream);
    case 256: hipLaunchKernelGGL((prefill_rs_kernel<MT, FP8, 256>), dim3(grid), dim3(512), 0, stream, pp); break;
    default: return MI_ERR_UNSUPPORTED;
  }
  return MI_OK;
}

// Merge of split tiles, after the prefill kernel.  A wavefront merges NV output
// tiles of one (split tile, kv-head, row group): row r is
// sum_i 2^(lse_i - max) o_i / sum_i 2^(lse_i - max), in piece order, up to 8
// pieces (4 at head_dim 256) loaded together.  HBM/latency bound: 64 tiles cut
// in four (33 MB of partials) 8 us.  (Merged by the
// prefill kernel's own workgroups once all pieces were done, the partials
// crossing the XCDs' L2 caches by agent-scope stores or by fences, the same 64
// tiles took 63 and 84 us of kernel against 44 + 8.)
constexpr int kPfMergeThreads = 512;
template <typename MT, int D>
MI_DEVICE void prefill_merge_body(const PrefillParams& p, int first_wave, int waves) {
  constexpr int VW = D / 16, NV = D / 64, ROWS = pf_rows(D), NG = ROWS / 16, U = D > 128 ? 4 : 8;
  constexpr float kNegInf = -__builtin_inff();
  const int nkv = p.num_kv_heads, G = p.group;
  const int lane = lane_id(), col = lane & 15, grp = lane >> 4;
  const int total = pf_fits(p) ? p.hdr[kPfSplitTiles] * nkv * NG * 4 : 0;
  for (int w = uniform(first_wave + ((int)threadIdx.x >> 6)); w < total; w += waves) {
    const int part = w & 3, rgi = (w >> 2) % NG, th = (w >> 2) / NG;
    const int h = th % nkv;
    const int4 st = p.split_tiles[th / nkv];
    const int b = uniform(st.x), n = uniform(st.z), slot = uniform(st.w) + h * n;
    const int qo_start = p.qo_indptr[b];
    const int rows_total = (p.qo_indptr[b + 1] - qo_start) * G;
    const int row = uniform(st.y) + 16 * rgi + col;
    if (row >= rows_total) continue;
    float4 acc[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) acc[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    float M = kNegInf, wsum = 0.f;
    for (int c = 0; c < n; c += U) {
      float lse[U];
      float4 o[U][NV];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        lse[u] = kNegInf;
        if (c + u < n) {
          const int64_t s = slot + c + u;
          lse[u] = p.part_lse[s * ROWS + 16 * rgi + col];
          const float4* src = p.part_o + ((s * NG + rgi) * VW + NV * part) * 64 + lane;
#pragma unroll
          for (int i = 0; i < NV; ++i) o[u][i] = src[64 * i];
        }
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (lse[u] == kNegInf) continue;  // past the last piece, or one that this row sees no key of
        if (lse[u] > M) {
          const float sc = fast_exp2(M - lse[u]);
          wsum *= sc;
#pragma unroll
          for (int i = 0; i < NV; ++i) {
            acc[i].x *= sc;
            acc[i].y *= sc;
            acc[i].z *= sc;
            acc[i].w *= sc;
          }
          M = lse[u];
        }
        const float g = fast_exp2(lse[u] - M);  // a NaN lse makes the row NaN
        wsum += g;
#pragma unroll
        for (int i = 0; i < NV; ++i) {
          acc[i].x += g * o[u][i].x;
          acc[i].y += g * o[u][i].y;
          acc[i].z += g * o[u][i].z;
          acc[i].w += g * o[u][i].w;
        }
      }
    }
    const float inv = wsum > 0.f ? 1.f / wsum : 0.f;
    const int tok = row / G, g = row - tok * G;
    uint16_t* orow = (uint16_t*)p.out + (int64_t)(qo_start + tok) * p.out_stride_tok + (int64_t)(h * G + g) * p.out_stride_head;
#pragma unroll
    for (int i = 0; i < NV; ++i)
      *(uint2*)(orow + 16 * (NV * part + i) + 4 * grp) =
          make_uint2(MT::pack2(acc[i].x * inv, acc[i].y * inv), MT::pack2(acc[i].z * inv, acc[i].w * inv));
  }
}

template <typename MT, int D>
__global__ __launch_bounds__(kPfMergeThreads) void prefill_merge_kernel(PrefillParams p) {
  constexpr int WAVES = kPfMergeThreads / 64;
  prefill_merge_body<MT, D>(p, (int)blockIdx.x * WAVES, (int)gridDim.x * WAVES);
}

// Both merges of a call that runs both parts in turn: workgroups below
// batch * nkv merge the short-query requests' split-KV items, the others the
// split tiles (8 wavefronts a CU at most, as in the launch of their own).  A
// dependent launch costs 4 us, whatever it does: two captured 50-token suffixes
// over 8 layers take 205 us against 221 with a launch each.  A batch whose
// decode plan pairs kv-heads keeps two launches.
template <typename MT, int D, int RUN>
__global__ __launch_bounds__(256) void both_merges_kernel(DecodeParams d, int32_t batch, PrefillParams p) {
  const int shorts = batch * d.num_kv_heads;
  if ((int)blockIdx.x < shorts)
    merge_body<MT, D, RUN>(d, batch, (int)blockIdx.x);
  else
    prefill_merge_body<MT, D>(p, ((int)blockIdx.x - shorts) * 4, ((int)gridDim.x - shorts) * 4);
}

template <typename MT, bool FP8>
static void launch_both_merges(const DecodeParams& d, int batch, const PrefillParams& p, int head_dim, int grid,
                               hipStream_t stream) {
  switch (head_dim) {
    case 64: hipLaunchKernelGGL((both_merges_kernel<MT, 64, lane_run(64, FP8 ? 1 : 2)>), dim3(grid), dim3(256), 0, stream, d, batch, p); break;
    case 128: hipLaunchKernelGGL((both_merges_kernel<MT, 128, lane_run(128, FP8 ? 1 : 2)>), dim3(grid), dim3(256), 0, stream, d, batch, p); break;
    default: hipLaunchKernelGGL((both_merges_kernel<MT, 256, lane_run(256, FP8 ? 1 : 2)>), dim3(grid), dim3(256), 0, stream, d, batch, p); break;
  }
}

template <typename MT>
static void launch_prefill_merge(const PrefillParams& pp, int head_dim, int grid, hipStream_t stream) {
  switch (head_dim) {
    case 64: hipLaunchKernelGGL((prefill_merge_kernel<MT, 64>), dim3(grid), dim3(kPfMergeThreads), 0, stream, pp); break;
    case 128: hipLaunchKernelGGL((prefill_merge_kernel<MT, 128>), dim3(grid), dim3(kPfMergeThreads), 0, stream, pp); break;
    default: hipLaunchKernelGGL((prefill_merge_kernel<MT, 256>), dim3(grid), dim3(kPfMergeThreads), 0, stream, pp); break;
  }
}

static bool ok_head_dim(int d) { return d == 64 || d == 128 || d == 256; }

}  // namespace mi

extern "C" int64_t mi_prefill_workspace_bytes(int32_t batch, int32_t max_qo_tokens, int32_t num_qo_heads,
                                              int32_t num_kv_heads, int32_t head_dim) {
  using namespace mi;
  if (batch < 0 || max_qo_tokens < 0 || num_kv_heads <= 0 || num_qo_heads <= 0 || num_qo_heads % num_kv_heads)
    return MI_ERR_INVALID;
  const PrefillLayout L = prefill_layout(batch, max_qo_tokens, num_qo_heads / num_kv_heads, num_kv_heads, head_dim);
  return pf_split_of(L, batch, num_qo_heads / num_kv_heads, num_kv_heads, head_dim, -1).total;
}

extern "C" int32_t mi_prefill_short_rows(int32_t batch, int32_t num_qo_heads, int32_t num_kv_heads,
                                         int32_t head_dim) {
  using namespace mi;
  if (batch < 0 || num_kv_heads <= 0 || num_qo_heads <= 0 || num_qo_heads % num_kv_heads) return MI_ERR_INVALID;
  const int32_t G = num_qo_heads / num_kv_heads;
  return pair_short_rows(pair_heads(nullptr, batch, num_kv_heads, G, head_dim, true));
}

namespace mi {

// host / pinned: the index arrays in the launch argument or in pinned memory (both NULL: the device arrays)
static int prefill_plan_impl(const int32_t* qo_indptr, const int32_t* kv_indptr, const int32_t* kv_indices,
                             const int32_t* last_page_len, int32_t batch, int32_t max_qo_tokens, int32_t page_size,
                             int32_t num_qo_heads, int32_t num_kv_heads, int32_t head_dim, int64_t* token_to_page,
                             int64_t* token_to_cache, int32_t token_map_len, void* workspace,
                             int64_t workspace_bytes, const HostIndices* host, PfPinned* pinned, void* stream) {
  if (batch < 0 || max_qo_tokens < 0 || token_map_len < 0 || !workspace) return MI_ERR_INVALID;
  if (!qo_indptr || !kv_indptr || !last_page_len || (batch > 0 && !kv_indices)) return MI_ERR_INVALID;
  if (token_map_len > 0 && (!token_to_page || !token_to_cache)) return MI_ERR_INVALID;
  if (num_kv_heads <= 0 || num_qo_heads <= 0 || num_qo_heads % num_kv_heads) return MI_ERR_INVALID;
  if (page_size <= 0) return MI_ERR_INVALID;
  if (page_size % 16 || !ok_head_dim(head_dim)) return MI_ERR_UNSUPPORTED;
  const int G = num_qo_heads / num_kv_heads;
  if (G > kShortRows) return MI_ERR_UNSUPPORTED;
  const PrefillLayout L = prefill_layout(batch, max_qo_tokens, G, num_kv_heads, head_dim);
  if (workspace_bytes < L.split) return MI_ERR_WORKSPACE;
  uint8_t* ws = (uint8_t*)workspace;
  PlanParams d{};
  const int st = decode_plan_params(qo_indptr, kv_indptr, kv_indices, last_page_len, batch, page_size, num_qo_heads,
                                    num_kv_heads, head_dim, nullptr, workspace, workspace_bytes, L.split, &d, true);
  if (st != MI_OK) return st;
  PfPlanArgs a;
  a.qo_indptr = qo_indptr;
  a.kv_indptr = kv_indptr;
  a.last_page_len = last_page_len;
  a.batch = batch;
  a.page_size = page_size;
  a.group = G;
  a.nkv = num_kv_heads;
  a.tile_rows = pf_rows(head_dim);
  a.max_tiles = L.max_tiles;
  a.causal = 1;  // cost model: causal
  a.short_rows = d.short_rows;  // the decode plan's threshold: every request goes to exactly one of the two
  a.hdr = (int32_t*)(ws + L.hdr);
  a.tiles = (int2*)(ws + L.tiles);
  a.tcum = (int32_t*)(ws + L.tcum);
  a.order = (int32_t*)(ws + L.order);
  a.ctr = (int32_t*)(ws + L.ctr);
  const PfSplitLayout P = pf_split_of(L, batch, G, num_kv_heads, head_dim, workspace_bytes);
  const PfSplitCosts costs = pf_split_costs(head_dim);
  a.max_parts = P.parts;
  a.workgroups = device_cu_count();
  a.unit_steps = costs.unit;
  a.part_steps = costs.part;
  a.merge_steps = costs.merge;
  a.merge_part_steps = costs.merge_part;
  a.pieces = (int4*)(ws + P.pieces);
  a.split_tiles = (int4*)(ws + P.split_tiles);
  TokenMapArgs m;
  m.qo_indptr = qo_indptr;
  m.kv_indptr = kv_indptr;
  m.kv_indices = kv_indices;
  m.last_page_len = last_page_len;
  m.batch = batch;
  m.page_size = page_size;
  m.t2p = token_to_page;
  m.t2c = token_to_cache;
  m.map_len = token_map_len;
  const int grid = 2 + (token_map_len + 1023) / 1024;
  if (host)
    hipLaunchKernelGGL(prefill_plan_host_kernel, dim3(grid), dim3(1024), 0, (hipStream_t)stream, a, d, m, *host);
  else if (pinned) {
    pinned->copy_blocks = (pinned->num_indices + 1023) / 1024;
    hipLaunchKernelGGL(prefill_plan_pinned_kernel, dim3(grid + pinned->copy_blocks), dim3(1024), 0, (hipStream_t)stream, a, d, m, *pinned);
  } else
    hipLaunchKernelGGL(prefill_plan_kernel, dim3(grid), dim3(1024), 0, (hipStream_t)stream, a, d, m);
  MI_CHECK_LAUNCH();
  return MI_OK;
}

}  // namespace mi

extern "C" int mi_prefill_plan(const int32_t* qo_indptr, const int32_t* kv_indptr,
                               const int32_t* kv_indices, const int32_t* last_page_len, int32_t batch,
                               int32_t max_qo_tokens, int32_t page_size, int32_t num_qo_heads,
                               int32_t num_kv_heads, int32_t head_dim, int64_t* token_to_page,
                               int64_t* token_to_cache, int32_t token_map_len, void* workspace,
                               int64_t workspace_bytes, void* stream) {
  return mi::prefill_plan_impl(qo_indptr, kv_indptr, kv_indices, last_page_len, batch, max_qo_tokens, page_size,
                               num_qo_heads, num_kv_heads, head_dim, token_to_page, token_to_cache, token_map_len,
                               workspace, workspace_bytes, nullptr, nullptr, stream);
}

extern "C" int mi_prefill_plan_host(const int32_t* qo_indptr_host, const int32_t* kv_indptr_host,
                                    const int32_t* kv_indices_host, const int32_t* last_page_len_host,
                                    int32_t num_indices, int32_t* qo_indptr, int32_t* kv_indptr, int32_t* kv_indices,
                                    int32_t* last_page_len, int32_t batch, int32_t max_qo_tokens, int32_t page_size,
                                    int32_t num_qo_heads, int32_t num_kv_heads, int32_t head_dim,
                                    int64_t* token_to_page, int64_t* token_to_cache, int32_t token_map_len,
                                    void* workspace, int64_t workspace_bytes, void* stream) {
  if (batch < 0) return MI_ERR_INVALID;
  const int32_t* const src[4] = {qo_indptr_host, kv_indptr_host, kv_indices_host, last_page_len_host};
  int32_t* const dst[4] = {qo_indptr, kv_indptr, kv_indices, last_page_len};
  const int32_t len[4] = {batch + 1, batch + 1, num_indices, batch};
  mi::HostIndices m;
  const int st = mi::host_indices(src, len, dst, 4, &m);
  if (st != MI_OK) return st;
  if (kv_indptr_host[batch] > num_indices) return MI_ERR_INVALID;  // pages past the argument's
  return mi::prefill_plan_impl(qo_indptr, kv_indptr, kv_indices, last_page_len, batch, max_qo_tokens, page_size,
                               num_qo_heads, num_kv_heads, head_dim, token_to_page, token_to_cache, token_map_len,
                               workspace, workspace_bytes, &m, nullptr, stream);
}

extern "C" int mi_prefill_plan_pinned(const int32_t* indices_pinned, int32_t num_indices, int32_t* qo_indptr,
                                      int32_t* kv_indptr, int32_t* kv_indices, int32_t* last_page_len, int32_t batch,
                                      int32_t max_qo_tokens, int32_t page_size, int32_t num_qo_heads,
                                      int32_t num_kv_heads, int32_t head_dim, int64_t* token_to_page,
                                      int64_t* token_to_cache, int32_t token_map_len, void* workspace,
                                      int64_t workspace_bytes, void* stream) {
  if (batch > MI_PLAN_PINNED_BATCH) return MI_ERR_UNSUPPORTED;
  if (num_indices < 0 || (num_indices > 0 && !kv_indices)) return MI_ERR_INVALID;  // copied also without requests
  if (!indices_pinned || !mi::device_reachable(indices_pinned)) return MI_ERR_INVALID;
  mi::PfPinned m{indices_pinned, num_indices, 0, qo_indptr, kv_indptr, last_page_len, kv_indices};
  return mi::prefill_plan_impl(qo_indptr, kv_indptr, kv_indices, last_page_len, batch, max_qo_tokens, page_size,
                               num_qo_heads, num_kv_heads, head_dim, token_to_page, token_to_cache, token_map_len,
                               workspace, workspace_bytes, nullptr, &m, stream);
}

namespace mi {

constexpr int kPhaseShort = 1;  // short-query requests: split-KV decode kernel + merge
constexpr int kPhaseTiles = 2;  // long-query requests: MFMA prefill tiles

static int prefill_run_impl(const void* q, int32_t q_dtype, int64_t q_stride_token, int64_t q_stride_head,
                            const mi_paged_kv* kv, const int32_t* qo_indptr, const int32_t* kv_indptr,
                            const int32_t* kv_indices, const int32_t* last_page_len, int32_t batch,
                            int32_t max_qo_tokens, int32_t num_qo_heads, int32_t causal, float sm_scale,
                            void* workspace, int64_t workspace_bytes, void* out, int64_t out_stride_token,
                            int64_t out_stride_head, int phases, void* stream) {
  if (!kv || batch < 0 || max_qo_tokens < 0 || !workspace) return MI_ERR_INVALID;
  if (batch == 0) return MI_OK;
  if (!q || !out || !kv->data || !qo_indptr || !kv_indptr || !kv_indices || !last_page_len) return MI_ERR_INVALID;
  const int nkv = kv->num_kv_heads, D = kv->head_dim;
  if (nkv <= 0 || num_qo_heads <= 0 || num_qo_heads % nkv) return MI_ERR_INVALID;
  const int G = num_qo_heads / nkv;
  if (G > kShortRows || kv->page_size % 16 || !ok_head_dim(D)) return MI_ERR_UNSUPPORTED;
  const bool fp8 = kv->dtype == MI_FP8_E4M3;
  if (q_dtype != MI_BF16 && q_dtype != MI_F16 && q_dtype != MI_F32) return MI_ERR_UNSUPPORTED;
  if (!fp8 && kv->dtype != q_dtype) return MI_ERR_UNSUPPORTED;
  if (fp8 && q_dtype == MI_F32) return MI_ERR_UNSUPPORTED;
  if (fp8 && (!kv->k_scale || !kv->v_scale)) return MI_ERR_INVALID;
  const int qesz = q_dtype == MI_F32 ? 4 : 2;
  if (!rows_aligned16(q, q_stride_token, q_stride_head, qesz) ||
      !rows_aligned16(out, out_stride_token, out_stride_head, qesz) || !kv_aligned16(kv))
    return MI_ERR_INVALID;
  // the tile loader keeps a chunk's offset within a page (K/V half, token
  // row, column) in 32 bits
  const int64_t kvesz = fp8 ? 1 : kv->dtype == MI_F32 ? 4 : 2;
  if (kv->kv_stride < 0 || kv->token_stride < 0 ||
      (kv->kv_stride + (int64_t)kv->page_size * kv->token_stride) * kvesz >= (1LL << 31))
    return MI_ERR_UNSUPPORTED;
  const PrefillLayout L = prefill_layout(batch, max_qo_tokens, G, nkv, D);
  if (workspace_bytes < L.split) return MI_ERR_WORKSPACE;
  hipStream_t s = (hipStream_t)stream;
  int st = MI_OK;
  const PfSplitLayout P = pf_split_of(L, batch, G, nkv, D, workspace_bytes);
  // both parts in one call: one launch merges both (both_merges_kernel)
  const bool both = phases == (kPhaseShort | kPhaseTiles) && P.parts > 0 && q_dtype != MI_F32 &&
                    !pair_heads(nullptr, batch, nkv, G, D, true);
  DecodeParams dmerge{};
  if (phases & kPhaseShort) {
    st = decode_run_impl(q, q_dtype, q_stride_token, q_stride_head, kv, qo_indptr, kv_indptr, kv_indices,
                         last_page_len, batch, num_qo_heads, causal, sm_scale, workspace, workspace_bytes,
                         L.split, out, out_stride_token, out_stride_head, kPhaseAttend | (both ? 0 : kPhaseMerge), s,
                         true, &dmerge);
    if (st != MI_OK) return st;
  }
  if (!(phases & kPhaseTiles)) return MI_OK;
  const uint8_t* ws = (const uint8_t*)workspace;
  if (q_dtype == MI_F32) {  // fp32 KV: the plan's tiles by blocks of rows
    DecodeParams dp{};
    dp.q = q;
    dp.q_stride_tok = q_stride_token;
    dp.q_stride_head = q_stride_head;
    dp.kv = kv->data;
    dp.page_stride = kv->page_stride;
    dp.kv_stride = kv->kv_stride;
    dp.token_stride = kv->token_stride;
    dp.head_stride = kv->head_stride;
    dp.qo_indptr = qo_indptr;
    dp.kv_indptr = kv_indptr;
    dp.kv_indices = kv_indices;
    dp.last_page_len = last_page_len;
    dp.out = out;
    dp.out_stride_tok = out_stride_token;
    dp.out_stride_head = out_stride_head;
    dp.num_kv_heads = nkv;
    dp.group = G;
    dp.page_size = kv->page_size;
    dp.causal = causal ? 1 : 0;
    dp.scale_log2 = sm_scale * 1.4426950408889634f;
    st = f32_prefill_launch(dp, (const int32_t*)(ws + L.hdr), (const int2*)(ws + L.tiles), L.max_tiles,
                            pf_rows(D), (int64_t)max_qo_tokens * G, D, s);
    if (st != MI_OK) return st;
    MI_CHECK_LAUNCH();
    return MI_OK;
  }
  // long-query requests: MFMA prefill tiles
  PrefillParams pp{};
  pp.q = q;
  pp.q_stride_tok = q_stride_token;
  pp.q_stride_head = q_stride_head;
  pp.kv = kv->data;
  pp.page_stride = kv->page_stride;
  pp.kv_stride = kv->kv_stride;
  pp.token_stride = kv->token_stride;
  pp.head_stride = kv->head_stride;
  pp.k_scale = kv->k_scale;
  pp.v_scale = kv->v_scale;
  pp.qo_indptr = qo_indptr;
  pp.kv_indptr = kv_indptr;
  pp.kv_indices = kv_indices;
  pp.last_page_len = last_page_len;
  pp.hdr = (const int32_t*)(ws + L.hdr);
  pp.tiles = (const int2*)(ws + L.tiles);
  pp.order = (const int32_t*)(ws + L.order);
  pp.ctr = (int32_t*)((uint8_t*)workspace + L.ctr);
  pp.pieces = (const int4*)(ws + P.pieces);
  pp.split_tiles = (const int4*)(ws + P.split_tiles);
  pp.part_lse = (float*)((uint8_t*)workspace + P.lse);
  pp.part_o = (float4*)((uint8_t*)workspace + P.o);
  pp.parts = P.parts;
  pp.out = out;
  pp.out_stride_tok = out_stride_token;
  pp.out_stride_head = out_stride_head;
  pp.num_kv_heads = nkv;
  pp.group = G;
  pp.page_size = kv->page_size;
  pp.causal = causal ? 1 : 0;
  pp.scale_log2 = sm_scale * 1.4426950408889634f;
  // persistent grid: one workgroup per CU (each holds two wavefronts per
  // SIMD), never more than there can be units
  const int ncu = device_cu_count();
  const int64_t units = (int64_t)(P.parts > 0 ? P.max_pieces : L.max_tiles) * nkv;
  const int grid = (int)(((units < ncu ? units : (int64_t)ncu) + 7) / 8 * 8);
  if (q_dtype == MI_BF16)
    st = fp8 ? launch_prefill<BF16, true>(pp, D, grid, s) : launch_prefill<BF16, false>(pp, D, grid, s);
  else
    st = fp8 ? launch_prefill<F16, true>(pp, D, grid, s) : launch_prefill<F16, false>(pp, D, grid, s);
  if (st != MI_OK) return st;
  // which tiles are split is the device's decision: the merge is launched
  // wherever a split is possible, and exits at once without one (4 us)
  if (both) {
    const int64_t waves = (int64_t)L.max_tiles * nkv * (pf_rows(D) / 16) * 4;
    const int grid2 = batch * nkv + (int)(waves < 8LL * ncu ? (waves + 3) / 4 : 2LL * ncu);
    if (q_dtype == MI_BF16)
      fp8 ? launch_both_merges<BF16, true>(dmerge, batch, pp, D, grid2, s) : launch_both_merges<BF16, false>(dmerge, batch, pp, D, grid2, s);
    else
      fp8 ? launch_both_merges<F16, true>(dmerge, batch, pp, D, grid2, s) : launch_both_merges<F16, false>(dmerge, batch, pp, D, grid2, s);
  } else if (P.parts > 0) {
    const int64_t waves = (int64_t)L.max_tiles * nkv * (pf_rows(D) / 16) * 4, per = kPfMergeThreads / 64;
    const int mgrid = (int)(waves < ncu * per ? (waves + per - 1) / per : ncu);
    if (q_dtype == MI_BF16) launch_prefill_merge<BF16>(pp, D, mgrid, s);
    else launch_prefill_merge<F16>(pp, D, mgrid, s);
  }
  MI_CHECK_LAUNCH();
  return MI_OK;
}

}  // namespace mi

#define MI_PREFILL_ARGS                                                                                          \
  const void *q, int32_t q_dtype, int64_t q_stride_token, int64_t q_stride_head, const mi_paged_kv *kv,          \
      const int32_t *qo_indptr, const int32_t *kv_indptr, const int32_t *kv_indices,                             \
      const int32_t *last_page_len, int32_t batch, int32_t max_qo_tokens, int32_t num_qo_heads, int32_t causal, \
      float sm_scale, void *workspace, int64_t workspace_bytes, void *out, int64_t out_stride_token,             \
      int64_t out_stride_head, void *stream
#define MI_PREFILL_FWD(phases)                                                                                    \
  mi::prefill_run_impl(q, q_dtype, q_stride_token, q_stride_head, kv, qo_indptr, kv_indptr, kv_indices,          \
                       last_page_len, batch, max_qo_tokens, num_qo_heads, causal, sm_scale, workspace,           \
                       workspace_bytes, out, out_stride_token, out_stride_head, phases, stream)

extern "C" int mi_prefill_run(MI_PREFILL_ARGS) { return MI_PREFILL_FWD(mi::kPhaseShort | mi::kPhaseTiles); }
extern "C" int mi_prefill_short(MI_PREFILL_ARGS) { return MI_PREFILL_FWD(mi::kPhaseShort); }
extern "C" int mi_prefill_tiles(MI_PREFILL_ARGS) { return MI_PREFILL_FWD(mi::kPhaseTiles); }
