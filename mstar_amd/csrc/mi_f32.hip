// fp32 paged attention (fp32 KV cache, fp32 q and output) for MI355X (gfx950).
//
// The reference allocates the KV pool in the model's autocast dtype, fp32
// included (mstar/engine/kv_cache_engine.py:104-105, 132-136; Pi0.5 runs its
// real weights with kv_cache_type=torch.float32), and plans its wrappers in
// the cache's dtype (mstar/engine/cache_manager.py:241-247), so q, K, V and
// the output are fp32.  This file computes that case in fp32 throughout with
// the fp32 matrix instruction v_mfma_f32_16x16x4_f32:
//
//   decode  (the decode plan's split-KV items: decode steps and the
//           short-query requests of a ragged batch): one workgroup per
//           (item, kv-head), its 4 wavefronts over contiguous quarters of
//           the item's 16-token tiles; partials in the bf16 decode kernel's
//           layout, so its merge (with fp32 output) finishes split requests;
//   prefill (the long-query requests): one workgroup per (tile of the
//           prefill plan, kv-head, 16-row block), its 4 wavefronts over
//           contiguous quarters of the keys the block's rows can see.
//
// Per 16-token tile, a wavefront holds 16 (query token, q-head) rows of one
// kv-head as the 16 MFMA columns (GQA rows packed token-major, so a K/V row
// is read once per q-head group):
//   S^T[16 keys x 16 rows] = K . Q^T     D/4 MFMAs; k slot g of step s is dim
//                                         (D/4)*g + s, so a lane's Q and K
//                                         operands are D/4 consecutive floats
//                                         of one row
//   online softmax in fp32 (exp2 domain), causal limit aligned to the end of
//   the KV
//   O^T[16 dims x 16 rows] += V^T . P^T  4 MFMAs per 16-dim output tile; k
//                                         slot g of step t is key 4g + t, so
//                                         the B operand is the lane's own
//                                         probability of key 4g + t; output
//                                         row i of tile m is the dim that
//                                         lane i loaded as its element m, so
//                                         the A operand is one of the lane's
//                                         own V floats
// Each lane loads, for its 4 keys 4g..4g+3, D/16 floats with 16-byte loads,
// each load instruction covering 256 contiguous bytes of the key row
// (dim_of in mi_plan.h).  K takes the same load layout and passes through a
// per-wavefront LDS buffer in natural dim order, where each lane reads back
// its key's D/4-float operand run.
#include "mi_common.h"
#include "mi_internal.h"
#include "mi_plan.h"

namespace mi {

struct F32Tiles {
  const int32_t* hdr;  // [0]: tiles listed by the prefill plan
  const int2* tiles;   // (request, first row)
  int32_t tile_rows;
  int32_t from = 0, to = 0x7fffffff;  // the launch acts if the plan has from <= tiles < to
};

template <int D>
struct F32Regs {  // lane: keys 4*grp + r, dims dim_of(lane_run(D, 4), col, j), j < D/16
  float4 k[4][D / 64];
  float4 v[4][D / 64];
};

template <int N>
MI_DEVICE void load_f4(float4 (&dst)[N], const uint8_t* src) {  // float4 i: 256*i bytes into the row (dim_of)
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const uint4 u = nt_load16(src + 256 * i);
    dst[i] = make_float4(bitcast<float>(u.x), bitcast<float>(u.y), bitcast<float>(u.z), bitcast<float>(u.w));
  }
}

MI_DEVICE float f4_at(const float4& v, int i) { return i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w; }

MI_DEVICE f32x4 mma_f32(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

template <int D, bool PREFILL>
__global__ __launch_bounds__(256) void attend_f32_kernel(DecodeParams p, F32Tiles pt) {
  constexpr int VW = D / 16;      // output dim tiles; floats per lane of a key row
  constexpr int NV = VW / 4;      // float4 per lane of a key row
  constexpr int KQ = D / 4;       // S MFMA steps; floats of a lane's Q / K operand run
  constexpr int KRS = D * 4 + 16;  // LDS row stride of the K staging buffer (bytes): rows 4 banks apart
  constexpr int RUN = lane_run(D, 4);  // consecutive floats per lane (dim_of)
  constexpr float kNegInf = -__builtin_inff();
  constexpr int kStageBytes = 4 * 16 * KRS;
  constexpr int kMergeBytes = 4 * (4 * NV * 64 * 16);
  __shared__ __attribute__((aligned(16))) uint8_t lds[kStageBytes > kMergeBytes ? kStageBytes : kMergeBytes];
  __shared__ float lds_m[4][kRows], lds_l[4][kRows];

  const int lane = lane_id();
  const int wave = uniform((int)threadIdx.x >> 6);
  const int nkv = p.num_kv_heads;
  const int G = p.group;
  const int ps = p.page_size;
  int b, h, row0, kidx = 0, nitems_b = 1, pg_end;
  if constexpr (PREFILL) {
    const int bpt = pt.tile_rows / kRows;  // 16-row blocks per tile
    const int x = (int)blockIdx.x;
    const int j = x % bpt, rest = x / bpt;
    h = uniform(rest % nkv);
    const int t = rest / nkv;
    const int planned = pt.hdr[0];
    if (t >= planned || planned >= pt.to) return;  // uniform
    const int2 tile = pt.tiles[t];
    b = uniform(tile.x);
    row0 = uniform(tile.y + kRows * j);
  } else {
    // the decode kernel's XCD-aware mapping: the kv-heads of an item share an XCD
    const int gsz = 8 * nkv;
    const int gi = uniform((int)blockIdx.x / gsz);
    const int gr = (int)blockIdx.x - gi * gsz;
    h = uniform(gr >> 3);
    const int item = uniform(gi * 8 + (gr & 7));
    if (item >= p.hdr[kHdrChunks]) return;
    const int4 wk = p.work[item];
    b = uniform(wk.x);
    kidx = uniform(wk.y);
    nitems_b = uniform(wk.w);
    row0 = 0;
    pg_end = uniform(wk.z);
  }
  const int page_base = p.kv_indptr[b];
  const int np = p.kv_indptr[b + 1] - page_base;
  const int kv_len = (np - 1) * ps + p.last_page_len[b];
  int qo_start = b, qo_len = 1;
  if (p.qo_indptr) {
    qo_start = p.qo_indptr[b];
    qo_len = p.qo_indptr[b + 1] - qo_start;
  }
  const int rows = min(qo_len * G - row0, kRows);  // rows of this block
  if (rows <= 0) return;                           // uniform: past the request's last row
  const int first_qtok = row0 / G, last_qtok = (row0 + rows - 1) / G;
  int tok0, tok1;  // key range of the unit
  if constexpr (PREFILL) {
    pg_end = np;
    tok0 = 0;
    tok1 = p.causal ? min(kv_len, kv_len - qo_len + last_qtok + 1) : kv_len;
  } else {
    tok0 = kidx * p.hdr[kHdrChunkPages] * ps;
    tok1 = min(pg_end * ps, kv_len);
  }
  const int unit_tiles = tok1 > tok0 ? (tok1 - tok0 + 15) >> 4 : 0;
  const int tq = unit_tiles >> 2, trem = unit_tiles & 3;
  const int my_t0 = wave * tq + min(wave, trem);
  const int ntiles = tq + (wave < trem ? 1 : 0);
  const int tok_begin = tok0 + 16 * my_t0;

  const int col = lane & 15;  // MFMA column = row of the block
  const int grp = lane >> 4;
  const int row = row0 + col;
  const int qtok = row / G;
  const int g = row - qtok * G;
  const bool row_valid = col < rows;
  int lim = p.causal ? (kv_len - qo_len + qtok) : (kv_len - 1);
  lim = min(lim, kv_len - 1);
  const int mask_from = p.causal ? (kv_len - qo_len + first_qtok + 1) : kv_len;  // keys >= this need a row check

  // Q as the B operand of S^T = K Q^T: lane holds Q[row][KQ*grp, +KQ)
  float4 qf[KQ / 4];
  {
    const float* qrow = (const float*)p.q + (int64_t)(qo_start + qtok) * p.q_stride_tok +
                        (int64_t)(h * G + g) * p.q_stride_head + KQ * grp;
#pragma unroll
    for (int i = 0; i < KQ / 4; ++i) qf[i] = row_valid ? *(const float4*)(qrow + 4 * i) : make_float4(0.f, 0.f, 0.f, 0.f);
  }
  const float sl2 = p.scale_log2;

  const uint8_t* kv = (const uint8_t*)p.kv;
  const int64_t head_off = (int64_t)h * p.head_stride * 4;
  const uint32_t voff0 = (uint32_t)((4 * grp) * p.token_stride + RUN * col) * 4;
  const uint32_t vrow = (uint32_t)(p.token_stride * 4);
  const int64_t kvhalf = p.kv_stride * 4;
  auto tile_base = [&](int page, int r0) -> const uint8_t* {
    return kv + (int64_t)page * p.page_stride * 4 + (int64_t)r0 * p.token_stride * 4 + head_off;
  };
  auto load_tile = [&](F32Regs<D>& t, const uint8_t* base) {
    const uint8_t* kb = base + voff0;
#pragma unroll
    for (int r = 0; r < 4; ++r) load_f4(t.k[r], kb + r * vrow);
    const uint8_t* vb = kb + kvhalf;
#pragma unroll
    for (int r = 0; r < 4; ++r) load_f4(t.v[r], vb + r * vrow);
  };
  uint8_t* kst = &lds[wave * 16 * KRS];

  f32x4 acc[VW];
#pragma unroll
  for (int m = 0; m < VW; ++m) acc[m] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m_run = kNegInf, l_run = 0.f;

  auto compute_tile = [&](F32Regs<D>& t, int ti) {
    const int tb = tok_begin + 16 * ti;
    // K rows -> LDS (row 4*grp + r, dims [VW*col, +VW)) -> A operand runs
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float* dst = (float*)(kst + (4 * grp + r) * KRS);  // row in natural dim order
#pragma unroll
      for (int i = 0; i < NV; ++i) *(float4*)(dst + dim_of(RUN, col, 4 * i)) = t.k[r][i];
    }
    f32x4 s = {0.f, 0.f, 0.f, 0.f};
    const float4* krun = (const float4*)(kst + col * KRS + KQ * grp * 4);
#pragma unroll
    for (int i = 0; i < KQ / 4; ++i) {
      const float4 a = krun[i];
      s = mma_f32(a.x, qf[i].x, s);
      s = mma_f32(a.y, qf[i].y, s);
      s = mma_f32(a.z, qf[i].z, s);
      s = mma_f32(a.w, qf[i].w, s);
    }
    float sv[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) sv[r] = s[r] * sl2;
    if (tb + 16 > mask_from) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int key = tb + 4 * grp + r;
        if (key > lim) sv[r] = kNegInf;
        if (key >= kv_len) {  // slots past the end hold stale data: keep NaN/Inf out of P.V
#pragma unroll
          for (int i = 0; i < NV; ++i) t.v[r][i] = make_float4(0.f, 0.f, 0.f, 0.f);
        }
      }
    }
    const float mt = rows4_max(fmaxf(fmaxf(sv[0], sv[1]), fmaxf(sv[2], sv[3])));
    const float m_new = fmaxf(m_run, mt);
    const float m_use = m_new == kNegInf ? 0.f : m_new;
    const float alpha = fast_exp2(m_run - m_use);
    float pr[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) pr[r] = fast_exp2(sv[r] - m_use);
    l_run = l_run * alpha + ((pr[0] + pr[1]) + (pr[2] + pr[3]));
    if (__builtin_amdgcn_ballot_w64(m_new > m_run)) {
#pragma unroll
      for (int m = 0; m < VW; ++m) acc[m] *= alpha;
    }
    m_run = m_new;
#pragma unroll
    for (int m = 0; m < VW; ++m)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[m] = mma_f32(f4_at(t.v[r][m >> 2], m & 3), pr[r], acc[m]);
  };

  // Tile loop in windows of 64 pages: the window's page ids sit in one VGPR
  // (lane i: page i of the window) and v_readlane hands each tile's page to
  // the scalar unit; loads run one tile ahead of the MFMA work.
  for (int w0 = 0; w0 < ntiles;) {
    const int wtok = tok_begin + 16 * w0;
    const int first = wtok / ps;
    const int wt = min(ntiles - w0, ((first + 64) * ps - wtok) >> 4);
    const int pwin = first + lane < pg_end ? p.kv_indices[page_base + first + lane] : 0;
    auto tile_ptr = [&](int t) -> const uint8_t* {
      const int tok = wtok + 16 * t;
      return tile_base(__builtin_amdgcn_readlane(pwin, tok / ps - first), tok % ps);
    };
    F32Regs<D> A, B;
    load_tile(A, tile_ptr(0));
    int t = 0;
    for (; t + 2 < wt; t += 2) {  // every load in range: exact vmcnt waits
      load_tile(B, tile_ptr(t + 1));
      compute_tile(A, w0 + t);
      load_tile(A, tile_ptr(t + 2));
      compute_tile(B, w0 + t + 1);
    }
    if (t + 1 < wt) {
      load_tile(B, tile_ptr(t + 1));
      compute_tile(A, w0 + t);
      compute_tile(B, w0 + t + 1);
    } else {
      compute_tile(A, w0 + t);
    }
    w0 += wt;
  }

  // Merge the 4 wavefronts' states in LDS (same register layout in every
  // wavefront: lane -> row col, dims VW*(4*grp + r) + m); wavefront w
  // finishes the dims with r == w.
  __syncthreads();
  {
    const float l_row = rows4_sum(l_run);
    if (grp == 0) {
      lds_m[wave][col] = m_run;
      lds_l[wave][col] = l_row;
    }
    float4* st = (float4*)lds + (size_t)wave * 4 * NV * 64 + lane;
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int m = 0; m < VW; m += 4)
        st[(r * NV + m / 4) * 64] = make_float4(acc[m][r], acc[m + 1][r], acc[m + 2][r], acc[m + 3][r]);
  }
  __syncthreads();
  float M = kNegInf;
#pragma unroll
  for (int w = 0; w < 4; ++w) M = fmaxf(M, lds_m[w][col]);
  const float M_use = M == kNegInf ? 0.f : M;
  float sc[4], L = 0.f;
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    sc[w] = fast_exp2(lds_m[w][col] - M_use);
    L += sc[w] * lds_l[w][col];
  }
  float4 o[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) o[i] = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    const float4* src = (const float4*)lds + (size_t)w * 4 * NV * 64 + (size_t)wave * NV * 64 + lane;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const float4 v = src[i * 64];
      o[i].x += sc[w] * v.x;
      o[i].y += sc[w] * v.y;
      o[i].z += sc[w] * v.z;
      o[i].w += sc[w] * v.w;
    }
  }
  const float inv = L > 0.f ? 1.f / L : (L == 0.f ? 0.f : __builtin_nanf(""));  // NaN L: keep the row NaN
  if (!row_valid) return;
  if (nitems_b == 1) {  // dims dim_of(RUN, 4*grp + wave, j) of row col
    float* dst = (float*)p.out + (int64_t)(qo_start + qtok) * p.out_stride_tok +
                 (int64_t)(h * G + g) * p.out_stride_head;
#pragma unroll
    for (int i = 0; i < NV; ++i)
      *(float4*)(dst + dim_of(RUN, 4 * grp + wave, 4 * i)) = make_float4(o[i].x * inv, o[i].y * inv, o[i].z * inv, o[i].w * inv);
  } else {  // partial (o, lse) in the split-KV layout of the decode kernel
    const int64_t unit_idx = (int64_t)(p.chunk_indptr[b] + kidx) * nkv + h;
    float* ob = p.o_part + unit_idx * kRows * D + 4 * lane;
#pragma unroll
    for (int i = 0; i < NV; ++i)
      *(float4*)(ob + 256 * (wave * NV + i)) = make_float4(o[i].x * inv, o[i].y * inv, o[i].z * inv, o[i].w * inv);
    if (wave == 0 && grp == 0)  // -inf: empty partial; NaN: the row met a NaN or +inf score
      p.lse_part[unit_idx * kRows + col] = L > 0.f ? M + fast_log2(L) : (L == 0.f ? kNegInf : __builtin_nanf(""));
  }
}

// Prefill with K and V shared by the workgroup: 64 rows of one (tile,
// kv-head), 16 per wavefront, and every wavefront goes over all the keys its
// rows can see.  Steps of KT keys (64 rows of K and V together are 32 KB at
// any head_dim) go through two LDS stages, filled from registers that were
// loaded a step ahead, page ids a step before that; each 16-byte LDS read of a
// K or V fragment feeds four MFMAs.  attend_f32_kernel<D, true> reads each K/V
// row from L2 once per 16 rows and keys' quarter instead: on 4 prefixes of
// 800-1000 tokens at 8 q / 1 kv / 256 its 3.3 GB of L2 reads, not the MFMAs,
// set the time: 409 us on 4 x 900 keys, 303 here (88 TFLOP/s).  Bound by the
// fp32 MFMAs and the vector work beside them, which add up: a step's 64 FMAs
// into O at head_dim 256 take 7 %, so its address arithmetic, bounds and masks
// are kept out of the steps that lie wholly within the rows' keys (5 %).
// S^T, the softmax and O^T use the same operand layouts as there (S^T in two
// chains over the head_dim); V rows past kv_len are stored as zeros.
template <int D>
__global__ __launch_bounds__(256, 2) void prefill_f32_kernel(DecodeParams p, F32Tiles pt) {
  constexpr int VW = D / 16, NV = VW / 4, KQ = D / 4, RUN = lane_run(D, 4);
  constexpr int KT = 16 * (256 / D), NS = KT / 16;  // keys and 16-key groups per step
  constexpr int KRS = D * 4 + 16;   // LDS row stride of K: rows 4 banks apart for the fragment reads
  constexpr int CPR = D / 4;        // 16-byte chunks per row
  constexpr int NL = KT * CPR / 256;  // chunks of K (and of V) per thread
  constexpr int CPG = 16 * CPR / 256;  // of them in one 16-key group
  constexpr float kNegInf = -__builtin_inff();
  __shared__ __attribute__((aligned(16))) uint8_t lds_k[2][KT * KRS];
  __shared__ __attribute__((aligned(16))) uint8_t lds_v[2][KT * D * 4];

  const int tid = (int)threadIdx.x, lane = lane_id(), wave = uniform(tid >> 6);
  const int col = lane & 15, grp = lane >> 4;
  const int nkv = p.num_kv_heads, G = p.group, ps = p.page_size;
  const int bpt = pt.tile_rows / 64;  // 64-row blocks per tile
  const int x = (int)blockIdx.x;
  const int j = x % bpt, rest = x / bpt, t_idx = rest / nkv;
  const int h = uniform(rest - t_idx * nkv);
  const int planned = pt.hdr[0];
  if (t_idx >= planned || planned < pt.from) return;  // uniform
  const int2 tile = pt.tiles[t_idx];
  const int b = uniform(tile.x), row_wg = uniform(tile.y + 64 * j);
  const int page_base = p.kv_indptr[b];
  const int np = p.kv_indptr[b + 1] - page_base;
  const int kv_len = (np - 1) * ps + p.last_page_len[b];
  const int qo_start = p.qo_indptr[b], qo_len = p.qo_indptr[b + 1] - qo_start;
  const int rows_wg = min(qo_len * G - row_wg, 64);
  if (rows_wg <= 0) return;  // uniform: past the request's last row
  const int last_qtok = (row_wg + rows_wg - 1) / G;
  const int kv_end = p.causal ? min(kv_len, kv_len - qo_len + last_qtok + 1) : kv_len;
  const int steps = kv_end > 0 ? (kv_end + KT - 1) / KT : 0;
  // keys that the wavefront's own 16 rows see
  const int last_w = row_wg + min(rows_wg, 16 * wave + 16) - 1;
  const int wave_end = p.causal ? min(kv_len, kv_len - qo_len + last_w / G + 1) : kv_len;

  const int row = row_wg + 16 * wave + col, qtok = row / G, g = row - qtok * G;
  const bool row_valid = row < qo_len * G;
  int lim = p.causal ? (kv_len - qo_len + qtok) : (kv_len - 1);
  lim = min(lim, kv_len - 1);
  const int mask_from = p.causal ? (kv_len - qo_len + row_wg / G + 1) : kv_len;  // keys >= this need a row check

  float4 qf[KQ / 4];
  {
    const float* qrow = (const float*)p.q + (int64_t)(qo_start + qtok) * p.q_stride_tok +
                        (int64_t)(h * G + g) * p.q_stride_head + KQ * grp;
#pragma unroll
    for (int i = 0; i < KQ / 4; ++i) qf[i] = row_valid ? *(const float4*)(qrow + 4 * i) : make_float4(0.f, 0.f, 0.f, 0.f);
  }
  const float sl2 = p.scale_log2;

  // loader: chunk tid + 256 i of the step's K rows and of its V rows; a
  // wavefront's 64 chunks lie in one 16-key group, hence in one page
  const uint8_t* kvb = (const uint8_t*)p.kv + (int64_t)h * p.head_stride * 4;
  const int64_t tok_bytes = p.token_stride * 4, page_bytes = p.page_stride * 4, kvhalf = p.kv_stride * 4;
  const int key_cap = np * ps - 16;  // last group inside the request's pages
  int pg[NS], slot[NS];  // page and slot of the groups of the step to load next
  auto find_pages = [&](int t) {
#pragma unroll
    for (int k = 0; k < NS; ++k) {
      const int key = min(t * KT + 16 * k, key_cap), pidx = (int)((unsigned)key / (unsigned)ps);
      pg[k] = p.kv_indices[page_base + pidx];
      slot[k] = key - pidx * ps;
    }
  };
  f32x4 rk[NL], rv[NL];
  constexpr int RPC = 256 / CPR;  // rows between a thread's chunks
  const int64_t own = (int64_t)(tid / CPR) * tok_bytes + 16 * (tid % CPR);
  auto load_step = [&]() {
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int k = i / CPG;
      const uint8_t* src = kvb + (int64_t)pg[k] * page_bytes + (int64_t)(slot[k] + i % CPG * RPC) * tok_bytes;  // scalar
      rk[i] = *(const f32x4*)(src + own);
      rv[i] = *(const f32x4*)(src + kvhalf + own);
    }
  };
  auto store_step = [&](int t, int st, auto tail) {
    uint8_t* kdst = lds_k[st] + tid / CPR * KRS + 16 * (tid % CPR);
    uint8_t* vdst = lds_v[st] + 16 * tid;
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      *(f32x4*)(kdst + i * RPC * KRS) = rk[i];
      if (decltype(tail)::value && t * KT + tid / CPR + i * RPC >= kv_len) rv[i] = f32x4{0.f, 0.f, 0.f, 0.f};  // slots past the end hold stale data
      *(f32x4*)(vdst + i * 16 * 256) = rv[i];
    }
  };

  f32x4 acc[VW];
#pragma unroll
  for (int m = 0; m < VW; ++m) acc[m] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m_run = kNegInf, l_run = 0.f;

  // One key step.  TAIL: it may end past the wavefront's keys, whose 16-key
  // groups are left out one by one: a masked key's V is multiplied by zero,
  // which a NaN or Inf in it survives, so a row meets no key beyond its 16-row
  // block's last group.
  auto compute = [&](int t, int st, auto tail) {
    constexpr bool TAIL = decltype(tail)::value;
    auto used = [&](int k) { return !TAIL || t * KT + 16 * k < wave_end; };  // uniform
    if (!used(0)) return;
    float sv[NS][4];
#pragma unroll
    for (int k = 0; k < NS; ++k) {
      if (!used(k)) {
#pragma unroll
        for (int r = 0; r < 4; ++r) sv[k][r] = kNegInf;
        continue;
      }
      f32x4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};
      const float4* krun = (const float4*)(lds_k[st] + (16 * k + col) * KRS + KQ * grp * 4);
#pragma unroll
      for (int i = 0; i < KQ / 4; ++i) {
        const float4 a = krun[i];
        s0 = mma_f32(a.x, qf[i].x, s0);
        s1 = mma_f32(a.y, qf[i].y, s1);
        s0 = mma_f32(a.z, qf[i].z, s0);
        s1 = mma_f32(a.w, qf[i].w, s1);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) sv[k][r] = (s0[r] + s1[r]) * sl2;
    }
    if (TAIL && (t + 1) * KT > mask_from) {
#pragma unroll
      for (int k = 0; k < NS; ++k)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (t * KT + 16 * k + 4 * grp + r > lim) sv[k][r] = kNegInf;
    }
    float ml = kNegInf;  // this lane's share of the row
#pragma unroll
    for (int k = 0; k < NS; ++k) ml = fmaxf(ml, fmaxf(fmaxf(sv[k][0], sv[k][1]), fmaxf(sv[k][2], sv[k][3])));
    const float m_new = fmaxf(m_run, rows4_max(ml));
    const float alpha = m_new > m_run ? fast_exp2(m_run - m_new) : 1.f;
    m_run = m_new;
    const float m_use = m_run == kNegInf ? 0.f : m_run;
    float ls = 0.f;
#pragma unroll
    for (int k = 0; k < NS; ++k) {
#pragma unroll
      for (int r = 0; r < 4; ++r) sv[k][r] = fast_exp2(sv[k][r] - m_use);
      ls += (sv[k][0] + sv[k][1]) + (sv[k][2] + sv[k][3]);
    }
    l_run = fmaf(l_run, alpha, ls);
    // The step's P.V is summed by itself, then added: O is rounded at its own size
    // once a step.  (Summed key by key into O, with a max that was raised only past
    // 2^8, 2048 keys were 1.3-1.7x as far from 64 bits as attend_f32_kernel's four
    // shorter sums over exact maxima.)
    f32x4 o[2][4];
    auto add = [&](int i) {
#pragma unroll
      for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[4 * i + m][e] = fmaf(acc[4 * i + m][e], alpha, o[i & 1][m][e]);
    };
    // at head_dim 256 a group of dims late, so that the matrix core's latency is
    // not waited for (296 us instead of 300 on 4 x 900 keys; slower below)
    constexpr int LATE = D > 128 ? 1 : 0;
#pragma unroll
    for (int i = 0; i < NV; ++i) {  // elements 4i..4i+3 of the lane: dims dim_of(RUN, col, 4i)
#pragma unroll
      for (int m = 0; m < 4; ++m) o[i & 1][m] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < NS; ++k) {
        if (!used(k)) continue;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float4 a = *(const float4*)(lds_v[st] + (16 * k + 4 * grp + r) * D * 4 + 16 * col + 256 * i);
          o[i & 1][0] = mma_f32(a.x, sv[k][r], o[i & 1][0]);
          o[i & 1][1] = mma_f32(a.y, sv[k][r], o[i & 1][1]);
          o[i & 1][2] = mma_f32(a.z, sv[k][r], o[i & 1][2]);
          o[i & 1][3] = mma_f32(a.w, sv[k][r], o[i & 1][3]);
        }
      }
      if (i >= LATE) add(i - LATE);
    }
    if (LATE) add(NV - 1);
  };
  static_assert(RUN == 4, "a lane's dims: one float4 per 64");

  if (steps > 0) {
    find_pages(0);
    load_step();
    find_pages(1);
    store_step(0, 0, std::true_type{});
    __syncthreads();
    auto step = [&](int t, auto tail) {
      constexpr bool TAIL = decltype(tail)::value;
      if (!TAIL || t + 1 < steps) {
        load_step();  // step t + 1
        find_pages(t + 2);
      }
      compute(t, t & 1, tail);
      if (!TAIL || t + 1 < steps) store_step(t + 1, (t + 1) & 1, tail);  // the stage of step t - 1
      __syncthreads();
    };
    int t = 0;
    for (const int whole = mask_from > 0 ? mask_from / KT - 1 : 0; t < whole; ++t) step(t, std::false_type{});
    for (; t < steps; ++t) step(t, std::true_type{});
  }
  const float L = rows4_sum(l_run);
  const float inv = L > 0.f ? 1.f / L : (L == 0.f ? 0.f : __builtin_nanf(""));  // NaN L: keep the row NaN
  if (!row_valid) return;
  float* dst = (float*)p.out + (int64_t)(qo_start + qtok) * p.out_stride_tok + (int64_t)(h * G + g) * p.out_stride_head;
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int i = 0; i < NV; ++i)
      *(float4*)(dst + dim_of(RUN, 4 * grp + r, 4 * i)) = make_float4(acc[4 * i][r] * inv, acc[4 * i + 1][r] * inv,
                                                                       acc[4 * i + 2][r] * inv, acc[4 * i + 3][r] * inv);
}

template <int D, bool PREFILL>
static void launch_f32(const DecodeParams& dp, const F32Tiles& pt, int grid, hipStream_t stream) {
  hipLaunchKernelGGL((attend_f32_kernel<D, PREFILL>), dim3(grid), dim3(256), 0, stream, dp, pt);
}

template <bool PREFILL>
static int dispatch_f32(const DecodeParams& dp, const F32Tiles& pt, int head_dim, int grid, hipStream_t stream) {
  switch (head_dim) {
    case 64: launch_f32<64, PREFILL>(dp, pt, grid, stream); break;
    case 128: launch_f32<128, PREFILL>(dp, pt, grid, stream); break;
    case 256: launch_f32<256, PREFILL>(dp, pt, grid, stream); break;
    default: return MI_ERR_UNSUPPORTED;
  }
  return MI_OK;
}

int f32_attend_launch(const DecodeParams& dp, int head_dim, int grid, hipStream_t stream) {
  if (grid <= 0) return MI_OK;
  return dispatch_f32<false>(dp, F32Tiles{nullptr, nullptr, 0}, head_dim, grid, stream);
}

// From how many of its 64-row blocks per CU on the shared-K/V kernel is the
// faster one: a block of it is a long serial job and a CU runs two at a time, so
// its time goes in steps (900 keys at head_dim 256: up to 1 block a CU 168 us, up
// to 2 278), where the other kernel has four times the workgroups and cuts each
// block's keys in four.  Under a causal mask the longest blocks set the step, so
// the line lies higher; where the caller's graph forks the short-query part onto
// another stream, that launch takes CUs in between and it lies higher still.
// us, other -> shared, 900 keys, at 0.9 / 1.0 / 1.25 / 1.6 / 1.8 / 2.2 / 2.5 / 4 blocks a CU:
//   head_dim 256  195 -> 168, 239 -> 272, 287 -> 276, 336 -> 278, 383 -> 280, 433 -> 444, 522 -> 464, 807 -> 676
//     causal      143 -> 163, 149 -> 231, 163 -> 232, 218 -> 233, 248 -> 233, 300 -> 234, 322 -> 288, 505 -> 433
//   head_dim 128  109 ->  85, 130 -> 136, 156 -> 137, 187 -> 138, 213 -> 140, 261 -> 208, 287 -> 208, 466 -> 330
//     causal       83 ->  84,  85 -> 119,  92 -> 120, 124 -> 124, 145 -> 125, 173 -> 131, 185 -> 145, 296 -> 223
//   head_dim 64    49 ->  48,  56 ->  74,  65 ->  75,  78 ->  76,  90 ->  77, 110 -> 115, 123 -> 115, 198 -> 180
//     causal       44 ->  46,  50 ->  68,  53 ->  69,  55 ->  70,  65 ->  71,  78 ->  72,  79 ->  72, 126 -> 106
// and 1800 keys at 1.25 and 1.6, head_dim 256: 506 -> 532, 593 -> 535.
// Without a mask the end of a step pays as well: [low, low_end), below the first
// (head_dim 64: the second) full step.
struct SharedFrom {
  double low, low_end, plain, causal, forked, forked_causal;
};
static SharedFrom shared_from(int head_dim) {
  if (head_dim == 64) return {1.6, 1.9, 2.3, 2.2, 4.0, 4.0};
  if (head_dim == 128) return {0.8, 0.96, 1.4, 1.7, 1.8, 2.0};
  return {0.8, 0.96, 1.6, 1.8, 1.6, 2.2};
}

// `rows` are exact in a plain call.  A captured one is replayed over plans of
// fewer rows, so where the most rows would take the shared kernel it records
// both, and the plan's tiles say which of them acts; the other exits at once (4
// us).  A graph of up to 4096 tokens at 8 q / 1 kv / 256 over one request of 900:
// 104 us a layer, 220 with the kernel chosen by the most rows.
int f32_prefill_launch(const DecodeParams& dp, const int32_t* tile_hdr, const int2* tiles, int max_tiles,
                       int tile_rows, int64_t rows, int head_dim, hipStream_t stream) {
  if (tile_rows <= 0 || tile_rows % 64) return MI_ERR_INVALID;
  const int64_t blocks = (int64_t)max_tiles * dp.num_kv_heads * (tile_rows / 64);
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(stream, &status) != hipSuccess) (void)hipGetLastError();
  const bool captured = status == hipStreamCaptureStatusActive;
  const SharedFrom line = shared_from(head_dim);
  const double cus = device_cu_count(), have = (double)rows / 64 * dp.num_kv_heads;
  const double from = cus * (captured ? (dp.causal ? line.forked_causal : line.forked)
                                      : (dp.causal ? line.causal : line.plain));
  const bool low = !captured && !dp.causal && have >= line.low * cus && have < line.low_end * cus;
  F32Tiles other{tile_hdr, tiles, tile_rows};
  if ((have >= from || low) && blocks <= 0x7fffffff) {
    F32Tiles pt{tile_hdr, tiles, tile_rows};
    if (captured) pt.from = other.to = (int)(from * 64 / ((double)dp.num_kv_heads * tile_rows)) + 1;
    switch (head_dim) {
      case 64: hipLaunchKernelGGL((prefill_f32_kernel<64>), dim3((int)blocks), dim3(256), 0, stream, dp, pt); break;
      case 128: hipLaunchKernelGGL((prefill_f32_kernel<128>), dim3((int)blocks), dim3(256), 0, stream, dp, pt); break;
      case 256: hipLaunchKernelGGL((prefill_f32_kernel<256>), dim3((int)blocks), dim3(256), 0, stream, dp, pt); break;
      default: return MI_ERR_UNSUPPORTED;
    }
    if (!captured) return MI_OK;
  }
  const int64_t grid = (int64_t)max_tiles * dp.num_kv_heads * (tile_rows / kRows);
  if (grid <= 0) return MI_OK;
  if (grid > 0x7fffffff) return MI_ERR_UNSUPPORTED;
  return dispatch_f32<true>(dp, other, head_dim, (int)grid, stream);
}

}  // namespace mi
