// Internal interfaces shared between the decode and prefill translation units.
#pragma once

#include "mi_common.h"

namespace mi {

// Compute units of the current device (cached per device).
inline int device_cu_count() {
  static int cached[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (!cached[dev]) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    cached[dev] = n;
  }
  return cached[dev];
}

// Memory a kernel may touch: HIP device memory, or host memory that HIP
// allocated pinned (reachable over the bus at the same address).  Pageable
// host memory is not.
inline bool device_reachable(const void* ptr) {
  hipPointerAttribute_t a;
  if (hipPointerGetAttributes(&a, ptr) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return a.type == hipMemoryTypeDevice || a.type == hipMemoryTypeHost || a.type == hipMemoryTypeManaged;
}

// Workspace layout of a split-KV plan (decode kernel + merge).
struct SplitLayout {
  int64_t hdr, chunk_indptr, work, lse, opart, total;
  int32_t max_chunks;
};
// ws_avail: bytes the caller's workspace offers from the layout's start (-1:
// unbounded, giving the recommended size); the chunk budget shrinks to fit.
// pair: the plan is for paired kv-heads (see pair_heads); it only sets the
// chunk target, the buffers are sized for nkv heads of head_dim either way.
SplitLayout split_layout(int32_t batch, int32_t nkv, int32_t head_dim, int64_t ws_avail, bool pair = false);

// Decode over head_dim 128 with at most 8 query heads per kv-head reads two
// adjacent kv-heads as one 256-element row (512 contiguous bytes of a token
// row instead of 256): each query row takes the 128 elements of its own head
// and zeros in the other half, the score MFMAs accumulate the two halves in
// separate registers and each row keeps its own head's (so its scores see
// only its head, non-finite keys of the other head included), and it keeps
// only its half of the output.  Decided from the call's shapes alone, so a
// plan and the run that consumes it agree; decode calls only (no qo_indptr),
// and batches of at least kPairMinBatch requests, whose items are long enough
// for the one-workgroup-per-CU head_dim 256 kernel (c3, B=256: 542 -> 515 us;
// c2, B=64, min-chunk items: 57 -> 60 us).  The run uses the paired kernel
// for 16-bit caches only (fp8 pairs are 256-byte rows: c5 400 -> 410 us).
// A ragged batch (qo_indptr given) pairs only on the prefill path (`ragged`),
// where a request that does not fit a paired row block has somewhere else to
// go: there the short-query threshold halves (pair_short_rows) and the MFMA
// tiles take the requests between the two thresholds.
constexpr int32_t kPairMinBatch = 128;
inline bool pair_heads(const int32_t* qo_indptr, int32_t batch, int32_t num_kv_heads, int32_t group,
                       int32_t head_dim, bool ragged = false) {
  return (!qo_indptr || ragged) && batch >= kPairMinBatch && head_dim == 128 && num_kv_heads % 2 == 0 &&
         group >= 1 && 2 * group <= 16;
}
// Short-query requests of a ragged batch (qo_len * group <= this many rows)
// run on the split-KV decode kernels, longer ones on the MFMA prefill tiles.
// 16 rows (one MFMA column block); 8 for a paired plan, whose column block
// holds a request's rows of both heads of a pair.
constexpr int32_t kShortRowsMax = 16;
inline int32_t pair_short_rows(bool pair) { return pair ? kShortRowsMax / 2 : kShortRowsMax; }

int decode_plan_impl(const int32_t* qo_indptr, const int32_t* kv_indptr, const int32_t* kv_indices,
                     const int32_t* last_page_len, int32_t batch, int32_t page_size,
                     int32_t num_qo_heads, int32_t num_kv_heads, int32_t head_dim,
                     int64_t* kv_locations, void* workspace, int64_t workspace_bytes,
                     int64_t ws_offset, hipStream_t stream);

// Checks the arguments and fills the plan kernel's parameters (no launch).
struct PlanParams;
int decode_plan_params(const int32_t* qo_indptr, const int32_t* kv_indptr, const int32_t* kv_indices,
                       const int32_t* last_page_len, int32_t batch, int32_t page_size,
                       int32_t num_qo_heads, int32_t num_kv_heads, int32_t head_dim,
                       int64_t* kv_locations, void* workspace, int64_t workspace_bytes,
                       int64_t ws_offset, PlanParams* out, bool ragged_pair = false);

// Index arrays of a plan call as a kernel argument (mi_decode_plan_host,
// mi_prefill_plan_host): one after the other, and where the device copies go.
constexpr int kHostParts = 4;
struct HostIndices {
  int32_t v[MI_PLAN_HOST_ARGS];
  int32_t end[kHostParts];  // part k is v[end[k - 1], end[k])
  int32_t* dst[kHostParts];
};
// Fills one; MI_ERR_UNSUPPORTED when the parts do not fit.
inline int host_indices(const int32_t* const* src, const int32_t* len, int32_t* const* dst, int parts, HostIndices* out) {
  int64_t at = 0;
  for (int k = 0; k < kHostParts; ++k) {
    const int32_t n = k < parts ? len[k] : 0;
    if (n < 0 || (n > 0 && (!src[k] || !dst[k]))) return MI_ERR_INVALID;
    if (at + n > MI_PLAN_HOST_ARGS) return MI_ERR_UNSUPPORTED;
    for (int32_t i = 0; i < n; ++i) out->v[at + i] = src[k][i];
    at += n;
    out->end[k] = (int32_t)at;
    out->dst[k] = k < parts ? dst[k] : nullptr;
  }
  return MI_OK;
}
// The workgroup's copy of the argument in LDS, and, by one workgroup of the
// launch (write), the device arrays.
__device__ __forceinline__ void host_indices_copy(const HostIndices& m, int32_t* s_idx, bool write) {
  const int total = m.end[kHostParts - 1];
  for (int i = (int)threadIdx.x; i < total; i += (int)blockDim.x) {
    const int32_t v = m.v[i];
    s_idx[i] = v;
    if (write) {
      int first = 0;
      int32_t* d = m.dst[0];
#pragma unroll
      for (int k = 1; k < kHostParts; ++k)
        if (i >= m.end[k - 1]) {
          first = m.end[k - 1];
          d = m.dst[k];
        }
      d[i - first] = v;
    }
  }
  __syncthreads();
}

enum : int { kPhaseAttend = 1, kPhaseMerge = 2 };

// The attention kernels move q / out rows and KV rows in 16-byte pieces: a
// tensor qualifies when its base is 16-byte aligned and each element stride
// spans a whole number of 16-byte pieces.
inline bool rows_aligned16(const void* base, int64_t stride_a, int64_t stride_b, int elem_bytes) {
  return ((uintptr_t)base & 15) == 0 && (stride_a * elem_bytes) % 16 == 0 && (stride_b * elem_bytes) % 16 == 0;
}
inline bool kv_aligned16(const mi_paged_kv* kv) {
  const int esz = kv->dtype == MI_FP8_E4M3 ? 1 : kv->dtype == MI_F32 ? 4 : 2;
  return rows_aligned16(kv->data, kv->page_stride, kv->kv_stride, esz) &&
         rows_aligned16(kv->data, kv->token_stride, kv->head_stride, esz);
}

// Arguments of the split-KV decode kernels (decode, merge, and their fp32
// variants): q/out rows, the KV layer, the packed batch and the plan in the
// workspace.
struct DecodeParams {
  const void* q;
  int64_t q_stride_tok, q_stride_head;
  const void* kv;
  int64_t page_stride, kv_stride, token_stride, head_stride;
  const float* k_scale;
  const float* v_scale;
  const int32_t* qo_indptr;
  const int32_t* kv_indptr;
  const int32_t* kv_indices;
  const int32_t* last_page_len;
  const int32_t* hdr;
  const int4* work;
  const int32_t* chunk_indptr;
  float* lse_part;
  float* o_part;
  void* out;
  int64_t out_stride_tok, out_stride_head;
  int32_t num_kv_heads, group, page_size, causal;
  float scale_log2;
  int32_t short_rows = kShortRowsMax;  // ragged batches: requests with qo_len * group above this are not ours
};

// fp32 KV (q, cache and output in fp32): the attend phase of a split-KV plan
// (mi_f32.hip), and the merge with fp32 output (mi_decode.hip).
int f32_attend_launch(const DecodeParams& dp, int head_dim, int grid, hipStream_t stream);
int merge_launch(const DecodeParams& dp, int head_dim, int out_dtype, int batch, hipStream_t stream);
// fp32 ragged prefill over the prefill plan's tile list, one workgroup per
// (tile, kv-head, block of 16 or 64 rows); rows: the most (token, q-head) rows
// the batch can have.
int f32_prefill_launch(const DecodeParams& dp, const int32_t* tile_hdr, const int2* tiles, int max_tiles,
                       int tile_rows, int64_t rows, int head_dim, hipStream_t stream);

int decode_run_impl(const void* q, int32_t q_dtype, int64_t q_stride_token, int64_t q_stride_head,
                    const mi_paged_kv* kv, const int32_t* qo_indptr, const int32_t* kv_indptr,
                    const int32_t* kv_indices, const int32_t* last_page_len, int32_t batch,
                    int32_t num_qo_heads, int32_t causal, float sm_scale, void* workspace,
                    int64_t workspace_bytes, int64_t ws_offset, void* out,
                    int64_t out_stride_token, int64_t out_stride_head, int phases, hipStream_t stream,
                    bool ragged_pair = false, DecodeParams* merge_args = nullptr);

// Wavefront scans and reductions on the VALU's cross-lane paths: one row_shr
// per power of two within a 16-lane row, then two row broadcasts.  (__shfl
// goes through the LDS crossbar with address arithmetic around it; a plan
// workgroup runs four wavefronts per SIMD, so every instruction of its scans
// costs 16 cycles.)
template <int CTRL, int ROWS>
__device__ __forceinline__ int dpp_move(int old, int x) {
  return __builtin_amdgcn_update_dpp(old, x, CTRL, ROWS, 0xf, false);
}
__device__ __forceinline__ int wave_inclusive_sum(int x) {
  x += dpp_move<0x111, 0xf>(0, x);  // row_shr:1, 2, 4, 8
  x += dpp_move<0x112, 0xf>(0, x);
  x += dpp_move<0x114, 0xf>(0, x);
  x += dpp_move<0x118, 0xf>(0, x);
  x += dpp_move<0x142, 0xa>(0, x);  // row_bcast:15 into rows 1 and 3
  x += dpp_move<0x143, 0xc>(0, x);  // row_bcast:31 into rows 2 and 3
  return x;
}
__device__ __forceinline__ int wave_sum(int x) { return __builtin_amdgcn_readlane(wave_inclusive_sum(x), 63); }
__device__ __forceinline__ int wave_max(int x) {
  constexpr int kMin = -0x7fffffff - 1;
  x = max(x, dpp_move<0x111, 0xf>(kMin, x));
  x = max(x, dpp_move<0x112, 0xf>(kMin, x));
  x = max(x, dpp_move<0x114, 0xf>(kMin, x));
  x = max(x, dpp_move<0x118, 0xf>(kMin, x));
  x = max(x, dpp_move<0x142, 0xa>(kMin, x));
  x = max(x, dpp_move<0x143, 0xc>(kMin, x));
  return __builtin_amdgcn_readlane(x, 63);
}

// Exclusive prefix sum over a 1024-thread block; `smem` holds >= 16 ints.
__device__ __forceinline__ int block_exclusive_scan_1024(int v, int& total, int* smem) {
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int x = wave_inclusive_sum(v);
  if (lane == 63) smem[w] = x;
  __syncthreads();
  const int t = wave_inclusive_sum(lane < 16 ? smem[lane] : 0);  // every wavefront scans the 16 sums
  total = __builtin_amdgcn_readlane(t, 15);
  const int before = w ? __builtin_amdgcn_readlane(t, w - 1) : 0;
  __syncthreads();
  return before + x - v;
}

// Sum and max of v over a 1024-thread workgroup, returned to every thread
// (smem: 16 ints, free again on return).
__device__ __forceinline__ int block_sum_1024(int v, int* smem) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  v = wave_sum(v);
  if (lane == 0) smem[w] = v;
  __syncthreads();
  const int t = wave_sum(lane < 16 ? smem[lane] : 0);
  __syncthreads();
  return t;
}

// The max of v and, in sum, the sum of sum (smem: 32 ints).
__device__ __forceinline__ int block_max_sum_1024(int v, int& sum, int* smem) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  v = wave_max(v);
  sum = wave_sum(sum);
  if (lane == 0) {
    smem[w] = v;
    smem[16 + w] = sum;
  }
  __syncthreads();
  const int t = wave_max(smem[lane & 15]);
  sum = wave_sum(lane < 16 ? smem[16 + lane] : 0);
  __syncthreads();
  return t;
}

__device__ __forceinline__ int block_max_1024(int v, int* smem) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  v = wave_max(v);
  if (lane == 0) smem[w] = v;
  __syncthreads();
  const int t = wave_max(smem[lane & 15]);
  __syncthreads();
  return t;
}

}  // namespace mi
