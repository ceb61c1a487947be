// Small device-side bookkeeping kernels.
#include "common.h"

namespace dsk {

__global__ void lens_add_kernel(int32_t* __restrict__ lens, const int32_t* __restrict__ n, int B, int add) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b < B) lens[b] += (n ? n[b] : 0) + add;
}

// one workgroup per logits row; the row's CSR entries are applied in order by one lane each
// (ids within a row are distinct, so there are no write conflicts)
__global__ void penalize_kernel(float* __restrict__ logits, int64_t ldl, const int32_t* __restrict__ row_ptr,
                                const int32_t* __restrict__ ids, const float* __restrict__ vals) {
  const int r = blockIdx.x;
  for (int j = row_ptr[r] + threadIdx.x; j < row_ptr[r + 1]; j += blockDim.x) logits[(int64_t)r * ldl + ids[j]] -= vals[j];
}

// One workgroup per row: a max / sum-of-exp pass for the log-normaliser, then top_k
// selection passes, each taking the largest entry that ranks below the previous pick in the
// order (value descending, index ascending), so ties resolve to the lowest index.
constexpr int kLpThreads = 1024;

__device__ __forceinline__ bool lp_before(float va, int64_t ia, float vb, int64_t ib) {
  return va > vb || (va == vb && ia < ib);
}

__global__ __launch_bounds__(kLpThreads) void row_logprobs_kernel(const float* __restrict__ logits, int64_t ldl,
                                                                  int64_t V, const int32_t* __restrict__ tokens,
                                                                  int top_k, float* __restrict__ chosen,
                                                                  int32_t* __restrict__ top_ids,
                                                                  float* __restrict__ top_vals) {
  __shared__ float sv[kLpThreads / 64];
  __shared__ int64_t si[kLpThreads / 64];
  const int r = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const float* x = logits + (int64_t)r * ldl;
  float m = -__builtin_inff();
  for (int64_t j = tid; j < V; j += kLpThreads) m = fmaxf(m, x[j]);
  m = wave_max(m);
  if (lane == 0) sv[wv] = m;
  __syncthreads();
  m = -__builtin_inff();
  for (int i = 0; i < kLpThreads / 64; ++i) m = fmaxf(m, sv[i]);
  __syncthreads();
  float se = 0.0f;
  for (int64_t j = tid; j < V; j += kLpThreads) se += expf(x[j] - m);
  se = wave_sum(se);
  if (lane == 0) sv[wv] = se;
  __syncthreads();
  se = 0.0f;
  for (int i = 0; i < kLpThreads / 64; ++i) se += sv[i];
  const float lse = m + logf(se);
  if (tid == 0) {
    int64_t t = tokens[r];
    t = t < 0 ? 0 : (t >= V ? V - 1 : t);
    chosen[r] = x[t] - lse;
  }
  float pv = __builtin_inff();
  int64_t pi = -1;
  for (int k = 0; k < top_k; ++k) {
    float bv = -__builtin_inff();
    int64_t bi = V;
    for (int64_t j = tid; j < V; j += kLpThreads) {
      const float v = x[j];
      if (lp_before(pv, pi, v, j) && lp_before(v, j, bv, bi)) {
        bv = v;
        bi = j;
      }
    }
    for (int o = 32; o > 0; o >>= 1) {
      const float ov = __shfl_xor(bv, o, 64);
      const int64_t oi = __shfl_xor(bi, o, 64);
      if (lp_before(ov, oi, bv, bi)) {
        bv = ov;
        bi = oi;
      }
    }
    __syncthreads();
    if (lane == 0) {
      sv[wv] = bv;
      si[wv] = bi;
    }
    __syncthreads();
    bv = sv[0];
    bi = si[0];
    for (int i = 1; i < kLpThreads / 64; ++i)
      if (lp_before(sv[i], si[i], bv, bi)) {
        bv = sv[i];
        bi = si[i];
      }
    if (tid == 0) {
      top_ids[(int64_t)r * top_k + k] = (int32_t)(bi < V ? bi : 0);
      top_vals[(int64_t)r * top_k + k] = bi < V ? bv - lse : -__builtin_inff();
    }
    pv = bv;
    pi = bi;
  }
}

// The same over many workgroups, for callers with scratch (dsk_row_logprobs_ws). One workgroup per
// row is bound by one CU's load rate and runs 2 + top_k passes over the row (16 rows of 151936, five
// alternatives: 185 us a call, back to back). Here a workgroup holds kLpSpan elements of a row in
// registers: one read of the logits, its waves' maxima and sums of exp against their own maximum, and each
// wave's top_k entries in order (each pass over registers). A second kernel, one wave per row, merges the sums and
// the waves' sorted lists: 20.1 us a call on the same rows (in a graph 6.8 without alternatives and 2.6 for
// each, picked one after the other; the host's part of a call takes about as long as the five).
constexpr int kLpBlock = 256;
constexpr int kLpEpt = 16;                          // elements per thread
constexpr int kLpSpan = kLpBlock * kLpEpt;          // elements per workgroup
constexpr int kLpWaves = kLpBlock / 64;
constexpr int64_t kLpMaxV = 1 << 19;                // at most 128 workgroups, 512 lists per row
constexpr int kLpMaxLists = (int)(kLpMaxV / kLpSpan) * kLpWaves;

// wave-wide first of (v, i) in the order of lp_before; every lane ends with it
__device__ __forceinline__ void lp_wave_first(float& v, int& i) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const float ov = __shfl_xor(v, o, 64);
    const int oi = __shfl_xor(i, o, 64);
    if (lp_before(ov, oi, v, i)) {
      v = ov;
      i = oi;
    }
  }
}

struct LpScratch {
  float2* ms;    // [rows][lists]: a list's max and its sum of exp(x - max) (max -inf: sum of exp(x))
  float* val;    // [rows][lists][top_k]: values in order, -inf / index V past the last entry
  int32_t* idx;
};

__global__ __launch_bounds__(kLpBlock) void lp_slices_kernel(const float* __restrict__ logits, int64_t ldl, int V,
                                                             int top_k, LpScratch ws) {
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, r = blockIdx.y;
  const float* x = logits + (int64_t)r * ldl;
  // wave wv of the workgroup holds a contiguous run, so its list's ties resolve by index anyway
  const int j0 = blockIdx.x * kLpSpan + wv * 64 * kLpEpt + lane;
  float v[kLpEpt];
#pragma unroll
  for (int e = 0; e < kLpEpt; ++e) v[e] = x[min(j0 + e * 64, V - 1)];  // past the row: not used below
  float m = -__builtin_inff();
#pragma unroll
  for (int e = 0; e < kLpEpt; ++e)
    if (j0 + e * 64 < V) m = fmaxf(m, v[e]);
  m = wave_max(m);
  const float mb = m == -__builtin_inff() ? 0.0f : m;
  float se = 0.0f;
#pragma unroll
  for (int e = 0; e < kLpEpt; ++e)
    if (j0 + e * 64 < V) se += expf(v[e] - mb);
  se = wave_sum(se);
  const int64_t list = (int64_t)r * (gridDim.x * kLpWaves) + blockIdx.x * kLpWaves + wv;
  if (lane == 0) ws.ms[list] = float2{m, se};
  float pv = __builtin_inff();
  int pi = -1;
  for (int k = 0; k < top_k; ++k) {
    float bv = -__builtin_inff();
    int bi = V;
#pragma unroll
    for (int e = 0; e < kLpEpt; ++e) {
      const int j = j0 + e * 64;
      if (j < V && lp_before(pv, pi, v[e], j) && lp_before(v[e], j, bv, bi)) {
        bv = v[e];
        bi = j;
      }
    }
    lp_wave_first(bv, bi);
    if (lane == 0) {
      ws.val[list * top_k + k] = bv;
      ws.idx[list * top_k + k] = bi;
    }
    pv = bv;
    pi = bi;
    if (bi >= V) {  // nothing left: the rest of the list is empty
      for (int q = k + 1 + lane; q < top_k; q += 64) {
        ws.val[list * top_k + q] = -__builtin_inff();
        ws.idx[list * top_k + q] = V;
      }
      break;
    }
  }
}

__global__ __launch_bounds__(64) void lp_merge_kernel(const float* __restrict__ logits, int64_t ldl, int V, int lists,
                                                      const int32_t* __restrict__ tokens, int top_k,
                                                      float* __restrict__ chosen, int32_t* __restrict__ top_ids,
                                                      float* __restrict__ top_vals, LpScratch ws) {
  constexpr int PER = kLpMaxLists / 64;
  const int lane = threadIdx.x, r = blockIdx.x;
  int64_t t = tokens[r];
  t = t < 0 ? 0 : (t >= V ? V - 1 : t);
  const float xt = logits[(int64_t)r * ldl + t];
  const float2* ms = ws.ms + (int64_t)r * lists;
  float m = -__builtin_inff(), lm[PER], ls[PER];
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const float2 q = ms[min(lane + 64 * u, lists - 1)];
    const bool in = lane + 64 * u < lists;
    lm[u] = in ? q.x : -__builtin_inff();
    ls[u] = in ? q.y : 0.0f;
    m = fmaxf(m, lm[u]);
  }
  m = wave_max(m);
  float se = 0.0f;
#pragma unroll
  for (int u = 0; u < PER; ++u)  // a list of -inf alone adds its sum as it is (0, or NaN)
    se += lm[u] == -__builtin_inff() ? ls[u] : ls[u] * expf(lm[u] - m);
  se = wave_sum(se);
  // a row without a value above -inf has no distribution (exp(-inf - -inf))
  const float lse = m == -__builtin_inff() ? __builtin_nanf("") : m + logf(se);
  if (lane == 0) chosen[r] = xt - lse;
  if (top_k == 0) return;
  // k-way merge: each lane's heads of the lists lane, lane + 64, ... and how far each has got
  const float* val = ws.val + (int64_t)r * lists * top_k;
  const int32_t* idx = ws.idx + (int64_t)r * lists * top_k;
  float hv[PER];
  int hi[PER], at[PER];
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int l = lane + 64 * u;
    const int64_t o = (int64_t)min(l, lists - 1) * top_k;
    hv[u] = val[o];
    hi[u] = idx[o];
    at[u] = 0;
    if (l >= lists) {
      hv[u] = -__builtin_inff();
      hi[u] = V;
    }
  }
  for (int k = 0; k < top_k; ++k) {
    float bv = hv[0];
    int bi = hi[0];
#pragma unroll
    for (int u = 1; u < PER; ++u)
      if (lp_before(hv[u], hi[u], bv, bi)) {
        bv = hv[u];
        bi = hi[u];
      }
    lp_wave_first(bv, bi);
    if (lane == 0) {
      top_ids[(int64_t)r * top_k + k] = bi < V ? bi : 0;
      top_vals[(int64_t)r * top_k + k] = bi < V ? bv - lse : -__builtin_inff();
    }
    if (bi >= V) continue;
#pragma unroll
    for (int u = 0; u < PER; ++u)
      if (hi[u] == bi) {  // this list's head was taken (indices are unique)
        const bool more = ++at[u] < top_k;
        const int64_t o = (int64_t)(lane + 64 * u) * top_k + (more ? at[u] : 0);
        hv[u] = more ? val[o] : -__builtin_inff();
        hi[u] = more ? idx[o] : V;
      }
  }
}

static int lp_lists(int64_t V) { return (int)ceil_div(V, kLpSpan) * kLpWaves; }

// Reads [p, p + n16 * 16) and keeps nothing: the bytes pass through the memory-side cache on
// their way, so a kernel that reads them soon after finds them there. Each thread issues
// kPrefetchLoads 16-byte loads before it uses any (a lane past the end re-reads the last chunk),
// so a workgroup keeps 32 KB in flight. The xor of everything read is stored only if it equals a
// value no real weight image produces in practice, and then into the caller's 16-byte sink, so
// the loads cannot be dropped.
constexpr int kPrefetchLoads = 8;

__global__ __launch_bounds__(256) void prefetch_kernel(const uint4* __restrict__ p, int64_t n16,
                                                       uint4* __restrict__ sink) {
  uint4 acc = {0, 0, 0, 0};
  const int64_t step = (int64_t)gridDim.x * 256 * kPrefetchLoads;
  for (int64_t base = (int64_t)blockIdx.x * 256 * kPrefetchLoads + threadIdx.x; base < n16; base += step) {
    uint4 v[kPrefetchLoads];
#pragma unroll
    for (int u = 0; u < kPrefetchLoads; ++u) v[u] = p[min(base + u * 256, n16 - 1)];
#pragma unroll
    for (int u = 0; u < kPrefetchLoads; ++u) {
      acc.x ^= v[u].x;
      acc.y ^= v[u].y;
      acc.z ^= v[u].z;
      acc.w ^= v[u].w;
    }
  }
  if (acc.x == 0x9e3779b9u && acc.y == 0x7f4a7c15u && acc.z == 0xf39cc060u && acc.w == 0x5ced1a3bu) *sink = acc;
}

}  // namespace dsk

using namespace dsk;

extern "C" int dsk_row_logprobs(const float* logits, int64_t ldl, int R, int64_t V, const int32_t* tokens,
                                int top_k, float* chosen, int32_t* top_ids, float* top_vals, dsk_stream_t stream) {
  DSK_REQUIRE(logits && tokens && chosen && R > 0 && V > 0 && ldl >= V, "dsk_row_logprobs: bad arguments");
  DSK_REQUIRE(top_k >= 0 && top_k <= 64 && (top_k == 0 || (top_ids && top_vals)),
              "dsk_row_logprobs: top_k=%d outside [0, 64] or no output", top_k);
  hipLaunchKernelGGL(row_logprobs_kernel, dim3((unsigned)R), dim3(kLpThreads), 0, as_stream(stream), logits, ldl, V,
                     tokens, top_k, chosen, top_ids, top_vals);
  DSK_LAUNCH_CHECK("dsk_row_logprobs");
  return DSK_OK;
}

extern "C" size_t dsk_row_logprobs_ws_bytes(int R, int64_t V, int top_k) {
  if (R <= 0 || R > 65535 || V <= 0 || V > kLpMaxV || top_k < 0 || top_k > 64) return 0;
  return (size_t)R * lp_lists(V) * (sizeof(float2) + (size_t)top_k * (sizeof(float) + sizeof(int32_t)));
}

extern "C" int dsk_row_logprobs_ws(const float* logits, int64_t ldl, int R, int64_t V, const int32_t* tokens,
                                   int top_k, float* chosen, int32_t* top_ids, float* top_vals, void* workspace,
                                   size_t ws_bytes, dsk_stream_t stream) {
  DSK_REQUIRE(logits && tokens && chosen && R > 0 && V > 0 && ldl >= V, "dsk_row_logprobs_ws: bad arguments");
  DSK_REQUIRE(top_k >= 0 && top_k <= 64 && (top_k == 0 || (top_ids && top_vals)),
              "dsk_row_logprobs_ws: top_k=%d outside [0, 64] or no output", top_k);
  const size_t need = dsk_row_logprobs_ws_bytes(R, V, top_k);
  DSK_REQUIRE(need > 0, "dsk_row_logprobs_ws: R=%d V=%lld outside (65535, %lld)", R, (long long)V, (long long)kLpMaxV);
  DSK_REQUIRE(workspace && ((uintptr_t)workspace & 7) == 0 && ws_bytes >= need,
              "dsk_row_logprobs_ws: workspace %zu < %zu or not 8-byte aligned", ws_bytes, need);
  const int lists = lp_lists(V);
  LpScratch ws;
  ws.ms = reinterpret_cast<float2*>(workspace);
  ws.val = reinterpret_cast<float*>(ws.ms + (size_t)R * lists);
  ws.idx = reinterpret_cast<int32_t*>(ws.val + (size_t)R * lists * top_k);
  hipLaunchKernelGGL(lp_slices_kernel, dim3((unsigned)(lists / kLpWaves), (unsigned)R), dim3(kLpBlock), 0,
                     as_stream(stream), logits, ldl, (int)V, top_k, ws);
  hipLaunchKernelGGL(lp_merge_kernel, dim3((unsigned)R), dim3(64), 0, as_stream(stream), logits, ldl, (int)V, lists,
                     tokens, top_k, chosen, top_ids, top_vals, ws);
  DSK_LAUNCH_CHECK("dsk_row_logprobs_ws");
  return DSK_OK;
}

extern "C" int dsk_logits_penalize(float* logits, int64_t ldl, int R, const int32_t* row_ptr, const int32_t* ids,
                                   const float* vals, dsk_stream_t stream) {
  DSK_REQUIRE(logits && row_ptr && ids && vals && R > 0, "dsk_logits_penalize: bad arguments");
  hipLaunchKernelGGL(penalize_kernel, dim3((unsigned)R), dim3(64), 0, as_stream(stream), logits, ldl, row_ptr, ids,
                     vals);
  DSK_LAUNCH_CHECK("dsk_logits_penalize");
  return DSK_OK;
}

extern "C" int dsk_prefetch(const void* p, size_t bytes, int workgroups, void* sink, dsk_stream_t stream) {
  DSK_REQUIRE(p && sink && workgroups > 0, "dsk_prefetch: bad arguments");
  DSK_REQUIRE(((uintptr_t)p & 15) == 0 && bytes % 16 == 0 && ((uintptr_t)sink & 15) == 0,
              "dsk_prefetch: 16-byte aligned pointers and a multiple of 16 bytes");
  if (bytes == 0) return DSK_OK;
  hipLaunchKernelGGL(prefetch_kernel, dim3((unsigned)workgroups), dim3(256), 0, as_stream(stream),
                     reinterpret_cast<const uint4*>(p), (int64_t)(bytes / 16), reinterpret_cast<uint4*>(sink));
  DSK_LAUNCH_CHECK("dsk_prefetch");
  return DSK_OK;
}

extern "C" int dsk_lens_add(int32_t* lens, const int32_t* n, int B, int add, dsk_stream_t stream) {
  DSK_REQUIRE(lens && B > 0, "dsk_lens_add: bad arguments");
  hipLaunchKernelGGL(lens_add_kernel, dim3((unsigned)ceil_div(B, 256)), dim3(256), 0, as_stream(stream), lens, n,
                     B, add);
  DSK_LAUNCH_CHECK("dsk_lens_add");
  return DSK_OK;
}
