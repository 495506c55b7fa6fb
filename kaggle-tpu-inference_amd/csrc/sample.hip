// Top-k / nucleus sampling of one logits row on the device (model.py:414-424).
//
// The reference: greedy = argmax(logits) (first index of the maximum) when
// temperature <= 0; otherwise v = logits / max(T, 1e-6), keep the top_k
// largest v (jax.lax.top_k: descending, ties to the lower index), p =
// softmax(v), keep entries whose exclusive prefix sum (csum - p) < top_p,
// renormalise and draw one.
//
// Candidates are ranked by a 64-bit key: the order-preserving bits of v in
// the high word and the complement of the index in the low word, so "larger
// key" means "larger value, then lower index", exactly top_k's order, and all
// keys are distinct.  Two launches: group_max_kernel writes the largest key of
// each of at most 1,024 groups of the row; sample_pick_kernel (one block) takes
// the 64 groups with the largest maxima, reads those groups again and sorts the
// keys that reach the smallest of the 64 maxima (at least 64 do, typically
// under 100), then draws.  What bounds it is latency: two launches and, in the
// second, two memory round trips and the sort.  A sort of 64 keys per wave and
// a tree of merges of the 64 largest need no barrier inside a list.  At 262,144
// logits 86 -> 18 us (before: three launches of 1,024-key bitonic sorts in
// LDS, 55 barriers each, and the softmax, cut and draw on one lane).  The
// softmax's exps and divisions run one entry per lane; its sums stay in the
// order of the entries.  The uniform comes from
// Philox4x32-10 under the caller's 64-bit seed at counter (step, 0x53414D50,
// 0, 0), where step is the decode position (the reference folds the position
// into its key, engine.py:80) or 0 for the sample after a prefill
// (engine.py:66).  The stream is this library's own, not JAX's.
//
// Like the greedy argmax kernel, the second kernel writes the token and, when
// `pos` is given, advances the device position and records the token in the
// history, so a captured decode step needs no host round trip.
#include "capi_util.h"
#include "common.h"
#include "philox.h"

namespace g4mi {

constexpr int kSortN = 1024;   // keys sorted per block of topk_stage_kernel; groups of a row at most
constexpr int kKeep = 64;      // keys that are kept (>= top_k)
constexpr uint32_t kSampleTag = 0x53414D50u;

struct SampleParams {
  float temperature;
  float top_p;
  uint64_t seed;
};

__device__ __forceinline__ uint32_t ord_bits(float v) {
  const uint32_t b = __float_as_uint(v);
  return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
__device__ __forceinline__ float from_ord(uint32_t o) {
  return __uint_as_float((o & 0x80000000u) ? (o & 0x7FFFFFFFu) : ~o);
}
__device__ __forceinline__ uint64_t make_key(float v, int i) {
  if (v != v) return 0ull;  // NaN ranks last
  return ((uint64_t)ord_bits(v) << 32) | (uint64_t)(0xFFFFFFFFu - (uint32_t)i);
}
__device__ __forceinline__ int key_index(uint64_t k) { return (int)(0xFFFFFFFFu - (uint32_t)k); }
__device__ __forceinline__ float key_value(uint64_t k) { return from_ord((uint32_t)(k >> 32)); }

// Descending bitonic sort of kSortN keys in LDS by 256 threads.
__device__ __forceinline__ void sort_desc(uint64_t* s) {
  for (int k = 2; k <= kSortN; k <<= 1) {
    for (int j = k >> 1; j > 0; j >>= 1) {
#pragma unroll
      for (int h = 0; h < kSortN / 2 / 256; ++h) {
        const int q = threadIdx.x + 256 * h;        // pair index
        const int i = 2 * j * (q / j) + (q % j);    // lower element of the pair
        const int l = i + j;
        const uint64_t a = s[i], b = s[l];
        const bool desc = (i & k) == 0;
        if (desc ? (a < b) : (a > b)) {
          s[i] = b;
          s[l] = a;
        }
      }
      __syncthreads();
    }
  }
}

// One reduction stage: block b sorts keys [b*1024, (b+1)*1024) and writes its
// 64 largest to out[b*64 ..].  FROM_LOGITS: the keys are built from logits / t.
template <bool FROM_LOGITS>
__global__ __launch_bounds__(256) void topk_stage_kernel(const float* __restrict__ logits,
                                                         const uint64_t* __restrict__ in, int n,
                                                         const SampleParams* __restrict__ prm,
                                                         uint64_t* __restrict__ out) {
  __shared__ uint64_t s[kSortN];
  const int base = blockIdx.x * kSortN;
  // greedy (temperature <= 0) ranks the raw logits: dividing by 1e-6 could
  // merge neighbouring floats and move the first-index argmax
  const float T = FROM_LOGITS ? prm->temperature : 0.0f;
  const float t = (T > 0.0f) ? fmaxf(T, 1e-6f) : 1.0f;
#pragma unroll
  for (int h = 0; h < kSortN / 256; ++h) {
    const int j = threadIdx.x + 256 * h;
    const int i = base + j;
    uint64_t key = 0ull;
    if (i < n) {
      if constexpr (FROM_LOGITS) key = make_key(logits[i] / t, i);
      else key = in[i];
    }
    s[j] = key;
  }
  __syncthreads();
  sort_desc(s);
  if (threadIdx.x < kKeep) out[(size_t)blockIdx.x * kKeep + threadIdx.x] = s[threadIdx.x];
}

// The candidates: logits / t (greedy, temperature <= 0, ranks the raw logits:
// dividing by 1e-6 could merge neighbouring floats and move the first-index
// argmax), or keys that topk_stage_kernel left.
template <bool FROM_LOGITS>
struct Candidates {
  const float* logits;
  const uint64_t* keys;
  int n;
  __device__ __forceinline__ uint64_t at(int i, float t) const {
    const int c = min(i, n - 1);  // unconditional load
    uint64_t k;
    if constexpr (FROM_LOGITS) k = make_key(logits[c] / t, i);
    else k = keys[c];
    return i < n ? k : 0ull;
  }
};
__device__ __forceinline__ float sample_divisor(const SampleParams* prm) {
  const float T = prm->temperature;
  return (T > 0.0f) ? fmaxf(T, 1e-6f) : 1.0f;
}
__device__ __forceinline__ uint64_t max_u64(uint64_t a, uint64_t b) { return a > b ? a : b; }
// x of lane l ^ J: DPP moves inside a row of 16 lanes (l ^ 4 and l ^ 8 are two
// mirrors), ds_bpermute across rows
template <int CTRL>
__device__ __forceinline__ int dpp_i(int x) {
  return __builtin_amdgcn_update_dpp(0, x, CTRL, 0xF, 0xF, false);
}
template <int J>
__device__ __forceinline__ int xor_lane(int x) {
  if constexpr (J == 1) return dpp_i<kDppXor1>(x);
  else if constexpr (J == 2) return dpp_i<kDppXor2>(x);
  else if constexpr (J == 4) return dpp_i<kDppHalfMirror>(dpp_i<0x1B>(x));  // 0x1B: quad_perm [3,2,1,0]
  else if constexpr (J == 8) return dpp_i<kDppMirror>(dpp_i<kDppHalfMirror>(x));
  else return __shfl_xor(x, J, kWave);
}
template <int J>
__device__ __forceinline__ uint64_t xor_lane_u64(uint64_t v) {
  return ((uint64_t)(uint32_t)xor_lane<J>((int)(v >> 32)) << 32) | (uint32_t)xor_lane<J>((int)(uint32_t)v);
}

// Groups of a row: wave w holds candidates [w * 256 m, (w + 1) * 256 m), lane l
// those at 64 j + l; 2^ll consecutive lanes of it are one group.  ll and m are
// the smallest that leave at most 1,024 groups (sample_groups), so a group is
// 2^ll * 4 m >= 16 candidates.
struct Groups {
  int ll, m;
};
static Groups sample_groups(int64_t n) {
  Groups g;
  g.ll = n <= 16 * kSortN ? 2 : n <= 64 * kSortN ? 4 : 6;
  g.m = (int)((n + 256 * kSortN - 1) / (256 * kSortN));
  return g;
}

// grid: 4 waves per block; out[group] = the group's largest key
template <bool FROM_LOGITS>
__global__ __launch_bounds__(256) void group_max_kernel(Candidates<FROM_LOGITS> c, Groups g, int ngroups,
                                                        const SampleParams* __restrict__ prm,
                                                        uint64_t* __restrict__ out) {
  const int lane = threadIdx.x & 63, w = blockIdx.x * 4 + wave_id();
  const float t = FROM_LOGITS ? sample_divisor(prm) : 1.0f;
  uint64_t best = 0ull;
  for (int q = 0; q < g.m; ++q) {
    uint64_t k[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) k[j] = c.at(((w * g.m + q) * 4 + j) * 64 + lane, t);
#pragma unroll
    for (int j = 0; j < 4; ++j) best = max_u64(best, k[j]);
  }
  best = max_u64(best, xor_lane_u64<1>(best));
  best = max_u64(best, xor_lane_u64<2>(best));
  if (g.ll >= 4) {
    best = max_u64(best, xor_lane_u64<4>(best));
    best = max_u64(best, xor_lane_u64<8>(best));
  }
  if (g.ll >= 6) {
    best = max_u64(best, xor_lane_u64<16>(best));
    best = max_u64(best, xor_lane_u64<32>(best));
  }
  const int id = (w << (6 - g.ll)) + (lane >> g.ll);
  if ((lane & ((1 << g.ll) - 1)) == 0 && id < ngroups) out[id] = best;
}

// Bitonic networks over the lanes of a wave: descending blocks of KK lanes where
// (lane & KK) == 0, from blocks of KK / 2; J the compare distance.
template <int KK, int J>
__device__ __forceinline__ void bitonic_step(uint64_t& v, int lane) {
  const uint64_t o = xor_lane_u64<J>(v);
  const bool keep_larger = ((lane & J) == 0) == (KK == 64 || (lane & KK) == 0);
  v = keep_larger == (v > o) ? v : o;
  if constexpr (J > 1) bitonic_step<KK, J / 2>(v, lane);
}
__device__ __forceinline__ uint64_t wave_merge_desc(uint64_t v, int lane) {  // v bitonic -> descending
  bitonic_step<64, 32>(v, lane);
  return v;
}
__device__ __forceinline__ uint64_t wave_sort_desc(uint64_t v, int lane) {
  bitonic_step<2, 1>(v, lane);
  bitonic_step<4, 2>(v, lane);
  bitonic_step<8, 4>(v, lane);
  bitonic_step<16, 8>(v, lane);
  bitonic_step<32, 16>(v, lane);
  return wave_merge_desc(v, lane);
}

// The 64 largest of the block's keys (one per thread, in the first nl waves;
// nl uniform), descending, in lists[0] and every lane of wave 0; ends with a
// barrier.  lists: nl x 64.
__device__ __forceinline__ uint64_t block_top64(uint64_t v, int nl, uint64_t (*lists)[64]) {
  const int lane = threadIdx.x & 63, w = wave_id();
  if (w < nl) {
    v = wave_sort_desc(v, lane);
    lists[w][lane] = v;
  }
  for (int s = 1; s < nl; s <<= 1) {
    __syncthreads();
    if (w % (2 * s) == 0 && w + s < nl) {  // the 64 largest of two descending lists are bitonic
      v = wave_merge_desc(max_u64(v, lists[w + s][63 - lane]), lane);
      lists[w][lane] = v;
    }
  }
  __syncthreads();
  return v;
}

__device__ __forceinline__ float lane_f(float v, int i) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), i));
}

// One block: the 64 largest candidates, then the token (see the top of the file).
constexpr int kPickThreads = 1024;
constexpr int kPickList = 6 * kPickThreads;  // keys that wait for a sort
template <bool FROM_LOGITS>
__global__ __launch_bounds__(kPickThreads) void sample_pick_kernel(Candidates<FROM_LOGITS> c, Groups gr, int ngroups,
                                                                   const uint64_t* __restrict__ gmax, int top_k,
                                                                   int V, const SampleParams* __restrict__ prm,
                                                                   int counter_mode, int32_t* __restrict__ tok,
                                                                   int32_t* __restrict__ pos,
                                                                   int32_t* __restrict__ hist, int hist_len) {
  __shared__ uint64_t lists[kPickThreads / 64 + 1][64];
  __shared__ uint64_t list[kPickList];
  __shared__ int gid[kKeep];
  __shared__ int ng, cnt;
  const int tid = threadIdx.x, lane = tid & 63, w = wave_id();
  const float t = FROM_LOGITS ? sample_divisor(prm) : 1.0f;
  const uint64_t gk = tid < ngroups ? gmax[tid] : 0ull;
  if (tid == 0) ng = cnt = 0;
  block_top64(gk, (ngroups + 63) / 64, lists);
  // a group takes part when its maximum is among the 64 largest (all nonzero
  // ones when there are fewer); so does every key that is at least the smallest
  // of those maxima (NaN has key 0 and never does)
  const uint64_t least = max_u64(lists[0][63], 1ull);
  if (gk >= least) gid[atomicAdd(&ng, 1)] = tid;
  __syncthreads();
  const int lg = gr.ll + 2, total = (ng << lg) * gr.m;  // a group: gr.m runs of 2^lg
  uint64_t top = 0ull;  // wave 0: the 64 largest so far, descending
  bool any = false;
  // the first nk keys of the list into `top`
  auto sort_list = [&](int nk) {
    for (int b = 0; b < nk; b += kPickThreads - 64) {  // 15 lists of new keys and, as list 15, the old ones
      const int left = min(nk - b, kPickThreads - 64), nl = (left + 63) / 64;
      uint64_t v = tid < left ? list[b + tid] : 0ull;
      if (any && w == nl) v = lists[kPickThreads / 64][lane];
      top = block_top64(v, nl + (any ? 1 : 0), lists);
      any = true;
      if (w == 0) lists[kPickThreads / 64][lane] = top;
      __syncthreads();
    }
  };
  for (int e0 = 0; e0 < total; e0 += 4 * kPickThreads) {
    uint64_t k[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int e = e0 + u * kPickThreads + tid, ec = min(e, total - 1);
      const int run = ec >> lg, q = gr.m == 1 ? run : run / gr.m;  // group q of gid, its run run - q m
      const int g = gid[q], o = ec & ((1 << lg) - 1), gw = 6 - gr.ll;
      const int i = ((g >> gw) * gr.m + (run - q * gr.m)) * 256 + ((o >> gr.ll) << 6) +
                    ((g & ((1 << gw) - 1)) << gr.ll) + (o & ((1 << gr.ll) - 1));
      k[u] = e < total ? c.at(i, t) : 0ull;
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (k[u] >= least) list[atomicAdd(&cnt, 1)] = k[u];
    __syncthreads();
    const int have = cnt;
    __syncthreads();  // (the next round's keys come after every thread has read the count)
    if (have > kPickList - 4 * kPickThreads) {  // the next round might not fit (uniform)
      sort_list(have);
      if (tid == 0) cnt = 0;
      __syncthreads();
    }
  }
  sort_list(cnt);
  if (w != 0) return;

  // ---- wave 0: lane i holds the i-th largest candidate
  const SampleParams P = *prm;
  const int K = min(top_k, min(c.n, V));
  int choice = key_index(__shfl(top, 0, kWave));  // greedy: the largest logit, lowest index on ties
  if (P.temperature > 0.0f && K > 1) {
    // entries from K on are 0: they change no sum
    const float val = key_value(top);
    float p = lane < K ? expf(val - lane_f(val, 0)) : 0.0f;
    float z = 0.0f;
#pragma unroll
    for (int i = 0; i < kKeep; ++i) z += lane_f(p, i);
    p = lane < K ? p / z : 0.0f;
    float csum = 0.0f, kept = 0.0f;
    float cut = 0.0f, upto = 0.0f;  // this lane's p after the nucleus cut on the exclusive prefix sum, and their sum so far
#pragma unroll
    for (int i = 0; i < kKeep; ++i) {
      float pi = lane_f(p, i);
      csum += pi;
      if (!(csum - pi < P.top_p)) pi = 0.0f;
      kept += pi;
      cut = lane == i ? pi : cut;
      upto = lane == i ? kept : upto;
    }
    const int p0 = (pos != nullptr) ? pos[0] : 0;
    const uint32_t step = counter_mode ? (uint32_t)p0 : 0u;
    const Philox4 r = philox4x32_10(step, kSampleTag, 0u, 0u, (uint32_t)P.seed, (uint32_t)(P.seed >> 32));
    const float u = (float)(r.v[0] >> 8) * (1.0f / 16777216.0f);  // [0, 1)
    const float target = u * kept;
    // the first kept entry whose sum passes the target, else the last kept one
    const unsigned long long some = __ballot(cut > 0.0f), past = __ballot(cut > 0.0f && upto > target);
    const int last = past != 0ull ? (int)__builtin_ctzll(past) : some != 0ull ? 63 - (int)__builtin_clzll(some) : 0;
    choice = key_index(__shfl(top, last, kWave));
  }
  if (lane != 0) return;
  tok[0] = choice;
  if (pos != nullptr) {
    const int np = pos[0] + 1;
    pos[0] = np;
    if (hist != nullptr && np >= 0 && np < hist_len) hist[np] = choice;
  }
}

// Rows above this many candidates are first reduced by topk_stage_kernel (16 to
// 1): one block would read too much of them (64 groups of n / 1,024 candidates).
constexpr int64_t kPickMax = (int64_t)1 << 22;

template <bool FROM_LOGITS>
static void launch_pick(const Candidates<FROM_LOGITS>& c, uint64_t* gmax, int64_t V, int64_t top_k,
                        const SampleParams* prm, int counter_mode, int32_t* tok, int32_t* pos, int32_t* hist,
                        int hist_len, hipStream_t st) {
  const Groups g = sample_groups(c.n);
  const int64_t waves = ((int64_t)c.n + 256 * g.m - 1) / (256 * g.m), all = waves << (6 - g.ll);  // groups, <= kSortN
  hipLaunchKernelGGL((group_max_kernel<FROM_LOGITS>), dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, st, c, g,
                     (int)all, prm, gmax);
  hipLaunchKernelGGL((sample_pick_kernel<FROM_LOGITS>), dim3(1), dim3(kPickThreads), 0, st, c, g, (int)all, gmax,
                     (int)top_k, (int)V, prm, counter_mode, tok, pos, hist, hist_len);
}

static int64_t stage_keys(int64_t n) { return ((n + kSortN - 1) / kSortN) * kKeep; }

}  // namespace g4mi

using namespace g4mi;

// ------------------------------------------------------------------ batched head
// Rows b of bf16 logits [B, V] (x . embed^T rounded to bf16, model.py:381):
// v = f32 logit, softcap c*tanh(v/c) when c > 0 (model.py:382-385), optional
// f32 copy, then the first index of the maximum (model.py:416 greedy).  Stage
// 1: grid (kArgParts, B), each block the best (value, index) of its slice of
// the row; stage 2: one block per row reduces the slices and writes tok[b] =
// it; pos[b] += 1; hist[b][pos[b]] = it.
constexpr int kArgParts = 64;

__device__ __forceinline__ void better_vi(float& bv, int& bi, float v, int i) {
  if (v > bv || (v == bv && i < bi)) {
    bv = v;
    bi = i;
  }
}

__global__ __launch_bounds__(256) void argmax_rows_part_kernel(const uint16_t* __restrict__ logits, int V, float cap,
                                                               float* __restrict__ out_f32, float* __restrict__ pv,
                                                               int* __restrict__ pi) {
  __shared__ float vs[4];
  __shared__ int is[4];
  const int part = blockIdx.x, b = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int span = (V + kArgParts - 1) / kArgParts;
  const int j0 = part * span, j1 = min(V, j0 + span);
  const uint16_t* row = logits + (size_t)b * V;
  float bv = -INFINITY;
  int bi = 0x7fffffff;
  for (int j = j0 + tid; j < j1; j += 256) {
    float v = bf2f(row[j]);
    if (cap > 0.0f) v = tanhf(v / cap) * cap;
    if (out_f32 != nullptr) out_f32[(size_t)b * V + j] = v;
    better_vi(bv, bi, v, j);
  }
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) better_vi(bv, bi, __shfl_xor(bv, m, kWave), __shfl_xor(bi, m, kWave));
  if (lane == 0) {
    vs[wave] = bv;
    is[wave] = bi;
  }
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w < 4; ++w) better_vi(bv, bi, vs[w], is[w]);
    pv[b * kArgParts + part] = bv;
    pi[b * kArgParts + part] = bi;
  }
}

__global__ __launch_bounds__(64) void argmax_rows_final_kernel(const float* __restrict__ pv, const int* __restrict__ pi,
                                                               int32_t* tok, int32_t* pos, int32_t* hist,
                                                               int hist_len) {
  const int b = blockIdx.x, lane = threadIdx.x;
  float bv = pv[b * kArgParts + lane];
  int bi = pi[b * kArgParts + lane];
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) better_vi(bv, bi, __shfl_xor(bv, m, kWave), __shfl_xor(bi, m, kWave));
  if (lane == 0) {
    bi = (bi == 0x7fffffff) ? 0 : bi;
    tok[b] = bi;
    if (pos != nullptr) {
      const int p = pos[b] + 1;
      pos[b] = p;
      if (hist != nullptr && p >= 0 && p < hist_len) hist[(size_t)b * hist_len + p] = bi;
    }
  }
}

extern "C" {

int64_t g4mi_argmax_rows_workspace_bytes(int64_t B) { return B * kArgParts * 8; }

int g4mi_argmax_rows(const uint16_t* logits, int64_t B, int64_t V, float softcap, float* logits_f32, int32_t* tok,
                     int32_t* pos, int32_t* hist, int64_t hist_len, void* ws, int64_t ws_bytes, void* stream) {
  G4MI_REQUIRE(logits && tok && B >= 1 && B <= 65535 && V >= 1 && V <= 2147483647, G4MI_EINVAL,
               "argmax_rows: bad arguments (B=%lld V=%lld)", (long long)B, (long long)V);
  G4MI_REQUIRE(hist == nullptr || (pos && hist_len >= 1), G4MI_EINVAL, "argmax_rows: hist needs pos and hist_len");
  G4MI_REQUIRE(ws && ws_bytes >= g4mi_argmax_rows_workspace_bytes(B), G4MI_EWORKSPACE,
               "argmax_rows: workspace too small");
  float* pv = (float*)ws;
  int* pi = (int*)((char*)ws + B * kArgParts * 4);
  hipStream_t st = as_stream(stream);
  hipLaunchKernelGGL(argmax_rows_part_kernel, dim3(kArgParts, (unsigned)B), dim3(256), 0, st, logits, (int)V,
                     softcap, logits_f32, pv, pi);
  int rc = check_launch("argmax_rows (slices)");
  if (rc) return rc;
  hipLaunchKernelGGL(argmax_rows_final_kernel, dim3((unsigned)B), dim3(64), 0, st, pv, pi, tok, pos, hist,
                     (int)hist_len);
  return check_launch("argmax_rows");
}


int64_t g4mi_sample_workspace_bytes(int64_t V) {
  const int64_t a = stage_keys(V);
  return 2 * ((a * 8 + 255) / 256) * 256;
}

int g4mi_sample(const float* logits, int64_t V, int64_t top_k, const void* params, int32_t counter_mode,
                int32_t* tok, int32_t* pos, int32_t* hist, int64_t hist_len, void* ws, int64_t ws_bytes,
                void* stream) {
  G4MI_REQUIRE(logits && params && tok && ws, G4MI_EINVAL, "sample: null pointer argument");
  G4MI_REQUIRE(V >= 1 && V <= ((int64_t)1 << 30), G4MI_EINVAL, "sample: bad vocab %lld", (long long)V);
  G4MI_REQUIRE(top_k >= 1 && top_k <= kKeep, G4MI_EUNSUPPORTED, "sample: top_k %lld not in [1, %d]",
               (long long)top_k, kKeep);
  G4MI_REQUIRE(ws_bytes >= g4mi_sample_workspace_bytes(V), G4MI_EWORKSPACE, "sample: workspace too small");
  G4MI_REQUIRE(((uintptr_t)params & 7u) == 0 && ((uintptr_t)ws & 7u) == 0, G4MI_EALIGN,
               "sample: params and workspace must be 8-byte aligned");
  hipStream_t st = as_stream(stream);
  const SampleParams* prm = (const SampleParams*)params;
  uint64_t* buf[2];
  buf[0] = (uint64_t*)ws;
  buf[1] = (uint64_t*)((char*)ws + g4mi_sample_workspace_bytes(V) / 2);
  if (V <= kPickMax) {
    launch_pick(Candidates<true>{logits, nullptr, (int)V}, buf[0], V, top_k, prm, counter_mode, tok, pos, hist,
                (int)hist_len, st);
    return check_launch("sample");
  }
  int64_t n = V;
  int cur = 0;
  bool from_logits = true;
  while (n > kPickMax) {
    const int64_t blocks = (n + kSortN - 1) / kSortN;
    if (from_logits)
      hipLaunchKernelGGL((topk_stage_kernel<true>), dim3((unsigned)blocks), dim3(256), 0, st, logits, nullptr,
                         (int)n, prm, buf[cur]);
    else
      hipLaunchKernelGGL((topk_stage_kernel<false>), dim3((unsigned)blocks), dim3(256), 0, st, nullptr,
                         buf[cur ^ 1], (int)n, prm, buf[cur]);
    n = blocks * kKeep;
    cur ^= 1;
    from_logits = false;
  }
  launch_pick(Candidates<false>{nullptr, buf[cur ^ 1], (int)n}, buf[cur], V, top_k, prm, counter_mode, tok, pos, hist,
              (int)hist_len, st);
  return check_launch("sample");
}

}  // extern "C"
