// On-device sampling (InferenceEngine::sample_current_logits,
// src/engine.rs:253-325): repetition penalty and temperature per token, the
// candidates in descending f32::total_cmp order, top-k truncation, softmax,
// the top-p cutoff and the draw, with the uniform number supplied by the
// caller.
//
// Two routes give the same sorted candidates (equal values keep ascending
// token order; the reference's sort_unstable_by leaves it unspecified):
//   - top-k (or greedy) with far fewer candidates than tokens: the keys'
//     kernel also writes the maximum of every group of tokens, and one
//     workgroup takes the m-th largest group maximum as a threshold (at least
//     m tokens reach it), collects the tokens that do and orders them;
//   - otherwise hipCUB's stable radix sort of all (order key, token) pairs.
// The softmax, the top-p cumulative sum and the draw run in one workgroup:
// each thread owns a contiguous slice of the sorted candidates, the slices'
// sums are scanned across the workgroup, and the thread whose slice holds a
// crossing walks it in order.  The sums are the reference's f32 sums in
// another association, so a draw can differ from the reference's only when
// it falls within rounding of a boundary between two candidates.
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <mutex>

#include "common.h"
#include "sampling.h"

namespace llrs {

namespace {

// Monotone map of f32::total_cmp order onto uint32 (and back).
__device__ __forceinline__ uint32_t order_key(float f) {
  const int32_t b = __float_as_int(f);
  return (uint32_t)(b ^ (int32_t)((uint32_t)(b >> 31) >> 1)) ^ 0x80000000u;
}
__device__ __forceinline__ float key_value(uint32_t k) {
  const int32_t b = (int32_t)(k ^ 0x80000000u);
  return __int_as_float(b ^ (int32_t)((uint32_t)(b >> 31) >> 1));
}

constexpr int kKeyBlock = 1024;  // tokens per workgroup of sample_keys_kernel

// The repeat window as a kernel argument (most windows; a copy to the device
// costs a call several microseconds), or on the device when longer.
struct RecentArg {
  const uint32_t *dev;
  int n;
  uint32_t tok[kArgRecent];
};

// src/engine.rs:262-278: the penalty for tokens of the repeat window
// (positive values divided, the others multiplied), then the temperature;
// a non-finite result becomes -inf.  A thread holds four consecutive tokens.
// With idx: the token of every key, for the sort.  With gmax: the largest key
// of every `group` tokens (16, 64, 256 or 1,024).  The window marks its
// tokens in LDS once per workgroup; testing it per token took 7.5 us at 64
// tokens over a 152,064-token vocabulary, this 4.2 us.
__global__ __launch_bounds__(256) void sample_keys_kernel(const float *__restrict__ logits, int n, RecentArg recent,
                                                          float penalty, float temperature,
                                                          uint32_t *__restrict__ keys, uint32_t *__restrict__ idx,
                                                          uint32_t *__restrict__ gmax, int group) {
  __shared__ uint32_t seen[kKeyBlock / 4];  // a byte per token
  __shared__ uint32_t wmax[4];
  const int base = blockIdx.x * kKeyBlock, t0 = base + 4 * (int)threadIdx.x, lane = threadIdx.x & 63;
  uint32_t mine = 0;
  if (penalty != 1.0f) {
    seen[threadIdx.x] = 0;
    __syncthreads();
    for (int i = threadIdx.x; i < recent.n; i += 256) {
      const uint32_t r = (recent.dev ? recent.dev[i] : recent.tok[i]) - (uint32_t)base;
      if (r < (uint32_t)kKeyBlock) reinterpret_cast<uint8_t *>(seen)[r] = 1;
    }
    __syncthreads();
    mine = seen[threadIdx.x];
  }
  uint32_t top = 0;  // below every token's key
#pragma unroll
  for (int e = 0; e < 4; e++) {
    const int t = t0 + e;
    if (t >= n) break;
    float v = logits[t];
    if ((mine >> (8 * e)) & 1) v = v > 0.0f ? v / penalty : v * penalty;
    if (temperature > 0.0f) v /= temperature;
    if (!isfinite(v)) v = -INFINITY;
    const uint32_t k = order_key(v);
    keys[t] = k;
    if (idx) idx[t] = (uint32_t)t;
    top = max(top, k);
  }
  if (!gmax) return;
#pragma unroll
  for (int b = 1; b < 64; b <<= 1) {
    if (4 * b >= group) break;
    top = max(top, (uint32_t)__shfl_xor((int)top, b));
  }
  if (group == kKeyBlock) {
    if (lane == 0) wmax[threadIdx.x >> 6] = top;
    __syncthreads();
    if (threadIdx.x == 0) gmax[blockIdx.x] = max(max(wmax[0], wmax[1]), max(wmax[2], wmax[3]));
  } else if (t0 % group == 0 && t0 < n) {
    gmax[t0 / group] = top;
  }
}

constexpr int kSelectThreads = 1024;

// Inclusive scan of one float per thread (Hillis-Steele in LDS).
__device__ float block_scan(float v, float *sh) {
  const int tid = threadIdx.x;
  sh[tid] = v;
  __syncthreads();
  for (int o = 1; o < kSelectThreads; o <<= 1) {
    const float a = tid >= o ? sh[tid - o] : 0.f;
    __syncthreads();
    sh[tid] += a;
    __syncthreads();
  }
  return sh[tid];
}

// src/engine.rs:286-324 over the sorted candidates.
__global__ __launch_bounds__(kSelectThreads) void sample_select_kernel(
    const uint32_t *__restrict__ keys, const uint32_t *__restrict__ idx, int n, int top_k, float top_p,
    float temperature, float u, uint32_t *__restrict__ out) {
  __shared__ float sh[kSelectThreads];
  __shared__ int cut, pick;
  __shared__ float kept_exp;
  const int tid = threadIdx.x;
  if (temperature <= 0.0f) {  // the first candidate
    if (tid == 0) *out = idx[0];
    return;
  }
  const int m = (top_k > 0 && top_k < n) ? top_k : n;
  const float top = key_value(keys[0]);
  const int per = (m + kSelectThreads - 1) / kSelectThreads;
  const int b = min(m, tid * per), e = min(m, b + per);
  float s = 0.f;
  for (int i = b; i < e; i++) s += expf(key_value(keys[i]) - top);
  const float incl = block_scan(s, sh);
  const float sum = sh[kSelectThreads - 1], before = incl - s;
  if (!isfinite(sum) || sum <= 0.0f) {  // src/engine.rs:299-301
    if (tid == 0) *out = idx[0];
    return;
  }
  if (tid == 0) {
    cut = m;
    pick = m;
  }
  __syncthreads();
  // The top-p cutoff: the first candidate whose cumulative probability
  // reaches top_p (all of them if none does).
  {
    float c = before;
    for (int i = b; i < e; i++) {
      c += expf(key_value(keys[i]) - top);
      if (c / sum >= top_p) {
        atomicMin(&cut, i + 1);
        break;
      }
    }
  }
  __syncthreads();
  const int kept = cut;
  // Probability mass of the kept candidates, from the slice that ends them.
  if (kept == m) {
    if (tid == 0) kept_exp = sum;
  } else if (b < kept && kept <= e) {
    float c = before;
    for (int i = b; i < kept; i++) c += expf(key_value(keys[i]) - top);
    kept_exp = c;
  }
  __syncthreads();
  // The draw: the first kept candidate whose cumulative mass reaches
  // u * (kept mass), i.e. where random - sum(p) first drops to <= 0.
  const float r = u * kept_exp;
  {
    float c = before;
    for (int i = b; i < min(e, kept); i++) {
      c += expf(key_value(keys[i]) - top);
      if (c >= r) {
        atomicMin(&pick, i);
        break;
      }
    }
  }
  __syncthreads();
  if (tid == 0) {
    const int i = pick < kept ? pick : kept - 1;  // no crossing: the last kept candidate
    *out = idx[i];
  }
}

// The draw among m <= 64 sorted candidates, a lane of one wave each: the
// sums, crossings and rounding of sample_select_kernel at one candidate per
// thread (its 1,024-wide scan over zeros past the 64th is this one).
__device__ uint32_t draw_wave(float v, float top, int m, float top_p, float u, const uint32_t *sidx) {
  const int lane = threadIdx.x & 63;
  const float s = lane < m ? expf(v - top) : 0.f;
  float incl = s;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const float a = __shfl_up(incl, o);
    incl += lane >= o ? a : 0.f;
  }
  const float sum = __shfl(incl, 63);
  if (!isfinite(sum) || sum <= 0.0f) return sidx[0];  // src/engine.rs:299-301
  const float c = (incl - s) + s;
  const unsigned long long over = __ballot(lane < m && c / sum >= top_p);
  const int kept = over ? __ffsll(over) : m;
  const float kept_exp = kept == m ? sum : __shfl(c, kept - 1);
  const unsigned long long hit = __ballot(lane < kept && c >= u * kept_exp);
  return sidx[hit ? __ffsll(hit) - 1 : kept - 1];
}

constexpr int kMaxCand = 1024;  // candidates the top-k workgroup orders in LDS

// src/engine.rs:286-324 for the m <= kSelectThreads largest keys (m = 1 for
// temperature <= 0), one workgroup.  Its bound is latency: two passes over
// the groups' maxima and one over the hot groups, 11.6 us at 152,064 tokens
// and top-k 40 where the full sort's ten launches take ~60 and more between them.  Keys and tokens form one
// 64-bit word, key << 32 | ~token, whose descending order is the sort's.
__global__ __launch_bounds__(kSelectThreads) void sample_topk_kernel(
    const uint32_t *__restrict__ keys, const uint32_t *__restrict__ gmax, int n, int group, int m, float top_p,
    float temperature, float u, uint32_t *__restrict__ out) {
  __shared__ __align__(16) unsigned long long cand[kMaxCand + 4];
  __shared__ __align__(16) uint32_t gm[kSelectThreads];
  __shared__ uint32_t skey[kSelectThreads], sidx[kSelectThreads];
  __shared__ float sh[kSelectThreads];
  __shared__ uint32_t thr;
  __shared__ int ncand, nhot, cut, pick, left;
  __shared__ float kept_exp;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int ng = (n + group - 1) / group;  // m <= ng <= kSelectThreads (the launcher's rule)
  const uint32_t mine = tid < ng ? gmax[tid] : 0;
  gm[tid] = mine;  // zeros past the groups: below every maximum
  if (tid == 0) ncand = nhot = 0;
  __syncthreads();
  if (tid < ng) {  // ranks are distinct: equal maxima rank in group order
    int rank = 0;
#pragma unroll 4
    for (int j = 0; j < ng; j += 4) {
      const uint4 g = *reinterpret_cast<const uint4 *>(gm + j);
      rank += (g.x > mine || (g.x == mine && j < tid)) + (g.y > mine || (g.y == mine && j + 1 < tid)) +
              (g.z > mine || (g.z == mine && j + 2 < tid)) + (g.w > mine || (g.w == mine && j + 3 < tid));
    }
    if (rank == m - 1) thr = mine;
  }
  __syncthreads();
  const uint32_t t = thr;
  __syncthreads();  // every thread has gm's maxima and thr
  if (tid < ng && mine >= t) gm[atomicAdd(&nhot, 1)] = (uint32_t)tid;
  __syncthreads();
  // The hot groups' tokens that reach the threshold: four keys a load (the
  // key array is padded to a multiple of four) and four loads in flight a
  // thread; one key at a time, each round waits for memory (21.6 against
  // 11.6 us for the kernel).
  auto word = [](uint32_t k, int i) { return ((unsigned long long)k << 32) | (uint32_t)~(uint32_t)i; };
  const int quads = nhot * (group >> 2), sh_q = __ffs(group) - 3;  // group is a power of two
  for (int i0 = tid; i0 < quads; i0 += 4 * kSelectThreads) {
    uint4 q[4];
    int tok[4];
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int i = i0 + r * kSelectThreads;
      tok[r] = i < quads ? (int)(gm[i >> sh_q] << (sh_q + 2)) + 4 * (i & ((group >> 2) - 1)) : n;
      q[r] = tok[r] < n ? *reinterpret_cast<const uint4 *>(keys + tok[r]) : uint4{0, 0, 0, 0};
    }
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const uint32_t k[4] = {q[r].x, q[r].y, q[r].z, q[r].w};
#pragma unroll
      for (int e = 0; e < 4; e++)
        if (k[e] >= t && tok[r] + e < n) {
          const int at = atomicAdd(&ncand, 1);
          if (at < kMaxCand) cand[at] = word(k[e], tok[r] + e);
        }
    }
  }
  __syncthreads();
  int nc = ncand;
  if (nc > kMaxCand) {
    // Too many equal or close keys: the m-th largest word over all tokens by
    // its eight bytes, from the highest (words are distinct).
    unsigned long long prefix = 0;
    if (tid == 0) left = m;
    for (int shift = 56; shift >= 0; shift -= 8) {
      __syncthreads();
      if (tid < 256) gm[tid] = 0;
      __syncthreads();
      for (int i = tid; i < n; i += kSelectThreads) {
        const unsigned long long w = word(keys[i], i);
        if (shift == 56 || (w >> (shift + 8)) == prefix) atomicAdd(&gm[(w >> shift) & 255], 1u);
      }
      __syncthreads();
      if (tid == 0) {
        int b = 255, l = left;
        while (b > 0 && (int)gm[b] < l) l -= (int)gm[b--];
        left = l;
        thr = (uint32_t)b;
      }
      __syncthreads();
      prefix = (prefix << 8) | thr;
    }
    if (tid == 0) ncand = 0;
    __syncthreads();
    for (int i = tid; i < n; i += kSelectThreads) {
      const unsigned long long w = word(keys[i], i);
      if (w >= prefix) cand[atomicAdd(&ncand, 1)] = w;  // exactly m of them
    }
    __syncthreads();
    nc = ncand;
  }
  if (tid < 4) cand[nc + tid] = 0;  // below every word
  __syncthreads();
  if (tid < nc) {
    const unsigned long long w = cand[tid];
    int rank = 0;
#pragma unroll 4
    for (int j = 0; j < nc; j += 4) rank += (cand[j] > w) + (cand[j + 1] > w) + (cand[j + 2] > w) + (cand[j + 3] > w);
    if (rank < m) {
      skey[rank] = (uint32_t)(w >> 32);
      sidx[rank] = ~(uint32_t)w;
    }
  }
  __syncthreads();
  if (temperature <= 0.0f) {  // the first candidate
    if (tid == 0) *out = sidx[0];
    return;
  }
  const float top = key_value(skey[0]);
  if (m <= 64) {
    if (wave == 0) {
      const uint32_t r = draw_wave(lane < m ? key_value(skey[lane]) : 0.f, top, m, top_p, u, sidx);
      if (lane == 0) *out = r;
    }
    return;
  }
  // sample_select_kernel's sums and crossings with one candidate per thread.
  const float s = tid < m ? expf(key_value(skey[tid]) - top) : 0.f;
  const float incl = block_scan(s, sh);
  const float sum = sh[kSelectThreads - 1], c = (incl - s) + s;
  if (!isfinite(sum) || sum <= 0.0f) {  // src/engine.rs:299-301
    if (tid == 0) *out = sidx[0];
    return;
  }
  if (tid == 0) cut = pick = m;
  __syncthreads();
  if (tid < m && c / sum >= top_p) atomicMin(&cut, tid + 1);
  __syncthreads();
  const int kept = cut;
  if (tid == kept - 1) kept_exp = kept == m ? sum : c;
  __syncthreads();
  if (tid < kept && c >= u * kept_exp) atomicMin(&pick, tid);
  __syncthreads();
  if (tid == 0) *out = sidx[pick < kept ? pick : kept - 1];
}

// Tokens per group for the top-k route, 0 for the sort: the largest group
// whose maxima still outnumber the m candidates by a tenth (so that the
// threshold leaves about ng * ln(ng / (ng - m)) tokens, at most 2.4 a group)
// and number at most kSelectThreads.
int topk_group(int n, int m) {
  for (int g : {1024, 256, 64, 16}) {
    const int ng = (n + g - 1) / g;
    if (ng <= kSelectThreads && 10 * (long)m <= 9 * (long)ng) return g;
  }
  return 0;
}

}  // namespace

namespace {

// The allocation-free sampler's scratch: keys, sorted keys, indices, sorted
// indices (kNoAllocMaxVocab words each), the repeat window,
// then the radix sort's temporary storage.  In host code `scratch` names a
// host-side stand-in, never the device memory: kernels and copies get the
// address hipGetSymbolAddress returns for the current device.
constexpr size_t kNoAllocWords = 4 * (size_t)kNoAllocMaxVocab + kNoAllocMaxRecent + 64;
constexpr size_t kNoAllocBytes = kNoAllocWords * 4 + kNoAllocSortBytes;
static __device__ __align__(256) uint8_t scratch[kNoAllocBytes];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
uint8_t *g_scratch_dev[kMaxDevices] = {};  // per device: its copy of `scratch`

}  // namespace

int sample_noalloc_scratch(SampleScratch &w) {
  int dev = 0;
  LLRS_HIP(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDevices) return set_error(LLRS_E_UNSUPPORTED, "device %d", dev);
  uint8_t *base = nullptr;
  {
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_dev[dev]) {
      void *p = nullptr;
      LLRS_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
      const size_t need = sample_sort_bytes(kNoAllocMaxVocab);
      if (need > kNoAllocSortBytes)
        return set_error(LLRS_E_UNSUPPORTED, "the radix sort needs %zu temporary bytes, %zu reserved", need,
                         kNoAllocSortBytes);
      g_scratch_dev[dev] = static_cast<uint8_t *>(p);
    }
    base = g_scratch_dev[dev];
  }
  uint32_t *words = reinterpret_cast<uint32_t *>(base);
  w.n = kNoAllocMaxVocab;
  w.max_recent = kNoAllocMaxRecent;
  w.keys = words;
  w.keys_sorted = words + kNoAllocMaxVocab;
  w.idx = words + 2 * (size_t)kNoAllocMaxVocab;
  w.idx_sorted = words + 3 * (size_t)kNoAllocMaxVocab;
  w.recent = words + 4 * (size_t)kNoAllocMaxVocab;
  w.tmp = base + kNoAllocWords * 4;
  w.tmp_bytes = kNoAllocSortBytes;
  return LLRS_OK;
}

size_t sample_sort_bytes(int n) {
  size_t bytes = 0;
  (void)hipcub::DeviceRadixSort::SortPairsDescending(nullptr, bytes, (const uint32_t *)nullptr,
                                                     (uint32_t *)nullptr, (const uint32_t *)nullptr,
                                                     (uint32_t *)nullptr, n, 0, 32);
  return bytes;
}

int launch_sample(const float *logits, int n, const SampleParams &p, const uint32_t *recent, int n_recent, float u,
                  SampleScratch &w, uint32_t *out, hipStream_t s) {
  if (n <= 0 || n > w.n || n_recent < 0 || n_recent > w.max_recent)
    return set_error(LLRS_E_INVALID, "sampling over %d tokens with %d recent ones", n, n_recent);
  RecentArg r{};
  if (p.penalty != 1.0f) {
    r.n = n_recent;
    if (n_recent <= kArgRecent) {
      for (int i = 0; i < n_recent; i++) r.tok[i] = recent[i];
    } else {
      LLRS_HIP(hipMemcpyAsync(w.recent, recent, (size_t)n_recent * 4, hipMemcpyHostToDevice, s));
      r.dev = w.recent;
    }
  }
  // Greedy takes the first candidate whatever top_k is; the penalty and the
  // temperature have been applied by the keys.
  const int m = p.temperature <= 0.0f ? 1 : (p.top_k > 0 && p.top_k < n ? p.top_k : n);
  const int group = topk_group(n, m);
  const dim3 grid((unsigned)((n + kKeyBlock - 1) / kKeyBlock));
  // The sorted-keys array is free on the top-k route: the groups' maxima.
  hipLaunchKernelGGL(sample_keys_kernel, grid, dim3(256), 0, s, logits, n, r, p.penalty, p.temperature, w.keys,
                     group ? nullptr : w.idx, group ? w.keys_sorted : nullptr, group);
  LLRS_HIP(hipGetLastError());
  if (group) {
    hipLaunchKernelGGL(sample_topk_kernel, dim3(1), dim3(kSelectThreads), 0, s, w.keys, w.keys_sorted, n, group, m,
                       p.top_p, p.temperature, u, out);
    LLRS_HIP(hipGetLastError());
    return LLRS_OK;
  }
  size_t bytes = w.tmp_bytes;
  LLRS_HIP(hipcub::DeviceRadixSort::SortPairsDescending(w.tmp, bytes, w.keys, w.keys_sorted, w.idx,
                                                        w.idx_sorted, n, 0, 32, s));
  hipLaunchKernelGGL(sample_select_kernel, dim3(1), dim3(kSelectThreads), 0, s, w.keys_sorted,
                     w.idx_sorted, n, p.top_k, p.top_p, p.temperature, u, out);
  LLRS_HIP(hipGetLastError());
  return LLRS_OK;
}

}  // namespace llrs
