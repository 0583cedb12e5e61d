// Next-token choice on the device, in two kernels (one where the vocabulary is one chunk) so that a 128k vocabulary is read by
// many workgroups: (1) per chunk of the vocabulary, the maximum with its lowest index and
// the sum of exponentials relative to it; (2) per sequence, the chunks combined and, for
// temperature sampling, the chunk that holds the target walked element by element.
//
// Reference (llama/runtime.rs:81-107): temperature <= 0 -> the index of the greatest logit
// with NaN counted as -inf; otherwise z = logit / T, e = exp(z - max z), r = u * sum(e) and
// the first index whose running sum (in index order) reaches r, the last index if none does.
// Among equal maxima the lowest index is taken.  Sums are kept in double, so that the order
// of summation (chunks, segments) cannot move the chosen index.
#include <math.h>

#include <mutex>

#include "api.h"
#include "common.h"

#define SAMPLE_CHUNK 4096
#define SAMPLE_THREADS 256
#define SAMPLE_SEG (SAMPLE_CHUNK / SAMPLE_THREADS)
#define SAMPLE_MAX_CHUNKS 1024

struct ChunkStat {
  float max;
  int arg;
  double sum;       // sum over the chunk of exp(z / T - max / T); 0 for greedy rows
};

__device__ __forceinline__ float clean(float v) { return v != v ? -INFINITY : v; }

// The chosen chunk c in index order: `before` is the sum over the chunks in front of it.  A thread adds up a segment of its own, the segments'
// running sums are a scan over the workgroup, and the first segment that reaches the target is walked by its thread, which holds its values.
// (One thread walking 256 segments' sums: 5 us of a step's last 6.)
__device__ __forceinline__ void sample_walk(const float* __restrict__ row, int vocab, int c, float temp, float zmax, double before, double target,
                                            int32_t* __restrict__ token) {
  __shared__ double s_wave[SAMPLE_THREADS / RB_WAVE];
  __shared__ int s_first;
  const int tid = threadIdx.x, lane = tid & (RB_WAVE - 1), wave = tid / RB_WAVE;
  const int i0 = c * SAMPLE_CHUNK + tid * SAMPLE_SEG;
  const int cend = (c + 1) * SAMPLE_CHUNK < vocab ? (c + 1) * SAMPLE_CHUNK : vocab;
  float v[SAMPLE_SEG];
#pragma unroll
  for (int k = 0; k < SAMPLE_SEG; ++k) v[k] = i0 + k < cend ? row[i0 + k] : 0.f;
  double part = 0.0;
#pragma unroll
  for (int k = 0; k < SAMPLE_SEG; ++k) {
    v[k] = i0 + k < cend ? expf(clean(v[k]) / temp - zmax) : 0.f;
    part += (double)v[k];
  }
  double upto = part;
#pragma unroll
  for (int o = 1; o < RB_WAVE; o <<= 1) {
    const double below = __shfl_up(upto, o, RB_WAVE);
    if (lane >= o) upto += below;
  }
  if (lane == RB_WAVE - 1) s_wave[wave] = upto;
  if (tid == 0) s_first = SAMPLE_THREADS;
  __syncthreads();
  for (int w = 0; w < wave; ++w) before += s_wave[w];
  if (i0 < cend && before + upto >= target) atomicMin(&s_first, tid);
  __syncthreads();
  if (s_first == SAMPLE_THREADS) {                           // rounding kept the running sum just below the target
    if (tid == 0) *token = cend - 1;
    return;
  }
  if (tid != s_first) return;
  double run = before + (upto - part);
  int pick = i0 + SAMPLE_SEG < cend ? i0 + SAMPLE_SEG - 1 : cend - 1;
  bool reached = false;
#pragma unroll
  for (int k = 0; k < SAMPLE_SEG; ++k) {
    run += (double)v[k];
    if (!reached && i0 + k < cend && run >= target) {
      pick = i0 + k;
      reached = true;
    }
  }
  *token = pick;
}

// WHOLE: the vocabulary is one chunk, and the choice is made here, in one launch.
template <bool WHOLE>
__global__ __launch_bounds__(SAMPLE_THREADS) void sample_chunk_kernel(const float* __restrict__ logits, int vocab,
                                                                      const float* __restrict__ temperature, const float* __restrict__ u,
                                                                      ChunkStat* __restrict__ stats, int n_chunks,
                                                                      int32_t* __restrict__ tokens) {
  __shared__ float s_val[SAMPLE_THREADS / RB_WAVE];
  __shared__ int s_idx[SAMPLE_THREADS / RB_WAVE];
  __shared__ double s_sum[SAMPLE_THREADS / RB_WAVE];
  const int c = blockIdx.x, r = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & (RB_WAVE - 1), wave = tid / RB_WAVE;
  const float* row = logits + (size_t)r * vocab;
  const int i0 = c * SAMPLE_CHUNK;
  const int i1 = i0 + SAMPLE_CHUNK < vocab ? i0 + SAMPLE_CHUNK : vocab;
  const float temp = temperature ? temperature[r] : 0.f;
  float v[SAMPLE_SEG];
  float best = -INFINITY;
  int best_i = 0x7fffffff;
#pragma unroll
  for (int k = 0; k < SAMPLE_SEG; ++k) {          // strided: coalesced loads
    const int i = i0 + tid + k * SAMPLE_THREADS;
    v[k] = i < i1 ? clean(row[i]) : -INFINITY;
    if (i < i1 && (v[k] > best || (v[k] == best && i < best_i))) {
      best = v[k];
      best_i = i;
    }
  }
#pragma unroll
  for (int o = RB_WAVE / 2; o > 0; o >>= 1) {
    const float ov = __shfl_xor(best, o, RB_WAVE);
    const int oi = __shfl_xor(best_i, o, RB_WAVE);
    if (ov > best || (ov == best && oi < best_i)) {
      best = ov;
      best_i = oi;
    }
  }
  if (lane == 0) {
    s_val[wave] = best;
    s_idx[wave] = best_i;
  }
  __syncthreads();
#pragma unroll
  for (int w = 0; w < SAMPLE_THREADS / RB_WAVE; ++w)         // every thread: the chunk's maximum and its lowest index
    if (s_val[w] > best || (s_val[w] == best && s_idx[w] < best_i)) {
      best = s_val[w];
      best_i = s_idx[w];
    }
  const bool sums = temp > 0.f && best > -INFINITY;
  const float zmax = sums ? best / temp : 0.f;
  double total = 0.0;
  if (sums) {
#pragma unroll
    for (int k = 0; k < SAMPLE_SEG; ++k) total += (double)expf(v[k] / temp - zmax);      // exp(-inf) = 0 beyond the end
#pragma unroll
    for (int o = RB_WAVE / 2; o > 0; o >>= 1) total += __shfl_xor(total, o, RB_WAVE);
    if (lane == 0) s_sum[wave] = total;
    __syncthreads();
    total = 0.0;
    for (int w = 0; w < SAMPLE_THREADS / RB_WAVE; ++w) total += s_sum[w];
  }
  if (!WHOLE) {
    if (tid == 0) stats[(size_t)r * n_chunks + c] = ChunkStat{best, best_i, total};
    return;
  }
  if (!sums) {
    if (tid == 0) tokens[r] = best_i == 0x7fffffff ? 0 : best_i;      // every logit NaN or -inf: index 0
    return;
  }
  sample_walk(row, vocab, 0, temp, zmax, 0.0, (double)u[r] * total, tokens + r);
}

// The chunks of a row combined by one wave, a lane a run of neighbouring chunks: their maximum; for temperature sampling, the running sums in
// index order as a scan over the lanes, and the chunk in which they reach the target.  (A thread that walks the chunks alone has a trip to
// memory for each: 4 rows of 128,256 logits 5.1 us, and 12 to 15 for both launches in a captured step with the cap on the logits in front of them; now 6.6.)
__global__ __launch_bounds__(SAMPLE_THREADS) void sample_pick_kernel(const float* __restrict__ logits, int vocab,
                                                                     const float* __restrict__ temperature,
                                                                     const float* __restrict__ u,
                                                                     const ChunkStat* __restrict__ stats, int n_chunks,
                                                                     int32_t* __restrict__ tokens) {
  __shared__ int s_chunk;
  __shared__ double s_before, s_target;
  __shared__ float s_gmax;
  const int r = blockIdx.x, tid = threadIdx.x;
  const float temp = temperature ? temperature[r] : 0.f;
  if (tid < RB_WAVE) {
    const ChunkStat* st = stats + (size_t)r * n_chunks;
    const int each = (n_chunks + RB_WAVE - 1) / RB_WAVE, c0 = tid * each, c1 = c0 + each < n_chunks ? c0 + each : n_chunks;
    float gmax = -INFINITY;
    int garg = 0x7fffffff;
    for (int c = c0; c < c1; ++c)
      if (st[c].max > gmax || (st[c].max == gmax && st[c].arg < garg)) {
        gmax = st[c].max;
        garg = st[c].arg;
      }
#pragma unroll
    for (int o = RB_WAVE / 2; o > 0; o >>= 1) {
      const float ov = __shfl_xor(gmax, o, RB_WAVE);
      const int oi = __shfl_xor(garg, o, RB_WAVE);
      if (ov > gmax || (ov == gmax && oi < garg)) {
        gmax = ov;
        garg = oi;
      }
    }
    int pick = -1;
    double before = 0.0, target = 0.0;
    if (!(temp > 0.f) || gmax == -INFINITY) {
      if (tid == 0) tokens[r] = garg == 0x7fffffff ? 0 : garg;          // every logit NaN or -inf: index 0
    } else {
      const double top = (double)(gmax / temp);
      auto share = [&](const ChunkStat& s) { return s.max > -INFINITY ? s.sum * exp((double)(s.max / temp) - top) : 0.0; };
      double mine = 0.0;
      bool any = false;
      for (int c = c0; c < c1; ++c) {
        mine += share(st[c]);
        any = any || st[c].max > -INFINITY;
      }
      double upto = mine;
#pragma unroll
      for (int o = 1; o < RB_WAVE; o <<= 1) {
        const double below = __shfl_up(upto, o, RB_WAVE);
        if (tid >= o) upto += below;
      }
      target = (double)u[r] * __shfl(upto, RB_WAVE - 1, RB_WAVE);
      const unsigned long long reach = __ballot(any && upto >= target);
      const int owner = reach ? __ffsll((long long)reach) - 1 : -1;
      if (tid == owner) {
        before = upto - mine;
        double run = before;
        for (int c = c0; c < c1; ++c) {
          if (!(st[c].max > -INFINITY)) continue;
          const double sum = share(st[c]);
          pick = c;                                          // (the last of them, should rounding leave the sum below the target)
          before = run;
          if (run + sum >= target) break;
          run += sum;
        }
        s_chunk = pick;
        s_before = before;
        s_target = target;
        s_gmax = gmax;
      }
      if (owner < 0 && tid == 0) tokens[r] = vocab - 1;
      if (owner >= 0) pick = 0;
    }
    if (pick < 0 && tid == 0) s_chunk = -1;
  }
  __syncthreads();
  const int c = s_chunk;
  if (c < 0) return;
  // sums inside the chunk are relative to the row's maximum, as the target is
  sample_walk(logits + (size_t)r * vocab, vocab, c, temp, s_gmax / temp, s_before, s_target, tokens + r);
}

static void launch_sample(const float* logits, int n_rows, int vocab, const float* temperature, const float* u, ChunkStat* stats, int n_chunks,
                          int32_t* tokens, hipStream_t s) {
  if (n_chunks == 1) {
    sample_chunk_kernel<true><<<dim3(1, n_rows), SAMPLE_THREADS, 0, s>>>(logits, vocab, temperature, u, stats, 1, tokens);
    return;
  }
  sample_chunk_kernel<false><<<dim3(n_chunks, n_rows), SAMPLE_THREADS, 0, s>>>(logits, vocab, temperature, u, stats, n_chunks, tokens);
  sample_pick_kernel<<<n_rows, SAMPLE_THREADS, 0, s>>>(logits, vocab, temperature, u, stats, n_chunks, tokens);
}

extern "C" int rb_sample_workspace_bytes(int n_rows, int vocab) {
  const int n_chunks = (vocab + SAMPLE_CHUNK - 1) / SAMPLE_CHUNK;
  return (int)((size_t)n_rows * n_chunks * sizeof(ChunkStat));
}

extern "C" int rb_sample(const float* logits, int n_rows, int vocab, const float* temperature, const float* u,
                         int32_t* tokens, void* workspace, void* stream) {
  RB_RECORDED(rb_sample(logits, n_rows, vocab, temperature, u, tokens, workspace, stream));
  RB_REQUIRE(n_rows >= 0 && vocab > 0, "rb_sample: bad sizes %d x %d", n_rows, vocab);
  RB_REQUIRE(temperature == nullptr || u != nullptr, "rb_sample: temperature given without uniform numbers");
  RB_REQUIRE(workspace != nullptr, "rb_sample: no workspace");
  if (n_rows == 0) return 0;
  const int n_chunks = (vocab + SAMPLE_CHUNK - 1) / SAMPLE_CHUNK;
  RB_REQUIRE(n_chunks <= SAMPLE_MAX_CHUNKS && n_rows <= 65535, "rb_sample: vocabulary %d or batch %d too large", vocab,
             n_rows);
  hipStream_t s = (hipStream_t)stream;
  ChunkStat* stats = (ChunkStat*)workspace;
  launch_sample(logits, n_rows, vocab, temperature, u, stats, n_chunks, tokens, s);
  RB_LAUNCH_CHECK();
  return 0;
}

// ---------------------------------------------------------------- the variant that allocates nothing
// rb_sample_static is rb_sample with the chunk statistics in device memory that the library
// itself holds: a file-scope array, one copy on every GPU the library runs on, kept until the
// process ends.  Nothing in it has to start at zero: the first kernel writes every entry
// [row, chunk] that the second reads.  The array's name is only a host-side handle; the
// address that kernels get is asked for once per device with hipGetSymbolAddress and kept.
#define SAMPLE_STATIC_MAX_STATS 16384      // entries of 16 bytes: 256 KiB per GPU
#define SAMPLE_STATIC_MAX_DEVICES 64
static __device__ __align__(256) unsigned char scratch[SAMPLE_STATIC_MAX_STATS * sizeof(ChunkStat)];
static void* g_scratch_ptr[SAMPLE_STATIC_MAX_DEVICES];
static std::mutex g_scratch_mutex;

static int scratch_of_current_device(void** out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  RB_REQUIRE(e == hipSuccess, "rb_sample_static: hipGetDevice failed: %s", hipGetErrorString(e));
  RB_REQUIRE(dev >= 0 && dev < SAMPLE_STATIC_MAX_DEVICES, "rb_sample_static: device %d beyond the %d this library keeps scratch for",
             dev, SAMPLE_STATIC_MAX_DEVICES);
  std::lock_guard<std::mutex> guard(g_scratch_mutex);
  if (g_scratch_ptr[dev] == nullptr) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    RB_REQUIRE(e == hipSuccess && p != nullptr, "rb_sample_static: hipGetSymbolAddress failed on device %d: %s", dev,
               hipGetErrorString(e));
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return 0;
}

// Also the set-up call: it asks for the current device's copy of the scratch array, so that a first
// rb_sample_static under stream capture finds the address known (the runtime may refuse the query
// while a stream captures).
extern "C" int rb_sample_static_max_stats(void) {
  void* ptr = nullptr;
  (void)scratch_of_current_device(&ptr);
  return SAMPLE_STATIC_MAX_STATS;
}

extern "C" int rb_sample_static(const float* logits, int n_rows, int vocab, const float* temperature, const float* u,
                                int32_t* tokens, void* stream) {
  RB_REQUIRE(n_rows >= 0 && vocab > 0, "rb_sample_static: bad sizes %d x %d", n_rows, vocab);
  RB_REQUIRE(temperature == nullptr || u != nullptr, "rb_sample_static: temperature given without uniform numbers");
  if (n_rows == 0) return 0;
  const long long n_chunks = ((long long)vocab + SAMPLE_CHUNK - 1) / SAMPLE_CHUNK;
  RB_REQUIRE(n_chunks <= SAMPLE_MAX_CHUNKS && n_rows <= 65535 && (long long)n_rows * n_chunks <= SAMPLE_STATIC_MAX_STATS,
             "rb_sample_static: %d rows of %d logits need %lld chunk entries, the built-in scratch holds %d "
             "(use rb_sample with a workspace)",
             n_rows, vocab, (long long)n_rows * n_chunks, SAMPLE_STATIC_MAX_STATS);
  void* ptr = nullptr;
  if (int rc = scratch_of_current_device(&ptr)) return rc;
  hipStream_t s = (hipStream_t)stream;
  ChunkStat* stats = (ChunkStat*)ptr;
  launch_sample(logits, n_rows, vocab, temperature, u, stats, (int)n_chunks, tokens, s);
  RB_LAUNCH_CHECK();
  return 0;
}

// ---------------------------------------------------------------- a captured step's inputs and its end
// n words from pinned host memory: what changes between the replays of a captured step, read when the kernel runs.  Loads at the scope of
// the whole system: no cache of the GPU may answer with the words of the replay before.  One launch at the head of the graph in place of
// a copy in front of it (10 us a step between the call and the first kernel).
__global__ __launch_bounds__(256) void fetch_words_kernel(const int32_t* host, int32_t* __restrict__ out, size_t n) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    out[i] = __hip_atomic_load(host + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
extern "C" int rb_fetch_words(const int32_t* host, int32_t* out, long long n, void* stream) {
  RB_RECORDED(rb_fetch_words(host, out, n, stream));
  RB_REQUIRE(n >= 0, "rb_fetch_words: negative count");
  if (n == 0) return 0;
  const long long blocks = (n + 255) / 256;
  fetch_words_kernel<<<(int)(blocks < 256 ? blocks : 256), 256, 0, (hipStream_t)stream>>>(host, out, (size_t)n);
  RB_LAUNCH_CHECK();
  return 0;
}

extern "C" int rb_stream_wait(void* stream) {
  const hipError_t e = hipStreamSynchronize((hipStream_t)stream);
  RB_REQUIRE(e == hipSuccess, "rb_stream_wait: %s", hipGetErrorString(e));
  return 0;
}
