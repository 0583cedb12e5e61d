// A step of one token per sequence through a layer that carries a matrix S [key size, value size] per head, in one launch: the short
// convolution in front of q, k and v, the unit vectors and decays, the recurrence, the read-out norm and its gate.  As launches of their
// own (rb_short_conv, rb_recurrence_prep, rb_linear_recurrence, rb_gated_rmsnorm and the like, which stay for steps of several tokens
// and for other sizes) they are a chain of up to four that hand a few KB on, and such a launch costs its boundary and a trip or two to
// memory whatever it does: 2.5 to 5 us each.  All arithmetic in float32.
//
// A workgroup takes a sequence and a q/k head with all R heads that read it, so that whoever reads the convolution's state of a channel
// is also who moves it on, and a norm over all of them is the workgroup's own.  That is few workgroups (4 sequences, 16 heads: 64), but
// up to 16 waves each, all of whose loads (the columns of S into registers, the window, the projections, the gate) are in flight together.
// A column of S lies in dim numbers in a row; RG = dim / 8 lanes hold 8 of them each, rows 4 rg .. + 3 of either half, so that a wave's load
// is whole columns; a wave has 64 / RG columns at a time and P times as many in all.
//
// Measured in a captured step, 4 sequences, launches of their own -> this one: 16 heads of 128 x 128 with decays per channel and a
// convolution 15.7 -> 7.9 us (64 workgroups); 64 heads of 128 x 64 in 8 groups, selective, 13.8 -> 10.3 (32 workgroups of 256 KB of state
// each, which is what they wait for).
#include <math.h>

#include "api.h"
#include "common.h"

namespace {

__device__ __forceinline__ float sigmoid_of(float v) { return 1.0f / (1.0f + expf(-v)); }
__device__ __forceinline__ float softplus_of(float v) { return v > 20.0f ? v : log1pf(expf(v)); }

// the sum over each group of RG neighbouring lanes (8 or 16), in every lane of it, by moves inside a row of 16 lanes
template <int RG>
__device__ __forceinline__ float group_sum(float v) {
  v += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0xB1, 0xF, 0xF, true));   // quad_perm [1,0,3,2]
  v += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x4E, 0xF, 0xF, true));   // quad_perm [2,3,0,1]
  v += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x141, 0xF, 0xF, true));  // row_half_mirror
  if (RG == 16) v += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x140, 0xF, 0xF, true));  // row_mirror
  return v;
}

enum { DELTA = 0, PLAIN = 1, BONUS = 2, SELECTIVE = 3 };

template <int DIM, int P, int MODE, typename TO>
__global__ __launch_bounds__(1024) void recurrence_step_kernel(const RbRecurrenceStep a) {
  constexpr int RG = DIM / 8, CPW = RB_WAVE / RG, MAX_C = 16 * CPW * P, MAX_R = MAX_C / 64;
  __shared__ __attribute__((aligned(16))) float sq[DIM], sk[DIM], sg[MODE == SELECTIVE ? 1 : MAX_R][DIM], sv[MAX_C];
  __shared__ float so[MAX_C], ssum[16], sb[MAX_R], sdecay[MAX_R], part_q[2], part_k[2];
  const int t = blockIdx.x, grp = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & (RB_WAVE - 1), wave = tid / RB_WAVE, rg = lane % RG;
  const int reads = a.n_heads / a.n_kv_heads;                // heads of this workgroup
  const int cols = reads * a.vdim;                           // at most MAX_C, a multiple of 64
  const int h0 = grp * reads;
  const int slot = a.slots[t];

  // ---- asked for together: what this thread turns into a number of q, k or v (the first 2 DIM + cols threads have one each), the gate and
  // the norm's weight of the column that it finishes, its part of S
  const int what = tid < DIM ? 0 : tid < 2 * DIM ? 1 : 2, e = what == 0 ? tid : what == 1 ? tid - DIM : tid - 2 * DIM;
  const bool makes = e < cols || what < 2;
  const int place = what == 2 ? h0 * a.vdim + e : grp * DIM + e;
  const int keep = a.taps - 1, channel = (what == 0 ? a.conv_q : what == 1 ? a.conv_k : a.conv_v) + place;
  float x = 0.f, w_cur = 0.f, w_bias = 0.f, win[3] = {0.f, 0.f, 0.f}, wt[3] = {0.f, 0.f, 0.f}, gate = 0.f, weight = 0.f;
  if (makes) {
    x = (what == 0 ? a.q + (size_t)t * a.q_stride : what == 1 ? a.k + (size_t)t * a.k_stride : a.v + (size_t)t * a.v_stride)[place];
    if (a.conv_w) {
      const float* w = a.conv_w + (size_t)channel * a.taps;
      w_cur = w[keep];
      if (a.conv_bias) w_bias = a.conv_bias[channel];
#pragma unroll
      for (int j = 0; j < 3; ++j) wt[j] = j < keep ? w[j] : 0.f;
    }
  }
  if (tid < cols) {
    gate = a.gate[(size_t)t * a.gate_stride + (size_t)h0 * a.vdim + tid];
    weight = a.norm_part ? a.norm[(size_t)h0 * a.vdim + tid] : a.norm[(size_t)(h0 + tid / a.vdim) * a.norm_head_stride + tid % a.vdim];
  }
  float* window = a.conv_w ? a.conv_state + (size_t)slot * keep * a.conv_channels + channel : nullptr;
  if (makes && a.conv_w) {
#pragma unroll
    for (int j = 0; j < 3; ++j) win[j] = j < keep ? window[(size_t)j * a.conv_channels] : 0.f;
  }
  float* S = a.state + ((size_t)slot * a.n_heads + h0) * a.vdim * DIM;
  float4 s[P][2];
#pragma unroll
  for (int p = 0; p < P; ++p) {
    const int col = (wave * P + p) * CPW + lane / RG;
    const float* at = S + (size_t)(col < cols ? col : 0) * DIM + 4 * rg;
    s[p][0] = *reinterpret_cast<const float4*>(at);
    s[p][1] = *reinterpret_cast<const float4*>(at + DIM / 2);
  }
  __builtin_amdgcn_sched_barrier(0);

  // ---- q, k and v: the projections, or what the convolution makes of them (and its state moves on)
  if (makes) {
    if (a.conv_w) {
      float acc = fmaf(w_cur, x, w_bias);
#pragma unroll
      for (int j = 0; j < 3; ++j) acc = fmaf(wt[j], win[j], acc);
#pragma unroll
      for (int j = 0; j < 3; ++j)
        if (j < keep) window[(size_t)j * a.conv_channels] = j + 1 < keep ? win[j + 1 < 3 ? j + 1 : 2] : x;
      x = acc * sigmoid_of(acc);
    }
    (what == 0 ? sq : what == 1 ? sk : sv)[e] = x;
    if (what < 2 && a.unit) {                                // (DIM is 64 or 128: a wave has one head's numbers)
      const float sum = wave_sum(x * x);
      if (lane == 0) (what == 0 ? part_q : part_k)[e / RB_WAVE] = sum;
    }
  }
  // ---- decays, and what weighs the write
  if (MODE == SELECTIVE || a.a_per_head) {
    if (tid < reads) {
      const int h = h0 + tid;
      const float z = a.a[(size_t)t * a.a_stride + h] + (a.a_bias ? a.a_bias[h] : 0.f);
      const float sp = softplus_of(z);
      sdecay[tid] = expf(-expf(a.a_log[h]) * sp);
      if (MODE == SELECTIVE) sb[tid] = sp;
    }
  } else {
    for (int i = tid; i < reads * DIM; i += blockDim.x) {
      const int at = h0 * DIM + i;
      const float z = a.a[(size_t)t * a.a_stride + at] + (a.a_bias ? a.a_bias[at] : 0.f);
      const float g = a.decay == 0   ? expf(-expf(a.a_log[at / DIM]) * softplus_of(z))
                      : a.decay == 1 ? expf(-softplus_of(-z) / a.tau)
                                     : expf(-expf(z));
      sg[MODE == SELECTIVE ? 0 : i / DIM][i % DIM] = g;
    }
  }
  if (MODE == DELTA && tid < reads) sb[tid] = sigmoid_of(a.b[(size_t)t * a.b_stride + h0 + tid]);
  __syncthreads();

  // ---- the recurrence: with D = diag(g) S and u = beta (v - D^T k), o = (D + k u^T)^T q = D^T q + u (k . q)
  float fq = a.q_scale, fk = 1.f;
  if (a.unit) {
    fq = a.q_scale / sqrtf(part_q[0] + (DIM > 64 ? part_q[1] : 0.f) + a.unit_eps);
    fk = 1.0f / sqrtf(part_k[0] + (DIM > 64 ? part_k[1] : 0.f) + a.unit_eps);
  }
  float q[8], k[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int r = 4 * rg + i % 4 + (i / 4) * (DIM / 2);
    q[i] = sq[r] * fq;
    k[i] = sk[r] * fk;
  }
  float kq_all = 0.f;
  if (MODE != BONUS) {
#pragma unroll
    for (int i = 0; i < 8; ++i) kq_all = fmaf(k[i], q[i], kq_all);
    kq_all = group_sum<RG>(kq_all);
  }
#pragma unroll
  for (int p = 0; p < P; ++p) {
    const int col = (wave * P + p) * CPW + lane / RG, c = col < cols ? col : 0, r = c / a.vdim;
    float m[8] = {s[p][0].x, s[p][0].y, s[p][0].z, s[p][0].w, s[p][1].x, s[p][1].y, s[p][1].z, s[p][1].w};
    const bool one = MODE == SELECTIVE || a.a_per_head;
    const float g1 = one ? sdecay[r] : 0.f;
    float kv = 0.f, dq = 0.f, kq = kq_all;
    if (MODE == BONUS) {                                     // read before the write; the token's own k v^T with a weight per channel
      kq = 0.f;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int row = 4 * rg + i % 4 + (i / 4) * (DIM / 2);
        kq = fmaf(a.bonus[(size_t)(h0 + r) * DIM + row] * k[i], q[i], kq);
        dq = fmaf(m[i], q[i], dq);
      }
      kq = group_sum<RG>(kq);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int row = 4 * rg + i % 4 + (i / 4) * (DIM / 2);
      m[i] *= one ? g1 : sg[MODE == SELECTIVE ? 0 : r][row];
      if (MODE == DELTA) kv = fmaf(m[i], k[i], kv);
      if (MODE != BONUS) dq = fmaf(m[i], q[i], dq);
    }
    if (MODE == DELTA) kv = group_sum<RG>(kv);
    dq = group_sum<RG>(dq);
    const float v = sv[c];
    const float u = MODE == DELTA ? sb[r] * (v - kv) : MODE == SELECTIVE ? sb[r] * v : v;
    if (rg == 0 && col < cols) so[col] = MODE == SELECTIVE ? fmaf(a.d[h0 + r], v, fmaf(u, kq, dq)) : fmaf(u, kq, dq);
    if (col < cols) {
      float* at = S + (size_t)col * DIM + 4 * rg;
      *reinterpret_cast<float4*>(at) = make_float4(fmaf(k[0], u, m[0]), fmaf(k[1], u, m[1]), fmaf(k[2], u, m[2]), fmaf(k[3], u, m[3]));
      *reinterpret_cast<float4*>(at + DIM / 2) =
          make_float4(fmaf(k[4], u, m[4]), fmaf(k[5], u, m[5]), fmaf(k[6], u, m[6]), fmaf(k[7], u, m[7]));
    }
  }
  __syncthreads();

  // ---- the norm over a head's numbers, then the gate; or the gate, then the norm over `norm_part` numbers.  Both sizes are multiples of 64
  const float act = a.gate_act == 1 ? gate * sigmoid_of(gate) : sigmoid_of(gate);
  float o = 0.f;
  if (tid < cols) {
    o = so[tid];
    if (a.norm_part) o *= act;
    const float sum = wave_sum(o * o);
    if (lane == 0) ssum[wave] = sum;
  }
  __syncthreads();
  if (tid >= cols) return;
  const int part = a.norm_part ? a.norm_part : a.vdim, w0 = tid / part * (part / RB_WAVE);
  float ss = 0.f;
  for (int w = w0; w < w0 + part / RB_WAVE; ++w) ss += ssum[w];
  const float f = 1.0f / sqrtf(ss / (float)part + a.eps);
  const float y = a.norm_part ? o * f * weight : o * f * weight * act;
  Num<TO>::store((TO*)a.out + (size_t)t * a.n_heads * a.vdim + (size_t)h0 * a.vdim + tid, y);
}

// columns of S a wave has at a time; how often (P): the fewest that 16 waves hold
int columns_at_once(int dim) { return dim == 128 ? 4 : 8; }
constexpr int MOST_COLUMNS = 512;
int passes(int dim, int cols) {
  int p = 1;
  while (cols > 16 * columns_at_once(dim) * p) p *= 2;
  return p;
}

}  // namespace

// Whether the kernel takes these sizes: key heads of 64 or 128, value sizes and norms in multiples of 64 (whole waves), all columns of a
// q/k head's readers in one workgroup's registers (at most 64 a lane), with a thread for each of them and for each number of q and k.
extern "C" int rb_recurrence_step_ok(int n_heads, int n_kv_heads, int dim, int vdim, int taps, int norm_part) {
  if (n_heads <= 0 || n_kv_heads <= 0 || n_heads % n_kv_heads != 0 || n_kv_heads > 65535 || (dim != 64 && dim != 128) || vdim <= 0 ||
      vdim % 64 != 0 || taps < 0 || taps > 4)
    return 0;
  const long long cols = (long long)(n_heads / n_kv_heads) * vdim;
  if (cols > MOST_COLUMNS) return 0;
  if (norm_part != 0 && (norm_part < 0 || norm_part % 64 != 0 || cols % norm_part != 0)) return 0;
  return 1;
}

extern "C" int rb_recurrence_step(const RbRecurrenceStep* args, void* stream) {
  RB_REQUIRE(args != nullptr, "rb_recurrence_step: no arguments");
  const RbRecurrenceStep a = *args;
  RB_RECORDED(rb_recurrence_step(&a, stream));
  RB_REQUIRE(a.n_tokens >= 0 && rb_recurrence_step_ok(a.n_heads, a.n_kv_heads, a.dim, a.vdim, a.taps, a.norm_part),
             "rb_recurrence_step: %d heads on %d of %d x %d, %d taps, norm over %d are not for it", a.n_heads, a.n_kv_heads, a.dim, a.vdim,
             a.taps, a.norm_part);
  RB_REQUIRE(a.mode >= DELTA && a.mode <= SELECTIVE && (a.out_dtype == RB_F32 || a.out_dtype == RB_BF16), "rb_recurrence_step: unknown mode or dtype");
  RB_REQUIRE(a.q && a.k && a.v && a.a && a.state && a.slots && a.norm && a.out && a.gate, "rb_recurrence_step: a tensor is missing");
  RB_REQUIRE(a.conv_w ? a.taps >= 1 && (a.taps == 1 || a.conv_state) : a.taps == 0, "rb_recurrence_step: the convolution lacks its weight or state");
  const bool per_head = a.mode == SELECTIVE || a.a_per_head;
  RB_REQUIRE(!per_head || (a.a_log && a.decay == 0), "rb_recurrence_step: decays per head are made with A_log");
  RB_REQUIRE((a.decay == 0 && a.a_log) || (a.decay == 1 && a.tau > 0.f) || a.decay == 2, "rb_recurrence_step: decay %d lacks its constants", a.decay);
  RB_REQUIRE((a.mode != DELTA || a.b) && (a.mode != BONUS || a.bonus) && (a.mode != SELECTIVE || a.d), "rb_recurrence_step: a mode lacks its tensor");
  RB_REQUIRE((reinterpret_cast<uintptr_t>(a.state) & 15) == 0, "rb_recurrence_step: the state is not aligned to 16 bytes");
  if (a.n_tokens == 0) return 0;
  const int cols = a.n_heads / a.n_kv_heads * a.vdim, p = passes(a.dim, cols), cpw = columns_at_once(a.dim);
  const int for_state = (cols + cpw * p - 1) / (cpw * p), for_inputs = (2 * a.dim + cols) / RB_WAVE;
  const int waves = for_state > for_inputs ? for_state : for_inputs;      // (at most 16: 512 columns and two heads of 128 are 12 waves' inputs)
  const dim3 grid(a.n_tokens, a.n_kv_heads);
  hipStream_t s = (hipStream_t)stream;
#define RS_GO(DIM, P, MODE)                                                                                  \
  do {                                                                                                       \
    if (a.out_dtype == RB_F32) recurrence_step_kernel<DIM, P, MODE, float><<<grid, waves * RB_WAVE, 0, s>>>(a); \
    else recurrence_step_kernel<DIM, P, MODE, bf16_t><<<grid, waves * RB_WAVE, 0, s>>>(a);                   \
  } while (0)
#define RS_MODE(DIM, P)                               \
  do {                                                \
    if (a.mode == DELTA) RS_GO(DIM, P, DELTA);        \
    else if (a.mode == PLAIN) RS_GO(DIM, P, PLAIN);   \
    else if (a.mode == BONUS) RS_GO(DIM, P, BONUS);   \
    else RS_GO(DIM, P, SELECTIVE);                    \
  } while (0)
#define RS_PASSES(DIM)              \
  do {                              \
    if (p == 1) RS_MODE(DIM, 1);    \
    else if (p == 2) RS_MODE(DIM, 2); \
    else if (p == 4) RS_MODE(DIM, 4); \
    else RS_MODE(DIM, DIM == 128 ? 8 : 4); \
  } while (0)
  if (a.dim == 128) RS_PASSES(128);
  else RS_PASSES(64);
#undef RS_PASSES
#undef RS_MODE
#undef RS_GO
  RB_LAUNCH_CHECK();
  return 0;
}
