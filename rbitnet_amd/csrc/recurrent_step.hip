// A step of one token per sequence through a layer that carries a matrix S [key size, value size] per head, in one launch: the short
// convolution in front of q, k and v, the unit vectors and decays, the recurrence, the read-out norm and its gate.  As launches of their
// own (rb_short_conv, rb_recurrence_prep, rb_linear_recurrence, rb_gated_rmsnorm and the like, which stay for steps of several tokens
// and for other sizes) they are a chain of up to four that hand a few KB on, and such a launch costs its boundary and a trip or two to
// memory whatever it does: 2.5 to 5 us each.  All arithmetic in float32.
//
// A workgroup takes a sequence and a q/k head with all R heads that read it, so that whoever reads the convolution's state of a channel
// is also who moves it on, and a norm over all of them is the workgroup's own.  That is few workgroups (4 sequences, 16 heads: 64), but
// up to 16 waves each, all of whose loads (the columns of S into registers, the window, the projections, the gate) are in flight together.
// A column of S lies in dim numbers in a row; RG lanes hold dim / RG of them each, 4 or 8, a wave has 64 / RG columns at a time and P times as
// many in all.
//
// Every sum is taken in the order of the launches it stands for, so that a token gives the same bits whether it comes alone or in a step
// that takes those: a lane's rows of a column and its two chains, the lanes a column is dealt to (by the number of sequences, as there), the
// squares of a unit vector and of a norm.  Where those give a lane 16 rows, two lanes have them here (PAIR), and the second one's chains go on
// from the first one's: 16 rows a lane are four loads 64 bytes apart, and 64 heads of 128 x 64 of 4 sequences took 16.9 us for 11.2.
//
// Measured in a chain of launches with the same products in front and behind, 1 / 4 / 16 / 64 sequences, launches of their own -> this one: 16 heads
// of 128 x 128 with decays per channel and a convolution 19.5 / 22.5 / 31.5 / 83.2 -> 13.8 / 16.3 / 22.0 / 70.1 us (this launch alone: 6.2 / 7.0 / 11.6 /
// 43.3); 64 heads of 128 x 64 in 8 groups, selective, 15.1 / 21.6 / 37.5 / 154.2 -> 16.7 / 21.3 / 28.6 / 87.9 (alone 10.5 / 12.7 / 18.3 / 71.6): with one
// sequence that is 8 workgroups of 256 KB of state each, which they wait for (Kernels.recurrence_step_pays).
#include <math.h>

#include "api.h"
#include "common.h"
#include "mfma.h"

namespace {

__device__ __forceinline__ float sigmoid_of(float v) { return 1.0f / (1.0f + expf(-v)); }
__device__ __forceinline__ float softplus_of(float v) { return v > 20.0f ? v : log1pf(expf(v)); }

// another lane's number, by a move inside a row of 16 lanes
template <int MOVE>
__device__ __forceinline__ float moved(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), MOVE, 0xF, 0xF, true));
}
// the sum over each group of RG neighbouring lanes (8 or 16), in every lane of it
template <int RG>
__device__ __forceinline__ float group_sum(float v) {
  v += moved<0xB1>(v);                       // quad_perm [1,0,3,2]
  v += moved<0x4E>(v);                       // quad_perm [2,3,0,1]
  v += moved<0x141>(v);                      // row_half_mirror
  if (RG == 16) v += moved<0x140>(v);        // row_mirror
  return v;
}

// the same sum as wave_sum's, added up in the same order (lanes 32 apart first, then 16, 8, 4, 2 and 1), without trips through LDS: lanes that
// differ in a bit already summed over hold the same number, so a turn of a row of 16 lanes stands for the exchange
__device__ __forceinline__ float wave_sum_moves(float v) {
  const unsigned u = __builtin_bit_cast(unsigned, v);
  const auto far = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  v = __builtin_bit_cast(float, (unsigned)far[0]) + __builtin_bit_cast(float, (unsigned)far[1]);
  const unsigned w = __builtin_bit_cast(unsigned, v);
  const auto rows = __builtin_amdgcn_permlane16_swap(w, w, false, false);
  v = __builtin_bit_cast(float, (unsigned)rows[0]) + __builtin_bit_cast(float, (unsigned)rows[1]);
  v += moved<0x128>(v);                      // row_ror:8
  v += moved<0x124>(v);                      // row_ror:4
  v += moved<0x4E>(v);
  v += moved<0xB1>(v);
  return v;
}

enum { DELTA = 0, PLAIN = 1, BONUS = 2, SELECTIVE = 3 };

template <int DIM, int RG, int P, int MODE, bool PAIR>
__global__ __launch_bounds__(1024) void recurrence_step_kernel(const RbRecurrenceStep a) {
  constexpr int DKL = DIM / RG, CPW = RB_WAVE / RG, MAX_C = 16 * CPW * P < 512 ? 16 * CPW * P : 512, MAX_R = MAX_C / 64;
  __shared__ __attribute__((aligned(16))) float sq[DIM], sk[DIM], sg[MODE == SELECTIVE ? 1 : MAX_R][DIM], sv[MAX_C];
  __shared__ __attribute__((aligned(16))) float so[MAX_C], sgate[MAX_C], sact[MAX_C];
  __shared__ float ssum[16], sb[MAX_R], sdecay[MAX_R];
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
  f32x4_t s[P][DKL / 4];
#pragma unroll
  for (int p = 0; p < P; ++p) {
    const int col = (wave * P + p) * CPW + lane / RG;
    const float* at = S + (size_t)(col < cols ? col : 0) * DIM + DKL * rg;
#pragma unroll
    for (int i = 0; i < DKL / 4; ++i) s[p][i] = *reinterpret_cast<const f32x4_t*>(at + 4 * i);
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
  }
  const float turn = sigmoid_of(gate), times = a.gate_act == 1 ? gate : 1.f;
  if (tid < cols && a.norm_part) {
    sgate[tid] = times;
    sact[tid] = turn;
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
    const float q0 = sq[lane], k0 = sk[lane], q1 = DIM > RB_WAVE ? sq[lane + DIM - RB_WAVE] : 0.f, k1 = DIM > RB_WAVE ? sk[lane + DIM - RB_WAVE] : 0.f;
    fq = a.q_scale / sqrtf(wave_sum_moves(fmaf(q1, q1, q0 * q0)) + a.unit_eps);
    fk = 1.0f / sqrtf(wave_sum_moves(fmaf(k1, k1, k0 * k0)) + a.unit_eps);
  }
  float q[DKL], k[DKL];
#pragma unroll
  for (int i = 0; i < DKL; ++i) {
    q[i] = sq[DKL * rg + i] * fq;
    k[i] = sk[DKL * rg + i] * fk;
  }
  // sum of x y over a column's rows: two chains over a lane's rows, as in delta_rule_kernel, then the lanes
  auto dot = [](auto x, auto y) __attribute__((always_inline)) {
    float c0 = 0.f, c1 = 0.f;
#pragma unroll
    for (int i = 0; i < DKL; i += 2) {
      c0 = fmaf(x(i), y(i), c0);
      c1 = fmaf(x(i + 1), y(i + 1), c1);
    }
    if (!PAIR) return group_sum<RG>(c0 + c1);
    c0 = moved<0xA0>(c0);                                    // quad_perm [0,0,2,2]: the second lane goes on where the first one ended
    c1 = moved<0xA0>(c1);
#pragma unroll
    for (int i = 0; i < DKL; i += 2) {
      c0 = fmaf(x(i), y(i), c0);
      c1 = fmaf(x(i + 1), y(i + 1), c1);
    }
    float v = moved<0xF5>(c0 + c1);                          // quad_perm [1,1,3,3]: the second lane's, in both
    v += moved<0x4E>(v);                                     // quad_perm [2,3,0,1]
    v += moved<0x141>(v);                                    // row_half_mirror
    v += moved<0x140>(v);                                    // row_mirror
    return v;
  };
  auto of_k = [&](int i) { return k[i]; };
  auto of_q = [&](int i) { return q[i]; };
  const float kq_all = MODE != BONUS ? dot(of_k, of_q) : 0.f;
#pragma unroll
  for (int p = 0; p < P; ++p) {
    const int col = (wave * P + p) * CPW + lane / RG, c = col < cols ? col : 0, r = c / a.vdim;
    const bool one = MODE == SELECTIVE || a.a_per_head;
    const float g1 = one ? sdecay[r] : 0.f;
    auto of_s = [&](int i) { return s[p][i / 4][i % 4]; };
    float kv = 0.f, dq = 0.f, kq = kq_all;
    if (MODE == BONUS) {                                     // read before the write; the token's own k v^T with a weight per channel
      kq = dot([&](int i) { return a.bonus[(size_t)(h0 + r) * DIM + DKL * rg + i] * k[i]; }, of_q);
      dq = dot(of_s, of_q);
    }
#pragma unroll
    for (int i = 0; i < DKL; ++i) s[p][i / 4][i % 4] *= one ? g1 : sg[MODE == SELECTIVE ? 0 : r][DKL * rg + i];
    if (MODE == DELTA) kv = dot(of_s, of_k);
    if (MODE != BONUS) dq = dot(of_s, of_q);
    const float v = sv[c];
    const float u = MODE == DELTA ? sb[r] * (v - kv) : MODE == SELECTIVE ? sb[r] * v : v;
    if (rg == 0 && col < cols) so[col] = MODE == SELECTIVE ? fmaf(a.d[h0 + r], v, fmaf(u, kq, dq)) : fmaf(u, kq, dq);
    if (col < cols) {
      float* at = S + (size_t)col * DIM + DKL * rg;
#pragma unroll
      for (int i = 0; i < DKL / 4; ++i) {
#pragma unroll
        for (int j = 0; j < 4; ++j) s[p][i][j] = fmaf(k[4 * i + j], u, s[p][i][j]);
        *reinterpret_cast<f32x4_t*>(at + 4 * i) = s[p][i];
      }
    }
  }
  __syncthreads();

  // ---- the norm over a head's numbers, then the gate; or the gate, then the norm over `norm_part` numbers.  Both sizes are multiples of 64.
  // The squares: of a head by one wave, lane after lane; of a part four in a row by each lane, 256 by a wave
  const int part = a.norm_part ? a.norm_part : a.vdim, per = a.norm_part ? (part + 255) / 256 : 1;
  if (wave < cols / part * per) {
    float ss = 0.f;
    if (a.norm_part) {
      const int i = 4 * (lane + RB_WAVE * (wave % per)), at = wave / per * part + i;
      if (i < part) {
        const float4 o = *reinterpret_cast<const float4*>(so + at), g = *reinterpret_cast<const float4*>(sgate + at),
                     f = *reinterpret_cast<const float4*>(sact + at);
        const float4 v = make_float4(o.x * g.x * f.x, o.y * g.y * f.y, o.z * g.z * f.z, o.w * g.w * f.w);
        ss += (v.x * v.x + v.y * v.y) + (v.z * v.z + v.w * v.w);
      }
    } else {
      for (int i = lane; i < part; i += RB_WAVE) ss = fmaf(so[wave * part + i], so[wave * part + i], ss);
    }
    ss = wave_sum_moves(ss);
    if (lane == 0) ssum[wave] = ss;
  }
  __syncthreads();
  if (tid >= cols) return;
  const int w0 = tid / part * per;
  float ss = a.norm_part ? 0.f : ssum[w0];
  if (a.norm_part)
    for (int w = w0; w < w0 + per; ++w) ss += ssum[w];
  const float f = 1.0f / sqrtf(ss / (float)part + a.eps);
  const float y = a.norm_part ? so[tid] * times * turn * f * weight : so[tid] * f * weight * (times * turn);
  const size_t to = (size_t)t * a.n_heads * a.vdim + (size_t)h0 * a.vdim + tid;
  if (a.out_dtype == RB_F32) ((float*)a.out)[to] = y;
  else Num<bf16_t>::store((bf16_t*)a.out + to, y);
}

// whether rb_linear_recurrence deals a column to 8 lanes and not to 16: once its waves fill the GPU's SIMDs
bool to_few_lanes(const RbRecurrenceStep& a) { return (long long)a.n_tokens * a.n_heads * ((a.vdim + 7) / 8) >= 4LL * rb_compute_units(); }
// how often a wave has 64 / lanes columns: the fewest times with which 16 waves hold all
constexpr int MOST_COLUMNS = 512;
int passes(int lanes, int cols) {
  int p = 1;
  while (cols > 16 * (RB_WAVE / lanes) * p) p *= 2;
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
  const bool few_lanes = to_few_lanes(a);
  const int lanes = few_lanes && a.dim == 64 ? 8 : 16, cols = a.n_heads / a.n_kv_heads * a.vdim, p = passes(lanes, cols), cpw = RB_WAVE / lanes;
  const int for_state = (cols + cpw * p - 1) / (cpw * p), for_inputs = (2 * a.dim + cols) / RB_WAVE;
  const int waves = for_state > for_inputs ? for_state : for_inputs;      // (at most 16: 512 columns and two heads of 128 are 12 waves' inputs)
  const dim3 grid(a.n_tokens, a.n_kv_heads);
  hipStream_t s = (hipStream_t)stream;
#define RS_GO(DIM, RG, P, MODE, PAIR) recurrence_step_kernel<DIM, RG, P, MODE, PAIR><<<grid, waves * RB_WAVE, 0, s>>>(a)
#define RS_MODE(DIM, RG, P, PAIR)                               \
  do {                                                          \
    if (a.mode == DELTA) RS_GO(DIM, RG, P, DELTA, PAIR);        \
    else if (a.mode == PLAIN) RS_GO(DIM, RG, P, PLAIN, PAIR);   \
    else if (a.mode == BONUS) RS_GO(DIM, RG, P, BONUS, PAIR);   \
    else RS_GO(DIM, RG, P, SELECTIVE, PAIR);                    \
  } while (0)
#define RS_PASSES(DIM, RG, PAIR)                       \
  do {                                                 \
    if (p == 1) RS_MODE(DIM, RG, 1, PAIR);             \
    else if (p == 2) RS_MODE(DIM, RG, 2, PAIR);        \
    else if (p == 4) RS_MODE(DIM, RG, 4, PAIR);        \
    else RS_MODE(DIM, RG, RG == 16 ? 8 : 4, PAIR);     \
  } while (0)
  if (a.dim == 128 && few_lanes) RS_PASSES(128, 16, true);
  else if (a.dim == 128) RS_PASSES(128, 16, false);
  else if (few_lanes) RS_PASSES(64, 8, false);
  else RS_PASSES(64, 16, false);
#undef RS_PASSES
#undef RS_MODE
#undef RS_GO
  RB_LAUNCH_CHECK();
  return 0;
}
