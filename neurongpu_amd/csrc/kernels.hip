// Per-timestep kernels for gfx950 (MI355X).
//
// Step sequence launched by the engine (one HIP stream, no host syncs):
//   node updates   one launch per node group.  Each first folds the port
//                  input of the previous step (delivery accumulators plus
//                  the Poisson draws of that step) into its state, then
//                  advances the state by dt and appends its spikes to the
//                  spike ring slot of this step (wavefront ballot + one
//                  atomic per wavefront).
//   record         gathers recorded variables into a device row buffer
//   delivery       flattened CSR-by-source gather over all (spike, delay)
//                  pairs due this step, float atomics into acc[port][node]
//   post STDP      (plastic networks only) reverse-index sweep
//
// Reference behaviour followed (file:line in the NeuronGPU sources):
//   fold            src/get_spike.cu:116-140, src/poiss_gen.cu:43-74
//   RK5             src/rk5.h:57-195, src/rk5.cu:23-60
//   AdEx RHS/reset  src/aeif_cond_beta_kernel.h:153-214,
//                   src/aeif_cond_alpha_kernel.h:149-211
//   iaf_psc_exp     src/iaf_psc_exp.cu:94-119
//   PushSpike       src/spike_buffer.cu:143-228
//   delivery        src/spike_buffer.cu:233-302, src/nested_loop.cu:96-167,
//                   src/get_spike.cu:48-85
//   post STDP       src/rev_spike.cu:41-75, src/stdp.cu:24-51
#include <hip/hip_runtime.h>

#include <type_traits>

#include "ngpu_device.h"
#include "ngpu_kernels.h"
#include "proposer.h"
#include "rk5_quads.h"
#include "step_common.h"

namespace ngpu {

namespace {

// ---------------------------------------------------------------------
// AdEx conductance neurons (aeif_cond_beta / aeif_cond_alpha), RK5.
// ---------------------------------------------------------------------
template <int P>
struct AeifLocal {
  float V_th, Delta_T, inv_Delta_T, g_L, E_L, inv_C_m, a, b, inv_tau_w, I_e,
      V_peak, V_reset, t_ref;
  float E_rev[P], inv_tau_rise[P], inv_tau_decay[P], g0[P];
};

template <int P>
__device__ __forceinline__ void aeif_rhs(const AeifLocal<P> &p, float refr,
                                         const float (&y)[2 + 2 * P],
                                         float (&dy)[2 + 2 * P]) {
  bool rf = refr > 0.0f;
  // (the minimum returns V_peak for a NaN, as y < V_peak ? y : V_peak does)
  float V = rf ? p.V_reset : __builtin_fminf(y[0], p.V_peak);
  // refractory: dV = 0, by a zero factor rather than a branch (a wave never
  // splits on the refractory state); (t/C_m)*0 and t*0 agree bit for bit
  const float inv_C_m = rf ? 0.0f : p.inv_C_m;
  float I_syn = 0.0f;
#pragma unroll
  for (int i = 0; i < P; i++)
    I_syn = __builtin_fmaf(y[2 + 2 * i], p.E_rev[i] - V, I_syn);
  float V_spike = p.Delta_T * dev_expf((V - p.V_th) * p.inv_Delta_T);
  float t = (V - p.E_L) - V_spike;
  t = (-p.g_L) * t;
  t = t + I_syn;
  t = t - y[1];
  t = t + p.I_e;
  dy[0] = t * inv_C_m;
  float u = p.a * (V - p.E_L);
  u = u - y[1];
  dy[1] = u * p.inv_tau_w;
#pragma unroll
  for (int i = 0; i < P; i++) {
    float g = y[2 + 2 * i], g1 = y[3 + 2 * i];
    dy[3 + 2 * i] = (-g1) * p.inv_tau_rise[i];
    dy[2 + 2 * i] = __builtin_fmaf(-g, p.inv_tau_decay[i], g1);
  }
}

// The AdEx RHS as a model of the generic RK5 attempt.
template <int P>
struct AeifModel {
  static constexpr int N = 2 + 2 * P;
  const AeifLocal<P> &p;
  __device__ __forceinline__ void rhs(float refr, const float (&y)[N],
                                      float (&dy)[N]) const {
    aeif_rhs<P>(p, refr, y, dy);
  }
};

template <int P>
__device__ __forceinline__ void aeif_rk5_begin(const AeifLocal<P> &p,
                                               float refr,
                                               const float (&y)[2 + 2 * P],
                                               float h,
                                               float (&k1)[2 + 2 * P],
                                               float (&scal)[2 + 2 * P]) {
  rk5_begin(AeifModel<P>{p}, refr, y, h, k1, scal);
}

template <int P>
__device__ __forceinline__ float aeif_rk5_attempt(
    const AeifLocal<P> &p, float refr, const float (&y)[2 + 2 * P],
    const float (&k1)[2 + 2 * P], const float (&scal)[2 + 2 * P],
    float hh, float eps, float (&yn)[2 + 2 * P]) {
  return rk5_attempt(AeifModel<P>{p}, refr, y, k1, scal, hh, eps, yn);
}

template <int P>
__device__ __forceinline__ bool aeif_rk5_step(const AeifLocal<P> &p, float refr,
                                              double &x, float (&y)[2 + 2 * P],
                                              float &h, float h_min,
                                              double h_min_acc, float h_max,
                                              float eps, int &n_att,
                                              int &n_acc, int &n_rej,
                                              unsigned long long *forced) {
  return rk5_step(AeifModel<P>{p}, refr, x, y, h, h_min, h_min_acc, h_max,
                  eps, n_att, n_acc, n_rej, forced);
}

template <int P>
__global__ __launch_bounds__(kBlock) void aeif_kernel(AeifArgs A) {
  const StepNow sn = step_now(A.out, &A.fold, A.clock);
  int i = blockIdx.x * kBlock + threadIdx.x;
  bool active = i < A.n;
  int ii = active ? i : 0;
  int node = A.i0 + ii;
  int nsp = 0;
  int n_acc = 0, n_rej = 0;
  if (active) {
    constexpr int N = 2 + 2 * P;
    AeifLocal<P> p;
    p.V_th = pf(A.p.V_th, i);
    p.Delta_T = pf(A.p.Delta_T, i);
    p.inv_Delta_T = pf(A.p.inv_Delta_T, i);
    p.g_L = pf(A.p.g_L, i);
    p.E_L = pf(A.p.E_L, i);
    p.inv_C_m = pf(A.p.inv_C_m, i);
    p.a = pf(A.p.a, i);
    p.b = pf(A.p.b, i);
    p.inv_tau_w = pf(A.p.inv_tau_w, i);
    p.I_e = pf(A.p.I_e, i);
    p.V_peak = pf(A.p.V_peak, i);
    p.V_reset = pf(A.p.V_reset, i);
    p.t_ref = pf(A.p.t_ref, i);
#pragma unroll
    for (int q = 0; q < P; q++) {
      p.E_rev[q] = pf(A.p.E_rev[q], i);
      p.inv_tau_rise[q] = pf(A.p.inv_tau_rise[q], i);
      p.inv_tau_decay[q] = pf(A.p.inv_tau_decay[q], i);
      p.g0[q] = pf(A.p.g0[q], i);
    }
    float y[N];
    y[0] = A.V[i];
    y[1] = A.w[i];
#pragma unroll
    for (int q = 0; q < P; q++) {
      y[2 + 2 * q] = A.g[q][i];
      y[3 + 2 * q] = A.g1[q][i];
    }
    // fold the previous step's port input into g1
    float in[P];
    gather_input<P>(A.fold, sn, node, in);
#pragma unroll
    for (int q = 0; q < P; q++)
      y[3 + 2 * q] = __builtin_fmaf(in[q], p.g0[q], y[3 + 2 * q]);
    if (A.do_step) {
      double x = A.x[i];
      float h = A.h[i];
      float refr = A.refr[i];
      double x1 = A.clock ? sn.t : A.x1;
      int n_att = 0;
      bool end = false;
      while (!end) {
        float hmax = (float)(x1 - x);
        if (!aeif_rk5_step<P>(p, refr, x, y, h, A.h_min, A.h_min_acc, hmax,
                              A.eps, n_att, n_acc, n_rej, A.forced))
          x = x1;
        end = (x >= x1 - (double)A.h_min);
        // ExternalUpdate
        if (y[0] < -1.0e3f) {
          y[0] = p.V_reset;
          y[1] = 0.0f;
          continue;
        }
        if (y[1] < -1.0e6f || y[1] > 1.0e6f) {
          y[0] = p.V_reset;
          y[1] = 0.0f;
          continue;
        }
        if (refr > 0.0f) {
          y[0] = p.V_reset;
          if (end) refr -= 1.0f;
        } else if (y[0] >= p.V_peak) {
          nsp++;
          y[0] = p.V_reset;
          y[1] = y[1] + p.b;
          float r = roundf(p.t_ref / A.dt);
          int ri = (int)r;
          refr = (float)(ri < 0 ? 0 : ri);
        }
      }
      A.x[i] = x;
      A.h[i] = h;
      A.refr[i] = refr;
    }
    A.V[i] = y[0];
    A.w[i] = y[1];
#pragma unroll
    for (int q = 0; q < P; q++) {
      A.g[q][i] = y[2 + 2 * q];
      A.g1[q][i] = y[3 + 2 * q];
    }
  }
  if (!A.do_step) return;
  emit_spikes(A.out, sn, active, ii, node, nsp, (float)nsp);
  // statistics: accepted / rejected RK5 attempts
  int sa = n_acc, sr = n_rej;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    sa += __shfl_xor(sa, off);
    sr += __shfl_xor(sr, off);
  }
  if (lane_id() == 0 && A.cnt && (sa | sr)) {
    unsigned long long *c = A.cnt + 2 * (blockIdx.x & (kCounterSlots - 1));
    atomicAdd(c, (unsigned long long)sa);
    atomicAdd(c + 1, (unsigned long long)sr);
  }
}

// UNI: every parameter of the group is uniform (PField::ptr == nullptr),
// so the values come straight from the kernel arguments
template <int P, bool UNI>
__device__ __forceinline__ void aeif_load_params(const AeifArgs &A, int i,
                                                 AeifLocal<P> &p) {
  if (UNI) {
    p.V_th = A.p.V_th.val;
    p.Delta_T = A.p.Delta_T.val;
    p.inv_Delta_T = A.p.inv_Delta_T.val;
    p.g_L = A.p.g_L.val;
    p.E_L = A.p.E_L.val;
    p.inv_C_m = A.p.inv_C_m.val;
    p.a = A.p.a.val;
    p.b = A.p.b.val;
    p.inv_tau_w = A.p.inv_tau_w.val;
    p.I_e = A.p.I_e.val;
    p.V_peak = A.p.V_peak.val;
    p.V_reset = A.p.V_reset.val;
    p.t_ref = A.p.t_ref.val;
#pragma unroll
    for (int q = 0; q < P; q++) {
      p.E_rev[q] = A.p.E_rev[q].val;
      p.inv_tau_rise[q] = A.p.inv_tau_rise[q].val;
      p.inv_tau_decay[q] = A.p.inv_tau_decay[q].val;
      p.g0[q] = A.p.g0[q].val;
    }
    return;
  }
  p.V_th = pf(A.p.V_th, i);
  p.Delta_T = pf(A.p.Delta_T, i);
  p.inv_Delta_T = pf(A.p.inv_Delta_T, i);
  p.g_L = pf(A.p.g_L, i);
  p.E_L = pf(A.p.E_L, i);
  p.inv_C_m = pf(A.p.inv_C_m, i);
  p.a = pf(A.p.a, i);
  p.b = pf(A.p.b, i);
  p.inv_tau_w = pf(A.p.inv_tau_w, i);
  p.I_e = pf(A.p.I_e, i);
  p.V_peak = pf(A.p.V_peak, i);
  p.V_reset = pf(A.p.V_reset, i);
  p.t_ref = pf(A.p.t_ref, i);
#pragma unroll
  for (int q = 0; q < P; q++) {
    p.E_rev[q] = pf(A.p.E_rev[q], i);
    p.inv_tau_rise[q] = pf(A.p.inv_tau_rise[q], i);
    p.inv_tau_decay[q] = pf(A.p.inv_tau_decay[q], i);
    p.g0[q] = pf(A.p.g0[q], i);
  }
}

// Resume record of a neuron whose step did not finish within the attempt
// budget of the first pass.  Its state (y, x, current h, refractory count)
// is in the group arrays; h_begin is the step size the current RK5 step
// started with, from which the second pass recomputes the step's first
// stage and error scale exactly.
// Learned step-size proposer (inference): features of a neuron at the
// start of an RK5 step and the MLP with BF16 weights, FP32 accumulation.
template <int P>
__device__ __forceinline__ void prop_features(const AeifLocal<P> &p,
                                              const float (&y)[2 + 2 * P],
                                              float h, float err_last,
                                              float inv_dt,
                                              float (&f)[kPropIn]) {
  f[0] = (y[0] - p.E_L) * 0.1f;
  f[1] = y[1] * 0.01f;
  f[2] = y[2];
  float gi = 0.0f;
#pragma unroll
  for (int q = 1; q < P; q++) gi += y[2 + 2 * q];
  f[3] = gi;
  f[4] = __log2f(h * inv_dt);
  float e = err_last > 1e-8f ? err_last : 1e-8f;
  f[5] = __log2f(e) * (0.30103f * 0.25f);
}

typedef short prop_s4 __attribute__((ext_vector_type(4)));
typedef float prop_f16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ short prop_bf16(float f) {
  uint32_t u = __float_as_uint(f);
  u += 0x7FFFu + ((u >> 16) & 1u);  // round to nearest even
  return (short)(u >> 16);
}

// The MLP for the 64 samples of a wavefront (one per lane) on the matrix
// cores: H1^T = W1 X^T and H2^T = W2 H1^T as 32x32x8 BF16 MFMAs with FP32
// accumulation, two 32-sample column blocks each; the accumulator layout of
// a layer is the B-operand layout of the next, so only the input features
// cross lanes.  Every lane of the wave must call it (wave-uniform branch);
// returns the output for the calling lane's own sample.
__device__ __forceinline__ float prop_mlp_mfma(const unsigned char *pk,
                                               const float (&f)[kPropIn]) {
  const uint32_t l = lane_id();
  const bool hi = l >= 32;
  float x[8], xs[8];
#pragma unroll
  for (int j = 0; j < 8; j++) x[j] = j < kPropIn ? f[j] : 0.0f;
#pragma unroll
  for (int j = 0; j < 8; j++) xs[j] = __shfl_xor(x[j], 32);
  prop_s4 b0, b1;
#pragma unroll
  for (int j = 0; j < 4; j++) {
    b0[j] = prop_bf16(hi ? xs[4 + j] : x[j]);  // samples 0-31
    b1[j] = prop_bf16(hi ? x[4 + j] : xs[j]);  // samples 32-63
  }
  const prop_s4 a1 = reinterpret_cast<const prop_s4 *>(pk + kPropPkW1)[l];
  const float *bp1 = reinterpret_cast<const float *>(pk + kPropPkB1) + l * 16;
  const float *bp2 = reinterpret_cast<const float *>(pk + kPropPkB2) + l * 16;
  const float *wp3 = reinterpret_cast<const float *>(pk + kPropPkW3) + l * 16;
  prop_f16 c1, c2;
#pragma unroll
  for (int r = 0; r < 16; r++) {
    c1[r] = bp1[r];
    c2[r] = bp2[r];
  }
  prop_f16 d0 = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(a1, b0, c1, 0, 0, 0);
  prop_f16 d1 = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(a1, b1, c1, 0, 0, 0);
  prop_f16 e0 = c2, e1 = c2;
#pragma unroll
  for (int c = 0; c < 4; c++) {
    const prop_s4 a2 =
        reinterpret_cast<const prop_s4 *>(pk + kPropPkW2)[c * 64 + l];
    prop_s4 h0, h1;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      float u0 = d0[4 * c + j], u1 = d1[4 * c + j];
      h0[j] = prop_bf16(u0 > 0.0f ? u0 : 0.0f);
      h1[j] = prop_bf16(u1 > 0.0f ? u1 : 0.0f);
    }
    e0 = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(a2, h0, e0, 0, 0, 0);
    e1 = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(a2, h1, e1, 0, 0, 0);
  }
  float p0 = 0.0f, p1 = 0.0f;
#pragma unroll
  for (int r = 0; r < 16; r++) {
    float w = wp3[r];
    p0 = __builtin_fmaf(w, e0[r] > 0.0f ? e0[r] : 0.0f, p0);
    p1 = __builtin_fmaf(w, e1[r] > 0.0f ? e1[r] : 0.0f, p1);
  }
  p0 += __shfl_xor(p0, 32);
  p1 += __shfl_xor(p1, 32);
  return (hi ? p1 : p0) + *reinterpret_cast<const float *>(pk + kPropPkB3);
}

// Inference on given feature vectors (n padded to whole waves); every
// lane runs the MLP, lanes beyond n use zero features and discard the
// output.
__global__ __launch_bounds__(kBlock) void prop_eval_kernel(
    const unsigned char *pk, const float *feat, int n, float *out) {
  int i = blockIdx.x * kBlock + threadIdx.x;
  float f[kPropIn];
#pragma unroll
  for (int k = 0; k < kPropIn; k++)
    f[k] = i < n ? feat[(size_t)i * kPropIn + k] : 0.0f;
  float o = prop_mlp_mfma(pk, f);
  if (i < n) out[i] = o;
}

constexpr int kStragLists = 64;  // sub-lists of resume records

struct StragRec {
  uint32_t i;
  uint32_t nsp;
  uint32_t n_att;
  uint32_t flags;     // bit 0: saved at an RK5 step boundary
  float h_begin;
  float err_last;     // scaled error of the neuron's last attempt
};
static_assert(sizeof(StragRec) == kStragRecBytes, "resume record size");

// One RK5 attempt of a neuron plus the step-boundary logic of RK5Update
// and ExternalUpdate (src/rk5.h:70-162, src/aeif_cond_beta_kernel.h:
// 178-214).  Same arithmetic, in the same order, as aeif_rk5_step and the
// loop of aeif_kernel.  Returns true when the neuron has reached the end of
// the time step.
template <int P>
__device__ __forceinline__ bool aeif_attempt_and_update(
    const AeifArgs &A, const double x1, const AeifLocal<P> &p,
    float (&y)[2 + 2 * P], const float (&k1)[2 + 2 * P],
    const float (&scal)[2 + 2 * P], double &x, float &h, float &refr,
    int &nsp, int &n_att, bool &need_k1, int &n_acc, int &n_rej,
    float &err_out, float &hh_out) {
  constexpr int N = 2 + 2 * P;
  float yn[N];
  float h_max = (float)(x1 - x);
  float hh = h;
  if (hh > h_max) hh = h_max;
  if (hh < A.h_min) hh = A.h_min;
  h = hh;
  float err = aeif_rk5_attempt<P>(p, refr, y, k1, scal, hh, A.eps, yn);
  err_out = err;
  hh_out = hh;
  n_att++;
  const bool accept = err <= 1.0f || (double)hh <= A.h_min_acc;
  // err^-1/5 (accepted) or err^-1/4 (rejected), one sequence for the wave
  const float pw = dev_pow_ctrl(err, accept ? -0.2f : -0.25f);
  if (accept) {
    n_acc++;
    if (err > 1.0f) count_forced(A.forced);
    x += (double)h;
    if (err > CK::err_min) {
      h = (h * CK::coeff) * pw;
    } else {
      h = 5.0f * h;
    }
#pragma unroll
    for (int k = 0; k < N; k++) y[k] = yn[k];
  } else {
    n_rej++;
    if (n_att > kMaxAttemptsPerStep) {
      x = x1;  // give up on this step
    } else {
      float h_new = (hh * CK::coeff) * pw;
      float h_lo = 0.1f * hh;
      h = (h_new > h_lo) ? h_new : h_lo;
      return false;  // retry with the smaller step
    }
  }
  bool end = (x >= x1 - (double)A.h_min);
  if (y[0] < -1.0e3f) {
    y[0] = p.V_reset;
    y[1] = 0.0f;
  } else if (y[1] < -1.0e6f || y[1] > 1.0e6f) {
    y[0] = p.V_reset;
    y[1] = 0.0f;
  } else if (refr > 0.0f) {
    y[0] = p.V_reset;
    if (end) refr -= 1.0f;
  } else if (y[0] >= p.V_peak) {
    nsp++;
    y[0] = p.V_reset;
    y[1] = y[1] + p.b;
    float r = roundf(p.t_ref / A.dt);
    int ri = (int)r;
    refr = (float)(ri < 0 ? 0 : ri);
  }
  if (!end) need_k1 = true;
  return end;
}

template <int P>
__device__ __forceinline__ void aeif_store_state(const AeifArgs &A, int i,
                                                 const float (&y)[2 + 2 * P],
                                                 double x, float h,
                                                 float refr) {
  const uint32_t u = (uint32_t)i;
  at(A.x, u) = x;
  at(A.h, u) = h;
  at(A.refr, u) = refr;
  at(A.V, u) = y[0];
  at(A.w, u) = y[1];
#pragma unroll
  for (int q = 0; q < P; q++) {
    at(A.g[q], u) = y[2 + 2 * q];
    at(A.g1[q], u) = y[3 + 2 * q];
  }
}

template <int P>
__device__ __forceinline__ void aeif_count(const AeifArgs &A, int n_acc,
                                           int n_rej) {
  rk5_count(A.cnt, n_acc, n_rej);
}

// Sub-list length set of the step (even / odd gs) and the other set.
__device__ __forceinline__ long long aeif_gs(const AeifArgs &A) {
  return A.clock ? A.clock->gs : A.gs;
}

// First pass: one neuron per lane, coalesced, at most A.budget RK5
// attempts.  Neurons that need more (those that spike or sit near
// threshold, which would otherwise hold their 63 wave neighbours idle)
// save their state and are listed per block for the second pass.
// W: the waves per SIMD the register allocation must allow (1: no
// constraint).  With group-uniform parameters and up to two ports the state
// fits in 80 VGPRs, which allows 6 wavefronts per SIMD instead of 5 (7 %
// faster on c1, measured); for more ports or per-neuron parameters the same
// limit would spill to scratch.
// B1: the attempt budget is 1 (the default), known at compile time, so the
// attempt loop is straight-line code.
template <int P, bool UNI, int W, bool OV, bool B1 = false>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(W)))
void aeif_pass1_kernel(AeifArgs A) {
  constexpr int N = 2 + 2 * P;
  const StepNow sn = step_now(A.out, &A.fold, A.clock);
  const double x1 = A.clock ? sn.t : A.x1;
  const long long gs = aeif_gs(A);
  const int sel = (int)(gs & 3);
  unsigned int *strag_n = A.strag_n2 + 2 * kStragLists * sel;
  unsigned int *strag_n_next = A.strag_n2 + 2 * kStragLists * ((gs + 1) & 3);
  StragRec *strag = reinterpret_cast<StragRec *>(A.strag) +
                    (size_t)sel * 2 * kStragLists * A.strag_cap;
  __shared__ uint32_t s_n, s_base, s_nc, s_basec;
  if (threadIdx.x == 0) {
    s_n = 0u;
    s_nc = 0u;
  }
  if (blockIdx.x == 0 && threadIdx.x < 2 * kStragLists)
    strag_n_next[threadIdx.x] = 0u;
  __syncthreads();
  uint32_t slot = 0xFFFFFFFFu;
  StragRec rec;
  int i = blockIdx.x * kBlock + threadIdx.x;
  bool active = i < A.n;
  int ii = active ? i : 0;
  int node = A.i0 + ii;
  int nsp = 0, n_acc = 0, n_rej = 0;
  bool finished = false, skipped = false;
  if (OV && active && A.skip_prev) {
    const unsigned long long m =
        A.mask[(size_t)((gs - 1) & 1) * A.n_waves + (i >> 6)];
    skipped = (m >> (i & 63)) & 1ull;
  }
  uint32_t cslot = 0xFFFFFFFFu;
  if (skipped) {
    // owned by the previous step's second pass, which may still run:
    // fold only the input, the second pass of this step runs the step
    float in[P];
    gather_input<P>(A.fold, sn, node, in);
    float *carry = A.carry + (size_t)(gs & 1) * P * A.n;
#pragma unroll
    for (int q = 0; q < P; q++) carry[(size_t)q * A.n + i] = in[q];
    cslot = atomicAdd(&s_nc, 1u);
  } else if (active) {
    AeifLocal<P> p;
    aeif_load_params<P, UNI>(A, i, p);
    float y[N], k1[N], scal[N];
    const uint32_t u = (uint32_t)i;
    y[0] = at(A.V, u);
    y[1] = at(A.w, u);
#pragma unroll
    for (int q = 0; q < P; q++) {
      y[2 + 2 * q] = at(A.g[q], u);
      y[3 + 2 * q] = at(A.g1[q], u);
    }
    float in[P];
    gather_input<P>(A.fold, sn, node, in);
#pragma unroll
    for (int q = 0; q < P; q++)
      y[3 + 2 * q] = __builtin_fmaf(in[q], p.g0[q], y[3 + 2 * q]);
    double x = at(A.x, u);
    float h = at(A.h, u);
    float refr = at(A.refr, u);
    int n_att = 0;
    bool need_k1 = true;
    float h_begin = h, err_last = 1.0f, hh_used = h;
    for (;;) {
      if (n_att >= (B1 ? 1 : A.budget)) break;
      if (need_k1) {
        h_begin = h;
        aeif_rk5_begin<P>(p, refr, y, h, k1, scal);
        need_k1 = false;
      }
      if (aeif_attempt_and_update<P>(A, x1, p, y, k1, scal, x, h, refr,
                                     nsp, n_att, need_k1, n_acc, n_rej,
                                     err_last, hh_used)) {
        finished = true;
        break;
      }
    }
    aeif_store_state<P>(A, i, y, x, h, refr);
    if (!finished) {
      slot = atomicAdd(&s_n, 1u);
      rec.i = (uint32_t)i;
      rec.nsp = (uint32_t)nsp;
      rec.n_att = (uint32_t)n_att;
      rec.flags = need_k1 ? 1u : 0u;
      rec.h_begin = need_k1 ? h : h_begin;
      rec.err_last = err_last;
    }
  }
  emit_spikes(A.out, sn, active && finished, ii, node, nsp, (float)nsp);
  if (B1)
    rk5_count_one(A.cnt1 ? A.cnt1 : A.cnt, n_acc, n_rej);
  else
    rk5_count(A.cnt1 ? A.cnt1 : A.cnt, n_acc, n_rej);
  if (OV && A.mask_write) {
    const unsigned long long m =
        __ballot(slot != 0xFFFFFFFFu || cslot != 0xFFFFFFFFu);
    if (lane_id() == 0 && (unsigned long long)(i >> 6) < A.n_waves)
      A.mask[(size_t)(gs & 1) * A.n_waves + (i >> 6)] = m;
  }
  // this block's resume records go to sub-list blockIdx % kStragLists,
  // at an offset reserved with one atomic per block (and its catch-up
  // entries to the same sub-list of the catch-up lists)
  __syncthreads();
  const uint32_t list = blockIdx.x % kStragLists;
  if (threadIdx.x == 0) {
    s_base = s_n ? atomicAdd(strag_n + list, s_n) : 0u;
    if (OV) s_basec = s_nc ? atomicAdd(strag_n + kStragLists + list, s_nc) : 0u;
  }
  __syncthreads();
  if (slot != 0xFFFFFFFFu)
    strag[(size_t)list * A.strag_cap + s_base + slot] = rec;
  if (OV && cslot != 0xFFFFFFFFu) {
    StragRec c;
    c.i = (uint32_t)i;
    c.nsp = 0u;
    c.n_att = 0u;
    c.flags = 1u;
    c.h_begin = 0.0f;
    c.err_last = 1.0f;
    strag[(size_t)(kStragLists + list) * A.strag_cap + s_basec + cslot] = c;
  }
}

// The AdEx conductance models' derivatives on a quad.
template <int P>
struct QuadModel {
  // parameters of the lane's role: lane 0 the membrane's, lane 1 + p port
  // p's (a = 0 makes lane 0's w equation the port's g1 equation)
  float V_th, Delta_T, inv_Delta_T, g_L, E_L, I_e, V_peak, V_reset;
  float E_rev[P];
  float a;          // 0 in the port lanes
  float ca, cb;     // 1/C_m and 1/tau_w, or 1/tau_decay and 1/tau_rise
  float V_b, n_refr;
  float ca_now;     // ca, 0 for a refractory membrane
  bool port;        // lane 1 and up
  bool clamp;       // V = V_reset: refractory, and in the port lanes

  __device__ __forceinline__ void refractory(bool rf) {
    clamp = port || rf;
    ca_now = !port && rf ? 0.0f : ca;
  }
  __device__ __forceinline__ void rhs(float ya, float yb, float &da,
                                      float &db) const {
    // (v_min_f32 returns V_peak for a NaN, as y < V_peak ? y : V_peak does;
    // spelled out, since the compiler's fmin quiets its operands first)
    float V;
    asm("v_min_f32 %0, %1, %2" : "=v"(V) : "v"(ya), "v"(V_peak));
    V = clamp ? V_reset : V;
    float I_syn = quad_get<1>(ya) * (E_rev[0] - V);
    if constexpr (P > 1)
      I_syn = __builtin_fmaf(quad_get<2>(ya), E_rev[1] - V, I_syn);
    if constexpr (P > 2)
      I_syn = __builtin_fmaf(quad_get<3>(ya), E_rev[2] - V, I_syn);
    const float V_spike = Delta_T * dev_expf((V - V_th) * inv_Delta_T);
    float t = (V - E_L) - V_spike;
    t = (-g_L) * t;
    t = t + I_syn;
    t = t - yb;
    t = t + I_e;
    da = __builtin_fmaf(port ? -ya : t, ca_now, port ? yb : -0.0f);
    float u = a * (V - E_L);
    u = u - yb;
    db = u * cb;
  }
};

template <int P, bool UNI>
__device__ __forceinline__ void aeif_quad_finish(
    const AeifArgs &A, const StepNow &sn, const double x1, bool have, int i1,
    const float (&y1)[2 + 2 * P], const float (&scal1)[2 + 2 * P], double xx,
    float h1, float refr1, int nsp1, int n_att1, bool need1, int &n_acc,
    int &n_rej) {
  QuadState<P, 2> st;
  st.take(have, i1, y1, scal1, xx, h1, refr1, nsp1, n_att1, need1);
  QuadModel<P> q;
  {
    AeifLocal<P> p;
    aeif_load_params<P, UNI>(A, st.i, p);
    q.V_th = p.V_th;
    q.Delta_T = p.Delta_T;
    q.inv_Delta_T = p.inv_Delta_T;
    q.g_L = p.g_L;
    q.E_L = p.E_L;
    q.I_e = p.I_e;
    q.V_peak = p.V_peak;
    q.V_reset = p.V_reset;
    q.port = st.role != 0;
    q.a = st.role == 0 ? p.a : 0.0f;
    q.ca = p.inv_C_m;
    q.cb = p.inv_tau_w;
#pragma unroll
    for (int k = 0; k < P; k++) {
      q.E_rev[k] = p.E_rev[k];
      if (st.rv == k + 1) {
        q.ca = p.inv_tau_decay[k];
        q.cb = p.inv_tau_rise[k];
      }
    }
    q.V_b = p.b;
    const int ri = (int)roundf(p.t_ref / A.dt);
    q.n_refr = (float)(ri < 0 ? 0 : ri);
  }
  const QuadStep step = {x1, A.h_min, A.h_min_acc, A.eps, A.forced};
  quad_run(q, st, step, n_acc, n_rej,
           [&](const QuadState<P, 2> &s, bool done) {
             if (done && s.own) {
               const uint32_t u = (uint32_t)s.i;
               if (s.role == 0) {
                 at(A.x, u) = s.x;
                 at(A.h, u) = s.h;
                 at(A.refr, u) = s.refr;
                 at(A.V, u) = s.ya;
                 at(A.w, u) = s.yb;
               } else {
                 // (selected, not indexed: the arguments stay in scalar
                 // registers)
                 float *ga = A.g[0], *gb = A.g1[0];
#pragma unroll
                 for (int k = 1; k < P; k++)
                   if (s.role == k + 1) {
                     ga = A.g[k];
                     gb = A.g1[k];
                   }
                 at(ga, u) = s.ya;
                 at(gb, u) = s.yb;
               }
             }
             const bool sp = done && s.role == 0;
             emit_spikes(A.out, sn, sp, sp ? s.i : 0, A.i0 + (sp ? s.i : 0),
                         s.nsp, (float)s.nsp);
           });
}

// Second pass: the listed neurons, run to the end of the step.  The
// sub-lists are concatenated (prefix over their counts, in LDS) and lane g
// of the grid takes entries g, g + G, ...; a lane moves on to its next
// entry as soon as the current neuron is done, so lanes stay busy while
// neurons need different numbers of attempts, and waves beyond the list
// end exit at once.
// PROP: the learned proposer's inference is compiled in (its weights in
// LDS, the MFMA registers); without it the pass keeps its occupancy.  Used
// for the sample log as well, with or without the proposer.
template <int P, bool UNI, bool PROP, bool CU>
__device__ __forceinline__ void aeif_pass2_body(const AeifArgs &A0,
                                                uint32_t vblock,
                                                uint32_t vgrid) {
  constexpr int N = 2 + 2 * P;
  const long long gs = aeif_gs(A0);
  // this step's set: resume records, then the catch-up entries (neurons
  // the first pass of this step skipped)
  const unsigned int *strag_n = A0.strag_n2 + 2 * kStragLists * (gs & 3);
  const unsigned int *strag_n_prev = strag_n + kStragLists;
  __shared__ uint32_t s_pre[kStragLists + 1], s_pre2[kStragLists + 1];
  if (threadIdx.x < (CU ? 128 : 64)) {  // exclusive scans of 64 lengths
    const int l = threadIdx.x & 63;
    const bool second = threadIdx.x >= 64;
    uint32_t c = second ? (A0.skip_prev ? strag_n_prev[l] : 0u) : strag_n[l];
    uint32_t incl = c;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      uint32_t v = __shfl_up(incl, off);
      if (l >= off) incl += v;
    }
    uint32_t *pre = second ? s_pre2 : s_pre;
    pre[l] = incl - c;
    if (l == 63) pre[kStragLists] = incl;
  }
  __syncthreads();
  const uint32_t n_cont = s_pre[kStragLists];
  const uint32_t total = n_cont + (CU ? s_pre2[kStragLists] : 0u);
  // Up to kQuadsPerWave entries for every wave of the grid: they start in
  // quads.  A longer list fills the waves' lanes, and a wave moves to quads
  // when its last kQuadsPerWave neurons are left.  (The proposer's stages
  // and its sample log work on whole lanes.)
  constexpr bool kQuad = P <= kQuadMaxPort && !PROP;
  const bool quads = kQuad && !A0.prop_log;
  const uint32_t per_wave =
      quads && total <= vgrid * (kBlock / 64) * kQuadsPerWave ? kQuadsPerWave
                                                              : 64u;
  const uint32_t per_block = per_wave * (kBlock / 64);
  if (vblock * per_block >= total) return;  // whole block beyond the list
  // With the proposer or its sample log every attempt runs in the lane loop
  // below, where late arguments would be read again after each store: it
  // takes them as passed (1e6 spiking neurons, tol 1e-6, 100 ms: 134 -> 132
  // ms in the mean).
  const AeifArgs &A = PROP ? A0 : late_args<AeifArgs>();
  // the pass is a few long dependent chains: its waves issue first when
  // they share a SIMD with the first pass or the delivery
  if (CU) __builtin_amdgcn_s_setprio(3);
  const StepNow sn = step_now(A.out, &A.fold, A.clock);
  const double x1 = A.clock ? sn.t : A.x1;
  // proposer weights, staged once per block (read at every step start)
  __shared__ __attribute__((aligned(16)))
  unsigned char s_pk[PROP ? kPropPkBytes : 16];
  if (PROP && A.prop_pk) {
    const uint4 *src = reinterpret_cast<const uint4 *>(A.prop_pk);
    uint4 *dst = reinterpret_cast<uint4 *>(s_pk);
    for (int k = threadIdx.x; k < kPropPkBytes / 16; k += kBlock)
      dst[k] = src[k];
    __syncthreads();
  }
  const uint32_t n_lanes = vgrid * per_block;
  uint32_t j = lane_id() < per_wave
                   ? vblock * per_block + (threadIdx.x / 64) * per_wave +
                         lane_id()
                   : total;
  const StragRec *list = reinterpret_cast<const StragRec *>(A.strag) +
                        (size_t)(gs & 3) * 2 * kStragLists * A.strag_cap;
  const StragRec *list_prev = list + (size_t)kStragLists * A.strag_cap;
  const float *carry = A.carry + (size_t)(gs & 1) * P * A.n;
  AeifLocal<P> p;
  float y[N], k1[N], scal[N];
  double x = 0.0;
  float h = 0.0f, refr = 0.0f;
  int nsp = 0, n_att = 0, n_acc = 0, n_rej = 0;
  int i = 0;
  float err_last = 1.0f;
  bool need_k1 = false, have = false;
  for (;;) {
    if (!have && j < total) {
      // entries [0, n_cont) resume this step's deferred neurons, the rest
      // are the catch-up neurons; sub-list of an entry: last l with
      // pre[l] <= its index
      const bool catch_up = CU && j >= n_cont;
      const uint32_t jj = catch_up ? j - n_cont : j;
      const uint32_t *pre = catch_up ? s_pre2 : s_pre;
      int lo = 0, hi = kStragLists;
      while (hi - lo > 1) {
        int mid = (lo + hi) >> 1;
        if (pre[mid] <= jj) lo = mid; else hi = mid;
      }
      StragRec r = (catch_up ? list_prev : list)[(size_t)lo * A.strag_cap +
                                                  (jj - pre[lo])];
      j += n_lanes;
      i = (int)r.i;
      nsp = catch_up ? 0 : (int)r.nsp;
      n_att = catch_up ? 0 : (int)r.n_att;
      err_last = catch_up ? 1.0f : r.err_last;
      aeif_load_params<P, UNI>(A, i, p);
      const uint32_t u = (uint32_t)i;
      y[0] = at(A.V, u);
      y[1] = at(A.w, u);
#pragma unroll
      for (int q = 0; q < P; q++) {
        y[2 + 2 * q] = at(A.g[q], u);
        y[3 + 2 * q] = at(A.g1[q], u);
      }
      x = at(A.x, u);
      h = at(A.h, u);
      refr = at(A.refr, u);
      if (catch_up) {
        // the whole step, as the first pass runs it: input fold, then
        // RK5 steps from the stored step size
#pragma unroll
        for (int q = 0; q < P; q++)
          y[3 + 2 * q] =
              __builtin_fmaf(carry[(size_t)q * A.n + i], p.g0[q], y[3 + 2 * q]);
        need_k1 = true;
      } else if (r.flags & 1u) {
        need_k1 = true;  // saved at a step boundary: a new RK5 step starts
      } else {
        aeif_rk5_begin<P>(p, refr, y, r.h_begin, k1, scal);
        need_k1 = false;
      }
      have = true;
    }
    const unsigned long long running = __ballot(have);
    if (running == 0ull) break;
    if constexpr (kQuad) {
      if (quads && __popcll(running) <= kQuadsPerWave &&
          __ballot(j < total) == 0ull) {
        aeif_quad_finish<P, UNI>(late_args<AeifArgs>(), sn, x1, have, i, y,
                                 scal, x, h, refr, nsp, n_att, need_k1, n_acc,
                                 n_rej);
        break;
      }
    }
    bool finished = false, attempted = false;
    float feat[kPropIn];
#pragma unroll
    for (int k = 0; k < kPropIn; k++) feat[k] = 0.0f;
    float err = 1.0f, hh = 0.0f;
    if (PROP && A.prop_pk) {
      // learned step size for the lanes that start an RK5 step; the MLP
      // runs on the whole wave
      bool want = have && need_k1;
      if (want) prop_features<P>(p, y, h, err_last, 1.0f / A.dt, feat);
      if (__ballot(want) != 0ull) {
        float o = prop_mlp_mfma(s_pk, feat);
        if (want) {
          // trust region around the plain controller's step
          float hp = A.dt * exp2f(o) * kPropSafety;
          float lo = h * kPropShrinkMax, hi = h * kPropGrowMax;
          hp = hp > lo ? hp : lo;   // also replaces a NaN output
          hp = hp < hi ? hp : hi;
          h = hp > A.h_min ? hp : A.h_min;
        }
      }
    }
    if (have) {
      if (need_k1) {
        aeif_rk5_begin<P>(p, refr, y, h, k1, scal);
        need_k1 = false;
      }
      if (A.prop_log) prop_features<P>(p, y, h, err_last, 1.0f / A.dt, feat);
      finished = aeif_attempt_and_update<P>(A, x1, p, y, k1, scal, x, h,
                                            refr, nsp, n_att, need_k1, n_acc,
                                            n_rej, err, hh);
      err_last = err;
      attempted = true;
      if (finished) aeif_store_state<P>(A, i, y, x, h, refr);
    }
    if (A.prop_log) {
      // sample: features before the attempt, target log2 of the step that
      // would have given a scaled error of 1
      unsigned long long m = __ballot(attempted);
      if (m != 0ull) {
        uint32_t leader = (uint32_t)(__ffsll((long long)m) - 1);
        unsigned long long base = 0;
        if (lane_id() == leader)
          base = atomicAdd(A.prop_log_n, (unsigned long long)__popcll(m));
        base = __shfl(base, (int)leader);
        unsigned long long slot2 = base + lanes_below(m);
        if (attempted && slot2 < A.prop_log_max) {
          float e = err > CK::err_min ? err : CK::err_min;
          float t = __log2f(hh / A.dt) - 0.2f * __log2f(e);
          float *o = A.prop_log + slot2 * kPropSample;
#pragma unroll
          for (int k = 0; k < kPropIn; k++) o[k] = feat[k];
          o[kPropIn] = t;
          o[kPropIn + 1] = 0.0f;
        }
      }
    }
    emit_spikes(A.out, sn, finished, finished ? i : 0,
                A.i0 + (finished ? i : 0),
                nsp, (float)nsp);
    if (finished) have = false;
  }
  aeif_count<P>(A, n_acc, n_rej);
}

// Overlapped steps: 4 waves per SIMD (128 VGPRs) where the state fits, as
// the pass shares the chip with the first pass and the delivery.  Else no
// limit: it would put some of the state in scratch, at the start of every
// chain.
template <int P, bool UNI, bool PROP, bool CU>
constexpr int kPass2Waves = P <= 2 && UNI && !PROP && CU ? 4 : 1;

template <int P, bool UNI, bool PROP, bool CU>
__global__ __launch_bounds__(kBlock)
__attribute__((amdgpu_waves_per_eu(kPass2Waves<P, UNI, PROP, CU>)))
void aeif_pass2_kernel(AeifArgs A) {
  aeif_pass2_body<P, UNI, PROP, CU>(A, blockIdx.x, gridDim.x);
}

template <bool PLASTIC>
__device__ __forceinline__ void delivery_body(const DeliveryArgs &A,
                                              uint32_t vblock,
                                              uint32_t vgrid);

// End of a captured step: block 0 of its last launch writes the next
// step's clock (computed as the host computes it in SimulationStep).
__device__ __forceinline__ void clock_step(const StepClock *c, StepClock *cn) {
  if (!cn || blockIdx.x != 0 || threadIdx.x != 0) return;
  StepClock v = *c;
  v.pois_T = v.T;
  v.pois_t = v.t;
  v.gs += 1;
  v.it += 1;
  v.T = v.T_base + v.it + 1;
  v.t = v.t0 + v.dt * (double)(v.it + 1);
  *cn = v;
}

// Arguments of a delivery or STDP launch with the step values of the
// clock, when the launch has one.
__device__ __forceinline__ DeliveryArgs clocked(const DeliveryArgs &D) {
  DeliveryArgs A = D;
  if (A.clock) {
    A.gs = A.clock->gs;
    A.slot = (int)(A.gs % A.R);
    A.T = A.clock->T;
  }
  return A;
}
__device__ __forceinline__ RevArgs clocked(const RevArgs &R) {
  RevArgs A = R;
  if (A.clock) {
    A.gs = A.clock->gs;
    A.slot = (int)(A.gs % A.R);
    A.T = A.clock->T;
  }
  return A;
}

// Ring slot of k steps before the step of slot `slot` (0 <= k < R).
__device__ __forceinline__ int slot_back(int slot, int k, int R) {
  const int s = slot - k;
  return s < 0 ? s + R : s;
}

// Second RK5 pass and the delivery of the same step in one launch: blocks
// [0, n2) run the second pass, the others the delivery.  The two are
// independent within a step when no synapse is plastic (the delivery reads
// spikes of earlier steps and writes only the input accumulators), so the
// latency-bound second pass and the atomic-bound delivery share the chip
// without a second stream.
template <int P, bool UNI, bool PROP, bool CU>
__global__ __launch_bounds__(kBlock)
__attribute__((amdgpu_waves_per_eu(kPass2Waves<P, UNI, PROP, CU>)))
void aeif_tail_kernel(AeifArgs A, DeliveryArgs D, uint32_t n2) {
  clock_step(D.clock, D.clock_next);
  if (blockIdx.x < n2)
    aeif_pass2_body<P, UNI, PROP, CU>(A, blockIdx.x, n2);
  else
    delivery_body<false>(clocked(D), blockIdx.x - n2, gridDim.x - n2);
}

// Whole time step of a group of at most kOneLaunchMax neurons: every attempt
// of its neurons, the last ones of a wave on quads of lanes.
template <int P, bool UNI>
__device__ __forceinline__ void aeif_step_body(const AeifArgs &A,
                                               uint32_t vblock) {
  constexpr int N = 2 + 2 * P;
  const StepNow sn = step_now(A.out, &A.fold, A.clock);
  const double x1 = A.clock ? sn.t : A.x1;
  // (the two-pass update finds the next step's list lengths cleared)
  if (vblock == 0 && threadIdx.x < 2 * kStragLists)
    A.strag_n2[2 * kStragLists * ((aeif_gs(A) + 1) & 3) + threadIdx.x] = 0u;
  int i = vblock * kBlock + threadIdx.x;
  const bool active = i < A.n;
  if (!active) i = 0;
  AeifLocal<P> p;
  aeif_load_params<P, UNI>(A, i, p);
  float y[N], k1[N], scal[N];
  const uint32_t u = (uint32_t)i;
  y[0] = at(A.V, u);
  y[1] = at(A.w, u);
#pragma unroll
  for (int q = 0; q < P; q++) {
    y[2 + 2 * q] = at(A.g[q], u);
    y[3 + 2 * q] = at(A.g1[q], u);
  }
  double x = at(A.x, u);
  float h = at(A.h, u);
  float refr = at(A.refr, u);
  if (active) {
    float in[P];
    gather_input<P>(A.fold, sn, A.i0 + i, in);
#pragma unroll
    for (int q = 0; q < P; q++)
      y[3 + 2 * q] = __builtin_fmaf(in[q], p.g0[q], y[3 + 2 * q]);
  }
  int nsp = 0, n_att = 0, n_acc = 0, n_rej = 0;
  bool need_k1 = true, run = active, first = true;
  float err = 1.0f, hh = 0.0f;
  for (;;) {
    const unsigned long long running = lanes_where(run);
    if (running == 0ull) break;
    if (!first && __popcll(running) <= kQuadsPerWave) {
      aeif_quad_finish<P, UNI>(late_args<AeifArgs>(), sn, x1, run, i, y, scal, x, h,
                               refr, nsp, n_att, need_k1, n_acc, n_rej);
      break;
    }
    bool done = false;
    if (run) {
      if (need_k1) {
        aeif_rk5_begin<P>(p, refr, y, h, k1, scal);
        need_k1 = false;
      }
      done = aeif_attempt_and_update<P>(A, x1, p, y, k1, scal, x, h, refr,
                                        nsp, n_att, need_k1, n_acc, n_rej,
                                        err, hh);
      if (done) {
        aeif_store_state<P>(A, i, y, x, h, refr);
        run = false;
      }
    }
    emit_spikes(A.out, sn, done, i, A.i0 + i, nsp, (float)nsp);
    if (first) {
      rk5_count_one(A.cnt1 ? A.cnt1 : A.cnt, n_acc, n_rej);
      n_acc = n_rej = 0;
      first = false;
    }
  }
  aeif_count<P>(A, n_acc, n_rej);
}

// The whole step of a small network in one launch: blocks [0, n1) the group,
// the others the step's atomic delivery, which reads earlier steps' spikes
// and adds to the accumulators that the next step reads (D.acc, not the ones
// that this step's fold reads).  A step of 1000 quiet neurons is two
// dependent launches of 6.6 and 2.8 us otherwise (first pass; empty second
// pass and delivery), and with spiking neurons the chain of the slowest one
// waits for every first attempt.
template <int P, bool UNI>
__global__ __launch_bounds__(kBlock) void aeif_step_kernel(AeifArgs A,
                                                           DeliveryArgs D,
                                                           uint32_t n1) {
  if (blockIdx.x < n1)
    aeif_step_body<P, UNI>(A, blockIdx.x);
  else
    delivery_body<false>(D, blockIdx.x - n1, gridDim.x - n1);
}

// ---------------------------------------------------------------------
// iaf_psc_exp, exact integration (src/iaf_psc_exp.cu:94-119)
// ---------------------------------------------------------------------
// (all threads of a block take part: the spikes leave with one atomic per
// block)
__device__ __forceinline__ void iaf_body(const IafArgs &A, uint32_t vblock) {
  const StepNow sn = step_now(A.out, &A.fold, A.clock);
  int i = vblock * kBlock + threadIdx.x;
  bool active = i < A.n;
  int ii = active ? i : 0;
  int node = A.i0 + ii;
  int nsp = 0;
  if (active) {
    float in[2];
    gather_input<2>(A.fold, sn, node, in);
    float I_ex = A.I_ex[i] + in[0];
    float I_in = A.I_in[i] + in[1];
    if (A.do_step) {
      float V = A.V[i];
      float refr = A.refr[i];
      if (refr > 0.0f) {
        refr -= 1.0f;
      } else {
        float v = V * pf(A.P22, i);
        v = __builtin_fmaf(I_ex, pf(A.P21ex, i), v);
        v = __builtin_fmaf(I_in, pf(A.P21in, i), v);
        v = __builtin_fmaf(pf(A.I_e, i), pf(A.P20, i), v);
        V = v;
      }
      I_ex = I_ex * pf(A.P11ex, i);
      I_in = I_in * pf(A.P11in, i);
      if (V >= pf(A.Theta, i)) {
        nsp = 1;
        V = pf(A.V_reset, i);
        refr = (float)(int)roundf(pf(A.t_ref, i) / A.dt);
      }
      A.V[i] = V;
      A.refr[i] = refr;
    }
    A.I_ex[i] = I_ex;
    A.I_in[i] = I_in;
  }
  if (!A.do_step) return;
  emit_spikes_block(A.out, sn, active, ii, node, nsp, 1.0f);
}

__global__ __launch_bounds__(kBlock) void iaf_kernel(IafArgs A) {
  iaf_body(A, blockIdx.x);
}

// Small networks: the update and the step's atomic delivery in one launch,
// as aeif_step_kernel.
__global__ __launch_bounds__(kBlock) void iaf_step_kernel(IafArgs A,
                                                          DeliveryArgs D,
                                                          uint32_t n1) {
  if (blockIdx.x < n1)
    iaf_body(A, blockIdx.x);
  else
    delivery_body<false>(D, blockIdx.x - n1, gridDim.x - n1);
}

// ---------------------------------------------------------------------
// spike_detector / parrot_neuron
// ---------------------------------------------------------------------
__global__ __launch_bounds__(kBlock) void relay_kernel(RelayArgs A) {
  const StepNow sn = step_now(A.out, &A.fold, A.clock);
  int i = blockIdx.x * kBlock + threadIdx.x;
  bool active = i < A.n;
  int ii = active ? i : 0;
  int node = A.i0 + ii;
  int nsp = 0;
  float height = 0.0f;
  if (active) {
    float in[2];
    if (A.parrot) {
      gather_input<2>(A.fold, sn, node, in);
    } else {
      float in1[1];
      gather_input<1>(A.fold, sn, node, in1);
      in[0] = in1[0];
    }
    float input = A.input[i] + in[0];
    if (A.do_step) {
      float sh = input;
      float hold = pf(A.hold, i);
      if (A.parrot) {
        A.out_var[i] = sh;
        if (sh != 0.0f) {
          if (hold == 0.0f) sh = 1.0f;
          input = 0.0f;
          nsp = 1;
          height = sh;
        }
      } else {
        if (sh != 0.0f) {
          if (hold == 0.0f) sh = 1.0f;
          input = 0.0f;
        }
        A.out_var[i] = sh;
      }
    }
    A.input[i] = input;
  }
  if (!A.do_step || !A.parrot) return;
  emit_spikes(A.out, sn, active, ii, node, nsp, height);
}

// ---------------------------------------------------------------------
// spike_generator (src/spike_generator.cu:37-55)
// ---------------------------------------------------------------------
__global__ __launch_bounds__(kBlock) void spikegen_kernel(SpikeGenArgs A) {
  const StepNow sn = step_now(A.out, nullptr, A.clock);
  const long long it = A.clock ? A.clock->it : A.it;
  int i = blockIdx.x * kBlock + threadIdx.x;
  bool active = i < A.n;
  int ii = active ? i : 0;
  int nsp = 0;
  float height = 0.0f;
  if (active) {
    int k = A.next[i];
    if (k < A.n_spikes[i] && (long long)A.time_idx[A.first[i] + k] == it) {
      nsp = 1;
      height = A.height[A.first[i] + k];
      A.next[i] = k + 1;
    }
  }
  emit_spikes(A.out, sn, active, ii, A.i0 + ii, nsp, height);
}

// ---------------------------------------------------------------------
// CreatePoissonGenerator nodes (src/poisson.cu:27-54): Threefry word at
// counter (node, T mod 2^32), key (seed_lo ^ kLegacyPoissonTag, seed_hi +
// T / 2^32), inverted through the CDF table.
// The reference pushes these spikes before it advances the step's time
// (src/neurongpu.cu:461-470), so they carry the previous step's time index
// and neural time; they enter the same ring slot as this step's spikes.
// ---------------------------------------------------------------------
__global__ __launch_bounds__(kBlock) void legacy_pois_kernel(LegacyPoisArgs A) {
  StepNow sn = step_now(A.out, nullptr, A.clock);
  const long long it = A.clock ? A.clock->it : A.it;
  const double t0 = A.clock ? A.clock->t0 : A.t0;
  const double dt = A.clock ? A.clock->dt : A.dt;
  const long long T = sn.T;
  sn.T = T - 1;
  sn.t = t0 + dt * (double)it;
  int i = blockIdx.x * kBlock + threadIdx.x;
  bool active = i < A.n;
  int ii = active ? i : 0;
  int node = A.i0 + ii;
  int nsp = 0;
  float height = 0.0f;
  if (active) {
    uint32_t u = dev_threefry2x32_w0(
        (uint32_t)node, (uint32_t)T, A.key0 ^ kLegacyPoissonTag,
        A.key1 + (uint32_t)((uint64_t)T >> 32));
    int k = 0;
    while (u > A.tab[k]) k++;   // the table ends with 0xFFFFFFFF
    if ((float)k > A.max_count) k = 0;
    if (k > 0) {
      nsp = 1;
      height = (float)k;
    }
  }
  emit_spikes(A.out, sn, active, ii, node, nsp, height);
}

// ---------------------------------------------------------------------
// Delivery.  Pairs (spike, delay slot d) due at global step gs are the
// spikes of ring slot gs-1-d combined with the source's synapse segment of
// delay index d.  Wavefronts take tiles of 64 pairs; a wavefront scans the
// 64 segment sizes, then its lanes stream the flattened synapse range of
// the tile (consecutive lanes read consecutive 8-byte records) and add
// height*weight into the target accumulators.
// ---------------------------------------------------------------------
constexpr int kMaxDelaySlots = 4096;  // checked on the host at calibration

// Block prologue of every delivery kernel: s_pre[d] = number of (spike,
// delay) pairs with delay slot < d due this step (d = 0..D), from the ring
// counts of slots gs-1-d.  Virtual block 0 also clears the ring counter of
// the slot the next step fills (slot gs+1 is never read in this step).
// Returns the number of pairs.  BS: threads per block; s_part holds BS
// entries and may be used again after the call.
template <int BS = kBlock>
__device__ __forceinline__ uint32_t delivery_prologue(const DeliveryArgs &A,
                                                      uint32_t vblock,
                                                      uint32_t *s_pre,
                                                      uint32_t *s_part) {
  const int D = A.D;
  const int tid = threadIdx.x;
  // spikes of delay slot d due this step (slot gs-1-d; D <= R - 2)
  auto due = [&](int d) -> uint32_t {
    return (long long)d < A.gs ? A.ring_n[slot_back(A.slot, d + 1, A.R)] : 0u;
  };
  const int next = A.slot + 1 == A.R ? 0 : A.slot + 1;
  if (D <= 64) {
    // one wave: scan of the D counts through cross-lane shuffles
    if (tid < 64) {
      const uint32_t n = tid < D ? due(tid) : 0u;
      uint32_t incl = n;
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        uint32_t v = __shfl_up(incl, off);
        if (tid >= off) incl += v;
      }
      if (tid < D) s_pre[tid] = incl - n;
      if (tid == 63) s_pre[D] = incl;
    }
    __syncthreads();
    if (vblock == 0 && tid == 0) A.ring_n[next] = 0u;
    return s_pre[D];
  }
  // per-thread partial sums of the due spike counts over d
  const int per = (D + BS - 1) / BS;
  uint32_t run = 0;
  for (int k = 0; k < per; k++) {
    int d = tid * per + k;
    if (d < D) run += due(d);
  }
  s_part[tid] = run;
  __syncthreads();
  // inclusive scan of the block partials (Hillis-Steele in LDS)
  for (int off = 1; off < BS; off <<= 1) {
    uint32_t v = (tid >= off) ? s_part[tid - off] : 0u;
    __syncthreads();
    s_part[tid] += v;
    __syncthreads();
  }
  {
    uint32_t acc = (tid > 0) ? s_part[tid - 1] : 0u;
    for (int k = 0; k < per; k++) {
      int d = tid * per + k;
      if (d < D) {
        s_pre[d] = acc;
        acc += due(d);
      }
    }
    if (tid == BS - 1) s_pre[D] = s_part[BS - 1];
  }
  __syncthreads();
  if (vblock == 0 && tid == 0) A.ring_n[next] = 0u;
  return s_pre[D];
}

// A wave tile whose segments average at least this many synapses is walked
// one (spike, delay) pair at a time.  Measured with 2e6 events per step:
// binned, segments of 48: 39.0 us with the line at 32, 37.2 at 128; tiled,
// segments of 31: 34.2 at 32, 31.7 at 128; of 63: 32.4 at 32, 32.1 at 64,
// 31.6 at 128; of 131: 31.5 at 128, 32.4 at 256.  The atomic delivery is
// the same with all of them.
constexpr uint32_t kLongSegment = 128;

// Synapse segment of (source, delay slot) in the canonical store: its
// records rec[start .. start + cnt).
struct SegLoc {
  __device__ __forceinline__ void operator()(const DeliveryArgs &A,
                                             uint32_t src, int d,
                                             uint32_t &cnt,
                                             unsigned long long &start) const {
    const uint32_t *sg = A.seg + (size_t)src * (A.D + 1) + d;
    const uint32_t o0 = sg[0], o1 = sg[1];
    cnt = o1 - o0;
    start = A.base[src] + o0;
  }
};

// A wave's table of the pairs of its tile, in LDS: per pair with synapses
// the start of its records minus its first event's number in the tile, and
// the spike's height (WIDE: and multiplicity); and one bit per event of the
// tile, set for the last event of each pair.  WIDE: records addressed by 64
// bits, else 32.
template <bool WIDE>
struct PairTable {
  static constexpr int kWords = WIDE ? 64 : 32;   // 64 events each
  struct Wide {
    unsigned long long start;
    float height;
    uint32_t mult;
  };
  struct Narrow {
    uint32_t start;
    float height;
  };
  typename std::conditional<WIDE, Wide, Narrow>::type pair[64];
  unsigned long long last[kWords];
};
static_assert(sizeof(PairTable<false>) * (kTiledBlock / 64) == kTiledScratch,
              "LDS of a tiled block");

// Inclusive sum over the wave by DPP (row shifts, then the row totals
// broadcast), without the LDS latency of shuffles.
__device__ __forceinline__ uint32_t wave_incl_sum(uint32_t v) {
#define NGPU_DPP_ADD(ctrl, rows)                                          \
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, ctrl, rows, 0xF,  \
                                             false)
  NGPU_DPP_ADD(0x111, 0xF);   // row_shr:1
  NGPU_DPP_ADD(0x112, 0xF);   // row_shr:2
  NGPU_DPP_ADD(0x114, 0xF);   // row_shr:4
  NGPU_DPP_ADD(0x118, 0xF);   // row_shr:8
  NGPU_DPP_ADD(0x142, 0xA);   // row_bcast:15 into rows 1 and 3
  NGPU_DPP_ADD(0x143, 0xC);   // row_bcast:31 into rows 2 and 3
#undef NGPU_DPP_ADD
  return v;
}

// Orders a wave's LDS writes before its lanes' later reads (LDS operations
// of a wave run in order; this keeps the compiler from moving them).
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The waves of the virtual grid take equal numbers of wave tiles of pt
// (spike, delay) pairs, pt at most tile_max.  Tile wt takes the pairs wt, wt
// + n_tiles, wt + 2 n_tiles, ...: pairs are numbered by delay slot, and a
// network's delays are rarely uniform, so that runs of consecutive pairs
// would differ in events many times over (1e6 neurons with normal delays:
// from 0 to over 8192 events per 8-wave block, scatter 47 us; with strided
// pairs 22 us).
//
// Plastic networks (not STRIDED) keep runs of consecutive pairs, of the
// largest power of two that still gives every wave a tile: their weights
// are not dyadic, so the order of the additions into an accumulator decides
// the last bit of its sum, and a spiking network amplifies it; this order
// keeps their runs as reproducible as the atomics allow (strided pairs would
// take 1 us off the 12 us delivery of 2e5 neurons).
template <bool STRIDED>
struct TileSplit {
  uint32_t total, pt, n_tiles, wave, n_waves;
  __device__ __forceinline__ uint32_t pair(uint32_t wt, uint32_t lane) const {
    return STRIDED ? lane * n_tiles + wt : wt * pt + lane;
  }
  template <int BS>
  static __device__ __forceinline__ TileSplit make(uint32_t total,
                                                   uint32_t tile_max,
                                                   uint32_t vblock,
                                                   uint32_t vgrid) {
    TileSplit t;
    t.total = total;
    t.wave = vblock * (BS / 64) + threadIdx.x / 64;
    t.n_waves = vgrid * (BS / 64);
    if (!STRIDED) {
      t.pt = 1u << (31 - __clz((int)tile_max));
      while (t.pt > 1 && (total + t.pt - 1) / t.pt < t.n_waves) t.pt >>= 1;
      t.n_tiles = (total + t.pt - 1) / t.pt;
      return t;
    }
    const uint32_t all = t.n_waves * tile_max;
    const uint32_t turns = total > all ? (total + all - 1) / all : 1u;
    t.pt = (total + t.n_waves * turns - 1) / (t.n_waves * turns);
    if (t.pt == 0u) t.pt = 1u;
    t.n_tiles = (total + t.pt - 1) / t.pt;
    return t;
  }
};

// One wave tile: the pairs of its lanes, and their events spread over the
// wave.  emit() calls f(ok, e, syn, rec, height, mult) for 64 events at a
// time (e: the event's number in the tile), in groups of U: the records of a
// group are loaded while the group before it is handed to f.  A lane finds
// its event's pair by counting the pairs that end before the event (the
// running count of the groups before, plus the set bits below its own in
// the group's 64-bit mask) and reads the pair's table entry: two LDS reads
// and a few VALU instructions per 64 events, where a search of the prefix by
// cross-lane reads took 11 of them.  Tiles of long segments (kLongSegment
// on average, or more events than the mask holds) are walked one pair at a
// time.
template <int U, bool WIDE>
struct WaveTile {
  uint32_t cnt = 0, incl = 0, mult = 0, E = 0;
  unsigned long long start = 0, nz = 0;
  float height = 0.0f;

  template <bool STRIDED, class Loc>
  __device__ __forceinline__ void fetch(const DeliveryArgs &A,
                                        const TileSplit<STRIDED> &t,
                                        uint32_t wt,
                                        const uint32_t *s_pre,
                                        const Loc &loc) {
    const uint32_t lane = lane_id();
    const uint32_t pidx = t.pair(wt, lane);
    cnt = 0;
    if (lane < t.pt && pidx < t.total) {
      // delay slot d of this pair: last d with s_pre[d] <= pidx
      int d = 0, hi = A.D;  // s_pre[d] <= pidx < s_pre[hi]
      while (hi - d > 1) {
        const int mid = (d + hi) >> 1;
        if (s_pre[mid] <= pidx) d = mid; else hi = mid;
      }
      const long long e =
          (long long)slot_back(A.slot, d + 1, A.R) * A.cap + (pidx - s_pre[d]);
      const uint32_t src = A.ring_src[e];
      height = A.ring_h[e];
      if (WIDE) mult = A.ring_cnt[e];
      loc(A, src, d, cnt, start);
    }
    incl = wave_incl_sum(cnt);
    E = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
    nz = __ballot(cnt > 0u);
  }

  // Walked one pair at a time (walk), else spread over the wave (spread).
  __device__ __forceinline__ bool long_segments() const {
    return E > 64u * PairTable<WIDE>::kWords ||
           E >= kLongSegment * (uint32_t)__popcll(nz);
  }

  template <class F>
  __device__ __forceinline__ void emit(PairTable<WIDE> &tab,
                                       const unsigned long long *recs,
                                       F &&f) const {
    if (E == 0u) return;
    if (long_segments())
      walk<false>(recs, 0u, E, f);
    else
      spread(tab, recs, f);
  }

  // Events lo .. hi-1 of the tile (PART, else all), one pair at a time, its
  // data broadcast through scalar registers, consecutive lanes on
  // consecutive records.
  template <bool PART, class F>
  __device__ __forceinline__ void walk(const unsigned long long *recs,
                                       uint32_t lo, uint32_t hi,
                                       F &&f) const {
    const uint32_t lane = lane_id();
    const uint32_t pre = incl - cnt;
    unsigned long long m = nz;
    while (m) {
      const int j = __ffsll((unsigned long long)m) - 1;
      m &= m - 1ull;
      const uint32_t c = (uint32_t)__builtin_amdgcn_readlane((int)cnt, j);
      const uint32_t pj = (uint32_t)__builtin_amdgcn_readlane((int)pre, j);
      uint32_t o0 = 0u, o1 = c;
      if (PART) {
        if (pj + c <= lo) continue;
        if (pj >= hi) break;
        o0 = pj < lo ? lo - pj : 0u;
        o1 = hi - pj < c ? hi - pj : c;
      }
      const uint32_t slo =
          (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)start, j);
      const uint32_t shi =
          (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(start >> 32), j);
      const unsigned long long st = ((unsigned long long)shi << 32) | slo;
      const float h = __uint_as_float((uint32_t)__builtin_amdgcn_readlane(
          (int)__float_as_uint(height), j));
      const uint32_t mu = (uint32_t)__builtin_amdgcn_readlane((int)mult, j);
      for (uint32_t o = o0; o < o1; o += 64u * U) {
        unsigned long long syn[U], r[U];
        bool ok[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
          const uint32_t e = o + 64u * u + lane;
          ok[u] = e < o1;
          syn[u] = st + e;
          r[u] = ok[u] ? recs[syn[u]] : 0ull;
        }
#pragma unroll
        for (int u = 0; u < U; u++)
          f(ok[u], pj + o + 64u * u + lane, syn[u], r[u], h, mu);
      }
    }
  }

  template <class F>
  __device__ __forceinline__ void spread(PairTable<WIDE> &tab,
                                         const unsigned long long *recs,
                                         F &&f) const {
    const uint32_t lane = lane_id();
    const uint32_t pre = incl - cnt;
    // the tile's table (every lane has read the one before: its last group
    // was handed over)
    if (lane < (E + 63u) / 64u) tab.last[lane] = 0ull;
    wave_lds_fence();
    if (cnt > 0u) {
      const uint32_t k = lanes_below(nz);
      tab.pair[k].height = height;
      if constexpr (WIDE) {
        tab.pair[k].start = start - pre;
        tab.pair[k].mult = mult;
      } else {
        tab.pair[k].start = (uint32_t)start - pre;
      }
      const uint32_t end = incl - 1u;
      atomicOr(reinterpret_cast<uint32_t *>(tab.last) + (end >> 5),
               1u << (end & 31u));
    }
    wave_lds_fence();
    struct Group {
      unsigned long long r[U];
      unsigned long long syn[U];
      float h[U];
      uint32_t m[U];
    };
    uint32_t before = 0;   // pairs that end before the next group
    auto load = [&](Group &g, uint32_t e0) {
#pragma unroll
      for (int u = 0; u < U; u++) {
        const uint32_t w = e0 / 64u + u;
        // (words past the tile's events are not read)
        const unsigned long long m64 = 64u * w < E ? tab.last[w] : 0ull;
        const uint32_t lo = (uint32_t)m64, hi = (uint32_t)(m64 >> 32);
        const uint32_t k = __builtin_amdgcn_mbcnt_hi(
            hi, __builtin_amdgcn_mbcnt_lo(lo, before));
        before += (uint32_t)__popcll(m64);
        const uint32_t e = 64u * w + lane;
        const bool ok = e < E;
        const auto p = tab.pair[ok ? k : 0u];
        g.h[u] = p.height;
        if constexpr (WIDE) {
          g.m[u] = p.mult;
          g.syn[u] = p.start + e;
        } else {
          g.m[u] = 0u;
          g.syn[u] = (uint32_t)(p.start + e);
        }
        g.r[u] = ok ? recs[g.syn[u]] : 0ull;
      }
    };
    auto give = [&](const Group &g, uint32_t e0) {
#pragma unroll
      for (int u = 0; u < U; u++) {
        const uint32_t e = e0 + 64u * u + lane;
        f(e < E, e, g.syn[u], g.r[u], g.h[u], g.m[u]);
      }
    };
    Group ga, gb;
    load(ga, 0u);
    for (uint32_t e0 = 0;;) {
      const bool more_b = e0 + 64u * U < E;
      if (more_b) load(gb, e0 + 64u * U);
      give(ga, e0);
      if (!more_b) break;
      e0 += 64u * U;
      const bool more_a = e0 + 64u * U < E;
      if (more_a) load(ga, e0 + 64u * U);
      give(gb, e0);
      if (!more_a) break;
      e0 += 64u * U;
    }
  }
};

// Hands the synaptic events of this wave's share of the step to
// f(ok, e, syn, rec, height, mult); returns their number.  BS: threads per
// block; tabs: one table per wave of the block; Loc(src, d, cnt, start)
// locates a pair's records in `recs`.
template <int U, int BS = kBlock, bool WIDE = true, bool STRIDED = true,
          class F, class Loc = SegLoc>
__device__ __forceinline__ unsigned long long deliver_events(
    const DeliveryArgs &A, uint32_t vblock, uint32_t vgrid,
    const uint32_t *s_pre, uint32_t total, PairTable<WIDE> *tabs, F &&f,
    const unsigned long long *recs = nullptr, Loc loc = Loc{}) {
  if (!recs) recs = A.rec;
  const TileSplit<STRIDED> t = TileSplit<STRIDED>::template make<BS>(
      total, (uint32_t)A.tile_max, vblock, vgrid);
  unsigned long long n_events = 0;
  for (uint32_t wt = t.wave; wt < t.n_tiles; wt += t.n_waves) {
    WaveTile<U, WIDE> w;
    w.fetch(A, t, wt, s_pre, loc);
    n_events += w.E;
    w.emit(tabs[threadIdx.x / 64], recs, f);
  }
  return n_events;
}

// Accumulator entry of a record's target and port: port * n_total + target,
// below 20 * 2^26.
__device__ __forceinline__ uint32_t acc_index(uint32_t tp, long long n_total) {
  return (tp >> kPortShift) * (uint32_t)n_total + (tp & kTargetMask);
}

// Dynamic LDS of the delivery kernels: s_pre[D + 1], then (binned
// phases) one counter per bin.
extern __shared__ __align__(16) uint32_t s_dyn[];

inline size_t delivery_lds_bytes(int D, int nb) {
  return sizeof(uint32_t) * ((size_t)D + 1 + (size_t)nb);
}

template <bool PLASTIC>
__device__ __forceinline__ void delivery_body(const DeliveryArgs &A,
                                              uint32_t vblock,
                                              uint32_t vgrid) {
  uint32_t *s_pre = s_dyn;
  __shared__ PairTable<true> s_tab[kBlock / 64];
  const uint32_t total = delivery_prologue(
      A, vblock, s_pre, reinterpret_cast<uint32_t *>(s_tab));
  unsigned long long n_events = deliver_events<2, kBlock, true, !PLASTIC>(
      A, vblock, vgrid, s_pre, total, s_tab,
      [&](bool ok, uint32_t, unsigned long long syn, unsigned long long r,
          float hj, uint32_t mj) {
        if (!ok) return;
        uint32_t tp = (uint32_t)r;
        float w = __uint_as_float((uint32_t)(r >> 32));
        uint32_t tgt = tp & kTargetMask;
        unsafeAtomicAdd(A.acc + acc_index(tp, A.n_total), hj * w);
        if (PLASTIC) {
          int sgp = A.syn_group[syn];
          if (sgp > 0) {
            int type = A.syn_type[sgp - 1];
            const float *prm = A.stdp_param + 8 * (sgp - 1);
            float wn = w;
            for (uint32_t rep = 0; rep < mj; rep++) {
              A.spike_time[syn] = (uint16_t)(A.T & 0xffff);
              long long Dt_int = A.T - A.last_rev[tgt];
              if (Dt_int > 0 && Dt_int < kMaxSynDt)
                wn = dev_syn_update(type, wn, -A.dt * (float)Dt_int, prm);
            }
            if (wn != w)
              reinterpret_cast<uint32_t *>(A.rec + syn)[1] =
                  __float_as_uint(wn);
          }
        }
      });
  if (lane_id() == 0 && n_events) {
    atomicAdd(A.events + (vblock & (kCounterSlots - 1)), n_events);
  }
}

template <bool PLASTIC>
__global__ __launch_bounds__(kBlock) void delivery_kernel(DeliveryArgs A) {
  clock_step(A.clock, A.clock_next);
  delivery_body<PLASTIC>(clocked(A), blockIdx.x, gridDim.x);
}

// ---------------------------------------------------------------------
// Binned delivery (non-plastic networks).  Float atomics on the
// accumulators run at a fixed rate per device whatever the address
// pattern, so when a step carries many events per accumulator entry the
// events are first grouped by accumulator range (bin of kBinLen entries):
//   1 scatter  enumerates the events once.  A block keeps its events
//              (accumulator entry, value) in LDS and counts them per bin;
//              then it reserves its run in every bin's buffer with one
//              atomic per bin and writes the events there, and goes on with
//              its next wave tiles if it has any.  Events beyond a bin's
//              capacity are added with float atomics instead.
//   2 reduce   one block per chunk of events of one bin sums them in LDS
//              (chunk size chosen from the step's event count, see
//              bin_chunk_size, or one chunk per bin when there are at
//              least kSingleChunkBins bins of about equal size; then the
//              sum phase has nothing to do); a bin of one chunk is added to
//              the accumulators directly, otherwise the partial sums are
//              written out
//   3 sum      bins of several chunks: accumulators += sum of partials;
//              clears the bins' counts for the next step.
// ---------------------------------------------------------------------

constexpr int kReduceBlock = 1024;
constexpr int kBinBlock = 512;  // threads per block of the scatter
// events of a tile of long segments that a wave buffers at a time: a
// wave's share of the block's buffer
constexpr uint32_t kBinPiece = kBinBuffer / (kBinBlock / 64);

// Float add into LDS by compare-and-swap.  On gfx950 the LDS float atomic
// add runs at about a twelfth of the rate of the integer atomics and of a
// plain read-modify-write; a CAS loop whose first attempt nearly always
// succeeds (random addresses in a table of kBinLen entries) is faster.
__device__ __forceinline__ void lds_add_f32(float *p, float v) {
  uint32_t *u = reinterpret_cast<uint32_t *>(p);
  uint32_t old = *u;
  for (;;) {
    uint32_t nw = __float_as_uint(__uint_as_float(old) + v);
    uint32_t prev = atomicCAS(u, old, nw);
    if (prev == old) break;
    old = prev;
  }
}

__device__ __forceinline__ uint32_t bin_chunk_size(unsigned long long n_ev) {
  unsigned long long ch = (n_ev + kReduceChunks - 1) / kReduceChunks;
  ch = (ch + 1023ull) & ~1023ull;
  if (ch < (unsigned long long)kBinChunkMin) ch = kBinChunkMin;
  if (ch > 0x40000000ull) ch = 0x40000000ull;
  return (uint32_t)ch;
}

// Exclusive scan of val(0..n-1) by one block of BS threads: put(b, sum of
// val(b') for b' < b).  Returns the total (below 2^32).  s_part: BS / 64
// entries; the values put are visible to the block after its next barrier.
template <int BS, class F, class G>
__device__ __forceinline__ uint32_t block_scan_excl(int n, F val, G put,
                                                    uint32_t *s_part) {
  const int tid = threadIdx.x;
  const int per = (n + BS - 1) / BS;
  uint32_t run = 0;
  for (int k = 0; k < per; k++) {
    const int b = tid * per + k;
    if (b < n) run += val(b);
  }
  const uint32_t incl = wave_incl_sum(run);
  __syncthreads();            // s_part may be in use from a call before
  if ((tid & 63) == 63) s_part[tid / 64] = incl;
  __syncthreads();
  uint32_t acc = incl - run, total = 0;
#pragma unroll
  for (int w = 0; w < BS / 64; w++) {
    const uint32_t v = s_part[w];
    acc += w < tid / 64 ? v : 0u;
    total += v;
  }
  for (int k = 0; k < per; k++) {
    const int b = tid * per + k;
    if (b < n) {
      const uint32_t v = val(b);
      put(b, acc);
      acc += v;
    }
  }
  return total;
}

// LDS of the scatter: events, pair prefix, counts and cursors of the bins.
inline size_t scatter_lds_bytes(int D, int nb) {
  return sizeof(unsigned long long) * kBinBuffer +
         sizeof(uint32_t) * ((size_t)D + 1 + 2 * (size_t)nb);
}

// What bounds it: the enumeration's chain of dependent loads (ring entry,
// segment bounds, records) and the stores to many bins.  A block of 8 waves
// with room for 8192 events in LDS, two blocks a CU; the host sizes the grid
// so that a block's events fit its buffer once.  The former version
// enumerated twice (counts, a scan over the blocks, then the events at
// their final places).
__global__ __launch_bounds__(kBinBlock) void bin_scatter_kernel(
    BinArgs B0, DeliveryArgs A0) {
  const DeliveryArgs A = clocked(A0);
  const int nb = B0.nb;
  unsigned long long *s_ev = reinterpret_cast<unsigned long long *>(s_dyn);
  uint32_t *s_pre = s_dyn + 2 * kBinBuffer;
  uint32_t *s_cnt = s_pre + A.D + 1;   // events of the round per bin; then
                                       // the next one's place in the order
  uint32_t *s_to = s_cnt + nb;       // from that place to the bin's buffer
  __shared__ PairTable<true> s_tab[kBinBlock / 64];
  __shared__ uint32_t s_part[kBinBlock / 64];
  __shared__ uint32_t s_n;             // events in the buffer
  for (int b = threadIdx.x; b < nb; b += kBinBlock) s_cnt[b] = 0u;
  if (threadIdx.x == 0) s_n = 0u;
  const uint32_t total = delivery_prologue<kBinBlock>(
      A, blockIdx.x, s_pre, reinterpret_cast<uint32_t *>(s_tab));
  TileSplit<true> t = TileSplit<true>::make<kBinBlock>(
      total, (uint32_t)A.tile_max, blockIdx.x, gridDim.x);
  // Tiles for at most half of the waves: spread over the blocks, whose
  // buffers then take them side by side (50 pairs of 20000 events: 206 us
  // per step in 7 blocks, 88 in 50).  More tiles stay in order, a block's
  // next to each other in the ring (1e6 neurons: 0.9 % of a step).
  if (t.n_tiles <= t.n_waves / 2u)
    t.wave = threadIdx.x / 64 * gridDim.x + blockIdx.x;
  unsigned long long n_events = 0;
  uint32_t wt = t.wave;
  WaveTile<4, true> w;
  bool loaded = false;
  uint32_t done = 0;                   // events of the tile in the buffer
  for (;;) {
    // round: every wave buffers its tiles until one does not fit
    bool waits = false;
    while (wt < t.n_tiles && !waits) {
      if (!loaded) {
        w.fetch(A, t, wt, s_pre, SegLoc{});
        n_events += w.E;
        loaded = true;
      }
      // Tiles of long segments go to the buffer in pieces, so that their
      // size is not limited and the waves of a block fill it together
      // (one step of 3e7 events in 40: 51 us per step when such a tile was
      // added with float atomics, 20 in pieces; 300 pairs of 6000 events:
      // 167 and 56 us).
      const bool whole = !w.long_segments();
      const uint32_t rest = w.E - done;
      const uint32_t c = whole || rest < kBinPiece ? rest : kBinPiece;
      uint32_t at0 = 0;
      if (lane_id() == 0) at0 = atomicAdd(&s_n, c);
      at0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)at0);
      if (at0 + c > (uint32_t)kBinBuffer) {
        // (the places from at0 on stay unused in this round)
        if (lane_id() == 0) atomicMin(&s_n, at0);
        waits = true;
        continue;
      }
      auto put = [&](bool ok, uint32_t e, unsigned long long,
                     unsigned long long r, float hj, uint32_t) {
        if (!ok) return;
        const uint32_t idx = acc_index((uint32_t)r, A.n_total);
        const float v = hj * __uint_as_float((uint32_t)(r >> 32));
        s_ev[at0 + (e - done)] =
            ((unsigned long long)__float_as_uint(v) << 32) | idx;
        atomicAdd(&s_cnt[idx >> kBinShift], 1u);
      };
      if (whole) {
        w.spread(s_tab[threadIdx.x / 64], A.rec, put);
      } else {
        w.template walk<true>(A.rec, done, done + c, put);
        done += c;
        if (done < w.E) continue;
        done = 0;
      }
      loaded = false;
      wt += t.n_waves;
    }
    const int more = __syncthreads_or(waits ? 1 : 0);
    // reserve the round's runs in the bins' buffers
    // (read here: through the enumeration they would be spilled)
    const BinArgs &L = late_args<BinArgs>();
    uint32_t *const tot = L.tot;
    const uint32_t *const off = L.off;
    unsigned long long *const out = L.ev;
    int full = 0;                      // some run leaves its bin's room
    (void)block_scan_excl<kBinBlock>(
        nb, [&](int b) -> uint32_t { return s_cnt[b]; },
        [&](int b, uint32_t first) {
          const uint32_t c = s_cnt[b];
          uint32_t to = 0u;
          if (c) {
            to = off[b] + atomicAdd(&tot[(size_t)b * kBinStride], c);
            full |= to + c > off[b + 1];
          }
          s_to[b] = to - first;
          s_cnt[b] = first;
        },
        s_part);
    const uint32_t n = s_n;
    full = __syncthreads_or(full);
    // order the events by bin, in place through registers, so that a bin's
    // run leaves as whole cache lines
    constexpr int kPer = kBinBuffer / kBinBlock;
    unsigned long long ev[kPer];
#pragma unroll
    for (int k = 0; k < kPer; k++) {
      const uint32_t j = k * kBinBlock + threadIdx.x;
      ev[k] = j < n ? s_ev[j] : 0ull;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kPer; k++)
      if (k * kBinBlock + threadIdx.x < n)
        s_ev[atomicAdd(&s_cnt[(uint32_t)ev[k] >> kBinShift], 1u)] = ev[k];
    __syncthreads();
    for (int b = threadIdx.x; b < nb; b += kBinBlock) s_cnt[b] = 0u;
    auto leave = [&](bool room) {
      for (uint32_t j = threadIdx.x; j < n; j += kBinBlock) {
        const unsigned long long e = s_ev[j];
        const uint32_t idx = (uint32_t)e, b = idx >> kBinShift;
        const uint32_t pos = j + s_to[b];
        if (room || pos < off[b + 1])
          out[pos] = (e & 0xFFFFFFFF00000000ull) | (idx & (kBinLen - 1));
        else
          unsafeAtomicAdd(A.acc + idx, __uint_as_float((uint32_t)(e >> 32)));
      }
    };
    // (one check for the round: with one per event the scatter of the
    // million spiking neurons took 34 us, 31.9 with this)
    if (full)
      leave(false);
    else
      leave(true);
    if (!more) break;
    __syncthreads();
    if (threadIdx.x == 0) s_n = 0u;
    __syncthreads();
  }
  if (lane_id() == 0 && n_events) {
    atomicAdd(A.events + (blockIdx.x & (kCounterSlots - 1)), n_events);
  }
}

// Events of bin b in its buffer.
__device__ __forceinline__ uint32_t bin_events(const BinArgs &B, int b) {
  const uint32_t n = B.tot[(size_t)b * kBinStride];
  const uint32_t room = B.off[b + 1] - B.off[b];
  return n < room ? n : room;
}

__global__ __launch_bounds__(kReduceBlock) void bin_reduce_kernel(BinArgs B,
                                                                  float *acc) {
  __shared__ float s_a[kBinLen];
  __shared__ uint32_t s_part[kReduceBlock / 64];
  __shared__ uint32_t s_red[2][kReduceBlock / 64];
  __shared__ int s_multi;              // some bin has more than one chunk
  uint32_t *s_c = s_dyn;               // first chunk of every bin [nb + 1]
  // events of the step and of the largest bin
  uint32_t n_ev = 0, mx = 0;
  for (int b = threadIdx.x; b < B.nb; b += kReduceBlock) {
    const uint32_t n = bin_events(B, b);
    n_ev += n;
    mx = n > mx ? n : mx;
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    n_ev += __shfl_xor(n_ev, off);
    const uint32_t o = __shfl_xor(mx, off);
    mx = o > mx ? o : mx;
  }
  if ((threadIdx.x & 63) == 0) {
    s_red[0][threadIdx.x / 64] = n_ev;
    s_red[1][threadIdx.x / 64] = mx;
  }
  if (threadIdx.x == 0) s_multi = 0;
  __syncthreads();
  n_ev = mx = 0;
#pragma unroll
  for (int w = 0; w < kReduceBlock / 64; w++) {
    n_ev += s_red[0][w];
    mx = s_red[1][w] > mx ? s_red[1][w] : mx;
  }
  // chunk size: about kReduceChunks chunks in all (at least kBinChunkMin
  // events each), so that the reduction fills the device whatever the
  // step's event count; with many bins of about equal size one chunk per
  // bin: the reduction still has a block for most CUs, and no partial sums
  // are written and summed
  uint32_t ch = bin_chunk_size(n_ev);
  const bool single =
      B.nb >= kSingleChunkBins &&
      (unsigned long long)mx * B.nb <= 2ull * n_ev && mx <= 0x40000000u;
  uint32_t n_chunk = (uint32_t)B.nb;   // chunk b is bin b
  if (single) {
    ch = mx;
  } else {
    n_chunk = block_scan_excl<kReduceBlock>(
        B.nb,
        [&](int b) -> uint32_t {
          const uint32_t c = (uint32_t)(
              ((unsigned long long)bin_events(B, b) + ch - 1u) / ch);
          if (c > 1u) s_multi = 1;
          return c;
        },
        [&](int b, uint32_t first) { s_c[b] = first; }, s_part);
    if (threadIdx.x == 0) s_c[B.nb] = n_chunk;
    __syncthreads();
  }
  if (blockIdx.x == 0) {     // for the sum phase
    if (!single)
      for (int b = threadIdx.x; b <= B.nb; b += kReduceBlock)
        B.cstart[b] = s_c[b];
    if (threadIdx.x == 0) B.meta[0] = (uint32_t)s_multi;
  }
  for (uint32_t w = blockIdx.x; w < n_chunk; w += gridDim.x) {
    int b = (int)w;
    uint32_t k = 0, nc = 1;
    if (!single) {
      // bin of chunk w: last b with s_c[b] <= w (it has >= 1 chunk)
      int lo = 0, hi = B.nb;  // s_c[lo] <= w < s_c[hi]
      while (hi - lo > 1) {
        int mid = (lo + hi) >> 1;
        if (s_c[mid] <= w) lo = mid; else hi = mid;
      }
      b = lo;
      k = w - s_c[b];
      nc = s_c[b + 1] - s_c[b];
    }
    const unsigned long long *ev = B.ev + B.off[b];
    const uint32_t e_end = bin_events(B, b);
    const uint32_t e0 = k * ch;
    const uint32_t e1 = (e_end - e0 < ch) ? e_end : e0 + ch;
    for (int i = threadIdx.x; i < kBinLen; i += kReduceBlock) s_a[i] = 0.0f;
    __syncthreads();
    uint32_t e = e0 + threadIdx.x;
    for (; e + 3u * kReduceBlock < e1; e += 4u * kReduceBlock) {
      unsigned long long v[4];
#pragma unroll
      for (int u = 0; u < 4; u++) v[u] = ev[e + (uint32_t)u * kReduceBlock];
#pragma unroll
      for (int u = 0; u < 4; u++)
        lds_add_f32(&s_a[(uint32_t)v[u]],
                    __uint_as_float((uint32_t)(v[u] >> 32)));
    }
    for (; e < e1; e += kReduceBlock) {
      unsigned long long v = ev[e];
      lds_add_f32(&s_a[(uint32_t)v], __uint_as_float((uint32_t)(v >> 32)));
    }
    __syncthreads();
    const long long a0 = (long long)b * kBinLen;
    const long long lim_ll = B.acc_n - a0;
    const int lim = lim_ll < kBinLen ? (int)lim_ll : kBinLen;
    if (nc == 1) {
      for (int i = threadIdx.x; i < lim; i += kReduceBlock) {
        float x = s_a[i];
        if (x != 0.0f) acc[a0 + i] += x;
      }
    } else {
      float *pp = B.part + (size_t)w * kBinLen;
      for (int i = threadIdx.x; i < kBinLen; i += kReduceBlock) pp[i] = s_a[i];
    }
    __syncthreads();
  }
}

__global__ __launch_bounds__(kBlock) void bin_sum_kernel(
    BinArgs B, float *acc, const StepClock *clock, StepClock *clock_next) {
  clock_step(clock, clock_next);
  for (long long b = (long long)blockIdx.x * kBlock + threadIdx.x; b < B.nb;
       b += (long long)gridDim.x * kBlock)
    B.tot[b * kBinStride] = 0u;
  if (B.meta[0] == 0u) return;  // every bin was summed by one chunk
  for (long long i = (long long)blockIdx.x * kBlock + threadIdx.x;
       i < B.acc_n; i += (long long)gridDim.x * kBlock) {
    const int b = (int)(i >> kBinShift);
    const uint32_t c0 = B.cstart[b], c1 = B.cstart[b + 1];
    if (c1 - c0 <= 1u) continue;
    const int j = (int)(i & (kBinLen - 1));
    float sum = 0.0f;
    for (uint32_t c = c0; c < c1; c++) sum += B.part[(size_t)c * kBinLen + j];
    acc[i] += sum;
  }
}

// ---------------------------------------------------------------------
// Tiled delivery (non-plastic).  Block b owns accumulator tile b / G in
// LDS and takes share b % G of the step's (spike, delay) pairs; for each
// pair it reads only the records of its tile (a contiguous group of the
// tile-major store), so every record is read once per step by one block.
// The same pair enumeration as the other delivery kernels, over the G
// blocks of the tile.
// ---------------------------------------------------------------------
struct TileLoc {
  const uint32_t *off;
  uint32_t T, t;
  __device__ __forceinline__ void operator()(const DeliveryArgs &A,
                                             uint32_t src, int d,
                                             uint32_t &cnt,
                                             unsigned long long &start) const {
    const size_t k = ((size_t)src * (size_t)A.D + (size_t)d) * T + t;
    const uint32_t o0 = off[k], o1 = off[k + T];
    cnt = o1 - o0;
    start = o0;
  }
};

// FIXED: 64-bit fixed-point sums with LDS integer atomics (no return
// value, no retry loop); else float sums by compare-and-swap.
template <bool FIXED>
__global__ __launch_bounds__(kTiledBlock) void tiled_delivery_kernel(
    DeliveryArgs A0, TileArgs B) {
  const DeliveryArgs A = clocked(A0);
  __shared__ PairTable<false> s_tab[kTiledBlock / 64];
  __shared__ int s_big;   // a float atomic went to the accumulator
  // dynamic LDS: the tile (2^tile_shift floats or 64-bit sums), then the
  // pair prefix
  const int TL = 1 << B.tile_shift;
  float *s_acc = reinterpret_cast<float *>(s_dyn);
  unsigned long long *s_q = reinterpret_cast<unsigned long long *>(s_dyn);
  uint32_t *s_pre = s_dyn + (FIXED ? 2 * TL : TL);
  const uint32_t tk = B.blk[blockIdx.x];
  const uint32_t t = tk & 0xFFFFu, k = tk >> 16;
  const uint32_t g0 = B.tg[t], G = B.tg[t + 1] - g0;
  for (int i = threadIdx.x; i < TL; i += kTiledBlock) {
    if (FIXED)
      s_q[i] = 0ull;
    else
      s_acc[i] = 0.0f;
  }
  if (threadIdx.x == 0) s_big = 0;
  // (the prologue's barriers order the clearing before the first add)
  const uint32_t total =
      delivery_prologue<kTiledBlock>(A, blockIdx.x, s_pre,
                                     reinterpret_cast<uint32_t *>(s_tab));
  const long long a0 = (long long)t << B.tile_shift;
  auto add = [&](bool ok, uint32_t, unsigned long long, unsigned long long r,
                 float hj, uint32_t) {
    if (!ok) return;
    const uint32_t loc = (uint32_t)r;   // entry of the tile
    const float v = hj * __uint_as_float((uint32_t)(r >> 32));
    if (FIXED) {
      if (fabsf(hj) <= B.h_max) {
        // exact: v * 2^F is v with a larger exponent, below 2^62
        const long long q = __float2ll_rn(v * B.q_scale);
        atomicAdd(&s_q[loc], (unsigned long long)q);
      } else {
        unsafeAtomicAdd(A.acc + a0 + loc, v);
        s_big = 1;
      }
    } else {
      lds_add_f32(&s_acc[loc], v);
    }
  };
  const unsigned long long n_events =
      deliver_events<4, kTiledBlock, false, true, decltype(add) &, TileLoc>(
          A, k, G, s_pre, total, s_tab, add, B.trec,
          TileLoc{B.off, (uint32_t)B.T, t});
  __syncthreads();
  const long long lim_ll = B.acc_n - a0;
  const int lim = lim_ll < TL ? (int)lim_ll : TL;
  if (G == 1) {
    // after a float atomic into this tile's entries the flush adds with
    // atomics too (they and plain accesses are not ordered)
    const bool big = FIXED && s_big;
    for (int i = threadIdx.x; i < lim; i += kTiledBlock) {
      const float x =
          FIXED ? (float)(long long)s_q[i] * B.q_inv : s_acc[i];
      if (x == 0.0f) continue;
      if (big)
        unsafeAtomicAdd(A.acc + a0 + i, x);
      else
        A.acc[a0 + i] += x;
    }
  } else if (FIXED) {
    long long *pq = B.part_q + (size_t)(g0 + k) * TL;
    for (int i = threadIdx.x; i < TL; i += kTiledBlock)
      pq[i] = (long long)s_q[i];
  } else {
    float *pp = B.part + (size_t)(g0 + k) * TL;
    for (int i = threadIdx.x; i < TL; i += kTiledBlock) pp[i] = s_acc[i];
  }
  if (lane_id() == 0 && n_events)
    atomicAdd(A.events + (blockIdx.x & (kCounterSlots - 1)), n_events);
}

// Sum of the G partial tiles of every accumulator entry (G > 1); the last
// launch of the step (writes the next step's clock when captured).
__global__ __launch_bounds__(kBlock) void tiled_sum_kernel(
    TileArgs B, float *acc, const StepClock *clock, StepClock *clock_next) {
  clock_step(clock, clock_next);
  if (!B.split) return;
  // four entries a thread (16-byte loads; a tile holds a multiple of 4),
  // the partials of each entry added in block order
  const long long TL = 1ll << B.tile_shift;
  const long long n4 = (B.acc_n + 3) >> 2;
  for (long long i4 = (long long)blockIdx.x * kBlock + threadIdx.x; i4 < n4;
       i4 += (long long)gridDim.x * kBlock) {
    const long long i = i4 << 2;
    const long long t = i >> B.tile_shift;
    const uint32_t g0 = B.tg[t], G = B.tg[t + 1] - g0;
    if (G <= 1) continue;   // that tile's block added its sums
    const size_t o = (size_t)g0 * TL + (size_t)(i & (TL - 1));
    float sum[4];
    if (B.fixed) {
      long long q[4] = {0, 0, 0, 0};
#pragma unroll 4
      for (uint32_t k = 0; k < G; k++) {
        const longlong2 *p =
            reinterpret_cast<const longlong2 *>(B.part_q + o + (size_t)k * TL);
        const longlong2 a = p[0], b = p[1];
        q[0] += a.x;
        q[1] += a.y;
        q[2] += b.x;
        q[3] += b.y;
      }
      for (int j = 0; j < 4; j++) sum[j] = (float)q[j] * B.q_inv;
    } else {
      float4 s = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll 8
      for (uint32_t k = 0; k < G; k++) {
        const float4 x =
            *reinterpret_cast<const float4 *>(B.part + o + (size_t)k * TL);
        s.x += x.x;
        s.y += x.y;
        s.z += x.z;
        s.w += x.w;
      }
      sum[0] = s.x;
      sum[1] = s.y;
      sum[2] = s.z;
      sum[3] = s.w;
    }
    for (int j = 0; j < 4; j++)
      if (i + j < B.acc_n && sum[j] != 0.0f) acc[i + j] += sum[j];
  }
}

// ---------------------------------------------------------------------
// Post-synaptic STDP (src/rev_spike.cu:41-75): every node whose spike
// reaches its dendrites this step updates its plastic incoming synapses.
// One wavefront per candidate node; lanes stride over its inputs.
// ---------------------------------------------------------------------
__global__ __launch_bounds__(kBlock) void rev_kernel(RevArgs A0) {
  clock_step(A0.clock, A0.clock_next);
  const RevArgs A = clocked(A0);
  // one block per spiking node: its incoming plastic synapses are
  // independent (each has this node as its only target), so all 256 lanes
  // walk the reverse index together
  for (int k = 0; k <= A.max_den; k++) {
    if (A.gs < k) break;
    const long long slot = slot_back(A.slot, k, A.R);
    uint32_t n = A.ring_n[slot];
    for (uint32_t e = blockIdx.x; e < n; e += gridDim.x) {
      uint32_t node = A.ring_src[slot * A.cap + e];
      if (A.den_idx[node] != k) continue;
      if (A.last_rev[node] != A.T) continue;
      unsigned long long r0 = A.rev_ptr[node], r1 = A.rev_ptr[node + 1];
      uint16_t ti = (uint16_t)(A.T & 0xffff);
      for (unsigned long long r = r0 + threadIdx.x; r < r1; r += kBlock) {
        uint32_t syn = A.rev_idx[r];
        int sgp = A.syn_group[syn];
        if (sgp <= 0) continue;
        uint16_t st = A.spike_time[syn];
        uint16_t Dt_int = (uint16_t)(ti - st);
        if (Dt_int < kMaxSynDt) {
          uint32_t *wp = reinterpret_cast<uint32_t *>(A.rec + syn) + 1;
          float w = __uint_as_float(*wp);
          float wn = dev_syn_update(A.syn_type[sgp - 1], w,
                                    A.dt * (float)Dt_int,
                                    A.stdp_param + 8 * (sgp - 1));
          *wp = __float_as_uint(wn);
        }
      }
    }
  }
}

// Spikes of nodes with a dendritic delay of k > 0 steps reach the
// dendrites k steps after emission (src/spike_buffer.cu:276-278,299-301):
// mark them before this step's delivery reads last_rev.
__global__ __launch_bounds__(kBlock) void den_rev_kernel(RevArgs A0) {
  const RevArgs A = clocked(A0);
  for (int k = 1; k <= A.max_den; k++) {
    if (A.gs < k) break;
    const long long slot = slot_back(A.slot, k, A.R);
    uint32_t n = A.ring_n[slot];
    for (uint32_t e = blockIdx.x * kBlock + threadIdx.x; e < n;
         e += gridDim.x * kBlock) {
      uint32_t node = A.ring_src[slot * A.cap + e];
      if (A.den_idx[node] == k) A.last_rev[node] = A.T;
    }
  }
}

// ---------------------------------------------------------------------
// Step clock of captured steps
// ---------------------------------------------------------------------
__global__ void clock_set_kernel(StepClock *c, StepClock v) {
  if (blockIdx.x == 0 && threadIdx.x == 0) *c = v;
}

__global__ void record_kernel(RecordArgs A) {
  int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= A.n_col) return;
  float v;
  float *p = A.ptr[c];
  if (p) {
    v = *p;
  } else {
    int node = A.node[c];
    v = (A.last_spike[node] == A.T) ? A.last_height[node] : 0.0f;
  }
  A.out[c] = v;
}

__global__ void wrap_kernel(uint16_t *st, unsigned long long n, int up) {
  unsigned long long i = (unsigned long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  uint16_t v = st[i];
  if (up) {
    if (v >= 0x8000) st[i] = 0;
  } else {
    if (v < 0x8000) st[i] = 0x8000;
  }
}

__global__ void fill_u16_kernel(uint16_t *p, unsigned long long n, uint16_t v) {
  unsigned long long i = (unsigned long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

template <int P>
void launch_aeif_p(const AeifArgs &a, hipStream_t s) {
  int grid = (a.n + kBlock - 1) / kBlock;
  if (grid <= 0) return;
  if (a.do_step && a.strag) {
    // the overlap bookkeeping is compiled in only where it is used (groups
    // of up to kOverlapMaxPort ports)
    // the default budget of one attempt, compiled in for uniform
    // parameters and up to two ports
    const bool b1 = a.uniform && a.budget == 1 && P <= 2;
    if constexpr (P <= kOverlapMaxPort) {
      if (a.skip_prev || a.mask_write) {
        if (b1)
          hipLaunchKernelGGL(
              (aeif_pass1_kernel<P, true, (P <= 2 ? 6 : 1), true, true>),
              dim3(grid), dim3(kBlock), 0, s, a);
        else if (a.uniform)
          hipLaunchKernelGGL((aeif_pass1_kernel<P, true, (P <= 2 ? 6 : 1), true>),
                             dim3(grid), dim3(kBlock), 0, s, a);
        else
          hipLaunchKernelGGL((aeif_pass1_kernel<P, false, 1, true>), dim3(grid),
                             dim3(kBlock), 0, s, a);
        return;
      }
    }
    if (b1)
      hipLaunchKernelGGL(
          (aeif_pass1_kernel<P, true, (P <= 2 ? 6 : 1), false, true>),
          dim3(grid), dim3(kBlock), 0, s, a);
    else if (a.uniform)
      hipLaunchKernelGGL((aeif_pass1_kernel<P, true, (P <= 2 ? 6 : 1), false>),
                         dim3(grid), dim3(kBlock), 0, s, a);
    else
      hipLaunchKernelGGL((aeif_pass1_kernel<P, false, 1, false>), dim3(grid),
                         dim3(kBlock), 0, s, a);
  } else {
    hipLaunchKernelGGL(aeif_kernel<P>, dim3(grid), dim3(kBlock), 0, s, a);
  }
}

template <int P, bool UNI, bool PROP, bool CU>
void launch_pass2_v(const AeifArgs &a, const DeliveryArgs *d, int grid2,
                    int d_grid, hipStream_t s) {
  if (d)
    hipLaunchKernelGGL((aeif_tail_kernel<P, UNI, PROP, CU>), dim3(grid2 + d_grid),
                       dim3(kBlock), delivery_lds_bytes(d->D, 0), s, a, *d,
                       (uint32_t)grid2);
  else
    hipLaunchKernelGGL((aeif_pass2_kernel<P, UNI, PROP, CU>), dim3(grid2),
                       dim3(kBlock), 0, s, a);
}

template <int P>
void launch_aeif_pass2_p(const AeifArgs &a, const DeliveryArgs *d,
                         int d_grid, hipStream_t s) {
  int grid2 = a.pass2_grid > 0 ? a.pass2_grid : 256;
  // the proposer's inference exists for groups of up to kPropMaxPort ports
  constexpr bool kProp = P <= kPropMaxPort;
  // the catch-up of neurons an overlapped step left
  if constexpr (P <= kOverlapMaxPort) {
    if (a.skip_prev || a.mask_write) {
      if (a.prop_pk && kProp) {
        if (a.uniform)
          launch_pass2_v<P, true, kProp, true>(a, d, grid2, d_grid, s);
        else
          launch_pass2_v<P, false, kProp, true>(a, d, grid2, d_grid, s);
      } else if (a.uniform) {
        launch_pass2_v<P, true, false, true>(a, d, grid2, d_grid, s);
      } else {
        launch_pass2_v<P, false, false, true>(a, d, grid2, d_grid, s);
      }
      return;
    }
  }
  // The sample log works on whole lanes too: the instance whose arguments
  // stay in registers (1e5 spiking neurons with the log on: 122 us per step
  // in the one made for quads, 114 in this one)
  if ((a.prop_pk || a.prop_log) && kProp) {
    if (a.uniform)
      launch_pass2_v<P, true, kProp, false>(a, d, grid2, d_grid, s);
    else
      launch_pass2_v<P, false, kProp, false>(a, d, grid2, d_grid, s);
  } else {
    if (a.uniform)
      launch_pass2_v<P, true, false, false>(a, d, grid2, d_grid, s);
    else
      launch_pass2_v<P, false, false, false>(a, d, grid2, d_grid, s);
  }
}

}  // namespace

void LaunchPropEval(const unsigned char *pk, const float *feat, int n,
                    float *out, void *stream) {
  int grid = (n + kBlock - 1) / kBlock;
  if (grid > 0)
    hipLaunchKernelGGL(prop_eval_kernel, dim3(grid), dim3(kBlock), 0,
                       (hipStream_t)stream, pk, feat, n, out);
}

// Staging of the allocation-free inference: the feature vectors and the
// outputs of one call, in a file-scope device array (one copy per GPU, held
// until the process ends).  Host code never uses the array's name as an
// address: each device's copy is found once with hipGetSymbolAddress.
namespace {
constexpr size_t kPropScratchFloats = (size_t)kPropEvalNoAllocMax * (kPropIn + 1);
__device__ __align__(256) float prop_scratch[kPropScratchFloats];
constexpr int kMaxDevices = 64;
float *prop_scratch_dev[kMaxDevices];   // per device, null until looked up
}  // namespace

const char *PropEvalNoAlloc(const unsigned char *pk, const float *feat,
                            int n, float *out, void *stream) {
  if (n < 0) return "negative number of feature vectors";
  if (n > kPropEvalNoAllocMax)
    return "more feature vectors than the allocation-free inference holds "
           "(kPropEvalNoAllocMax)";
  if (n == 0) return nullptr;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices)
    return "no usable HIP device";
  if (!prop_scratch_dev[dev]) {
    void *p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(prop_scratch)) != hipSuccess ||
        !p)
      return "hipGetSymbolAddress of the inference staging failed";
    prop_scratch_dev[dev] = static_cast<float *>(p);
  }
  float *f_dev = prop_scratch_dev[dev];
  float *o_dev = f_dev + (size_t)kPropEvalNoAllocMax * kPropIn;
  hipStream_t s = (hipStream_t)stream;
  if (hipMemcpyAsync(f_dev, feat, (size_t)n * kPropIn * sizeof(float),
                     hipMemcpyHostToDevice, s) != hipSuccess)
    return "copy of the feature vectors failed";
  LaunchPropEval(pk, f_dev, n, o_dev, stream);
  if (hipGetLastError() != hipSuccess) return "inference launch failed";
  if (hipMemcpyAsync(out, o_dev, (size_t)n * sizeof(float),
                     hipMemcpyDeviceToHost, s) != hipSuccess)
    return "copy of the outputs failed";
  if (hipStreamSynchronize(s) != hipSuccess) return "inference failed";
  return nullptr;
}

void LaunchAeifPass2(const AeifArgs &a, int n_port, const DeliveryArgs *d,
                     int d_grid, void *stream) {
  hipStream_t s = (hipStream_t)stream;
  switch (n_port) {
#define NGPU_CASE(P) \
  case P: launch_aeif_pass2_p<P>(a, d, d_grid, s); break;
    NGPU_CASE(1) NGPU_CASE(2) NGPU_CASE(3) NGPU_CASE(4) NGPU_CASE(5)
    NGPU_CASE(6) NGPU_CASE(7) NGPU_CASE(8) NGPU_CASE(9) NGPU_CASE(10)
    NGPU_CASE(11) NGPU_CASE(12) NGPU_CASE(13) NGPU_CASE(14) NGPU_CASE(15)
    NGPU_CASE(16) NGPU_CASE(17) NGPU_CASE(18) NGPU_CASE(19) NGPU_CASE(20)
#undef NGPU_CASE
    default: break;
  }
}

void LaunchAeifStep(const AeifArgs &a, int n_port, const DeliveryArgs *d,
                    int d_grid, void *stream) {
  hipStream_t s = (hipStream_t)stream;
  const uint32_t n1 = (uint32_t)((a.n + kBlock - 1) / kBlock);
  const DeliveryArgs da = d ? *d : DeliveryArgs{};
  const dim3 grid(n1 + (d ? (uint32_t)d_grid : 0u));
  const size_t lds = d ? delivery_lds_bytes(d->D, 0) : 0;
  if (n1 == 0) return;
#define NGPU_STEP(P)                                                        \
  case P:                                                                   \
    if (a.uniform)                                                          \
      hipLaunchKernelGGL((aeif_step_kernel<P, true>), grid, dim3(kBlock),   \
                         lds, s, a, da, n1);                                \
    else                                                                    \
      hipLaunchKernelGGL((aeif_step_kernel<P, false>), grid, dim3(kBlock),  \
                         lds, s, a, da, n1);                                \
    break;
  switch (n_port) {
    NGPU_STEP(1)
    NGPU_STEP(2)
    NGPU_STEP(3)
    default: break;
  }
#undef NGPU_STEP
}

void LaunchAeif(const AeifArgs &a, int n_port, void *stream) {
  hipStream_t s = (hipStream_t)stream;
  switch (n_port) {
#define NGPU_CASE(P) \
  case P: launch_aeif_p<P>(a, s); break;
    NGPU_CASE(1) NGPU_CASE(2) NGPU_CASE(3) NGPU_CASE(4) NGPU_CASE(5)
    NGPU_CASE(6) NGPU_CASE(7) NGPU_CASE(8) NGPU_CASE(9) NGPU_CASE(10)
    NGPU_CASE(11) NGPU_CASE(12) NGPU_CASE(13) NGPU_CASE(14) NGPU_CASE(15)
    NGPU_CASE(16) NGPU_CASE(17) NGPU_CASE(18) NGPU_CASE(19) NGPU_CASE(20)
#undef NGPU_CASE
    default: break;
  }
}

void LaunchIaf(const IafArgs &a, void *stream) {
  int grid = (a.n + kBlock - 1) / kBlock;
  if (grid > 0)
    hipLaunchKernelGGL(iaf_kernel, dim3(grid), dim3(kBlock), 0,
                       (hipStream_t)stream, a);
}

void LaunchIafStep(const IafArgs &a, const DeliveryArgs &d, int d_grid,
                   void *stream) {
  const uint32_t n1 = (uint32_t)((a.n + kBlock - 1) / kBlock);
  hipLaunchKernelGGL(iaf_step_kernel, dim3(n1 + (uint32_t)d_grid),
                     dim3(kBlock), delivery_lds_bytes(d.D, 0),
                     (hipStream_t)stream, a, d, n1);
}

void LaunchRelay(const RelayArgs &a, void *stream) {
  int grid = (a.n + kBlock - 1) / kBlock;
  if (grid > 0)
    hipLaunchKernelGGL(relay_kernel, dim3(grid), dim3(kBlock), 0,
                       (hipStream_t)stream, a);
}

void LaunchLegacyPoisson(const LegacyPoisArgs &a, void *stream) {
  int grid = (a.n + kBlock - 1) / kBlock;
  if (grid > 0)
    hipLaunchKernelGGL(legacy_pois_kernel, dim3(grid), dim3(kBlock), 0,
                       (hipStream_t)stream, a);
}

void LaunchSpikeGen(const SpikeGenArgs &a, void *stream) {
  int grid = (a.n + kBlock - 1) / kBlock;
  if (grid > 0)
    hipLaunchKernelGGL(spikegen_kernel, dim3(grid), dim3(kBlock), 0,
                       (hipStream_t)stream, a);
}

void LaunchDelivery(const DeliveryArgs &a, int grid, void *stream) {
  const size_t lds = delivery_lds_bytes(a.D, 0);
  if (a.syn_group)
    hipLaunchKernelGGL(delivery_kernel<true>, dim3(grid), dim3(kBlock), lds,
                       (hipStream_t)stream, a);
  else
    hipLaunchKernelGGL(delivery_kernel<false>, dim3(grid), dim3(kBlock), lds,
                       (hipStream_t)stream, a);
}

void LaunchDeliveryTiled(const DeliveryArgs &a, const TileArgs &b,
                         void *stream) {
  hipStream_t s = (hipStream_t)stream;
  const size_t lds =
      sizeof(uint32_t) * (((size_t)(b.fixed ? 2 : 1) << b.tile_shift) +
                          (size_t)a.D + 1);
  static bool lds_attr = false;   // the tile may exceed the default limit
  if (!lds_attr) {
    // the largest tiles: 2^15 floats, or 2^14 64-bit sums (the host uses
    // fixed-point sums only where the tile fits in LDS)
    const int most = (int)(sizeof(uint32_t) *
                           (((size_t)1 << kTileShiftMax) + kMaxDelaySlots + 1));
    (void)hipFuncSetAttribute(
        reinterpret_cast<const void *>(tiled_delivery_kernel<false>),
        hipFuncAttributeMaxDynamicSharedMemorySize, most);
    (void)hipFuncSetAttribute(
        reinterpret_cast<const void *>(tiled_delivery_kernel<true>),
        hipFuncAttributeMaxDynamicSharedMemorySize, most);
    lds_attr = true;
  }
  if (b.fixed)
    hipLaunchKernelGGL(tiled_delivery_kernel<true>, dim3((unsigned)b.n_blocks),
                       dim3(kTiledBlock), lds, s, a, b);
  else
    hipLaunchKernelGGL(tiled_delivery_kernel<false>,
                       dim3((unsigned)b.n_blocks), dim3(kTiledBlock), lds, s,
                       a, b);
  long long g = ((b.acc_n + 3) / 4 + kBlock - 1) / kBlock;
  if (g > 2048) g = 2048;
  if (!b.split) g = 1;
  hipLaunchKernelGGL(tiled_sum_kernel, dim3((unsigned)g), dim3(kBlock), 0, s,
                     b, a.acc, a.clock, a.clock_next);
}

void LaunchDeliveryBinned(const DeliveryArgs &a, const BinArgs &b,
                          int reduce_grid, void *stream) {
  hipStream_t s = (hipStream_t)stream;
  static bool lds_attr = false;   // both may exceed the default LDS limit
  if (!lds_attr) {
    (void)hipFuncSetAttribute(
        reinterpret_cast<const void *>(bin_scatter_kernel),
        hipFuncAttributeMaxDynamicSharedMemorySize,
        (int)scatter_lds_bytes(kMaxDelaySlots, kMaxBins));
    (void)hipFuncSetAttribute(
        reinterpret_cast<const void *>(bin_reduce_kernel),
        hipFuncAttributeMaxDynamicSharedMemorySize,
        (int)(sizeof(uint32_t) * (kMaxBins + 1)));
    lds_attr = true;
  }
  hipLaunchKernelGGL(bin_scatter_kernel, dim3(b.grid), dim3(kBinBlock),
                     scatter_lds_bytes(a.D, b.nb), s, b, a);
  hipLaunchKernelGGL(bin_reduce_kernel, dim3(reduce_grid), dim3(kReduceBlock),
                     sizeof(uint32_t) * ((size_t)b.nb + 1), s, b, a.acc);
  // Many bins of about equal size leave nothing to sum (128 blocks: the
  // million spiking neurons are 0.3 % slower with 512, 0.7 % with 2048;
  // unequal bins, 2e7 events on 14 of 245: 202 us per step with 128, 178
  // with 512); few bins leave a sum in most steps (25 bins, 2e6 events: 70
  // us with 128, 48 with 512, 42 with 2048).
  long long g = (b.acc_n + kBlock - 1) / kBlock;
  const long long most = b.nb >= kSingleChunkBins ? 128 : 2048;
  if (g > most) g = most;
  hipLaunchKernelGGL(bin_sum_kernel, dim3((unsigned)g), dim3(kBlock), 0, s, b,
                     a.acc, a.clock, a.clock_next);
}

void LaunchClockSet(StepClock *c, const StepClock &v, void *stream) {
  hipLaunchKernelGGL(clock_set_kernel, dim3(1), dim3(64), 0,
                     (hipStream_t)stream, c, v);
}

void LaunchRevStdp(const RevArgs &a, int grid, void *stream) {
  hipLaunchKernelGGL(rev_kernel, dim3(grid), dim3(kBlock), 0,
                     (hipStream_t)stream, a);
}

void LaunchDenRev(const RevArgs &a, int grid, void *stream) {
  hipLaunchKernelGGL(den_rev_kernel, dim3(grid), dim3(kBlock), 0,
                     (hipStream_t)stream, a);
}

void LaunchRecord(const RecordArgs &a, void *stream) {
  int grid = (a.n_col + 255) / 256;
  if (grid > 0)
    hipLaunchKernelGGL(record_kernel, dim3(grid), dim3(256), 0,
                       (hipStream_t)stream, a);
}

void LaunchSpikeTimeWrap(uint16_t *spike_time, unsigned long long n, int up,
                         void *stream) {
  unsigned long long grid = (n + 255) / 256;
  if (grid > 0)
    hipLaunchKernelGGL(wrap_kernel, dim3((unsigned)grid), dim3(256), 0,
                       (hipStream_t)stream, spike_time, n, up);
}

void LaunchFillU16(uint16_t *p, unsigned long long n, uint16_t v, void *stream) {
  unsigned long long grid = (n + 255) / 256;
  if (grid > 0)
    hipLaunchKernelGGL(fill_u16_kernel, dim3((unsigned)grid), dim3(256), 0,
                       (hipStream_t)stream, p, n, v);
}

}  // namespace ngpu
