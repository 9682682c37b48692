// The last neurons of a wave, one neuron per quad of lanes: the state's
// layout, the move from one neuron per lane, and the RK5 attempts.  Used by
// the second pass of the AdEx conductance models (kernels.hip) and by the
// current-based AdEx models (rk5_models.hip).
#pragma once
#include <hip/hip_runtime.h>

#include "ngpu_device.h"
#include "ngpu_kernels.h"
#include "step_common.h"

namespace ngpu {
namespace {

// ---------------------------------------------------------------------
// The last neurons of a wave, one neuron per quad of lanes.
//
// A spiking neuron takes 30 to 60 RK5 attempts in a time step, one after
// the other, and the second pass lasts as long as the longest of these
// chains.  A wave issues one instruction per 4 clocks whether 1 or 64 of
// its lanes are busy (measured on this chip: 4.24 clocks per dependent or
// independent VALU or scalar instruction of a lone wave, 58 clocks per
// divergent branch), so the chain is as long as its instruction count.
// Once at most 16 neurons of a wave are left, each moves to four lanes:
// lane 0 holds V and w, lane 1 + p the variables (g, g1; I, I1; or I alone)
// of port p.  The stage
// sums, the solution and the error then take 2 variables' instructions
// instead of 2 + 2P, and the quad exchanges values through DPP operands
// (quad_perm), at no cost in LDS latency.  The state update is written with
// selects, without divergent branches.  Every operation of a neuron is the
// one of the one-neuron-per-lane attempt, in its order, so the results are the same
// bit for bit (a product added to zero there is the product here; that can
// change only the sign of a zero).
// Measured, second pass per step: 10000 spiking neurons at tolerance 1e-6
// 90.5 -> 53.7 us, 2e5 plastic neurons 89.1 -> 52.7 us; 20001 aeif_psc_exp
// neurons, whole update: 66 -> 48 us.
constexpr int kQuadMaxPort = 3;    // 1 + P lanes hold the state
constexpr int kQuadsPerWave = 16;

// value of lane R of the quad
template <int R>
__device__ __forceinline__ float quad_get(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), R * 0x55,
                                                 0xF, 0xF, true));
}

__device__ __forceinline__ unsigned long long lanes_where(bool c) {
  return __builtin_amdgcn_ballot_w64(c);
}
constexpr unsigned long long kMemLanes = 0x1111111111111111ull;

// One link of the error norm's running maximum (rk5_attempt), taken by every
// lane of the quad: lane R's quotient v / s.
template <int R>
__device__ __forceinline__ void quad_max(float va, float sa, float &num,
                                         float &den) {
  const float v = quad_get<R>(va), s = quad_get<R>(sa);
  const bool keep = v * den <= num * s;
  num = keep ? num : v;
  den = keep ? den : s;
}

// A neuron's state spread over its quad.  VP: variables of a port (2: in ya
// and yb of its lane; 1: in ya, yb stays 0).
template <int P, int VP>
struct QuadState {
  static constexpr int N = 2 + VP * P;
  int i, role, rv;         // neuron; lane of the quad; lane whose role it has
  bool live, own;          // has a neuron; holds state variables
  float ya, yb, sa, sb;    // state and error scale
  double x;
  float h, refr;
  int nsp, n_att;
  bool need_k1;            // at the start of an RK5 step

  // From one neuron per lane (have: at most 16 lanes of the wave).
  __device__ __forceinline__ void take(bool have, int i1,
                                       const float (&y1)[N],
                                       const float (&scal1)[N], double x1,
                                       float h1, float refr1, int nsp1,
                                       int n_att1, bool need1) {
    const unsigned long long m = lanes_where(have);
    const int na = __popcll(m);
    const uint32_t lane = lane_id();
    role = (int)(lane & 3u);
    const int quad = (int)(lane >> 2);
    // the lane that held quad q's neuron: a permutation of the wave, the
    // lanes with a neuron first
    const uint32_t to =
        have ? lanes_below(m) : (uint32_t)na + lanes_below(~m);
    const int from_rank =
        __builtin_amdgcn_ds_permute((int)(to << 2), (int)lane);
    const int src = __shfl(from_rank, quad);
    live = quad < na;
    own = role <= P;
    rv = own ? role : P;     // idle lanes repeat the last port
    // (every lane takes part in every shuffle: a lane without a neuron to
    // finish may hold one to give away)
    const int i_src = __shfl(i1, src);
    i = live ? i_src : 0;
    ya = yb = 0.0f;
    sa = sb = 1.0f;
#pragma unroll
    for (int k = 0; k < N; k++) {
      const float v = __shfl(y1[k], src), s = __shfl(scal1[k], src);
      const int r = k < 2 ? 0 : 1 + (k - 2) / VP;
      const bool second = k < 2 ? k == 1 : (k - 2) % VP == 1;
      if (r == rv) {
        if (second) {
          yb = v;
          sb = s;
        } else {
          ya = v;
          sa = s;
        }
      }
    }
    x = __shfl(x1, src);
    h = __shfl(h1, src);
    refr = __shfl(refr1, src);
    nsp = __shfl(nsp1, src);
    n_att = __shfl(n_att1, src);
    need_k1 = __shfl(need1 ? 1 : 0, src) != 0;
  }
};

struct QuadStep {
  double x1;               // end of the time step
  float h_min;
  double h_min_acc;
  float eps;
  unsigned long long *forced;
};

// Runs the wave's quads to the end of the time step.  Q: the derivatives of
// a lane's pair, rhs(ya, yb, da, db) and refractory(bool), with V_peak,
// V_reset, port (lanes 1 and up), V_b (added to w at a spike) and n_refr
// (refractory steps after one).  finish(s, done) stores and sends the spikes
// of the neurons of the lanes with done; every lane calls it.
template <int P, int VP, class Q, class F>
__device__ __forceinline__ void quad_run(Q &q, QuadState<P, VP> &s,
                                         const QuadStep &A, int &n_acc,
                                         int &n_rej, F &&finish) {
  const double x1 = A.x1;
  const int role = s.role;
  float ya = s.ya, yb = s.yb, sa = s.sa, sb = s.sb, h = s.h, refr = s.refr;
  double x = s.x;
  int nsp = s.nsp;
  const int n_att = s.n_att;
  const bool live = s.live, need_k1 = s.need_k1;
  const double x_end = x1 - (double)A.h_min;
  // (double)hh <= h_min_acc for a float hh is hh <= the largest float that
  // does not exceed h_min_acc
  float h_acc = (float)A.h_min_acc;
  if ((double)h_acc > A.h_min_acc)
    h_acc = __uint_as_float(__float_as_uint(h_acc) - 1u);
  const float h_min = A.h_min, eps = A.eps;
  float ka1 = 0.0f, kb1 = 0.0f;
  q.refractory(refr > 0.0f);
  unsigned long long rf_m = lanes_where(refr > 0.0f);
  unsigned long long live_m = lanes_where(live), need_m = lanes_where(need_k1);
  // attempts of this phase, the same for every neuron still running, and
  // those accepted
  int tries = 0, accepted = 0;
  int most = live ? n_att : 0;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const int o = __shfl_xor(most, off);
    most = o > most ? o : most;
  }
  const int tries_max =
      kMaxAttemptsPerStep - __builtin_amdgcn_readfirstlane(most);
  bool first = true;
  for (;;) {
    // first stage and error scale of the neurons that start an RK5 step (a
    // retried neuron's first stage is the same function of the same state)
    if (first || (live_m & need_m)) {
      first = false;
      const bool need_k1 = __builtin_amdgcn_inverse_ballot_w64(need_m);
      q.rhs(ya, yb, ka1, kb1);
      const float ta = (fabsf(ya) + fabsf(ka1 * h)) + CK::scal_min;
      const float tb = (fabsf(yb) + fabsf(kb1 * h)) + CK::scal_min;
      sa = need_k1 ? ta : sa;
      sb = need_k1 ? tb : sb;
    }
    const float h_max = (float)(x1 - x);
    float hh = h;
    hh = hh > h_max ? h_max : hh;
    hh = hh < h_min ? h_min : hh;
    float ka2, kb2, ka3, kb3, ka4, kb4, ka5, kb5, ka6, kb6;
    float ta, tb;
    q.rhs(__builtin_fmaf(hh, CK::a21 * ka1, ya),
          __builtin_fmaf(hh, CK::a21 * kb1, yb), ka2, kb2);
    ta = __builtin_fmaf(CK::a32, ka2, CK::a31 * ka1);
    tb = __builtin_fmaf(CK::a32, kb2, CK::a31 * kb1);
    q.rhs(__builtin_fmaf(hh, ta, ya), __builtin_fmaf(hh, tb, yb), ka3, kb3);
    ta = __builtin_fmaf(CK::a42, ka2, CK::a41 * ka1);
    tb = __builtin_fmaf(CK::a42, kb2, CK::a41 * kb1);
    ta = __builtin_fmaf(CK::a43, ka3, ta);
    tb = __builtin_fmaf(CK::a43, kb3, tb);
    q.rhs(__builtin_fmaf(hh, ta, ya), __builtin_fmaf(hh, tb, yb), ka4, kb4);
    ta = __builtin_fmaf(CK::a52, ka2, CK::a51 * ka1);
    tb = __builtin_fmaf(CK::a52, kb2, CK::a51 * kb1);
    ta = __builtin_fmaf(CK::a53, ka3, ta);
    tb = __builtin_fmaf(CK::a53, kb3, tb);
    ta = __builtin_fmaf(CK::a54, ka4, ta);
    tb = __builtin_fmaf(CK::a54, kb4, tb);
    q.rhs(__builtin_fmaf(hh, ta, ya), __builtin_fmaf(hh, tb, yb), ka5, kb5);
    ta = __builtin_fmaf(CK::a62, ka2, CK::a61 * ka1);
    tb = __builtin_fmaf(CK::a62, kb2, CK::a61 * kb1);
    ta = __builtin_fmaf(CK::a63, ka3, ta);
    tb = __builtin_fmaf(CK::a63, kb3, tb);
    ta = __builtin_fmaf(CK::a64, ka4, ta);
    tb = __builtin_fmaf(CK::a64, kb4, tb);
    ta = __builtin_fmaf(CK::a65, ka5, ta);
    tb = __builtin_fmaf(CK::a65, kb5, tb);
    q.rhs(__builtin_fmaf(hh, ta, ya), __builtin_fmaf(hh, tb, yb), ka6, kb6);
    ta = __builtin_fmaf(CK::a73, ka3, CK::a71 * ka1);
    tb = __builtin_fmaf(CK::a73, kb3, CK::a71 * kb1);
    ta = __builtin_fmaf(CK::a74, ka4, ta);
    tb = __builtin_fmaf(CK::a74, kb4, tb);
    ta = __builtin_fmaf(CK::a76, ka6, ta);
    tb = __builtin_fmaf(CK::a76, kb6, tb);
    const float yna = __builtin_fmaf(hh, ta, ya);
    const float ynb = __builtin_fmaf(hh, tb, yb);
    ta = __builtin_fmaf(CK::e3, ka3, CK::e1 * ka1);
    tb = __builtin_fmaf(CK::e3, kb3, CK::e1 * kb1);
    ta = __builtin_fmaf(CK::e4, ka4, ta);
    tb = __builtin_fmaf(CK::e4, kb4, tb);
    ta = __builtin_fmaf(CK::e5, ka5, ta);
    tb = __builtin_fmaf(CK::e5, kb5, tb);
    ta = __builtin_fmaf(CK::e6, ka6, ta);
    tb = __builtin_fmaf(CK::e6, kb6, tb);
    const float va = fabsf(hh * ta), vb = fabsf(hh * tb);
    // (the first quotient needs no comparison with 0 / 1)
    float num = quad_get<0>(va), den = quad_get<0>(sa);
    quad_max<0>(vb, sb, num, den);
    quad_max<1>(va, sa, num, den);
    if constexpr (VP > 1) quad_max<1>(vb, sb, num, den);
    if constexpr (P > 1) {
      quad_max<2>(va, sa, num, den);
      if constexpr (VP > 1) quad_max<2>(vb, sb, num, den);
    }
    if constexpr (P > 2) {
      quad_max<3>(va, sa, num, den);
      if constexpr (VP > 1) quad_max<3>(vb, sb, num, den);
    }
    const float err = num / (den * eps);
    // acceptance, next step size, state at the step boundary (conditions as
    // lane masks in scalar registers, selects from them)
    tries++;
    const unsigned long long at_min = lanes_where(hh <= h_acc);
    const unsigned long long acc_m = lanes_where(err <= 1.0f) | at_min;
    const bool accept = __builtin_amdgcn_inverse_ballot_w64(acc_m);
    if (at_min & live_m & kMemLanes) {
      const bool mine =
          __builtin_amdgcn_inverse_ballot_w64(at_min & live_m & kMemLanes);
      if (mine && err > 1.0f) count_forced(A.forced);
    }
    const float pw = dev_pow_ctrl(err, accept ? -0.2f : -0.25f);
    const float hc = (hh * CK::coeff) * pw;
    const float h_up = err > CK::err_min ? hc : 5.0f * hh;
    const float h_lo = 0.1f * hh;
    const float h_dn = hc > h_lo ? hc : h_lo;
    h = accept ? h_up : h_dn;
    x += (double)(accept ? hh : 0.0f);
    ya = accept ? yna : ya;
    yb = accept ? ynb : yb;
    accepted += accept ? 1 : 0;
    unsigned long long upd_m = acc_m;
    if (tries > tries_max) {
      // some neuron may be at the attempt cap (the reference has none): it
      // gives up the step
      const bool over = !accept && n_att + tries > kMaxAttemptsPerStep;
      x = over ? x1 : x;
      h = over ? hh : h;
      upd_m |= lanes_where(over);
    }
    const unsigned long long end_m = lanes_where(x >= x_end);
    if (upd_m & kMemLanes &
        (lanes_where(ya < -1.0e3f) | lanes_where(fabsf(yb) > 1.0e6f) |
         lanes_where(ya >= q.V_peak) | rf_m)) {
      const bool rf = refr > 0.0f;
      const bool mem =
          __builtin_amdgcn_inverse_ballot_w64(upd_m & kMemLanes);
      const bool end = __builtin_amdgcn_inverse_ballot_w64(end_m);
      const bool bad = mem && (ya < -1.0e3f || fabsf(yb) > 1.0e6f);
      const bool ref = mem && !bad && rf;
      const bool spk = mem && !bad && !rf && ya >= q.V_peak;
      ya = (bad || ref || spk) ? q.V_reset : ya;
      yb = bad ? 0.0f : (spk ? yb + q.V_b : yb);
      refr = spk ? q.n_refr : (ref && end ? refr - 1.0f : refr);
      nsp += spk ? 1 : 0;
      q.refractory(refr > 0.0f);
      rf_m = lanes_where(refr > 0.0f);
    }
    need_m = upd_m & ~end_m;
    const unsigned long long done_m = live_m & upd_m & end_m;
    if (done_m) {
      const bool done = __builtin_amdgcn_inverse_ballot_w64(done_m);
      if (done && role == 0) {
        n_acc += accepted;
        n_rej += tries - accepted;
      }
      s.ya = ya;
      s.yb = yb;
      s.x = x;
      s.h = h;
      s.refr = refr;
      s.nsp = nsp;
      finish(s, done);
      live_m &= ~done_m;
      if (!live_m) break;
    }
  }
}

}  // namespace
}  // namespace ngpu
