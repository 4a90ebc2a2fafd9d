// resident_kernel.hip -- k_resident: a whole rollout, or K control steps on given actions, with two worlds
// per wave or one world on two waves (resident.h).
#include <hip/hip_runtime.h>

#include "resident.h"

namespace g1k {

// kDuo: one world on two waves, which share the physics of a substep (world_qacc); both carry the world's
// state, wave 0 (role 0) stores. Else two worlds on one wave: group g of block b has
// world 2 b + g. With one world both groups of a wave carry it and group 0 stores: the second group costs
// nothing (its lanes would idle), and the contact phases run at the world's own contact count instead of
// the larger of two. kPolicy: the actions come from the policy (K = H steps), else from ph.act.
template <bool kDuo, bool kPolicy>
__global__ void __launch_bounds__(resident_threads(kDuo)) k_resident(ResidentArgs ra) {
  constexpr int kW = kDuo ? 1 : 2;   // worlds per wave
  __shared__ __align__(16) WorldLds lds[2];
  __shared__ __align__(16) DuoLds duo[kDuo ? 2 : 1];
  __shared__ float acts[kGroup];   // kDuo: the policy's actions, from wave 0
  const int role = kDuo ? __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6) : 0;
  const int g = group_id(), l = group_lane();
  WorldLds& s = lds[g];
  const int N = ra.ph.N;
  const int w = kW == 2 ? 2 * (int)blockIdx.x + g : (int)blockIdx.x;
  const bool wvalid = kW == 2 ? w < N : g == 0 && role == 0;
  const int wc = w < N ? w : N - 1;   // an odd N's last group repeats world N - 1 and stores nothing
  const bool hinge = l >= 2 && l < kNBody;
  LaneState st;
  float pa;
  int step;
  unsigned rng;
  {
    const PhysArgs& a = ra.ph;
    const float* gq = a.qp + (long)wc * kNQ;
    const float* gv = a.qv + (long)wc * kNV;
#pragma unroll
    for (int m = 0; m < 7; ++m) st.bq[m] = gq[m];
#pragma unroll
    for (int m = 0; m < 6; ++m) st.bqd[m] = gv[m];
    st.jq = hinge ? gq[l + 5] : 0.f;
    st.jqd = hinge ? gv[l + 4] : 0.f;
    pa = hinge ? a.pa[(long)wc * kAct + l - 2] : 0.f;
    step = a.steps[wc];
    rng = a.rng[wc];
  }
  unsigned hcnt = 0;
  const int K = ra.ph.K;
#pragma unroll 1
  for (int k = 0;; ++k) {
    const ResidentArgs& rb = kernarg_reread<ResidentArgs>();
    float act = 0.f;
    if (kPolicy) {   // k == K: the bootstrap value of the state after the last step
      if (kDuo) __syncthreads();   // wave 1 has read the last substep's results: the policy takes their place
      act = wave_policy<kW, kDuo>(rb.po, st, pa, rng, rb.ph.seed, rb.ph.N, k, w, wc, wvalid,
                                  reinterpret_cast<float*>(lds), role);
      if (kDuo) {
        if (role == 0) acts[l] = act;
        __syncthreads();
        act = acts[l];
      }
    }
    if (k >= K) break;
    // the lane's model constants, formed here (opaque lane index) rather than held across steps
    int lo = l;
    __asm__ volatile("" : "+v"(lo));
    const LaneModel L = lane_model(lo);
    const PhysArgs& a = kernarg_reread<ResidentArgs>().ph;
    const int t = a.t0 + k * a.astep;
    if (!kPolicy) act = hinge ? a.act[((long)t * a.N + wc) * kAct + l - 2] : 0.f;
    float vx_sum = 0.f, energy = 0.f;
    const SolveParams P{a.pgs, a.mu, true, true};
    run_substeps<kDuo>(P, s, L, l, wvalid, pd_target(L, act), 0, a.S, st, energy, vx_sum, hcnt, role, duo + (kDuo ? g : 0));
    float r;
    const int done = finish_control_step(a, L, l, wc, t, act, vx_sum, energy, st, pa, step, rng, r);
    if (wvalid && l == 1) {
      const long o = (long)(a.t0 + k * a.rstep) * a.N + w;
      a.R[o] = r;
      a.D[o] = (float)done;
    }
    if (!kPolicy && k == K - 1 && a.obs && wvalid) store_observation(a.obs + (long)w * kObs, L, l, st, pa);
  }
  const PhysArgs& a = kernarg_reread<ResidentArgs>().ph;
  if (wvalid && a.K > 0) {
    const LaneModel L = lane_model(l);
    store_state(a, L, l, w, st);
    if (L.hinge) a.pa[(long)w * kAct + l - 2] = pa;
    if (l == 1) {
      a.steps[w] = step;
      a.rng[w] = rng;
    }
  }
  if (a.ncon_hist && l < 9 && hcnt) atomicAdd(&a.ncon_hist[l], (unsigned long long)hcnt);
}

void launch_resident_kernel(const ResidentArgs& ra, bool policy, bool duo) {
  const dim3 grid((unsigned)(duo ? ra.ph.N : (ra.ph.N + 1) / 2)), block(resident_threads(duo));
  if (duo && policy) hipLaunchKernelGGL((k_resident<true, true>), grid, block, 0, 0, ra);
  else if (duo) hipLaunchKernelGGL((k_resident<true, false>), grid, block, 0, 0, ra);
  else if (policy) hipLaunchKernelGGL((k_resident<false, true>), grid, block, 0, 0, ra);
  else hipLaunchKernelGGL((k_resident<false, false>), grid, block, 0, 0, ra);
}

const void* resident_kernel_fn(bool policy, bool duo) {
  if (duo) return policy ? (const void*)k_resident<true, true> : (const void*)k_resident<true, false>;
  return policy ? (const void*)k_resident<false, true> : (const void*)k_resident<false, false>;
}

}  // namespace g1k
