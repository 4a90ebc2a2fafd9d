// resident.h -- waves that keep their worlds for a whole launch (k_resident, resident_kernel.hip): every
// control step of two worlds on one wave, or of one world on two waves, the policy included, with the
// worlds' state in registers from the first step to the last.
//
// For batches of at most two worlds per resident wave of the chip (launch_form in g1env.hip). There
// the work queue of k_rollout has nothing to balance, and its 16-world policy tile costs more than it
// saves: one wave computes the tile in 43 us while the tile's other seven waves wait for it, each step
// of all 16 worlds starts when the slowest of the eight pairs has finished the last one, and state,
// actions and flags cross the L2 between the waves. Here nothing is waited for but the world's own work.
// Bound by one wave's instruction stream: with 256 worlds on two waves each the VALU is busy 17% of the time,
// and a wave that is not at a barrier issues in about 70% of its cycles and waits for LDS and memory in most
// of the others. A substep takes 8 us (19.4k cycles; standing worlds 35.5k), the policy 10.5 us per control
// step (25k cycles, 15.6k of them the hidden layers of 256-256: their weights' way from the L2), with two
// worlds per wave 10 and 15.5. Up to 1024 worlds a second wave, on a SIMD that would stand idle or carry one
// wave, takes part of each substep's physics (world_qacc<true>) and half of the policy's rows (16 steps of
// 256 worlds 1.51 -> 1.47 ms by the latter; 4 steps of 512 with the 512-512-256 policy 0.63 -> 0.57). Rollouts
// against the queue: 16 steps of 256 worlds 2.55 -> 1.48 ms, 32 steps of 1024 5.45 -> 3.17, 24 steps of 3001 (5
// substeps) 2.79 -> 1.72; 512-512-256 policy, 4 steps of 512 worlds 1.26 -> 0.57. One world's host step 149 ->
// 104 us; the other sizes and the control steps on given actions: launch_form.
#pragma once
#include <hip/hip_runtime.h>

#include "queue.h"

namespace g1k {

struct ResidentArgs {
  PhysArgs ph;   // K control steps (the queue's fields are unused)
  TileArgs po;   // weights packed in WideLayout wl in chain order, whatever the policy's shape (tl, scr unused)
};

// ---- the policy of the wave's kW worlds on the vector ALUs
//
// A dense layer of one or two worlds is a matrix-vector product: bound by the weights' way from the L2
// (400 KB per pass for 256-256), not by arithmetic, and an MFMA would leave 14 of its 16 columns idle.
// Each lane computes whole rows (neurons) of a layer: in a pass over the tiles T0 .. T0 + 4 R - 1 lane
// 16 tt + j takes row j of the tiles T0 + 4 r + tt, r < R. v_mfma_f32_16x16x4f32 adds its four products to
// the accumulator one after the other, each a fused multiply-add (the tests of the forms compare both bit for
// bit, with ordinary weights, weights spread over 2^80, subnormal sums and overflow), so a row's fma chain in
// the MFMA tile's order of inputs gives the tile's sums bit for bit. That order goes in units of four inputs, the four lane groups' of one
// k-step (unit 4 q + e: the inputs kappa(L, 4 q + e, g), g < 4), and the weights are packed for it
// (WideLayout with chain = 1): one float4 per unit and row. The inputs come from LDS, one float4 per unit
// at the same address on every lane.
constexpr int kNetBuf = kMaxHidden + 16;          // floats of one activation buffer
constexpr int kNetWorld = 2 * kNetBuf;            // two buffers per world (layers alternate)
constexpr int kNetTail = 2 * kNetWorld;           // log-prob terms [2][32], actions [2][32]
constexpr int kNetLds = kNetTail + 4 * 32;
static_assert(kNetLds * sizeof(float) <= 2 * sizeof(WorldLds), "the policy's scratch lies over the physics'");
static_assert(kNetWorld % 64 == 32, "the two worlds' inputs on different LDS banks");

// Slot of row j of a hidden layer's tile among the tile's 16 in an activation buffer, so that the four
// inputs of a unit of the next layer are one float4 (kappa(L, 4 q + e, g) = 16 q + 4 g + e). The
// observation's features lie in natural order (kappa(0, 4 q + e, g) = 16 q + 4 e + g).
__device__ __forceinline__ int net_slot(int j) { return 4 * (j & 3) + (j >> 2); }

// The weights of unit U past the row blocks' bases: uniform bases and a 32-bit lane offset (bytes), so
// that a load is one instruction with the unit as its immediate (a lane address of its own per load took
// as many instructions as the arithmetic).
template <int R, int U>
__device__ __forceinline__ void net_load(const char* const (&base)[R], unsigned off, float4 (&w)[R]) {
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int r = 0; r < R; ++r) w[r] = *reinterpret_cast<const float4*>(base[r] + off + 256 * U);
  __builtin_amdgcn_sched_barrier(0);
}
template <int V>
__device__ __forceinline__ void net_inputs(const float* x, float4 (&xu)[V]) {
#pragma unroll
  for (int v = 0; v < V; ++v) xu[v] = *reinterpret_cast<const float4*>(x + v * kNetWorld);
}

// R row blocks of a layer of nQ k-quads for V worlds (inputs at x, x + kNetWorld): acc starts from the
// bias. kAhead quads' weights are in flight, each unit's slot refilled kAhead quads on as soon as its
// arithmetic is issued (past the end with the last quad again, unused). kHead: the head's two tiles,
// whose 32 rows take half a wave: lanes 0..31 serve one world and lanes 32..63 the other (x is the
// lane's own world's).
static_assert(kNetBuf >= kMaxHidden + 4, "a unit past the inputs is inside the buffer");
template <int V, int R, bool kHead>
__device__ __forceinline__ void net_pass(const float4* W, const float* bias, int nQ, int T0, const float* x, int lane,
                                         float (&acc)[V][R]) {
  // four quads ahead in the head; one in the hidden layers, where two would take the kernel to the register limit
  // of two waves per SIMD, at which the physics' schedule is slower (32 steps of 1024 worlds 3.39 -> 3.55 ms)
  constexpr int kAhead = kHead ? 4 : 1;
  const int j = lane & 15, tt = kHead ? (lane >> 4) & 1 : lane >> 4;
  const char* base[R];
#pragma unroll
  for (int r = 0; r < R; ++r) base[r] = reinterpret_cast<const char*>(W + (long)(T0 + 4 * r) * nQ * 64);
  const unsigned off = (unsigned)(tt * nQ * 64 + j) * 16u;
  float4 w[kAhead][4][R], xc[V];
#pragma unroll
  for (int i = 0; i < kAhead; ++i) {   // (every layer has at least four k-quads)
    net_load<R, 0>(base, off, w[i][0]);
    net_load<R, 1>(base, off, w[i][1]);
    net_load<R, 2>(base, off, w[i][2]);
    net_load<R, 3>(base, off, w[i][3]);
#pragma unroll
    for (int r = 0; r < R; ++r) base[r] += 1024;
  }
  net_inputs<V>(x, xc);
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const float b = bias[16 * (T0 + 4 * r + tt) + j];
#pragma unroll
    for (int v = 0; v < V; ++v) acc[v][r] = b;
  }
  auto unit = [&](auto uc, float4 (&wq)[4][R]) {
    constexpr int U = decltype(uc)::value;
    float4 xn[V];
    net_inputs<V>(x + 4 * (U + 1), xn);
#pragma unroll
    for (int g = 0; g < 4; ++g)
#pragma unroll
      for (int v = 0; v < V; ++v)
#pragma unroll
        for (int r = 0; r < R; ++r) acc[v][r] = __builtin_fmaf((&wq[U][r].x)[g], (&xc[v].x)[g], acc[v][r]);
    net_load<R, U>(base, off, wq[U]);
#pragma unroll
    for (int v = 0; v < V; ++v) xc[v] = xn[v];
  };
#pragma unroll 1
  for (int q = 0; q < nQ; q += kAhead) {   // nQ is 7 (layer 0) or a multiple of 4 (all others, the head's too)
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
      if (q + i + kAhead >= nQ) {   // past the end: the last quad again
#pragma unroll
        for (int r = 0; r < R; ++r) base[r] -= 1024;
      }
      unit(std::integral_constant<int, 0>(), w[i]);
      unit(std::integral_constant<int, 1>(), w[i]);
      unit(std::integral_constant<int, 2>(), w[i]);
      unit(std::integral_constant<int, 3>(), w[i]);
#pragma unroll
      for (int r = 0; r < R; ++r) base[r] += 1024;
      x += 16;
    }
  }
}

// The rows of R row blocks for both worlds, activated, into the layer's output buffers.
template <int kW, int R>
__device__ __forceinline__ void net_rows(const float4* W, const float* bias, int nQ, int T0, const float* x, float* out,
                                         int act, int lane) {
  float acc[kW][R];
  net_pass<kW, R, false>(W, bias, nQ, T0, x, lane, acc);
#pragma unroll
  for (int v = 0; v < kW; ++v)
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const float h = act == 0 ? act_tile<0>(acc[v][r]) : act_tile<1>(acc[v][r]);
      out[v * kNetWorld + 16 * (T0 + 4 * r + (lane >> 4)) + net_slot(lane & 15)] = h;
    }
}

// Policy of control step t for the wave's worlds (t == a.H: the bootstrap value only): observation,
// normalisation, MLP, sampling and log-probability, with the values of the policy tiles (rollout.h) bit
// for bit. The worlds' state is in the lanes (st, pa, rng); w: the group's world, wvalid: its lanes store.
// Returns the lane's own action (hinge lanes; t < a.H). lds: kNetLds floats. kDuo: both waves of the world
// call it; wave 0 forms the observation, the head and the outputs, and each takes half of a hidden layer's
// rows, with a block barrier after the observation and after each layer (nl + 1 on either wave). The two waves
// together take 24 bytes of weights per clock (368 KB of 256-256 in 15.6k cycles). (Returns 0 on wave 1.)
template <int kW, bool kDuo>
__device__ __forceinline__ float wave_policy(const TileArgs& a, const LaneState& st, float pa, unsigned rng,
                                             unsigned long long seed, int N, int t, int w, int wc, bool wvalid,
                                             float* lds, int role) {
  int lane = threadIdx.x & 63;
  __asm__ volatile("" : "+v"(lane));
  const int l = lane & 31, v = kW == 2 ? lane >> 5 : 0;
  const WideLayout& T = a.wl;
  float* const mine = lds + v * kNetWorld;
  if (!kDuo || role == 0) {
  // ---- observation (raw to O) and frozen normalisation: the lanes put their world's features into the
  // second buffer, and lane l takes features l, 32 + l, 64 + l, 96 + l from there
  const float* const nrm = a.Wt + T.nrm_off;
  float c[4][3];
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    const int k = l + 32 * m, kc = k < 4 * kObsSteps ? k : 0;
#pragma unroll
    for (int e = 0; e < 3; ++e) c[m][e] = nrm[e * 4 * kObsSteps + kObsSteps * (kc & 3) + (kc >> 2)];
  }
  float* const raw = mine + kNetBuf;
  if (l == 1) {
#pragma unroll
    for (int i = 0; i < 6; ++i) raw[i] = st.bqd[i];
#pragma unroll
    for (int i = 6; i < 9; ++i) raw[i] = obs_value(0.f, st.bq[3], st.bq[4], st.bq[5], st.bq[6], i);
  }
  if (l >= 2 && l < kNBody) {
    raw[9 + l - 2] = st.jq; raw[38 + l - 2] = st.jqd; raw[67 + l - 2] = pa;
  }
  if (l == 0) { raw[96] = 0.8f; raw[97] = 0.f; raw[98] = 0.f; raw[99] = 0.f; }
  wave_sync();
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    const int k = l + 32 * m;
    if (k < 4 * kObsSteps) {
      float z = 0.f;
      if (k < kObs) {
        const float o = raw[k];
        if (wvalid && t < a.H) a.O[((long)t * N + w) * kObs + k] = o;
        z = div_rn_inf(o - c[m][0], c[m][1], c[m][2]);
        if (z < -10.f) z = -10.f; else if (z > 10.f) z = 10.f;
      }
      mine[k] = z;
    }
  }
  wave_sync();
  }
  if (kDuo) __syncthreads();
  // ---- hidden layers: four row blocks (256 rows) at a time, then two, then one
  const float4* const W = reinterpret_cast<const float4*>(a.Wt);
#pragma unroll 1
  for (int ly = 0; ly < T.nl; ++ly) {
    const float* const x = lds + (ly & 1) * kNetBuf;
    float* const out = lds + ((ly & 1) ^ 1) * kNetBuf;
    const float4* const Wl = W + T.woff[ly] / 4;
    const float* const bl = a.Wt + T.boff[ly];
    const int nT = T.nT[ly], nQ = T.nQ[ly];
    const int half = kDuo ? (nT / 4 + 1) / 2 * 4 : nT;   // a wave's tiles (whole row blocks)
    int T0 = kDuo && role != 0 ? half : 0;
    const int T1 = kDuo && role == 0 ? half : nT;
#pragma unroll 1
    for (; T0 + 16 <= T1; T0 += 16) net_rows<kW, 4>(Wl, bl, nQ, T0, x, out, T.act, lane);
    if (T0 + 8 <= T1) {
      net_rows<kW, 2>(Wl, bl, nQ, T0, x, out, T.act, lane);
      T0 += 8;
    }
    if (T0 < T1) net_rows<kW, 1>(Wl, bl, nQ, T0, x, out, T.act, lane);
    if (kDuo) __syncthreads();
    else wave_sync();
  }
  if (kDuo && role != 0) return 0.f;
  // ---- head: lane (v, 16 ht + j) has row i = 16 ht + j of world v (mu 0..28, value 29)
  float hd[1][1];
  net_pass<1, 1, true>(W + T.woff[T.nl] / 4, a.Wt + T.boff[T.nl], T.nQ[T.nl], 0, mine + (T.nl & 1) * kNetBuf, lane, hd);
  const int i = l;
  if (i == kAct && wvalid) {
    if (t == a.H) a.Vlast[w] = hd[0][0];
    else a.V[(long)t * N + w] = hd[0][0];
  }
  if (t == a.H) return 0.f;
  // ---- sampling and log-prob (reference: src/g1_env.cu:308-318)
  float* const lpt = lds + kNetTail + 32 * v;
  float* const acts = lpt + 64;
  const float LOG2PI = 1.8378770664093453f;
  const long ab = ((long)t * N + w) * kAct;
  if (i < kAct) {
    float nz[2];
    if (a.act_noise) {
      nz[0] = nz[1] = wvalid || kW == 1 ? a.act_noise[ab + i] : 0.f;
    } else {
      rng_normal2(seed, wc, rng, kStreamAction, i >> 1, nz[0], nz[1]);   // actions 2 p and 2 p + 1 of one draw
    }
    const float n = (i & 1) ? nz[1] : nz[0];
    const float lsi = a.Wt[T.ls_off + i];
    const float av = hd[0][0] + expf(lsi) * n;
    if (wvalid) a.A[ab + i] = av;
    acts[i] = av;
    lpt[i] = -0.5f * n * n - lsi - 0.5f * LOG2PI;
  }
  wave_sync();
  if (l == 0 && wvalid) {
    float lpsum = 0.f;
#pragma unroll
    for (int k = 0; k < kAct; ++k) lpsum += lpt[k];
    a.LP[(long)t * N + w] = lpsum;
  }
  const float act = (l >= 2 && l < kNBody) ? acts[l - 2] : 0.f;
  wave_sync();
  return act;
}

// The end of control step t (its action and noise row) of world wc: reward r (lane 1), termination and
// auto-reset (reference: src/g1_env.cu:164-211), lane 1 decides. pa, step, rng: the lane's previous
// action and the world's step and noise counters, updated in place. Returns the done flag.
__device__ __forceinline__ int finish_control_step(const PhysArgs& a, const LaneModel& L, int l, int wc, int t,
                                                   float act, float vx_sum, float energy, LaneState& st, float& pa,
                                                   int& step, unsigned& rng, float& r) {
  const int ai = L.hinge ? L.b - 2 : 0;
  const float da = L.hinge ? act - pa : 0.f;
  float act_pen = gsum(da * da);
  const float energy_tot = gsum(energy);
  int d_flag = 0;
  r = 0.f;
  if (l == 1) {
    const float vx = vx_sum / (float)a.S;
    const float height = st.bq[2];
    const float qx = st.bq[4], qy = st.bq[5];
    const float up = fmaf_(-2.f, fmaf_(qy, qy, qx * qx), 1.f);   // quat2mat(q)[2][2]
    const int alive = !(height < 0.45f || up < 0.5f);
    const float upc = up < 0.f ? 0.f : (up > 1.f ? 1.f : up);
    float vx_c = vx > 0.8f ? 0.8f : vx;
    if (vx_c < 0.f) vx_c = 0.f;
    const float r_vel = 1.0f * vx_c * upc;
    const float r_lat = -0.2f * fabsf(st.bqd[1]) - 0.05f * fabsf(st.bqd[5]);
    const float r_up = 0.3f * upc;
    const float r_h = -0.5f * fabsf(height - 0.78f);
    if (act_pen > 10.f) act_pen = 10.f;
    r = alive ? 1.0f + r_vel + r_lat + r_up + r_h - 0.005f * act_pen - 1e-4f * energy_tot : -5.0f;
    const int won = alive && st.bq[0] >= 5.0f;
    if (won) r += 50.0f;
    d_flag = (!alive || won || step + 1 >= 1000) ? 1 : 0;
  }
  d_flag = gshfl(d_flag, 1);
  step += 1;
  pa = act;
  if (d_flag) {
    const float u = a.reset_noise ? a.reset_noise[((long)t * a.N + wc) * kAct + ai]
                                  : rng_pm1(a.seed, wc, rng, kStreamReset, ai);
    if (L.hinge) { st.jq = L.qstand + 0.05f * u; st.jqd = 0.f; pa = 0.f; }
#pragma unroll
    for (int m = 0; m < 7; ++m) st.bq[m] = MF::qpos_stand[m];
#pragma unroll
    for (int m = 0; m < 6; ++m) st.bqd[m] = 0.f;
    step = 0;
  }
  rng += 1;
  return d_flag;
}

// Enqueue k_resident on the null stream (resident_kernel.hip) with one world on two waves (duo) or two
// worlds per wave: the policy's rollout of ra.ph.K control steps, or (policy false) K >= 1 control steps
// on ra.ph.act.
void launch_resident_kernel(const ResidentArgs& ra, bool policy, bool duo);
// The instantiations' handles and block sizes (occupancy).
const void* resident_kernel_fn(bool policy, bool duo);
constexpr int resident_threads(bool duo) { return duo ? 2 * kPhysThreads : kPhysThreads; }

}  // namespace g1k
