// Affine-reset LIF kernels for MI355X (gfx950).  Reference: lifscan/triton_affine.py.
//
//   v = fl(fl(beta*u) + x);  s = v >= theta;  u' = s ? fl(fl(gamma*v) + delta) : v
//                                                     (triton_affine.py:19-23, 0 <= gamma <= 1)
// gamma = 0, delta = u_r is the hard reset; gamma = 1, delta = -theta the soft reset.
//
// Forward: serial / replay (k_aff_fwd) and the exact two-level scan (triton_affine.py:165-199):
// lower and upper reachable-state envelopes in one pass over the inputs (k_aff_env) and their
// sequential carries (k_aff_env_carry), capacity-K chunk maps of unsorted pieces
// [xl, xr) -> a*u + c (k_aff_build), the verified carry with serial fallback (k_aff_carry), the
// replay, and Jacobi repair on device (k_aff_repair).  The adjoint is the hard-reset adjoint
// with J_t = s_t ? gamma : 1 (lsh_aff_bwd in lif_kernels.hip).
//
// Workspace layout: header, envelope maps and bounds [M, N], pieces [M, N, K] as float4
// (xl, xr, a, c; the 32 lanes of one neuron store 512 contiguous bytes), counts, overflow
// flags, chunk starts / ends [M, N], repair work lists.
#include "lsh_abi.h"
#include "lsh_common.h"

namespace lsh {

// ---------------------------------------------------------------------------------------
// Serial / replay over segments of Ls steps from su (triton_affine.py:143-162).
template <int D, bool NT>
__global__ __launch_bounds__(64) void k_aff_fwd(const float* __restrict__ I,
                                                const float* __restrict__ su, float* __restrict__ U,
                                                float* __restrict__ S, float* __restrict__ eu,
                                                int64_t N, int64_t Ls, int NB, float beta,
                                                float theta, float gamma, float delta) {
  const int64_t m = blockIdx.x / NB;
  const int nb = (int)(blockIdx.x - m * NB);
  const int64_t n = (int64_t)nb * WAVE + threadIdx.x;
  if (n >= N) return;
  float u = su[m * N + n];
  const size_t base = (size_t)m * (size_t)Ls * (size_t)N + (size_t)n;
  stream_rows<D>(I + base, (size_t)N, Ls, [&](int64_t j, float x) {
    bool s;
    u = aff_step(u, x, beta, theta, gamma, delta, s);
    const size_t o = base + (size_t)j * N;
    st_out<NT>(U + o, u);
    st_out<NT>(S + o, s ? 1.0f : 0.0f);
  });
  if (eu) eu[m * N + n] = u;
}

// ---------------------------------------------------------------------------------------
// Envelopes of the reachable states per chunk, both from one read of the inputs:
//  lower (triton_lif.py:699-719 with u_r = r(theta), as triton_affine.py:171-172):
//    l -> min(r, beta*l + x), composed as min(c, a*l + b);
//  upper (triton_affine.py:26-36): h -> max(theta, gamma*(beta*h + x) + delta), composed as
//    max(c, a*h + b) with a = (gamma*beta)^C.  From c = -inf, gamma = 0 gives 0*(-inf) = NaN,
//    which fmaxf drops (IEEE maxNum), leaving theta.
__global__ __launch_bounds__(64) void k_aff_env(const float* __restrict__ I,
                                                float* __restrict__ EC, float* __restrict__ EA,
                                                float* __restrict__ EB, float* __restrict__ HC,
                                                float* __restrict__ HA, float* __restrict__ HB,
                                                int64_t N, int NB, int C, float beta, float theta,
                                                float gamma, float delta, float r_theta) {
  const int64_t m = blockIdx.x / NB;
  const int nb = (int)(blockIdx.x - m * NB);
  const int64_t n = (int64_t)nb * WAVE + threadIdx.x;
  if (n >= N) return;
  const float gb = gamma * beta;
  float lc = INFINITY, la = 1.0f, lb = 0.0f;
  float hc = -INFINITY, ha = 1.0f, hb = 0.0f;
  stream_rows<16>(I + (size_t)m * C * N + n, (size_t)N, C, [&](int64_t, float x) {
    lc = fminf(r_theta, lif_v(lc, x, beta));
    la = beta * la;
    lb = lif_v(lb, x, beta);
    hc = fmaxf(theta, __fadd_rn(__fmul_rn(gamma, lif_v(hc, x, beta)), delta));
    ha = gb * ha;
    hb = __fadd_rn(__fmul_rn(gamma, lif_v(hb, x, beta)), delta);
  });
  const size_t o = (size_t)m * N + n;
  EC[o] = lc;
  EA[o] = la;
  EB[o] = lb;
  HC[o] = hc;
  HA[o] = ha;
  HB[o] = hb;
}

constexpr int kAffAhead = 8;  // chunks whose envelope maps the carry reads ahead

// Sequential envelope carries (triton_lif.py:723-733, triton_affine.py:39-48), margin 1e-5:
// LO[m] = l - 1e-5(|l| + 1), HI[m] = h + 1e-5(|h| + 1) with l, h the bounds at chunk m's start.
__global__ __launch_bounds__(64) void k_aff_env_carry(
    const float* __restrict__ u0, const float* __restrict__ EC, const float* __restrict__ EA,
    const float* __restrict__ EB, const float* __restrict__ HC, const float* __restrict__ HA,
    const float* __restrict__ HB, float* __restrict__ LO, float* __restrict__ HI, int64_t N, int M) {
  const int64_t n = (int64_t)blockIdx.x * WAVE + threadIdx.x;
  if (n >= N) return;
  const float margin = 1e-5f;
  float l = u0[n], h = l;
  // The maps of the next kAffAhead chunks are in flight while one is applied (index clamped, every
  // load unconditional): one chunk at a time waited for six loads per chunk, 23 us for 64 chunks.
  float ec[kAffAhead], ea[kAffAhead], eb[kAffAhead], hc[kAffAhead], ha[kAffAhead], hb[kAffAhead];
  const auto load = [&](int k, int m) {
    const size_t o = (size_t)min(m, M - 1) * N + n;
    ec[k] = EC[o];
    ea[k] = EA[o];
    eb[k] = EB[o];
    hc[k] = HC[o];
    ha[k] = HA[o];
    hb[k] = HB[o];
    __builtin_amdgcn_sched_barrier(0);  // issued in the chunks' order
  };
#pragma unroll
  for (int k = 0; k < kAffAhead; ++k) load(k, k);
  for (int m0 = 0; m0 < M; m0 += kAffAhead) {
#pragma unroll
    for (int k = 0; k < kAffAhead; ++k) {
      const int m = m0 + k;
      if (m < M) {
        const size_t o = (size_t)m * N + n;
        LO[o] = l - margin * (fabsf(l) + 1.0f);
        HI[o] = h + margin * (fabsf(h) + 1.0f);
        l = fminf(ec[k], __fadd_rn(__fmul_rn(ea[k], l), eb[k]));
        h = fmaxf(hc[k], __fadd_rn(__fmul_rn(ha[k], h), hb[k]));
      }
      load(k, m + kAffAhead);
    }
  }
}

// ---------------------------------------------------------------------------------------
// Chunk maps (triton_affine.py:51-111).  L lanes serve one neuron of one chunk: a 16-lane row (4
// neurons a wave, 16 a workgroup), lane i holding piece slots i and 16 + i, the second touched only
// while some neuron of the wave has more than 16 pieces; or 32 lanes with one slot each.  Inputs are
// staged through LDS in tiles of 32 steps together with ct = (theta - x)/beta, computed once per
// (neuron, step); the next tile's inputs are loaded while a tile runs.
// Per step every piece [xl, xr) with value a*u + c meets the threshold cut z = (ct - c)/a
// (u >= z spikes; a == 0: all or nothing); its left part [xl, min(xr, z)) and its spiking
// right part [z, xr) are kept when they meet [lo, hi].
// Between steps the slots are in no order: a piece that keeps one part stays where it is, one that
// dies leaves a free slot, and the right part of one that keeps both goes to a free slot (through
// the neuron's LDS row).  The pieces are disjoint intervals, so the reference's list is the slots
// sorted by xl; they are sorted at the end of the chunk, and in a step after which a neuron would
// hold more than K (the overflow flag is set and the parts beyond slot K are dropped, as the
// reference's compaction does).  Compacting on every birth and death ran on two steps of three.
// The tests are kept as wave masks (a ballot of one compare is the compare's own result); free
// slots drift with the others and the masks leave them out.
// Where the chunks and neurons fill the chip it is bound by VALU issue (a correctly rounded division
// per piece and step): most maps hold 3 to 9 pieces, so 32 lanes leave most lanes idle.  Measured, C
// 128, 32 lanes and compaction -> 16 lanes: T 8192, N 200 gamma 0.5 82 -> 51 us, N 333 soft reset 121
// -> 101 us; T 4096, N 4096 537 -> 284 and 543 -> 300 us (16 lanes with compaction 59, 111, 353, 367;
// 8 lanes and four slots 98, 177, 416, 492).  With few it is bound by a step's own latency, which a
// second slot and the sorts of overflowing maps lengthen: up to kAffWideBlocks workgroups of 16
// neurons take 32 lanes.  The scan, 32 lanes and compaction / 16 lanes / 32 lanes, us, with many pieces
// (beta 0.99, gamma 0.9) and few (0.9, 0.5): T 512, N 65, C 128, K 32 (20 workgroups) 71 / 103 / 69 and
// 62 / 58 / 52; T 2048, N 333, C 128 (336) 108 / 136 / 100 and 88 / 65 / 64; C 64, K 16 (672) 121 / 138 /
// 112 and 84 / 55 / 60; T 8192, N 200, C 128, K 32 (832) 234 / 238 / 198 and 158 / 95 / 105; T 4096, N
// 1000 (2016) 252 / 265 / 224 and 210 / 120 / 157.
constexpr int64_t kAffWideBlocks = 768;
constexpr int kAffWaves = 4;                 // waves per workgroup
constexpr int kAffTS = 32;                   // steps per staged tile
constexpr int aff_npw(int L) { return kAffWaves * (WAVE / L); }  // neurons per workgroup, L lanes each

// One piece slot's step: the cut, the masks of the kept left / right parts and the updated fields.
struct AffStepSlot {
  float z, xr, vns, c_sp, a_sp, a_ns;
  unsigned long long left, right, full;
};
__device__ __forceinline__ AffStepSlot aff_slot_step(float pxl, float pxr, float pa, float pc,
                                                     unsigned long long live, float x, float ct,
                                                     float lo, float hi, float beta, float gb,
                                                     float gamma, float delta) {
  AffStepSlot r;
  const float num = ct - pc;
  r.z = num / pa;
  if (wave_ballot(pa == 0.0f) != 0ull)
    r.z = pa == 0.0f ? (num > 0.0f ? INFINITY : -INFINITY) : r.z;
  const unsigned long long cut = live & wave_ballot(r.z > pxl) & wave_ballot(r.z < pxr);
  r.full = wave_ballot(r.z <= pxl);
  r.xr = __builtin_amdgcn_inverse_ballot_w64(cut) ? r.z : pxr;
  r.left = live & wave_ballot(r.xr > lo) & wave_ballot(pxl <= hi);
  r.right = cut & wave_ballot(pxr > lo) & wave_ballot(r.z <= hi);
  r.vns = lif_v(pc, x, beta);
  r.c_sp = __fadd_rn(__fmul_rn(gamma, r.vns), delta);
  r.a_sp = gb * pa;
  r.a_ns = beta * pa;
  return r;
}

template <int L>
__global__ __launch_bounds__(WAVE * kAffWaves, 7) void k_aff_build(  // 72 registers: 7 waves a SIMD
    const float* __restrict__ I, const float* __restrict__ LO, const float* __restrict__ HI,
    float4* __restrict__ PC, int* __restrict__ NP, int* __restrict__ OVF, int64_t N, int NBLK,
    int C, int K, float beta, float theta, float gamma, float delta) {
  static_assert(L == 16 || L == 32, "a row holds 32 pieces in one or two slots a lane");
  constexpr bool TWO = L == 16;  // a lane's second slot
  constexpr int NPW = aff_npw(L), LD = NPW * kAffTS / (kAffWaves * WAVE);  // LD: inputs a lane stages
  __shared__ float sX[NPW][kAffTS + 1], sCt[NPW][kAffTS + 1];
  __shared__ float4 sSlot[NPW][33];  // a neuron's slots, off the banks of the next neuron's
  // sort keys: at most 32 pieces, each with a new part, and three past the last one
  __shared__ __attribute__((aligned(16))) float sKey[NPW][TWO ? 65 : 68];
  const int64_t m = blockIdx.x / NBLK;
  const int blk = (int)(blockIdx.x - m * NBLK);
  const int tid = threadIdx.x;
  const int lane = tid % WAVE;
  const int i = lane & (L - 1);
  const int ln = tid / L;  // neuron of the workgroup
  const int64_t n0 = (int64_t)blk * NPW;
  const int64_t n = n0 + ln;
  const bool valid_n = n < N;
  const size_t o = (size_t)m * N + (valid_n ? n : N - 1);
  const float lo = LO[o], hi = HI[o];
  const float gb = gamma * beta;
  float pxl0 = i == 0 ? -INFINITY : INFINITY, pxr0 = INFINITY, pa0 = 1.0f, pc0 = 0.0f;
  float pxl1 = INFINITY, pxr1 = INFINITY, pa1 = 1.0f, pc1 = 0.0f;
  int cnt = 1, ovf = 0;
  unsigned long long live0 = wave_ballot(i < 1), live1 = 0ull;
  float4* slot = sSlot[ln];
  const unsigned below = (1u << i) - 1;  // the row's lanes before this one
  // the row's bits of a wave mask
  const auto row_of = [&](unsigned long long mask) {
    const unsigned w = lane < 32 ? (unsigned)mask : (unsigned)(mask >> 32);
    return TWO ? (w >> (lane & 16)) & 0xffffu : w;
  };
  const auto lane_of = [](unsigned long long mask) {
    return __builtin_amdgcn_inverse_ballot_w64(mask);
  };
  // The row's pieces (live0, live1) and, where the masks say so, the new parts n0, n1 of this
  // lane's slots into slots 0, 1, ... by ascending xl, the first K of them.  Same-wave LDS accesses
  // complete in order.
  const auto sort_row = [&](unsigned long long new0, unsigned long long new1, const float4& n0,
                            const float4& n1) {
    const unsigned l0 = row_of(live0), l1 = row_of(live1), b0 = row_of(new0), b1 = row_of(new1);
    const int o1 = __popc(l0), o2 = o1 + __popc(l1), o3 = o2 + __popc(b0), tot = o3 + __popc(b1);
    float* key = sKey[ln];
    const bool h0 = lane_of(live0), h1 = lane_of(live1), g0 = lane_of(new0), g1 = lane_of(new1);
    if (h0) key[__popc(l0 & below)] = pxl0;
    if (h1) key[o1 + __popc(l1 & below)] = pxl1;
    if (g0) key[o2 + __popc(b0 & below)] = n0.x;
    if (g1) key[o3 + __popc(b1 & below)] = n1.x;
    if (!TWO && i < 3) key[tot + i] = INFINITY;  // counted by nothing
    __builtin_amdgcn_wave_barrier();
    int k0 = 0, k1 = 0, m0 = 0, m1 = 0;  // ranks
    if constexpr (TWO) {
      for (int j = 0; j < tot; ++j) {
        const float v = key[j];
        k0 += v < pxl0 ? 1 : 0;
        k1 += v < pxl1 ? 1 : 0;
        m0 += v < n0.x ? 1 : 0;
        m1 += v < n1.x ? 1 : 0;
      }
    } else {  // a step's latency counts: four keys a load
      const auto count = [](int& k, const float4& v, float x) {
        k += (v.x < x ? 1 : 0) + (v.y < x ? 1 : 0) + (v.z < x ? 1 : 0) + (v.w < x ? 1 : 0);
      };
      for (int j = 0; j < tot; j += 4) {
        const float4 v = *reinterpret_cast<const float4*>(key + j);
        count(k0, v, pxl0);
        count(m0, v, n0.x);
      }
    }
    if (h0 && k0 < K) slot[k0] = make_float4(pxl0, pxr0, pa0, pc0);
    if (h1 && k1 < K) slot[k1] = make_float4(pxl1, pxr1, pa1, pc1);
    if (g0 && m0 < K) slot[m0] = n0;
    if (g1 && m1 < K) slot[m1] = n1;
    if (tot > K) ovf = 1;
    cnt = min(tot, K);
    __builtin_amdgcn_wave_barrier();
    const float4 q0 = slot[i];
    pxl0 = q0.x, pxr0 = q0.y, pa0 = q0.z, pc0 = q0.w;
    live0 = wave_ballot(i < cnt);
    if constexpr (TWO) {
      const float4 q1 = slot[L + i];
      pxl1 = q1.x, pxr1 = q1.y, pa1 = q1.z, pc1 = q1.w;
      live1 = wave_ballot(L + i < cnt);
    }
    __builtin_amdgcn_wave_barrier();
  };
  const float* __restrict__ Im = I + (size_t)m * C * N;
  float xr[LD];
  const auto load = [&](int j0) {  // this lane's inputs of the tile at j0 (rows past C: the last)
#pragma unroll
    for (int q = 0; q < LD; ++q) {
      const int e = tid + q * kAffWaves * WAVE;
      const int64_t ne = n0 + e % NPW;
      xr[q] = Im[(size_t)min(j0 + e / NPW, C - 1) * N + (ne < N ? ne : N - 1)];
    }
  };
  load(0);
  for (int j0 = 0; j0 < C; j0 += kAffTS) {
    const int ts = min(kAffTS, C - j0);
    __syncthreads();  // the previous tile has been read
#pragma unroll
    for (int q = 0; q < LD; ++q) {
      const int e = tid + q * kAffWaves * WAVE;
      sX[e % NPW][e / NPW] = xr[q];
      sCt[e % NPW][e / NPW] = (theta - xr[q]) / beta;
    }
    __syncthreads();
    load(j0 + kAffTS);
    // second slots that are no longer needed: back to one slot a lane
    if (TWO && live1 != 0ull &&
        wave_ballot(__popc(row_of(live0)) + __popc(row_of(live1)) > 16) == 0ull)
      sort_row(0ull, 0ull, make_float4(0, 0, 0, 0), make_float4(0, 0, 0, 0));
    float xs = sX[ln][0], cts = sCt[ln][0];
    for (int k = 0; k < ts; ++k) {
      const float x = xs, ct = cts;
      xs = sX[ln][k + 1];  // the next step's (behind the tile's last step: the padding)
      cts = sCt[ln][k + 1];
      const AffStepSlot r0 = aff_slot_step(pxl0, pxr0, pa0, pc0, live0, x, ct, lo, hi, beta, gb,
                                           gamma, delta);
      const unsigned long long new0 = r0.left & r0.right;
      const float4 n0 = make_float4(r0.z, pxr0, r0.a_sp, r0.c_sp);
      {
        const unsigned long long ro = r0.right & ~r0.left;
        const bool right = lane_of(ro), sp = lane_of(ro | r0.full);
        pxr0 = right ? pxr0 : r0.xr;
        pxl0 = right ? r0.z : pxl0;
        pa0 = sp ? r0.a_sp : r0.a_ns;
        pc0 = sp ? r0.c_sp : r0.vns;
        live0 = r0.left | r0.right;
      }
      unsigned long long new1 = 0ull;
      float4 n1 = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      if (TWO && live1 != 0ull) {
        const AffStepSlot r1 = aff_slot_step(pxl1, pxr1, pa1, pc1, live1, x, ct, lo, hi, beta, gb,
                                             gamma, delta);
        new1 = r1.left & r1.right;
        n1 = make_float4(r1.z, pxr1, r1.a_sp, r1.c_sp);
        const unsigned long long ro = r1.right & ~r1.left;
        const bool right = lane_of(ro), sp = lane_of(ro | r1.full);
        pxr1 = right ? pxr1 : r1.xr;
        pxl1 = right ? r1.z : pxl1;
        pa1 = sp ? r1.a_sp : r1.a_ns;
        pc1 = sp ? r1.c_sp : r1.vns;
        live1 = r1.left | r1.right;
      }
      if ((new0 | new1) == 0ull) continue;
      const unsigned b0 = row_of(new0), b1 = row_of(new1);
      constexpr unsigned row = TWO ? 0xffffu : 0xffffffffu;
      const unsigned f0 = ~row_of(live0) & row, f1 = TWO ? ~row_of(live1) & row : 0u;
      const int nb0 = __popc(b0), nb = nb0 + __popc(b1), nf0 = __popc(f0);
      if (wave_ballot(32 - nf0 - __popc(f1) + nb > K) != 0ull) {
        sort_row(new0, new1, n0, n1);
        continue;
      }
      // the j-th new part of the row to its j-th free slot
      if (lane_of(new0)) slot[__popc(b0 & below)] = n0;
      if (lane_of(new1)) slot[nb0 + __popc(b1 & below)] = n1;
      __builtin_amdgcn_wave_barrier();
      const int j = __popc(f0 & below);
      const bool take = ((f0 >> i) & 1u) != 0u && j < nb;
      const float4 q = slot[j];
      pxl0 = take ? q.x : pxl0;
      pxr0 = take ? q.y : pxr0;
      pa0 = take ? q.z : pa0;
      pc0 = take ? q.w : pc0;
      live0 |= wave_ballot(take);
      if (TWO && wave_ballot(nb > nf0) != 0ull) {
        const int j1 = nf0 + __popc(f1 & below);
        const bool take1 = ((f1 >> i) & 1u) != 0u && j1 < nb;
        const float4 q1 = slot[j1];
        pxl1 = take1 ? q1.x : pxl1;
        pxr1 = take1 ? q1.y : pxr1;
        pa1 = take1 ? q1.z : pa1;
        pc1 = take1 ? q1.w : pc1;
        live1 |= wave_ballot(take1);
      }
      __builtin_amdgcn_wave_barrier();
    }
  }
  sort_row(0ull, 0ull, make_float4(0, 0, 0, 0), make_float4(0, 0, 0, 0));
  if (!valid_n) return;
  if (i < K)
    PC[o * K + i] = i < cnt ? make_float4(pxl0, pxr0, pa0, pc0)
                            : make_float4(INFINITY, INFINITY, 1.0f, 0.0f);
  if (TWO && L + i < K)
    PC[o * K + L + i] = L + i < cnt ? make_float4(pxl1, pxr1, pa1, pc1)
                                    : make_float4(INFINITY, INFINITY, 1.0f, 0.0f);
  if (i == 0) {
    NP[o] = cnt;
    OVF[o] = ovf;
  }
}

// Verified carry (triton_affine.py:114-140), two neurons per wave, lane i = piece slot i: the
// start u must lie in exactly one piece of a map that did not overflow, and the chunk's end
// state is that piece's a*u + c (plus 0.0: the reference sums the hit lanes, so a -0.0 reads
// as +0.0); otherwise the chunk runs serially.  The next kAffMaps chunks' maps are in flight while
// one is evaluated (one ahead left the walk waiting for memory: 64 chunks of 200 neurons 39 -> 18 us).
constexpr int kAffMaps = 4;
constexpr int kAffCarryWaves = 4;  // waves of a workgroup, which adds its statistics once
__global__ __launch_bounds__(WAVE* kAffCarryWaves) void k_aff_carry(
    const float* __restrict__ I, const float* __restrict__ u0, const float4* __restrict__ PC,
    const int* __restrict__ NP, const int* __restrict__ OVF, float* __restrict__ STARTS,
    WsHeader* hdr, int64_t N, int M, int C, int K, float beta, float theta, float gamma,
    float delta) {
  const int lane = threadIdx.x % WAVE;
  const int half = lane >> 5;
  const int i = lane & 31;
  const int hb = half << 5;
  const int64_t n = ((int64_t)blockIdx.x * kAffCarryWaves + threadIdx.x / WAVE) * 2 + half;
  const bool valid_n = n < N;
  const int64_t nn = valid_n ? n : N - 1;
  const unsigned long long hmask = 0xffffffffull << hb;
  // lanes i >= K read slot K - 1 (never a hit: i >= K >= count)
  const int ks = i < K ? i : K - 1;
  float u = u0[nn];
  unsigned long long ovf_acc = 0, pcs_acc = 0;
  int pmax = 0;
  float4 qs[kAffMaps];
  int cnts[kAffMaps], ovfs[kAffMaps];
  const auto load = [&](int k, int m) {
    const size_t o = (size_t)min(m, M - 1) * N + nn;
    qs[k] = PC[o * K + ks];
    cnts[k] = NP[o];
    ovfs[k] = OVF[o];
    // the loads stay in the chunks' order: with a later chunk's issued first, the wait for the
    // current chunk covers them all
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
#pragma unroll
  for (int k = 0; k < kAffMaps; ++k) load(k, k);
  for (int m0 = 0; m0 < M; m0 += kAffMaps) {
#pragma unroll
    for (int k = 0; k < kAffMaps; ++k) {
      const int m = m0 + k;
      if (m < M) {
        const float4 q = qs[k];
        const int cnt = cnts[k], ovf = ovfs[k];
        if (valid_n && i == 0) STARTS[(size_t)m * N + nn] = u;
        const bool hit = i < cnt && q.x <= u && u < q.y;
        const unsigned long long hm = (wave_ballot(hit) & hmask) >> hb;
        const int nh = __builtin_popcountll(hm);
        const int hl = hm ? __builtin_ctzll(hm) : 0;
        const float val = __fadd_rn(__fmul_rn(q.z, u), q.w);
        float nu = __shfl(val, hl, 32) + 0.0f;  // all lanes shuffle
        if (ovf != 0 || nh != 1) {
          float w = u;
          stream_rows<16>(I + (size_t)m * C * N + nn, (size_t)N, C, [&](int64_t, float x) {
            bool s;
            w = aff_step(w, x, beta, theta, gamma, delta, s);
          });
          nu = w;
        }
        if (valid_n && i == 0) {
          ovf_acc += ovf ? 1ull : 0ull;
          pcs_acc += (unsigned long long)cnt;
          pmax = max(pmax, cnt);
        }
        u = nu;
      }
      load(k, m + kAffMaps);
    }
  }
  add_map_stats(hdr, ovf_acc, pcs_acc, pmax);
}

// Jacobi repair of the chunk starts on device (triton_affine.py:188-194): chunk m (> 0) whose
// start differs from chunk m-1's end is replayed from that end; a changed end queues chunk
// m+1.  One workgroup per 64 neurons with work lists in the workspace; the rounds counted are
// those the reference's loop counts (at most R).
__global__ __launch_bounds__(256) void k_aff_repair(
    const float* __restrict__ I, float* __restrict__ U, float* __restrict__ S,
    float* __restrict__ su, float* __restrict__ eu, int* __restrict__ list0,
    int* __restrict__ list1, WsHeader* hdr, int64_t N, int M, int C, int64_t R, float beta,
    float theta, float gamma, float delta) {
  __shared__ int s_nd, s_nc;
  const int nb = blockIdx.x;
  const int tid = threadIdx.x;
  const size_t cap = (size_t)M * WAVE;
  int* __restrict__ dl = list0 + (size_t)nb * cap;
  int* __restrict__ cl = list1 + (size_t)nb * cap;
  auto differs = [&](int m, int64_t n) {
    return eu[(size_t)(m - 1) * N + n] != su[(size_t)m * N + n];
  };
  if (tid == 0) s_nd = 0;
  __syncthreads();
  for (int e = tid + WAVE; e < M * WAVE; e += blockDim.x) {
    const int m = e / WAVE;
    const int64_t n = (int64_t)nb * WAVE + (e % WAVE);
    if (n < N && differs(m, n)) dl[atomicAdd(&s_nd, 1)] = e;
  }
  __syncthreads();
  int64_t rounds = 0;
  while (true) {
    const int nd = s_nd;
    if (nd == 0 || rounds >= R) break;
    ++rounds;
    for (int k = tid; k < nd; k += blockDim.x) {
      const int e = dl[k];
      const int m = e / WAVE;
      const int64_t n = (int64_t)nb * WAVE + (e % WAVE);
      su[(size_t)m * N + n] = eu[(size_t)(m - 1) * N + n];
    }
    __syncthreads();
    if (tid == 0) s_nc = 0;
    __syncthreads();
    for (int k = tid; k < nd; k += blockDim.x) {
      const int e = dl[k];
      const int m = e / WAVE;
      const int64_t n = (int64_t)nb * WAVE + (e % WAVE);
      float u = su[(size_t)m * N + n];
      const size_t base = (size_t)m * C * N + n;
      stream_rows<16>(I + base, (size_t)N, C, [&](int64_t j, float x) {
        bool s;
        u = aff_step(u, x, beta, theta, gamma, delta, s);
        U[base + (size_t)j * N] = u;
        S[base + (size_t)j * N] = s ? 1.0f : 0.0f;
      });
      const size_t oe = (size_t)m * N + n;
      if (u != eu[oe]) {
        eu[oe] = u;
        if (m + 1 < M) cl[atomicAdd(&s_nc, 1)] = e + WAVE;
      }
    }
    __syncthreads();
    if (tid == 0) s_nd = 0;
    __syncthreads();
    const int nc = s_nc;
    for (int k = tid; k < nc; k += blockDim.x) {
      const int e = cl[k];
      const int m = e / WAVE;
      const int64_t n = (int64_t)nb * WAVE + (e % WAVE);
      if (differs(m, n)) dl[atomicAdd(&s_nd, 1)] = e;
    }
    __syncthreads();
  }
  if (tid == 0) atomicMax(&hdr->repair_iters, (unsigned int)rounds);
}

// Reverse affine recurrence lam_t = a_t*lam_{t+1} + b_t, lam_T = 0, per column
// (triton_affine.py:202-211 reverse_affine_scan, there a Hillis-Steele scan over torch ops):
// one lane per column, rows consumed from the last in tiles of D loaded ahead.
template <int D>
__global__ __launch_bounds__(64) void k_rev_affine(const float* __restrict__ A,
                                                   const float* __restrict__ B,
                                                   float* __restrict__ L, int64_t T, int64_t N) {
  const int64_t n = (int64_t)blockIdx.x * WAVE + threadIdx.x;
  if (n >= N) return;
  float lam = 0.0f;
  const int64_t nt = T / D;
  auto row = [&](int64_t t) { return (size_t)t * (size_t)N + (size_t)n; };
  float a[D], b[D];
  if (nt > 0) {
#pragma unroll
    for (int k = 0; k < D; ++k) {
      a[k] = A[row(T - 1 - k)];
      b[k] = B[row(T - 1 - k)];
    }
  }
  for (int64_t g = 0; g < nt; ++g) {
    float an[D], bn[D];
    const bool more = g + 1 < nt;
    if (more) {
#pragma unroll
      for (int k = 0; k < D; ++k) {
        an[k] = A[row(T - 1 - (g + 1) * D - k)];
        bn[k] = B[row(T - 1 - (g + 1) * D - k)];
      }
    }
#pragma unroll
    for (int k = 0; k < D; ++k) {
      lam = __fadd_rn(__fmul_rn(a[k], lam), b[k]);
      L[row(T - 1 - g * D - k)] = lam;
    }
    if (more) {
#pragma unroll
      for (int k = 0; k < D; ++k) {
        a[k] = an[k];
        b[k] = bn[k];
      }
    }
  }
  for (int64_t t = T - nt * D - 1; t >= 0; --t) {
    lam = __fadd_rn(__fmul_rn(A[row(t)], lam), B[row(t)]);
    L[row(t)] = lam;
  }
}

static void aff_scan_layout(int64_t T, int64_t N, int C, int K, lsh_aff_layout* L) {
  const int64_t M = T / C;
  const size_t mn = (size_t)M * (size_t)N * 4;
  const size_t nb = (size_t)((N + WAVE - 1) / WAVE);
  Carver c;
  L->EC = c.take(mn);
  L->EA = c.take(mn);
  L->EB = c.take(mn);
  L->HC = c.take(mn);
  L->HA = c.take(mn);
  L->HB = c.take(mn);
  L->LO = c.take(mn);
  L->HI = c.take(mn);
  L->PIECES = c.take(mn * 4 * (size_t)K);
  L->NP = c.take(mn);
  L->OVF = c.take(mn);
  L->STARTS = c.take(mn);
  L->ENDS = c.take(mn);
  L->LIST0 = c.take(nb * (size_t)M * WAVE * 4);
  L->LIST1 = c.take(nb * (size_t)M * WAVE * 4);
  L->total = c.off;
}

static int aff_scan_check(int64_t T, int64_t N, int C, int K) {
  if (T < 0 || N < 0 || N > (int64_t)1 << 31) return LSH_ERR_SHAPE;
  if (C < 1 || K < 1 || K > 32) return LSH_ERR_SHAPE;
  if (T % C != 0) return LSH_ERR_DIVISIBILITY;
  const int64_t M = T / C;
  if (M * ((N + aff_npw(16) - 1) / aff_npw(16)) > ((int64_t)1 << 31) - 1) return LSH_ERR_SHAPE;
  return LSH_OK;
}

}  // namespace lsh

using namespace lsh;

extern "C" int lsh_aff_serial_fwd(const float* I, const float* u0, float* U, float* S, int64_t T,
                                  int64_t N, float beta, float theta, float gamma, float delta,
                                  void* stream) {
  if (bad_ptr(I) || bad_ptr(u0) || bad_ptr(U) || bad_ptr(S)) return LSH_ERR_ARG;
  if (!(gamma >= 0.0f && gamma <= 1.0f)) return LSH_ERR_ARG;
  if (T < 0 || N < 0 || N > (int64_t)1 << 31) return LSH_ERR_SHAPE;
  if (T == 0 || N == 0) return LSH_OK;
  aff_serial_fwd_pipe(I, u0, U, S, N, T, beta, theta, gamma, delta, (hipStream_t)stream);
  LSH_CHECK_LAUNCH();
  return LSH_OK;
}

extern "C" int lsh_aff_scan_layout(int64_t T, int64_t N, int C, int K, lsh_aff_layout* out) {
  if (bad_ptr(out)) return LSH_ERR_ARG;
  const int rc = aff_scan_check(T, N, C, K);
  if (rc != LSH_OK) return rc;
  aff_scan_layout(T, N, C, K, out);
  return LSH_OK;
}

extern "C" size_t lsh_aff_scan_workspace(int64_t T, int64_t N, int C, int K) {
  if (aff_scan_check(T, N, C, K) != LSH_OK) return 0;
  lsh_aff_layout L;
  aff_scan_layout(T, N, C, K, &L);
  return L.total;
}

extern "C" int lsh_aff_scan_fwd(const float* I, const float* u0, float* U, float* S, int64_t T,
                                int64_t N, float beta, float theta, float gamma, float delta,
                                float r_theta, int C, int K, int64_t repair, void* ws,
                                size_t ws_bytes, void* stream) {
  if (bad_ptr(I) || bad_ptr(u0) || bad_ptr(U) || bad_ptr(S) || bad_ptr(ws)) return LSH_ERR_ARG;
  if (repair < 0 || !(gamma >= 0.0f && gamma <= 1.0f)) return LSH_ERR_ARG;
  const int rc = aff_scan_check(T, N, C, K);
  if (rc != LSH_OK) return rc;
  lsh_aff_layout L;
  aff_scan_layout(T, N, C, K, &L);
  if (ws_bytes < L.total || (reinterpret_cast<uintptr_t>(ws) & 255u) != 0) return LSH_ERR_WORKSPACE;
  hipStream_t st = (hipStream_t)stream;
  char* w = static_cast<char*>(ws);
  WsHeader* h = reinterpret_cast<WsHeader*>(w);
  hipLaunchKernelGGL(k_ws_header_reset, dim3(1), dim3(64), 0, st, h);
  if (T == 0 || N == 0) {
    LSH_CHECK_LAUNCH();
    return LSH_OK;
  }
  const int M = (int)(T / C);
  const int NB = (int)((N + WAVE - 1) / WAVE);
  auto F = [&](size_t off) { return reinterpret_cast<float*>(w + off); };
  auto Iq = [&](size_t off) { return reinterpret_cast<int*>(w + off); };
  float4* PC = reinterpret_cast<float4*>(w + L.PIECES);
  hipLaunchKernelGGL(k_aff_env, dim3((unsigned)((int64_t)M * NB)), dim3(WAVE), 0, st, I, F(L.EC),
                     F(L.EA), F(L.EB), F(L.HC), F(L.HA), F(L.HB), N, NB, C, beta, theta, gamma,
                     delta, r_theta);
  hipLaunchKernelGGL(k_aff_env_carry, dim3((unsigned)NB), dim3(WAVE), 0, st, u0, F(L.EC), F(L.EA),
                     F(L.EB), F(L.HC), F(L.HA), F(L.HB), F(L.LO), F(L.HI), N, M);
  const auto build = [&](auto lanes) {
    constexpr int LN = decltype(lanes)::value;
    const int NBLK = (int)((N + aff_npw(LN) - 1) / aff_npw(LN));
    hipLaunchKernelGGL(k_aff_build<LN>, dim3((unsigned)((int64_t)M * NBLK)), dim3(WAVE * kAffWaves), 0, st,
                       I, F(L.LO), F(L.HI), PC, Iq(L.NP), Iq(L.OVF), N, NBLK, C, K, beta, theta, gamma,
                       delta);
  };
  if (M * ((N + aff_npw(16) - 1) / aff_npw(16)) <= kAffWideBlocks)
    build(std::integral_constant<int, 32>{});
  else
    build(std::integral_constant<int, 16>{});
  hipLaunchKernelGGL(k_aff_carry,
                     dim3((unsigned)((N + 2 * kAffCarryWaves - 1) / (2 * kAffCarryWaves))),
                     dim3(WAVE * kAffCarryWaves), 0, st, I, u0, PC,
                     Iq(L.NP), Iq(L.OVF), F(L.STARTS), h, N, M, C, K, beta, theta, gamma, delta);
  with_store_policy(rows_aligned(N), [&](auto nt) {
    hipLaunchKernelGGL((k_aff_fwd<16, decltype(nt)::value>), dim3((unsigned)((int64_t)M * NB)), dim3(WAVE), 0, st, I,
                     F(L.STARTS), U, S, F(L.ENDS), N, (int64_t)C, NB, beta, theta, gamma, delta);
  });
  if (repair > 0 && M > 1) {
    const int64_t rounds = repair < (int64_t)M ? repair : (int64_t)M;
    hipLaunchKernelGGL(k_aff_repair, dim3((unsigned)NB), dim3(256), 0, st, I, U, S, F(L.STARTS),
                       F(L.ENDS), Iq(L.LIST0), Iq(L.LIST1), h, N, M, C, rounds, beta, theta, gamma,
                       delta);
  }
  LSH_CHECK_LAUNCH();
  return LSH_OK;
}

extern "C" int lsh_reverse_affine_scan(const float* A, const float* B, float* L, int64_t T,
                                       int64_t N, void* stream) {
  if (bad_ptr(A) || bad_ptr(B) || bad_ptr(L)) return LSH_ERR_ARG;
  if (T < 0 || N < 0 || N > (int64_t)1 << 31) return LSH_ERR_SHAPE;
  if (T == 0 || N == 0) return LSH_OK;
  hipLaunchKernelGGL((k_rev_affine<16>), dim3((unsigned)((N + WAVE - 1) / WAVE)), dim3(WAVE), 0,
                     (hipStream_t)stream, A, B, L, T, N);
  LSH_CHECK_LAUNCH();
  return LSH_OK;
}
