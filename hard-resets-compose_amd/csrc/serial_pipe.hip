// Wave-specialised serial sweeps for few neurons (MI355X, gfx950).
//
// A serial recurrence over T steps for one block of 64 neurons is one chain of dependent steps.
// Run by a single wave, every instruction of a step (loads, address arithmetic, the surrogate's
// exp and division, stores) issues from that wave at 4 cycles per wave64 VALU instruction, so
// with few neurons the sweep is bound by one wave's issue rate while the rest of its CU idles.
// Here one workgroup per 64 neurons splits the work by role:
//   * PIPE_P producer waves load the inputs of a tile of PIPE_D rows one tile ahead, compute the
//     per-step coefficients (everything that does not depend on the recurrence) into an LDS
//     double buffer, and store the outputs of the tile the consumer finished one round earlier;
//   * one consumer wave (raised issue priority) runs only the recurrence, through LDS.
// One barrier per tile hands the buffers over.  The per-step arithmetic is the serial kernels'
// (same operations, same order, no contraction), so every output is bit-identical to theirs.
#include "lsh_abi.h"
#include "lsh_common.h"

namespace lsh {

// Every serial sweep of the library's serial entry points runs here, at every neuron count.
// Measured on MI355X (LIF adjoint, one wave -> pipe): N = 1024, T = 2^20: 172 -> 36.6 ms;
// N = 16384, T = 4096: 0.71 -> 0.26 ms; N = 65536, T = 4096: 1.13 -> 1.06 ms.

#ifndef LSH_PIPE_D
#define LSH_PIPE_D 64
#endif
// rows per tile of the adjoint, a multiple of 16 (LDS: 2 x D x 64 x 12 B).  96 rows measured
// 3 % faster at N = 1024, T = 2^20 (34.6 vs 35.7 ms) and no better at N = 16384.
constexpr int PIPE_D = LSH_PIPE_D;
constexpr int PIPE_P = 15;  // producer waves (16 waves per workgroup)
constexpr int PIPE_R = (PIPE_D + PIPE_P - 1) / PIPE_P;  // rows per producer per tile
// Rows per tile of the forward (LDS: 2 x D x 64 x 8 B = 128 KB).  Each tile costs a fixed
// ~0.35 us (barrier, load latency) besides ~14 ns per row at N = 1024: 32-row tiles were 28 %
// slower than 64-row ones, which longer tiles amortise further.
#ifndef LSH_PIPE_FD
#define LSH_PIPE_FD 128
#endif
constexpr int PIPE_FD = LSH_PIPE_FD;
constexpr int PIPE_FR = (PIPE_FD + PIPE_P - 1) / PIPE_P;

__device__ __forceinline__ int64_t pipe_tile_lo(int64_t T, int64_t k) {
  const int64_t hi = T - k * PIPE_D;
  return hi > PIPE_D ? hi - PIPE_D : 0;
}
__device__ __forceinline__ int pipe_tile_rows(int64_t T, int64_t k) {
  const int64_t hi = T - k * PIPE_D;
  return (int)(hi > PIPE_D ? PIPE_D : hi);
}

// Serial hard-reset LIF adjoint lam_t = b_t + a_t*lam_{t+1}, lam_T = 0 (triton_lif.py:54-72
// serial_bwd_kernel, :1088-1135 bwd_tiled_pf_kernel): tiles from the end of time, coefficients
// as k_lif_bwd's (v = fl(fl(beta*u_{t-1}) + x_t), sg = surrogate'(v - theta), J = 1 - s_t
// (+ (u_r - v)*sg when the reset is not detached), a = beta*J, b = gs*sg + J*gu).
template <bool DETACH, bool HAS_GU>
__global__ __launch_bounds__(WAVE*(PIPE_P + 1)) void k_lif_bwd_pipe(
    const float* __restrict__ I, const float* __restrict__ u0, const float* __restrict__ U,
    const float* __restrict__ S, const float* __restrict__ GS, const float* __restrict__ GU,
    float* __restrict__ Lam, int64_t N, int64_t T, float beta, float theta, float u_r,
    float alpha) {
  constexpr int D = PIPE_D, P = PIPE_P, R = PIPE_R;
  __shared__ float2 sAB[2][D][WAVE];
  __shared__ float sL[2][D][WAVE];
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const unsigned lane = threadIdx.x % WAVE;
  const int64_t nb0 = (int64_t)blockIdx.x * WAVE;
  const bool valid = nb0 + lane < N;
  const unsigned ln = valid ? lane : (unsigned)(N - 1 - nb0);
  const unsigned lb = ln * 4u, sb = lane * 4u;
  const int64_t ntiles = (T + D - 1) / D;

  if (w == 0) {  // consumer: tile k - 1 in round k
    __builtin_amdgcn_s_setprio(3);
    float lam = 0.0f;
    for (int64_t k = 0; k <= ntiles + 1; ++k) {
      if (k >= 1 && k <= ntiles) {
        const int buf = (int)((k - 1) & 1);
        const int nr = pipe_tile_rows(T, k - 1);
        if (nr == D) {
#pragma unroll
          for (int g = D - 16; g >= 0; g -= 16) {
            float2 ab[16];
#pragma unroll
            for (int i = 0; i < 16; ++i) ab[i] = sAB[buf][g + i][lane];
#pragma unroll
            for (int i = 15; i >= 0; --i) {
              lam = ab[i].y + ab[i].x * lam;
              sL[buf][g + i][lane] = lam;
            }
          }
        } else {
          for (int j = nr - 1; j >= 0; --j) {
            const float2 ab = sAB[buf][j][lane];
            lam = ab.y + ab.x * lam;
            sL[buf][j][lane] = lam;
          }
        }
      }
      __syncthreads();
    }
    return;
  }

  // producers: coefficients of tile k and the stores of tile k - 2 in round k
  const int p = w - 1;
  const float u0n = u0[nb0 + ln];
  float xr[R], sr[R], gr[R], hr[R], pr[R];
  auto load = [&](int64_t k) {
    const int64_t lo = pipe_tile_lo(T, k);
    const int nr = pipe_tile_rows(T, k);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int j = p + r * P;
      if (j < nr) {
        const int64_t t = lo + j;
        const size_t row = (size_t)t * (size_t)N + (size_t)nb0;
        xr[r] = ld_row(I + row, lb);
        sr[r] = ld_row(S + row, lb);
        gr[r] = ld_row(GS + row, lb);
        hr[r] = HAS_GU ? ld_row(GU + row, lb) : 0.0f;
        pr[r] = t > 0 ? ld_row(U + row - N, lb) : u0n;
      }
    }
  };
  if (ntiles > 0) load(0);
  for (int64_t k = 0; k <= ntiles + 1; ++k) {
    if (k < ntiles) {
      float x[R], s[R], g[R], h[R], up[R];
#pragma unroll
      for (int r = 0; r < R; ++r) {
        x[r] = xr[r];
        s[r] = sr[r];
        g[r] = gr[r];
        h[r] = hr[r];
        up[r] = pr[r];
      }
      if (k + 1 < ntiles) load(k + 1);
      const int buf = (int)(k & 1);
      const int nr = pipe_tile_rows(T, k);
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int j = p + r * P;
        if (j < nr) {
          const float v = lif_v(up[r], x[r], beta);
          const float sg = surrogate(v, theta, alpha);
          float J = 1.0f - s[r];
          if (!DETACH) J = J + (u_r - v) * sg;
          const float a = beta * J;
          const float bb = HAS_GU ? g[r] * sg + J * h[r] : g[r] * sg;
          sAB[buf][j][lane] = make_float2(a, bb);
        }
      }
    }
    if (k >= 2 && valid) {
      const int buf = (int)(k & 1);  // tile k - 2 has the parity of k
      const int64_t lo = pipe_tile_lo(T, k - 2);
      const int nr = pipe_tile_rows(T, k - 2);
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int j = p + r * P;
        if (j < nr) st_row(Lam + (size_t)(lo + j) * (size_t)N + (size_t)nb0, sb, sL[buf][j][lane]);
      }
    }
    __syncthreads();
  }
}

// The two serial forwards' steps: hard reset (triton_lif.py:21-25) and affine reset
// (triton_affine.py:20-24), with the values of the one-wave kernels' lif_step and aff_step.  A step
// takes the carried value p (start(u) from a state u) to the next one and gives its potential v;
// after(v) is the state u it leaves, spike(v) its decision.
struct LifStep {
  float beta, theta, u_r, kr;
  LifStep(float b, float t, float r) : beta(b), theta(t), u_r(r), kr(b * r) {}
  __device__ __forceinline__ float start(float u) const { return __fmul_rn(beta, u); }
  __device__ __forceinline__ float operator()(float& p, float x) const {
    return lif_walk(p, x, beta, theta, kr);
  }
  __device__ __forceinline__ float after(float v) const { return v >= theta ? u_r : v; }
  __device__ __forceinline__ bool spike(float v) const { return v >= theta; }
};
struct AffStep {
  float beta, theta, gamma, delta;
  __device__ __forceinline__ float start(float u) const { return u; }
  __device__ __forceinline__ float operator()(float& p, float x) const {
    const float v = lif_v(p, x, beta);
    p = after(v);
    return v;
  }
  __device__ __forceinline__ float after(float v) const {
    return v >= theta ? __fadd_rn(__fmul_rn(gamma, v), delta) : v;
  }
  __device__ __forceinline__ bool spike(float v) const { return v >= theta; }
};

// Serial forward over T rows of 64 neurons from the states us (triton_lif.py:30-39
// serial_fwd_kernel, :460-466 serial_forward_tiled; triton_affine.py:143-162), run by every wave of
// a workgroup of PIPE_P + 1: tiles in time order; the consumer runs the recurrence and writes v per
// step (and each tile's entry state), the producers stage I into LDS one tile ahead and store U, S
// of the tile finished one round earlier, both from its v, so the consumer's chain carries neither
// the selection of u nor a spike-to-float select.
// SO: no U; `U` is [ceil(T/32), N] and receives the state before rows 0, 32, 64, ... (NULL: not
// wanted), so the spikes alone are written per step.
struct FwdTiles {
  float X[2][PIPE_FD][WAVE];
  float V[2][PIPE_FD][WAVE];
  float entry[2][WAVE];  // u before row 0 of the tile in the same buffer
};
template <class Step, bool NT, bool SO>
__device__ __forceinline__ void serial_fwd_tiles(FwdTiles& sh, const float* __restrict__ I,
                                                 const float* us, float* __restrict__ U,
                                                 float* __restrict__ S, int64_t nb0, int64_t N,
                                                 int64_t T, Step step) {
  constexpr int D = PIPE_FD, P = PIPE_P, R = PIPE_FR;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const unsigned lane = threadIdx.x % WAVE;
  const bool valid = nb0 + lane < N;
  const unsigned ln = valid ? lane : (unsigned)(N - 1 - nb0);
  const unsigned lb = ln * 4u, sb = lane * 4u;
  const int64_t ntiles = (T + D - 1) / D;
  auto rows = [&](int64_t k) { return (int)(T - k * D > D ? D : T - k * D); };

  if (w == 0) {  // consumer: tile k - 1 in round k
    __builtin_amdgcn_s_setprio(3);
    const float u = us[nb0 + ln];
    float p = step.start(u), v = 0.0f;
    for (int64_t k = 0; k <= ntiles + 1; ++k) {
      if (k >= 1 && k <= ntiles) {
        const int buf = (int)((k - 1) & 1);
        const int nr = rows(k - 1);
        if constexpr (SO) sh.entry[buf][lane] = k == 1 ? u : step.after(v);
        if (nr == D) {
#pragma unroll
          for (int g = 0; g < D; g += 16) {
            float x[16];
#pragma unroll
            for (int i = 0; i < 16; ++i) x[i] = sh.X[buf][g + i][lane];
#pragma unroll
            for (int i = 0; i < 16; ++i) {
              v = step(p, x[i]);
              sh.V[buf][g + i][lane] = v;
            }
          }
        } else {
          for (int j = 0; j < nr; ++j) {
            v = step(p, sh.X[buf][j][lane]);
            sh.V[buf][j][lane] = v;
          }
        }
      }
      __syncthreads();
    }
    return;
  }

  // producers: I of tile k into LDS (loaded one round ahead) and U, S of tile k - 2 in round k
  const int p = w - 1;
  float xr[R];
  auto load = [&](int64_t k) {
    const int nr = rows(k);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int j = p + r * P;
      if (j < nr) xr[r] = ld_row(I + (size_t)(k * D + j) * (size_t)N + (size_t)nb0, lb);
    }
  };
  if (ntiles > 0) load(0);
  for (int64_t k = 0; k <= ntiles + 1; ++k) {
    if (k < ntiles) {
      const int buf = (int)(k & 1);
      const int nr = rows(k);
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int j = p + r * P;
        if (j < nr) sh.X[buf][j][lane] = xr[r];
      }
      if (k + 1 < ntiles) load(k + 1);
    }
    if (k >= 2 && valid) {
      const int buf = (int)(k & 1);
      const int nr = rows(k - 2);
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int j = p + r * P;
        if (j < nr) {
          const size_t row = (size_t)((k - 2) * D + j) * (size_t)N + (size_t)nb0;
          const float v = sh.V[buf][j][lane];
          if constexpr (SO) {
            static_assert(D % 32 == 0, "the states fall on rows 0, 32, ... of a tile");
            if (j % 32 == 0 && U != nullptr)
              st_row<NT>(U + (size_t)((k - 2) * (D / 32) + j / 32) * (size_t)N + (size_t)nb0, sb,
                         j == 0 ? sh.entry[buf][lane] : step.after(sh.V[buf][j - 1][lane]));
          } else {
            st_row<NT>(U + row, sb, step.after(v));
          }
          st_row<NT>(S + row, sb, step.spike(v) ? 1.0f : 0.0f);
        }
      }
    }
    __syncthreads();
  }
}

template <class Step, bool NT, bool SO = false>
__global__ __launch_bounds__(WAVE*(PIPE_P + 1)) void k_serial_fwd_pipe(
    const float* __restrict__ I, const float* __restrict__ u0, float* __restrict__ U,
    float* __restrict__ S, int64_t N, int64_t T, Step step) {
  __shared__ FwdTiles sh;
  serial_fwd_tiles<Step, NT, SO>(sh, I, u0, U, S, (int64_t)blockIdx.x * WAVE, N, T, step);
}

// What the warm-started chunks (lif_warm.hip) leave to repair, in linear work: chunks m >= 1 whose
// start is not the exit of the chunk before are replayed in Jacobi rounds, as k_lif_repair does, while
// the rounds' replays stay within a budget; then, if a start is still wrong, the rows from the
// block's first such chunk on are run once more by the serial sweep.  Every chunk below it has the
// bits of the exit before it as its start, so that exit is exact.  The rounds suit the few misses that
// noisy inputs leave (each meets its stored trajectory soon); with a nearly constant current no
// trajectory ever meets another one of a different phase, every round makes one more chunk exact,
// and rounds alone took M of them, some M^2/2 chunk replays.
// One workgroup per 64 neurons.  A round of nd replays takes 1 + nd/128 units of the budget: a few
// lanes walk a row in some 45 ns (the sweep in 17), all 1024 in 250, for their rows lie apart.
// Measured, N 64, T 50000, beta 0.93 (C 256; the serial sweep alone 0.86 ms), rounds alone -> this:
// constant current 104.8 -> 0.94 ms, current steps 12.5 -> 0.93 ms, noise 60 -> 39 us (the first
// comparison by 16 waves instead of 4); N 1000, T 60001, beta 0.95 (C 1888; sweep 1.20 ms) constant
// current 5.25 -> 2.24 ms; N 4096, T 16001 (C 2000; 0.30 ms) 1.41 -> 0.75 ms.
constexpr int kWarmScanAhead = 8;  // chunks a wave compares at once
__global__ __launch_bounds__(WAVE*(PIPE_P + 1)) void k_lif_warm_finish(
    const float* __restrict__ I, float* __restrict__ U, float* __restrict__ S, float* starts,
    float* ends, int* list0, int* list1, WsHeader* hdr, int64_t T, int64_t N, int M, int C,
    int budget, LifStep step) {
  constexpr int NW = PIPE_P + 1, NT = WAVE * NW;
  __shared__ FwdTiles sh;
  __shared__ int s_nd, s_nc, s_first;
  const int tid = threadIdx.x, lane = tid % WAVE;
  const int64_t nb0 = (int64_t)blockIdx.x * WAVE;
  const size_t cap = (size_t)M * WAVE;
  int* dl = list0 + (size_t)blockIdx.x * cap;  // chunks (as m*64 + lane) whose start is wrong
  int* cl = list1 + (size_t)blockIdx.x * cap;  // successors of chunks whose end changed
  if (tid == 0) {
    s_nd = 0;
    s_first = M;
  }
  __syncthreads();
  {
    const bool valid = nb0 + lane < N;
    const int64_t n = valid ? nb0 + lane : N - 1;
    for (int m0 = 1 + tid / WAVE; m0 < M; m0 += NW * kWarmScanAhead) {
      float st[kWarmScanAhead], en[kWarmScanAhead];
#pragma unroll
      for (int k = 0; k < kWarmScanAhead; ++k) {
        const size_t o = (size_t)min(m0 + k * NW, M - 1) * N + n;
        st[k] = starts[o];
        en[k] = ends[o - N];
      }
#pragma unroll
      for (int k = 0; k < kWarmScanAhead; ++k) {
        const int m = m0 + k * NW;
        if (valid && m < M && !same_bits(st[k], en[k])) dl[atomicAdd(&s_nd, 1)] = m * WAVE + lane;
      }
    }
  }
  __syncthreads();
  int rounds = 0, nd = s_nd;
  while (nd > 0) {
    const int units = 1 + nd / 128;
    if (units > budget) break;
    budget -= units;
    ++rounds;
    for (int i = tid; i < nd; i += NT) {
      const size_t o = (size_t)(dl[i] / WAVE) * N + (size_t)(nb0 + dl[i] % WAVE);
      starts[o] = ends[o - N];
    }
    if (tid == 0) s_nc = 0;
    __syncthreads();
    for (int i = tid; i < nd; i += NT) {
      const int e = dl[i], m = e / WAVE;
      const size_t o = (size_t)m * N + (size_t)(nb0 + e % WAVE);
      const size_t base = (size_t)m * C * N + (size_t)(nb0 + e % WAVE);
      float u = starts[o];
      const bool met = stream_rows_until<16>(
          I + base, U + base, (size_t)N, min<int64_t>(C, T - (int64_t)m * C),
          [&](int64_t j, float x, float u_old) {
            bool s;
            u = lif_step(u, x, step.beta, step.theta, step.u_r, s);
            U[base + (size_t)j * N] = u;
            S[base + (size_t)j * N] = s ? 1.0f : 0.0f;
            return same_bits(u, u_old);
          });
      if (!met && !same_bits(u, ends[o])) {
        ends[o] = u;
        if (m + 1 < M) cl[atomicAdd(&s_nc, 1)] = e + WAVE;
      }
    }
    if (tid == 0) s_nd = 0;
    __syncthreads();
    for (int i = tid; i < s_nc; i += NT) {
      const int e = cl[i];
      const size_t o = (size_t)(e / WAVE) * N + (size_t)(nb0 + e % WAVE);
      if (!same_bits(ends[o - N], starts[o])) dl[atomicAdd(&s_nd, 1)] = e;
    }
    __syncthreads();
    nd = s_nd;
  }
  if (tid == 0) atomicMax(&hdr->repair_iters, (unsigned int)(rounds + (nd > 0 ? 1 : 0)));
  if (nd == 0) return;
  for (int i = tid; i < nd; i += NT) atomicMin(&s_first, dl[i] / WAVE);
  __builtin_amdgcn_s_waitcnt(0);  // the rounds' stores land before the sweep's to the same rows
  __syncthreads();
  const int c0 = s_first;
  const size_t row0 = (size_t)c0 * C;
  serial_fwd_tiles<LifStep, true, false>(sh, I + row0 * N, ends + (size_t)(c0 - 1) * N, U + row0 * N,
                                       S + row0 * N, nb0, N, T - (int64_t)row0, step);
}

// The budget of the rounds: M/5 units, half the serial sweep's time.  Noisy inputs need up to 6 rounds
// with 32 chunks and 16 with 128 (beta 0.98 to 0.995); with M/16 units some were swept although two or
// three rounds more would have done (N 1024, T 32768, beta 0.995 529 -> 754 us).
void lif_warm_finish_launch(const float* I, float* U, float* S, float* starts, float* ends, int* list0,
                            int* list1, WsHeader* hdr, int64_t T, int64_t N, int M, int C, float beta,
                            float theta, float u_r, hipStream_t st) {
  const int NB = (int)((N + WAVE - 1) / WAVE);
  hipLaunchKernelGGL(k_lif_warm_finish, dim3((unsigned)NB), dim3(WAVE * (PIPE_P + 1)), 0, st, I, U, S,
                     starts, ends, list0, list1, hdr, T, N, M, C, M / 5, LifStep(beta, theta, u_r));
}

void lif_serial_fwd_pipe(const float* I, const float* u0, float* U, float* S, int64_t N, int64_t T,
                         float beta, float theta, float u_r, hipStream_t st) {
  const int NB = (int)((N + WAVE - 1) / WAVE);
  with_store_policy(nt_sweep(N), [&](auto nt) {
    hipLaunchKernelGGL((k_serial_fwd_pipe<LifStep, decltype(nt)::value>), dim3((unsigned)NB),
                       dim3(WAVE * (PIPE_P + 1)), 0, st, I, u0, U, S, N, T, LifStep(beta, theta, u_r));
  });
}

void lif_starts_fwd_pipe(const float* I, const float* u0, float* STARTS, float* S, int64_t N, int64_t T,
                         float beta, float theta, float u_r, hipStream_t st) {
  const int NB = (int)((N + WAVE - 1) / WAVE);
  hipLaunchKernelGGL((k_serial_fwd_pipe<LifStep, true, true>), dim3((unsigned)NB),
                     dim3(WAVE * (PIPE_P + 1)), 0, st, I, u0, STARTS, S, N, T, LifStep(beta, theta, u_r));
}

void aff_serial_fwd_pipe(const float* I, const float* u0, float* U, float* S, int64_t N, int64_t T,
                         float beta, float theta, float gamma, float delta, hipStream_t st) {
  const int NB = (int)((N + WAVE - 1) / WAVE);
  with_store_policy(nt_sweep(N), [&](auto nt) {
    hipLaunchKernelGGL((k_serial_fwd_pipe<AffStep, decltype(nt)::value>), dim3((unsigned)NB),
                       dim3(WAVE * (PIPE_P + 1)), 0, st, I, u0, U, S, N, T,
                       AffStep{beta, theta, gamma, delta});
  });
}

template <bool DETACH, bool HAS_GU>
static void launch_lif_bwd_pipe(const float* I, const float* u0, const float* U, const float* S,
                                const float* GS, const float* GU, float* Lam, int64_t N, int64_t T,
                                float beta, float theta, float u_r, float alpha, hipStream_t st) {
  const int NB = (int)((N + WAVE - 1) / WAVE);
  hipLaunchKernelGGL((k_lif_bwd_pipe<DETACH, HAS_GU>), dim3((unsigned)NB), dim3(WAVE * (PIPE_P + 1)),
                     0, st, I, u0, U, S, GS, GU, Lam, N, T, beta, theta, u_r, alpha);
}

void lif_serial_bwd_pipe(const float* I, const float* u0, const float* U, const float* S,
                         const float* GS, const float* GU, float* Lam, int64_t N, int64_t T,
                         float beta, float theta, float u_r, float alpha, bool detach,
                         hipStream_t st) {
  const bool gu = GU != nullptr;
  if (detach && gu)
    launch_lif_bwd_pipe<true, true>(I, u0, U, S, GS, GU, Lam, N, T, beta, theta, u_r, alpha, st);
  else if (detach)
    launch_lif_bwd_pipe<true, false>(I, u0, U, S, GS, GU, Lam, N, T, beta, theta, u_r, alpha, st);
  else if (gu)
    launch_lif_bwd_pipe<false, true>(I, u0, U, S, GS, GU, Lam, N, T, beta, theta, u_r, alpha, st);
  else
    launch_lif_bwd_pipe<false, false>(I, u0, U, S, GS, GU, Lam, N, T, beta, theta, u_r, alpha, st);
}

}  // namespace lsh
