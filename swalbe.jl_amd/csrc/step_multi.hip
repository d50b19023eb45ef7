// step_multi.hip -- several D2Q9 steps of one film per launch, for films too
// small to fill the chip one step at a time, and for FP32 films whose carried
// populations (τ ≠ 1) outgrow the caches.
//
// A workgroup owns a TX x TY tile and stages it with a halo of 3 K nodes in
// LDS; a step costs three nodes of halo at each side (one per stencil), so
// after K steps the tile is exact.  Per step: pressure, forces and collision
// at the source, stream and moments, a barrier after each; each phase spreads
// the rectangle it still needs over the threads.  The intermediate steps'
// populations and pressures never leave the chip; the launch that runs the
// loop's last step writes them.
//
// What bounds it: a 256 x 256 FP64 film has one 64 x 8 tile of k_step for half
// of the CUs, and a step of it 7.8 us, of which 2-3 are the launch and its
// loads and the rest the latency of one wave per SIMD going through four
// phases.  16 x 16 tiles use every CU and three steps share the launch; the
// FP64 issue of the tile and its halo (1.5 to 2.6 times the film's nodes) is
// then what is left: 3.1 us a step (9.4 per launch).  Keeping a thread's nodes
// fixed, with u and f_t in registers and no trimming of the rectangle's
// columns, took 3.7; 512 threads instead of 1024 for these tiles 3.4; two
// steps per launch 3.5.
//
// FP64 evaluates every expression in the reference's order (the bits of
// k_step and of the oracle).
#include "step_node.h"
#include "swalbe_internal.h"

namespace swalbe {

namespace {

struct MultiRun {
  int Lx, Ly, ntx, k;  // k <= K steps in this launch
  int64_t fstride;
  uint64_t step;       // number of the first step
  StepSeries ser;      // slots of the first step
  int write_f;         // the launch's last step writes f and p
};

// a, at most `reach` outside [0, L), wrapped into it
__device__ __forceinline__ int wrap(int a, int L, int reach) {
  if (reach > L) {  // a film smaller than its halo wraps more than once
    a %= L;
    return a < 0 ? a + L : a;
  }
  a = a < 0 ? a + L : a;
  return a >= L ? a - L : a;
}

// LDS planes of a tile and its halo: h, u, v, p, κ and the nine post-collision
// populations (with τ ≠ 1 a node's own nine streamed ones between steps).
enum { kH, kU, kV, kP, kK, kF, kPlanes = kF + kQ };

// This thread's nodes of the rectangle M nodes inside the RW x RH region, as
// offsets into a plane (-1: none): consecutive threads take consecutive nodes
// of a row.
template <int RW, int RH, int M, int NT>
struct Inner {
  static constexpr int W = RW - 2 * M, H = RH - 2 * M, N = W * H, NQ = (N + NT - 1) / NT;
  static __device__ __forceinline__ int off(int q) {
    const int e = threadIdx.x + q * NT;
    const int r = e / W, c = e - r * W;
    return e < N ? (r + M) * RW + c + M : -1;
  }
};

template <typename T, int TX, int TY, int K, int NT, bool RFT, bool TH, bool GRAV>
struct Multi {
  static constexpr bool F32 = sizeof(T) == 4;
  static constexpr int RW = TX + 6 * K, RH = TY + 6 * K, RN = RW * RH;

  const StepIO<T>& io;
  const StepParams& sp;
  const F32K& K32;
  const MultiRun& R;
  T* const lds;
  int x0, y0;

  __device__ __forceinline__ T* plane(int i) const { return lds + i * RN; }

  __device__ __forceinline__ void load(int margin) const {
    using I = Inner<RW, RH, 0, NT>;
    T h[I::NQ], u[I::NQ], v[I::NQ], kp[I::NQ], ft[I::NQ][kQ];
    int64_t g[I::NQ];
    int o[I::NQ];
#pragma unroll
    for (int q = 0; q < I::NQ; ++q) {
      o[q] = I::off(q);
      const int r = o[q] / RW, c = o[q] - r * RW;
      if (r < margin || r >= RH - margin || c < margin || c >= RW - margin) o[q] = -1;
      int gx = x0 - 3 * K + c, gy = y0 - 3 * K + r;
      gx = wrap(gx, R.Lx, RW);
      gy = wrap(gy, R.Ly, RH);
      g[q] = gx + (int64_t)R.Lx * gy;
    }
#pragma unroll
    for (int q = 0; q < I::NQ; ++q)
      if (o[q] >= 0) {
        h[q] = io.h_in[g[q]];
        u[q] = io.ux_in[g[q]];
        v[q] = io.uy_in[g[q]];
        if (io.kappa) kp[q] = io.kappa[g[q]];
        if constexpr (RFT) {
#pragma unroll
          for (int k = 0; k < kQ; ++k) ft[q][k] = io.ft[k * R.fstride + g[q]];
        }
      }
#pragma unroll
    for (int q = 0; q < I::NQ; ++q)
      if (o[q] >= 0) {
        plane(kH)[o[q]] = h[q];
        plane(kU)[o[q]] = u[q];
        plane(kV)[o[q]] = v[q];
        if (io.kappa) plane(kK)[o[q]] = kp[q];
        if constexpr (RFT) {
#pragma unroll
          for (int k = 0; k < kQ; ++k) plane(kF + k)[o[q]] = ft[q][k];
        }
      }
  }

  // max, min and count(> thresh) of the step's input height over the tile's nodes (NaN passed
  // over, as k_step's comparisons do; nothing but NaN: -inf and inf), gathered by
  // LDS atomics that nobody waits for before the next barrier (a shuffle tree per wave and one
  // thread walking the waves' results took 1.2 us a step, half a step of a 100 x 100 film);
  // eight addresses share the lanes of a wave
  __device__ __forceinline__ void series(unsigned long long* red) const {
    using I = Inner<RW, RH, 3 * K, NT>;
    unsigned long long kmax = kNoMax, kmin = kNoMin;
    unsigned int cnt = 0;
#pragma unroll
    for (int q = 0; q < I::NQ; ++q) {
      const int o = I::off(q);
      const int r = o / RW, c = o - r * RW;
      const bool own = o >= 0 && x0 + c - 3 * K < R.Lx && y0 + r - 3 * K < R.Ly;
      double hv = 0.0;
      if (own) {
        hv = (double)plane(kH)[o];
        if constexpr (F32) hv = (double)K32.href + hv;
        if (hv == hv) {
          const unsigned long long key = dkey(hv);
          kmax = key > kmax ? key : kmax;
          kmin = key < kmin ? key : kmin;
        }
      }
      cnt += (unsigned int)__popcll(__ballot(own && hv > sp.wet_thresh));
    }
    if (R.ser.dh && kmax >= kmin) {
      atomicMax(&red[2 * (threadIdx.x & 7)], kmax);
      atomicMin(&red[2 * (threadIdx.x & 7) + 1], kmin);
    }
    if ((threadIdx.x & 63) == 0 && cnt) atomicAdd(&red[16], (unsigned long long)cnt);
  }

  // after the barrier: the tile's result to the step's slot, the LDS words neutral again (the
  // next step's series comes after two more barriers)
  __device__ __forceinline__ void series_out(unsigned long long* red, int64_t i) const {
    if (threadIdx.x != 0) return;
    unsigned long long kmax = kNoMax, kmin = kNoMin;
    if (R.ser.dh)
      for (int w = 0; w < 8; ++w) {
        kmax = red[2 * w] > kmax ? red[2 * w] : kmax;
        kmin = red[2 * w + 1] < kmin ? red[2 * w + 1] : kmin;
      }
    R.ser.add(i, kmax, kmin, red[16]);
    series_clear(red);
  }
  static __device__ __forceinline__ void series_clear(unsigned long long* red) {
    for (int w = 0; w < 8; ++w) {
      red[2 * w] = kNoMax;
      red[2 * w + 1] = kNoMin;
    }
    red[16] = 0ull;
  }

  // film pressure (src/pressure.jl:119-155)
  template <int M>
  __device__ __forceinline__ void pressure(bool out) const {
    using I = Inner<RW, RH, M, NT>;
#pragma unroll
    for (int q = 0; q < I::NQ; ++q) {
      const int o = I::off(q);
      if (o < 0) continue;
      const T* hc = plane(kH) + o;
      const T hip = hc[-1], him = hc[1], hjp = hc[-RW], hjm = hc[RW], h = hc[0];
      const T hipjp = hc[-RW - 1], himjp = hc[-RW + 1], himjm = hc[RW + 1], hipjm = hc[RW - 1];
      T p;
      if constexpr (F32) {
#pragma clang fp contract(fast)
        const float L = (2.0f / 3.0f) * (((hjp + hip) + him) + hjm) +
                        (1.0f / 6.0f) * (((hipjp + himjp) + himjm) + hipjm) - (10.0f / 3.0f) * h;
        const float kap = io.kappa ? plane(kK)[o] : K32.kap;
        p = disjoining_f(K32, h, kap, io.kappa != nullptr) - K32.gamma * L;
      } else {
        const T L = (T(2.0 / 3.0) * (((hjp + hip) + him) + hjm) +
                     T(1.0 / 6.0) * (((hipjp + himjp) + himjm) + hipjm)) -
                    T(10.0 / 3.0) * h;
        const T kap = io.kappa ? plane(kK)[o] : (T)sp.kappa;
        const T a = Recip<false>(h + sp.hcrit).div(sp.hmin);
        const T p0 = -sp.gamma * (kap * powlaw(a, sp.n, sp.m, sp.powmode));
        p = p0 - sp.gamma * L;
      }
      plane(kP)[o] = p;
      if (out) {  // the launch writes p: this tile's nodes
        const int r = o / RW, c = o - r * RW;
        const int tx = c - 3 * K, ty = r - 3 * K;
        if (tx >= 0 && tx < TX && ty >= 0 && ty < TY && x0 + tx < R.Lx && y0 + ty < R.Ly)
          io.p_out[x0 + tx + (int64_t)R.Lx * (y0 + ty)] = p;
      }
    }
  }

  // forces (src/forcing.jl:42-46, 168-187, 297-311, 363-368) and the collision at the source
  // (src/equilibrium.jl:74-114, src/collide.jl:70-105)
  template <int M>
  __device__ __forceinline__ void collide(uint64_t step) const {
    using I = Inner<RW, RH, M, NT>;
#pragma unroll
    for (int q = 0; q < I::NQ; ++q) {
      const int o = I::off(q);
      if (o < 0) continue;
      const T* pc = plane(kP) + o;
      const T fip = pc[-1], fim = pc[1], fjp = pc[-RW], fjm = pc[RW];
      const T fipjp = pc[-RW - 1], fimjp = pc[-RW + 1], fimjm = pc[RW + 1], fipjm = pc[RW - 1];
      const T h = plane(kH)[o], u = plane(kU)[o], v = plane(kV)[o];
      T* const F = plane(kF) + o;
      uint32_t ni = 0;
      if constexpr (TH) {
        const int r = o / RW, c = o - r * RW;
        ni = noise_index(wrap(x0 - 3 * K + c, R.Lx, RW), wrap(y0 - 3 * K + r, R.Ly, RH), R.Lx);
      }
      if constexpr (F32) {
#pragma clang fp contract(fast)
        const float hh = K32.href + h;
        const float gx = (-1.0f / 3.0f) * (fip - fim) -
                         (1.0f / 12.0f) * (((fipjp - fimjp) - fimjm) + fipjm);
        const float gy = (-1.0f / 3.0f) * (fjp - fjm) -
                         (1.0f / 12.0f) * (((fipjp + fimjp) - fimjm) - fipjm);
        const float iden = __builtin_amdgcn_rcpf((2.0f * hh + K32.c6d) * hh + K32.c3dd);
        const float sl = K32.c6mu * hh * iden;
        float Fx = -hh * gx - sl * u;
        float Fy = -hh * gy - sl * v;
        if constexpr (TH) {
          uint32_t w[4];
          philox_ctr(sp.seed, step, ni >> 1, kTagThermal, w);
          float z0, z1;
          box_muller_f32((ni & 1) ? w[2] : w[0], (ni & 1) ? w[3] : w[1], &z0, &z1);
          const float amp = __builtin_amdgcn_sqrtf(K32.kb26 * hh * iden);
          Fx -= z0 * amp;
          Fy -= z1 * amp;
        }
        if (sp.body) {
          Fx += hh * K32.bfx;
          Fy += hh * K32.bfy;
        }
        const float w1 = 1.0f / 9.0f, w5 = 1.0f / 36.0f, c3 = 1.0f / 3.0f, c24 = 1.0f / 24.0f;
        const float usq = u * u + v * v;
        const float w1h = w1 * hh, w5h = w5 * hh;
        float b1 = -1.5f * w1h * usq, b5 = -1.5f * w5h * usq;
        float fe[kQ];
        fe[0] = h - (2.0f / 3.0f) * hh * usq;
        if constexpr (GRAV) {
          const float gg = h * (hh + K32.href);
          b1 += w1 * K32.g0 * gg;
          b5 += w5 * K32.g0 * gg;
          fe[0] -= K32.c56g * gg;
        }
        const float a5 = u + v, a6 = v - u;
        fe[1] = b1 + w1h * ((4.5f * u + 3.0f) * u);
        fe[2] = b1 + w1h * ((4.5f * v + 3.0f) * v);
        fe[3] = b1 + w1h * ((4.5f * u - 3.0f) * u);
        fe[4] = b1 + w1h * ((4.5f * v - 3.0f) * v);
        fe[5] = b5 + w5h * ((4.5f * a5 + 3.0f) * a5);
        fe[6] = b5 + w5h * ((4.5f * a6 + 3.0f) * a6);
        fe[7] = b5 + w5h * ((4.5f * a5 - 3.0f) * a5);
        fe[8] = b5 + w5h * ((4.5f * a6 - 3.0f) * a6);
        if constexpr (RFT) {
#pragma unroll
          for (int k = 0; k < kQ; ++k) fe[k] = K32.itau * fe[k] + K32.omeg * F[k * RN];
        }
        F[0 * RN] = fe[0];
        F[1 * RN] = fe[1] + c3 * Fx;
        F[2 * RN] = fe[2] + c3 * Fy;
        F[3 * RN] = fe[3] - c3 * Fx;
        F[4 * RN] = fe[4] - c3 * Fy;
        F[5 * RN] = fe[5] + c24 * (Fx + Fy);
        F[6 * RN] = fe[6] + c24 * (Fy - Fx);
        F[7 * RN] = fe[7] - c24 * (Fx + Fy);
        F[8 * RN] = fe[8] + c24 * (Fx - Fy);
      } else {
        const T gx = T(-1.0 / 3.0) * (fip - fim) -
                     T(1.0 / 12.0) * (((fipjp - fimjp) - fimjm) + fipjm);
        const T gy = T(-1.0 / 3.0) * (fjp - fjm) -
                     T(1.0 / 12.0) * (((fipjp + fimjp) - fimjm) - fipjm);
        const T hgx = h * gx, hgy = h * gy;
        const Recip<> iden((T(2) * (h * h) + sp.c6d * h) + sp.c3dd);
        const T sx = iden.div(sp.c6mu * h * u);
        const T sy = iden.div(sp.c6mu * h * v);
        T Fx = -hgx - sx;
        T Fy = -hgy - sy;
        if constexpr (TH) {
          double z0, z1;
          normal_pair(sp.seed, step, ni, kTagThermal, &z0, &z1);
          const T amp = sqrt(Recip<>(((T(2) * h) * h + (T(6) * h) * sp.delta) + sp.d3dd)
                                 .div(sp.kb26 * h));
          Fx = Fx - z0 * amp;
          Fy = Fy - z1 * amp;
        }
        if (sp.body) {
          Fx = Fx + (h * sp.bax) * sp.bfac;
          Fy = Fy + (h * sp.bay) * sp.bfac;
        }
        const T usq = u * u + v * v;
        const T c56g = (T)((5.0 / 6.0) * sp.g), g0 = (T)(1.5 * sp.g);
#pragma unroll
        for (int k = 0; k < kQ; ++k) {
          T f;
          // (k = 0: NaN for an infinite height, as the force makes the others)
          if (GRAV || k == 0) f = feq_k<T>(k, h, u, v, usq, c56g, g0);
          else f = feq_k0<T>(k, h, u, v, usq);
          if constexpr (RFT) f = sp.omeg * F[k * RN] + sp.itau * f;
          F[k * RN] = k > 0 ? f + force_term<T>(k, Fx, Fy) : f;
        }
      }
    }
  }

  // pull-stream and moments (src/collide.jl:92-100, src/moments.jl:43-52); OUT: the tile's nodes
  // to global memory (the launch's last step), else back to LDS
  template <int M, bool OUT>
  __device__ __forceinline__ void stream() const {
    using I = Inner<RW, RH, M, NT>;
    T h[I::NQ], u[I::NQ], v[I::NQ], f[I::NQ][kQ];
#pragma unroll
    for (int q = 0; q < I::NQ; ++q) {
      const int o = I::off(q);
      if (o < 0) continue;
      const T* F = plane(kF) + o;
#pragma unroll
      for (int k = 0; k < kQ; ++k) f[q][k] = F[k * RN - (cx(k) + RW * cy(k))];
      T sum = f[q][0];
#pragma unroll
      for (int k = 1; k < kQ; ++k) sum = sum + f[q][k];
      const T mx = ((((f[q][1] - f[q][3]) + f[q][5]) - f[q][6]) - f[q][7]) + f[q][8];
      const T my = ((((f[q][2] - f[q][4]) + f[q][5]) + f[q][6]) - f[q][7]) - f[q][8];
      h[q] = sum;
      if constexpr (F32) {
        const float ih = __builtin_amdgcn_rcpf(K32.href + sum);
        u[q] = mx * ih;
        v[q] = my * ih;
      } else {
        const Recip<> ih(sum);
        u[q] = ih.div(mx);
        v[q] = ih.div(my);
      }
      if constexpr (OUT) {
        const int r = o / RW, c = o - r * RW;
        const int gx = x0 + c - 3 * K, gy = y0 + r - 3 * K;
        if (gx < R.Lx && gy < R.Ly) {
          const int64_t g = gx + (int64_t)R.Lx * gy;
          io.h_out[g] = h[q];
          io.ux_out[g] = u[q];
          io.uy_out[g] = v[q];
          if (RFT || R.write_f) {
#pragma unroll
            for (int k = 0; k < kQ; ++k) io.f_out[k * R.fstride + g] = f[q][k];
          }
        }
      } else {
        plane(kH)[o] = h[q];
        plane(kU)[o] = u[q];
        plane(kV)[o] = v[q];
      }
    }
    if constexpr (RFT && !OUT) {  // a node's streamed populations are its next f_t
      __syncthreads();            // every wave has read its neighbours'
#pragma unroll
      for (int q = 0; q < I::NQ; ++q) {
        const int o = I::off(q);
        if (o < 0) continue;
#pragma unroll
        for (int k = 0; k < kQ; ++k) plane(kF + k)[o] = f[q][k];
      }
    }
  }

  // step S of K (those before K - R.k are not taken), then the ones after it
  template <int S>
  __device__ __forceinline__ void steps(unsigned long long* red) const {
    if constexpr (S < K) {
      const int64_t i = S - (K - R.k);
      if (i >= 0) {
        constexpr bool LAST = S == K - 1;
        const bool ser = R.ser.base != nullptr;
        if (ser) series(red);
        pressure<3 * S + 1>(LAST && R.write_f);
        __syncthreads();
        if (ser) series_out(red, i);
        collide<3 * S + 2>(R.step + (uint64_t)i);
        __syncthreads();
        stream<3 * S + 3, LAST>();
        if constexpr (!LAST) __syncthreads();
      }
      steps<S + 1>(red);
    }
  }
};

template <typename T, int TX, int TY, int K, int NT, bool RFT, bool TH, bool GRAV>
__global__ __launch_bounds__(NT) void k_multi(StepIO<T> io, StepParams sp, F32K K32, MultiRun R) {
  using M = Multi<T, TX, TY, K, NT, RFT, TH, GRAV>;
  __shared__ T lds[kPlanes * M::RN];
  __shared__ unsigned long long red[17];
  const int tile = blockIdx.x;
  const M m{io, sp, K32, R, lds, (tile % R.ntx) * TX, (tile / R.ntx) * TY};
  if (threadIdx.x == 0) M::series_clear(red);
  m.load(3 * (K - R.k));
  __syncthreads();
  m.template steps<0>(red);
}

// The tiles compiled and what a launch of each costs on films from 64 x 64 to
// 1024 x 1024 (no noise, τ = 1): fixed + body us per round of at most `wgs`
// workgroups per CU.  Noise and τ ≠ 1 scale all of them, and the one-step
// kernels, by about the same factor.
struct Geom {
  int tx, ty, k;
  double fixed, body;
  int wgs;
};
constexpr int kNGeoms = 5;  // those from kTwoStepGeom on have k = 2
constexpr Geom kGeoms64[kNGeoms] = {{8, 8, 3, 3.6, 3.2, 1},
                                    {16, 16, 3, 2.0, 7.5, 1},
                                    {24, 16, 2, 2.6, 5.9, 1},
                                    {32, 16, 2, 1e9, 0.0, 1},  // 512 threads: FP32 only
                                    {32, 16, 2, 3.2, 6.2, 1}};
constexpr Geom kGeoms32[kNGeoms] = {{8, 8, 3, 4.3, 1.5, 1},
                                    {16, 16, 3, 1.6, 5.6, 1},
                                    {24, 16, 2, 2.6, 5.2, 2},
                                    {32, 16, 2, 4.0, 6.1, 2},
                                    {32, 16, 2, 1.5, 5.1, 1}};

template <typename T, int TX, int TY, int K, int NT>
void launch_geom(const StepIO<T>& io, const StepParams& sp, const F32K& K32, MultiRun R,
                 hipStream_t s) {
  R.ntx = (R.Lx + TX - 1) / TX;
  const dim3 grid(R.ntx * ((R.Ly + TY - 1) / TY)), block(NT);
#define SW_K(RF, TH, GR)                                                                       \
  hipLaunchKernelGGL((k_multi<T, TX, TY, K, NT, RF, TH, GR>), grid, block, 0, s, io, sp, K32, R)
  if (sp.read_ft) {
    if (sp.thermal) SW_K(true, true, true);
    else SW_K(true, false, true);
  } else if (sp.thermal) {
    if (sp.g != 0.0) SW_K(false, true, true);
    else SW_K(false, true, false);
  } else {
    if (sp.g != 0.0) SW_K(false, false, true);
    else SW_K(false, false, false);
  }
#undef SW_K
}

}  // namespace

template <typename T>
void launch_multi(const StepIO<T>& io, const StepParams& sp, StepSeries ser, uint64_t step, int k,
                  bool write_f, int Lx, int Ly, int64_t fstride, Enc enc, int geom,
                  hipStream_t s) {
  MultiRun R{Lx, Ly, 0, k, fstride, step, ser, write_f ? 1 : 0};
  const F32K K32 = make_f32k(sp, enc);
  switch (geom) {
    case 0: launch_geom<T, 8, 8, 3, 512>(io, sp, K32, R, s); break;
    case 1: launch_geom<T, 16, 16, 3, 1024>(io, sp, K32, R, s); break;
    case 2: launch_geom<T, 24, 16, 2, 512>(io, sp, K32, R, s); break;
    case 3:
      if constexpr (sizeof(T) == 4) launch_geom<T, 32, 16, 2, 512>(io, sp, K32, R, s);
      break;
    default: launch_geom<T, 32, 16, 2, 1024>(io, sp, K32, R, s); break;
  }
}

// The shape with the smallest modelled time per step, unless one launch per
// step is faster: (FP64) 5.0 us and 2.1 us per round of its 64 x 8 tiles over
// the CUs, (FP32) 7.6 us and 1.05 us per round of 64 x 16 tiles (6 and 1.85
// beyond four), when it writes the moments only.  Measured, us per step (several / one per launch):
// FP64 64² 2.32 / 7.48, 256² 3.14 / 7.35, 512² 7.92 / 8.94, 700 x 640 13.9 /
// 12.7; FP32 64² 2.01 / 8.06, 256² 2.34 / 8.10, 512² 5.32 / 9.04, 850² 11.2 /
// 11.6, 1024² 14.2 / 11.9.
MultiShape multi_shape(int Lx, int Ly, bool f64, bool carried, int64_t nsteps) {
  const int64_t cus = device_cus();
  auto rounds = [&](int tx, int ty, int wgs) {
    const int64_t tiles = (int64_t)((Lx - 1) / tx + 1) * ((Ly - 1) / ty + 1);
    return (double)((tiles - 1) / (cus * wgs) + 1);
  };
  const double r = rounds(64, f64 ? 8 : 16, 1);
  double least = f64 ? 5.0 + 2.1 * r : r <= 4.0 ? 7.6 + 1.05 * r : 6.0 + 1.85 * r;
  // FP64 with τ ≠ 1: the halo's populations weigh more than the model's.  us per
  // step, one / several steps: 900 x 700 34.8 / 35.3, with noise 38.5 / 44.6;
  // 560² 21.0 / 20.4, 24.9 / 25.9; 500² (modelled at 0.85) 17.7 / 14.0, 21.0 / 18.0.
  if (carried && f64) least *= 0.9;
  MultiShape best{-1, 1, least};
  for (int i = 0; i < kNGeoms; ++i) {
    const Geom& g = f64 ? kGeoms64[i] : kGeoms32[i];
    const double t = (g.fixed + g.body * rounds(g.tx, g.ty, g.wgs)) / g.k;
    if (t < least) {
      least = t;
      best = MultiShape{i, g.k, t};
    }
  }
  // FP32 films that carry their populations (τ ≠ 1) outgrow the caches, where
  // two steps per launch halve the traffic of the 18 planes.  us per step, one
  // / two steps: 1000 x 1031 24.5 / 23.8, 1200² 32.7 / 33.5, 1300 x 1250 44.5 /
  // 35.8, 2000 x 1500 78 / 64, 3000² 256 / 180, 4096² 389 / 323, with noise 397
  // / 355.  FP64 tiles are bound by arithmetic: 2000 x 1500 118 / 141.
  // A launch of one of its two steps, which every loop ends with and a loop of
  // an even number takes twice, costs more than the one-step kernel's (us per
  // loop of one step, one / two: 750² 37 / 40, 1300 x 1250 62 / 76, 4096² 430 /
  // 610), and FP32 bits must not depend on where a launch falls, so short loops
  // stay with the one-step kernel (us per step of loops of 3 steps: 750² 26.3 /
  // 23.5, 4096² with noise 407 / 428).
  if (carried && !f64) {
    const bool large = best.geom < 0 && (int64_t)Lx * Ly >= 1600000;
    if (large) best = MultiShape{3, kGeoms32[3].k, least};
    if (best.geom >= kTwoStepGeom && nsteps < (large ? 9 : 4)) best = MultiShape{-1, 1, least};
  }
  return best;
}

template void launch_multi<double>(const StepIO<double>&, const StepParams&, StepSeries, uint64_t,
                                   int, bool, int, int, int64_t, Enc, int, hipStream_t);
template void launch_multi<float>(const StepIO<float>&, const StepParams&, StepSeries, uint64_t,
                                  int, bool, int, int, int64_t, Enc, int, hipStream_t);

}  // namespace swalbe
