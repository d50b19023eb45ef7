// ops.hip -- one kernel per reference op (the unfused, drop-in granularity).
//
// Every FP64 expression is written in the evaluation order of the reference
// broadcast it replaces and the library is built with -ffp-contract=off, so
// each op reproduces the reference's Float64 arithmetic bit for bit.  FP32
// arrays may carry the deviation encoding of Film (decode on load, encode on
// store); raw caller arrays use zero_enc().
#include "swalbe_internal.h"

namespace swalbe {

namespace {

constexpr int kBlock1D = 256;
constexpr int kBX = 64, kBY = 4;  // one wavefront per row for 2D stencils

template <typename T>
__device__ __forceinline__ T dec_h(T v, const Enc& e) {
  if constexpr (sizeof(T) == 4) return e.href + v;
  else return v;
}
template <typename T>
__device__ __forceinline__ T enc_h(T v, const Enc& e) {
  if constexpr (sizeof(T) == 4) return v - e.href;
  else return v;
}
template <typename T>
__device__ __forceinline__ T dec_f(T v, int k, const Enc& e) {
  if constexpr (sizeof(T) == 4) return e.R[k] + v;
  else return v;
}
template <typename T>
__device__ __forceinline__ T enc_f(T v, int k, const Enc& e) {
  if constexpr (sizeof(T) == 4) return v - e.R[k];
  else return v;
}

__device__ __forceinline__ int wrapi(int a, int L) {
  a %= L;
  return a < 0 ? a + L : a;
}

inline dim3 grid2d(int Lx, int Ly) { return dim3((Lx + kBX - 1) / kBX, (Ly + kBY - 1) / kBY); }
inline dim3 grid1d(int64_t N) {
  int64_t b = (N + kBlock1D - 1) / kBlock1D;
  if (b > 65535LL * 32) b = 65535LL * 32;
  return dim3((unsigned)(b < 1 ? 1 : b));
}

// ---------------------------------------------------------------- equilibrium
// src/equilibrium.jl:63-116
template <typename T>
__global__ void k_equilibrium(T* __restrict__ feq, const T* __restrict__ h,
                              const T* __restrict__ ux, const T* __restrict__ uy,
                              T* __restrict__ vsq, T g, int64_t N, int64_t fs, Enc e) {
  const T g0 = T(1.5) * g;
  const T w1 = T(1.0 / 9.0), w5 = T(1.0 / 36.0);
  for (int64_t x = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; x < N;
       x += (int64_t)gridDim.x * blockDim.x) {
    const T hh = dec_h(h[x], e), u = ux[x], v = uy[x];
    const T usq = u * u + v * v;
    vsq[x] = usq;
    T f[kQ];
    f[0] = hh * ((T(1) - T(5.0 / 6.0) * g * hh) - T(2.0 / 3.0) * usq);
    f[1] = w1 * hh * (((g0 * hh + T(3) * u) + T(4.5) * (u * u)) - T(1.5) * usq);
    f[2] = w1 * hh * (((g0 * hh + T(3) * v) + T(4.5) * (v * v)) - T(1.5) * usq);
    f[3] = w1 * hh * (((g0 * hh - T(3) * u) + T(4.5) * (u * u)) - T(1.5) * usq);
    f[4] = w1 * hh * (((g0 * hh - T(3) * v) + T(4.5) * (v * v)) - T(1.5) * usq);
    T a = u + v;
    f[5] = w5 * hh * (((g0 * hh + T(3) * a) + T(4.5) * (a * a)) - T(1.5) * usq);
    a = v - u;
    f[6] = w5 * hh * (((g0 * hh + T(3) * a) + T(4.5) * (a * a)) - T(1.5) * usq);
    a = u + v;
    f[7] = w5 * hh * (((g0 * hh - T(3) * a) + T(4.5) * (a * a)) - T(1.5) * usq);
    a = u - v;
    f[8] = w5 * hh * (((g0 * hh + T(3) * a) + T(4.5) * (a * a)) - T(1.5) * usq);
#pragma unroll
    for (int k = 0; k < kQ; ++k) feq[k * fs + x] = enc_f(f[k], k, e);
  }
}

// ---------------------------------------------------------------- BGK + stream
// src/collide.jl:70-105: collision with the force term, pull stream
// f_k(x) <- fo_k(x - c_k), written to fdst (the caller makes fout and ftemp
// both refer to it, as `fout .= ftemp` does).
template <typename T>
__device__ __forceinline__ T force_term(int k, T Fx, T Fy) {
  const T c3 = T(1.0 / 3.0), c24 = T(1.0 / 24.0);
  switch (k) {
    case 1: return c3 * Fx;
    case 2: return c3 * Fy;
    case 3: return -(c3 * Fx);
    case 4: return -(c3 * Fy);
    case 5: return c24 * (Fx + Fy);
    case 6: return c24 * (Fy - Fx);
    case 7: return -(c24 * (Fx + Fy));
    case 8: return c24 * (Fx - Fy);
    default: return T(0);
  }
}

template <typename T>
__global__ void k_bgk_stream(T* __restrict__ fdst, const T* __restrict__ feq,
                             const T* __restrict__ ftemp, const T* __restrict__ Fx,
                             const T* __restrict__ Fy, T omeg, T itau, int Lx, int Ly, int64_t fs,
                             Enc e) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int j = blockIdx.y * blockDim.y + threadIdx.y;
  if (i >= Lx || j >= Ly) return;
  const int64_t x = i + (int64_t)Lx * j;
#pragma unroll
  for (int k = 0; k < kQ; ++k) {
    const int is = wrapi(i - cx(k), Lx), js = wrapi(j - cy(k), Ly);
    const int64_t y = is + (int64_t)Lx * js;
    const T ft = dec_f(ftemp[k * fs + y], k, e);
    const T fe = dec_f(feq[k * fs + y], k, e);
    T fo = omeg * ft + itau * fe;
    // (a + b) - c*F is written as (a + b) + (-(c*F)); IEEE negation is exact
    if (k > 0) fo = fo + force_term<T>(k, Fx[y], Fy[y]);
    fdst[k * fs + x] = enc_f(fo, k, e);
  }
}

// ---------------------------------------------------------------- moments
// src/moments.jl:43-52: h = f0 + f1 + ... + f8 (sum!), u = Σ c f / h.
template <typename T>
__global__ void k_moments(T* __restrict__ h, T* __restrict__ ux, T* __restrict__ uy,
                          const T* __restrict__ f, int64_t N, int64_t fs, Enc e) {
  for (int64_t x = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; x < N;
       x += (int64_t)gridDim.x * blockDim.x) {
    T v[kQ];
#pragma unroll
    for (int k = 0; k < kQ; ++k) v[k] = dec_f(f[k * fs + x], k, e);
    T s = v[0];
#pragma unroll
    for (int k = 1; k < kQ; ++k) s = s + v[k];
    h[x] = enc_h(s, e);
    ux[x] = (((((v[1] - v[3]) + v[5]) - v[6]) - v[7]) + v[8]) / s;
    uy[x] = (((((v[2] - v[4]) + v[5]) + v[6]) - v[7]) - v[8]) / s;
  }
}

// ---------------------------------------------------------------- film pressure
// src/pressure.jl:72-155.  Neighbour names follow the reference: hip is
// circshift(h, (1,0)), i.e. h[i-1, j].
template <typename T>
__device__ __forceinline__ T lap9(T hip, T hjp, T him, T hjm, T hipjp, T himjp, T himjm, T hipjm,
                                  T hc) {
  return (T(2.0 / 3.0) * (((hjp + hip) + him) + hjm) +
          T(1.0 / 6.0) * (((hipjp + himjp) + himjm) + hipjm)) -
         T(10.0 / 3.0) * hc;
}

template <typename T>
__device__ __forceinline__ T power_broad(T a, int n) {
  T t = T(1);
  for (int i = 0; i < n; ++i) t *= a;
  return t;
}

template <typename T>
__device__ __forceinline__ T powlaw(T a, int n, int m, int mode) {
  if (mode == 1) {  // fast_93
    const T t = (a * a) * a;
    return ((t * t) * t) - t;
  }
  if (mode == 2) return ((a * a) * a) - (a * a);  // fast_32
  if (n == 9 && m == 3) {  // power_broad's products in its order, no loop
    const T a3 = (a * a) * a;
    const T a6 = ((a3 * a) * a) * a;
    return (((a6 * a) * a) * a) - a3;
  }
  return power_broad(a, n) - power_broad(a, m);
}

template <typename T>
__global__ void k_filmpressure(T* __restrict__ p, const T* __restrict__ h, T gamma, T kap,
                               const T* __restrict__ theta, const T* __restrict__ kapf, int n,
                               int m, T hmin, T hcrit, int mode, int Lx, int Ly, Enc e) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int j = blockIdx.y * blockDim.y + threadIdx.y;
  if (i >= Lx || j >= Ly) return;
  const int im = wrapi(i - 1, Lx), ip = wrapi(i + 1, Lx);
  const int jm = wrapi(j - 1, Ly), jp = wrapi(j + 1, Ly);
  auto H = [&](int a, int b) { return h[a + (int64_t)Lx * b]; };
  const int64_t x = i + (int64_t)Lx * j;
  // Laplacian of the stored values (the FP32 offset href cancels exactly).
  const T L = lap9(H(im, j), H(i, jm), H(ip, j), H(i, jp), H(im, jm), H(ip, jm), H(ip, jp),
                   H(im, jp), H(i, j));
  const T hh = dec_h(H(i, j), e);
  T k = kap;
  if (kapf) k = kapf[x];
  else if (theta) k = (T)kappa((double)theta[x], n, m, (double)hmin);
  const T a = hmin / (hh + hcrit);
  const T p0 = -gamma * (k * powlaw(a, n, m, mode));
  p[x] = p0 - gamma * L;
}

// ---------------------------------------------------------------- gradients
// ∇f! (src/differences.jl:153-206) and h∇p! (src/forcing.jl:168-187):
// out = a * (-1/3 (f[i-1]-f[i+1]) - 1/12 (...)); `a` is a field or absent.
template <typename T>
__global__ void k_grad(T* __restrict__ ox, T* __restrict__ oy, const T* __restrict__ f,
                       const T* __restrict__ a, const T* __restrict__ hh, int Lx, int Ly,
                       Enc e) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int j = blockIdx.y * blockDim.y + threadIdx.y;
  if (i >= Lx || j >= Ly) return;
  const int im = wrapi(i - 1, Lx), ip = wrapi(i + 1, Lx);
  const int jm = wrapi(j - 1, Ly), jp = wrapi(j + 1, Ly);
  auto F = [&](int u, int v) { return f[u + (int64_t)Lx * v]; };
  const T fip = F(im, j), fim = F(ip, j), fjp = F(i, jm), fjm = F(i, jp);
  const T fipjp = F(im, jm), fimjp = F(ip, jm), fimjm = F(ip, jp), fipjm = F(im, jp);
  const T gx = T(-1.0 / 3.0) * (fip - fim) - T(1.0 / 12.0) * (((fipjp - fimjp) - fimjm) + fipjm);
  const T gy = T(-1.0 / 3.0) * (fjp - fjm) - T(1.0 / 12.0) * (((fipjp + fimjp) - fimjm) - fipjm);
  const int64_t x = i + (int64_t)Lx * j;
  if (hh) {  // h∇p!: height * gradient
    const T hv = dec_h(hh[x], e);
    ox[x] = hv * gx;
    oy[x] = hv * gy;
  } else if (a) {
    ox[x] = a[x] * gx;
    oy[x] = a[x] * gy;
  } else {
    ox[x] = gx;
    oy[x] = gy;
  }
}

// ∇²f!(output, f, γ): src/differences.jl:57-75
template <typename T>
__global__ void k_laplacian(T* __restrict__ out, const T* __restrict__ f, T gamma, int Lx,
                            int Ly) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int j = blockIdx.y * blockDim.y + threadIdx.y;
  if (i >= Lx || j >= Ly) return;
  const int im = wrapi(i - 1, Lx), ip = wrapi(i + 1, Lx);
  const int jm = wrapi(j - 1, Ly), jp = wrapi(j + 1, Ly);
  auto F = [&](int u, int v) { return f[u + (int64_t)Lx * v]; };
  out[i + (int64_t)Lx * j] =
      gamma * lap9(F(im, j), F(i, jm), F(ip, j), F(i, jp), F(im, jm), F(ip, jm), F(ip, jp),
                   F(im, jp), F(i, j));
}

// ---------------------------------------------------------------- slip, noise, body force
// slippage!: src/forcing.jl:42-46
template <typename T>
__global__ void k_slippage(T* __restrict__ sx, T* __restrict__ sy, const T* __restrict__ h,
                           const T* __restrict__ ux, const T* __restrict__ uy, T c6mu, T c6d,
                           T c3dd, int64_t N, Enc e) {
  for (int64_t x = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; x < N;
       x += (int64_t)gridDim.x * blockDim.x) {
    const T hh = dec_h(h[x], e);
    const T den = (T(2) * (hh * hh) + c6d * hh) + c3dd;
    sx[x] = (c6mu * hh * ux[x]) / den;
    sy[x] = (c6mu * hh * uy[x]) / den;
  }
}

// thermal!: src/forcing.jl:297-311 with counter-based normals
template <typename T>
__global__ void k_thermal(T* __restrict__ kx, T* __restrict__ ky, const T* __restrict__ h,
                          T kb26, T delta, T d3dd, uint64_t seed, uint64_t step, int64_t N,
                          int Lx, Enc e) {
  for (int64_t x = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; x < N;
       x += (int64_t)gridDim.x * blockDim.x) {
    double z0, z1;
    normal_pair(seed, step, noise_index((int)(x % Lx), (int)(x / Lx), Lx), kTagThermal, &z0, &z1);
    const T hh = dec_h(h[x], e);
    const T amp = sqrt(kb26 * hh / (((T(2) * hh) * hh + (T(6) * hh) * delta) + d3dd));
    kx[x] = (T)z0 * amp;
    ky[x] = (T)z1 * amp;
  }
}

// inclination!: src/forcing.jl:363-368
template <typename T>
__global__ void k_inclination(T* __restrict__ Fx, T* __restrict__ Fy, const T* __restrict__ h,
                              T ax, T ay, T fac, int64_t N, Enc e) {
  for (int64_t x = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; x < N;
       x += (int64_t)gridDim.x * blockDim.x) {
    const T hh = dec_h(h[x], e);
    Fx[x] = Fx[x] + (hh * ax) * fac;
    Fy[x] = Fy[x] + (hh * ay) * fac;
  }
}

// F = -h∇p - slip [- kbt]: src/simulate.jl:18-19
template <typename T>
__global__ void k_force_sum(T* __restrict__ Fx, T* __restrict__ Fy, const T* __restrict__ hx,
                            const T* __restrict__ hy, const T* __restrict__ sx,
                            const T* __restrict__ sy, const T* __restrict__ kx,
                            const T* __restrict__ ky, int64_t N) {
  for (int64_t x = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; x < N;
       x += (int64_t)gridDim.x * blockDim.x) {
    T a = -hx[x] - sx[x];
    T b = -hy[x] - sy[x];
    if (kx) {
      a = a - kx[x];
      b = b - ky[x];
    }
    Fx[x] = a;
    Fy[x] = b;
  }
}

// ---------------------------------------------------------------- a step's two halves
// The op-by-op loop with a user's callback between the force sum and
// equilibrium! runs these instead of five and three op kernels: every field
// an op would write is written, with its bits, and a step costs two launches.
// A step of 512 x 512 FP64 with a reduction in the callback took 88 us with
// the eight op kernels (45 us of GPU time); with these two it takes 40 (24).

// filmpressure!, h∇p!, slippage!, [thermal!] and the force sum.  A workgroup
// takes 64 x kFY nodes; their pressures and a ring around them go through LDS.
// Bound by memory: three planes read and seven written (nine with noise) take
// 7.4 us at 512 x 512 FP64; as five kernels 25 us.
constexpr int kFY = 8;

struct ForceConst {
  double gamma, kap, hmin, hcrit, c6mu, c6d, c3dd, kb26, delta, d3dd;
  int n, m, thermal;
  uint64_t seed, step;
};

template <typename T>
struct ForceOut {
  T *p, *hx, *hy, *sx, *sy, *kx, *ky, *Fx, *Fy;
};

template <typename T>
__global__ __launch_bounds__(256) void k_forces(ForceOut<T> o, const T* __restrict__ h,
                                                const T* __restrict__ ux,
                                                const T* __restrict__ uy, ForceConst C, int Lx,
                                                int Ly, Enc e) {
  constexpr int PC = 66, PR = kFY + 2;
  __shared__ T sp[PR * PC];
  const int x0 = blockIdx.x * 64, y0 = blockIdx.y * kFY;
  const T gamma = (T)C.gamma, kap = (T)C.kap, hmin = (T)C.hmin, hcrit = (T)C.hcrit;
  for (int t = threadIdx.x; t < PR * PC; t += 256) {
    const int r = t / PC, c = t - r * PC;
    const int i = wrapi(x0 - 1 + c, Lx), j = wrapi(y0 - 1 + r, Ly);
    const int im = i == 0 ? Lx - 1 : i - 1, ip = i == Lx - 1 ? 0 : i + 1;
    const int jm = j == 0 ? Ly - 1 : j - 1, jp = j == Ly - 1 ? 0 : j + 1;
    auto H = [&](int a, int b) { return h[a + (int64_t)Lx * b]; };
    const T L = lap9(H(im, j), H(i, jm), H(ip, j), H(i, jp), H(im, jm), H(ip, jm), H(ip, jp),
                     H(im, jp), H(i, j));
    const T a = hmin / (dec_h(H(i, j), e) + hcrit);
    const T p0 = -gamma * (kap * powlaw(a, C.n, C.m, 0));
    sp[t] = p0 - gamma * L;
  }
  __syncthreads();
  for (int t = threadIdx.x; t < 64 * kFY; t += 256) {
    const int r = t >> 6, c = t & 63;
    const int i = x0 + c, j = y0 + r;
    if (i >= Lx || j >= Ly) continue;
    const int64_t x = i + (int64_t)Lx * j;
    const T* pc = &sp[(r + 1) * PC + c + 1];
    const T fip = pc[-1], fim = pc[1], fjp = pc[-PC], fjm = pc[PC];
    const T fipjp = pc[-PC - 1], fimjp = pc[-PC + 1], fimjm = pc[PC + 1], fipjm = pc[PC - 1];
    const T gx = T(-1.0 / 3.0) * (fip - fim) - T(1.0 / 12.0) * (((fipjp - fimjp) - fimjm) + fipjm);
    const T gy = T(-1.0 / 3.0) * (fjp - fjm) - T(1.0 / 12.0) * (((fipjp + fimjp) - fimjm) - fipjm);
    const T hh = dec_h(h[x], e);
    const T hx = hh * gx, hy = hh * gy;
    const T den = (T(2) * (hh * hh) + (T)C.c6d * hh) + (T)C.c3dd;
    const T sx = ((T)C.c6mu * hh * ux[x]) / den, sy = ((T)C.c6mu * hh * uy[x]) / den;
    o.p[x] = pc[0];
    o.hx[x] = hx;
    o.hy[x] = hy;
    o.sx[x] = sx;
    o.sy[x] = sy;
    T a = -hx - sx, b = -hy - sy;
    if (C.thermal) {
      double z0, z1;
      normal_pair(C.seed, C.step, noise_index(i, j, Lx), kTagThermal, &z0, &z1);
      const T amp = sqrt((T)C.kb26 * hh /
                         (((T(2) * hh) * hh + (T(6) * hh) * (T)C.delta) + (T)C.d3dd));
      const T kx = (T)z0 * amp, ky = (T)z1 * amp;
      o.kx[x] = kx;
      o.ky[x] = ky;
      a = a - kx;
      b = b - ky;
    }
    o.Fx[x] = a;
    o.Fy[x] = b;
  }
}

// feq_k of a node of height hh and velocity (u, v), as k_equilibrium forms it
template <typename T>
__device__ __forceinline__ T feq_of(int k, T hh, T u, T v, T usq, T g, T g0) {
  const T w1 = T(1.0 / 9.0), w5 = T(1.0 / 36.0);
  if (k == 0) return hh * ((T(1) - T(5.0 / 6.0) * g * hh) - T(2.0 / 3.0) * usq);
  const T a = k == 1 || k == 3 ? u : k == 2 || k == 4 ? v : k == 5 || k == 7 ? u + v
            : k == 6 ? v - u : u - v;
  const T lin = k == 3 || k == 4 || k == 7 ? g0 * hh - T(3) * a : g0 * hh + T(3) * a;
  return (k <= 4 ? w1 : w5) * hh * ((lin + T(4.5) * (a * a)) - T(1.5) * usq);
}

// equilibrium!, BGKandStream! and moments!: feq and |u|^2 of the old moments,
// the streamed populations, the new moments (to other buffers than the old).
// Bound by memory: 14 planes read and 22 written, 16.5 us at 512 x 512 FP64
// (4.6 TB/s); each source node's equilibrium is formed again by its neighbours
// instead of read back from feq.  As three kernels 25 us.
template <typename T>
struct Advance {
  const T *h, *ux, *uy, *Fx, *Fy, *ft;
  T *feq, *vsq, *f, *hn, *un, *vn;
};

template <typename T>
__global__ __launch_bounds__(kBX* kBY) void k_advance(Advance<T> a, T g, T omeg, T itau, int Lx,
                                                      int Ly, int64_t fs, Enc e) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int j = blockIdx.y * blockDim.y + threadIdx.y;
  if (i >= Lx || j >= Ly) return;
  const int64_t x = i + (int64_t)Lx * j;
  const int im = i == 0 ? Lx - 1 : i - 1, ip = i == Lx - 1 ? 0 : i + 1;
  const int jm = j == 0 ? Ly - 1 : j - 1, jp = j == Ly - 1 ? 0 : j + 1;
  const T g0 = T(1.5) * g;
  T f[kQ];
#pragma unroll
  for (int k = 0; k < kQ; ++k) {
    const int is = cx(k) > 0 ? im : cx(k) < 0 ? ip : i, js = cy(k) > 0 ? jm : cy(k) < 0 ? jp : j;
    const int64_t y = is + (int64_t)Lx * js;
    const T hh = dec_h(a.h[y], e), u = a.ux[y], v = a.uy[y];
    const T usq = u * u + v * v;
    if (k == 0) {  // the node's own equilibrium
      a.vsq[x] = usq;
#pragma unroll
      for (int q = 0; q < kQ; ++q) a.feq[q * fs + x] = enc_f(feq_of(q, hh, u, v, usq, g, g0), q, e);
    }
    // what k_equilibrium stores and k_bgk_stream reads back
    const T fe = dec_f(enc_f(feq_of(k, hh, u, v, usq, g, g0), k, e), k, e);
    T fo = omeg * dec_f(a.ft[k * fs + y], k, e) + itau * fe;
    if (k > 0) fo = fo + force_term<T>(k, a.Fx[y], a.Fy[y]);
    const T st = enc_f(fo, k, e);
    a.f[k * fs + x] = st;
    f[k] = dec_f(st, k, e);
  }
  T s = f[0];
#pragma unroll
  for (int k = 1; k < kQ; ++k) s = s + f[k];
  a.hn[x] = enc_h(s, e);
  a.un[x] = (((((f[1] - f[3]) + f[5]) - f[6]) - f[7]) + f[8]) / s;
  a.vn[x] = (((((f[2] - f[4]) + f[5]) + f[6]) - f[7]) - f[8]) / s;
}

template <typename T>
__global__ void k_kappa(T* __restrict__ kap, const T* __restrict__ theta, int n, int m,
                        double hmin, int64_t N) {
  for (int64_t x = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; x < N;
       x += (int64_t)gridDim.x * blockDim.x)
    kap[x] = (T)kappa((double)theta[x], n, m, hmin);
}

template <typename T>
__global__ void k_fill(T* __restrict__ p, T v, int64_t N) {
  for (int64_t x = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; x < N;
       x += (int64_t)gridDim.x * blockDim.x)
    p[x] = v;
}

template <typename T>
__global__ void k_init_random(T* __restrict__ h, int dist, uint64_t seed, double base,
                              double amp, double href, int64_t N, int Lx) {
  for (int64_t x = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; x < N;
       x += (int64_t)gridDim.x * blockDim.x) {
    double v;
    if (dist == 0) {
      v = base + amp * uniform(seed, 0, (uint32_t)x, kTagInitUniform);
    } else {
      double z0, z1;
      normal_pair(seed, 0, noise_index((int)(x % Lx), (int)(x / Lx), Lx), kTagInitNormal, &z0,
                  &z1);
      v = base + amp * z0;
    }
    h[x] = (T)(v - href);
  }
}

}  // namespace

// ---------------------------------------------------------------- launchers
template <typename T>
void launch_forces(const Film& F, const swalbe_params& p, int thermal, uint64_t seed, uint64_t step,
                   hipStream_t s) {
  ForceConst C{};
  C.gamma = p.gamma;
  C.kap = kappa(p.theta, p.n, p.m, p.hmin);
  C.hmin = p.hmin;
  C.hcrit = p.hcrit;
  C.c6mu = 6.0 * p.mu;
  C.c6d = 6.0 * p.delta;
  C.c3dd = 3.0 * (p.delta * p.delta);
  C.kb26 = ((2.0 * p.kbt) * p.mu) * 6.0;
  C.delta = p.delta;
  C.d3dd = (3.0 * p.delta) * p.delta;
  C.n = p.n;
  C.m = p.m;
  C.thermal = thermal;
  C.seed = seed;
  C.step = step;
  const ForceOut<T> o{(T*)F.pressure, (T*)F.hgpx, (T*)F.hgpy, (T*)F.slipx, (T*)F.slipy,
                      (T*)F.kbtx,     (T*)F.kbty, (T*)F.Fx,   (T*)F.Fy};
  const dim3 grid((F.Lx + 63) / 64, (F.Ly + kFY - 1) / kFY);
  hipLaunchKernelGGL(k_forces<T>, grid, dim3(256), 0, s, o, (const T*)F.height(),
                     (const T*)F.velx(), (const T*)F.vely(), C, F.Lx, F.Ly, F.enc);
}

template <typename T>
void launch_advance(Film& F, double g, double tau, hipStream_t s) {
  const int cur = F.hu_cur, dst = F.fout_buf != F.ftemp_buf ? F.fout_buf : 1 - F.ftemp_buf;
  const Advance<T> a{(const T*)F.hbuf[cur],     (const T*)F.uxbuf[cur], (const T*)F.uybuf[cur],
                     (const T*)F.Fx,            (const T*)F.Fy,         (const T*)F.f[F.ftemp_buf],
                     (T*)F.feq,                 (T*)F.vsq,              (T*)F.f[dst],
                     (T*)F.hbuf[1 - cur],       (T*)F.uxbuf[1 - cur],   (T*)F.uybuf[1 - cur]};
  const double omeg = 1.0 - 1.0 / tau, itau = 1.0 / tau;
  hipLaunchKernelGGL(k_advance<T>, grid2d(F.Lx, F.Ly), dim3(kBX, kBY), 0, s, a, (T)g, (T)omeg,
                     (T)itau, F.Lx, F.Ly, F.fstride, F.enc);
  F.fout_buf = F.ftemp_buf = dst;
  F.hu_cur = 1 - cur;
}
template void launch_forces<double>(const Film&, const swalbe_params&, int, uint64_t, uint64_t,
                                    hipStream_t);
template void launch_forces<float>(const Film&, const swalbe_params&, int, uint64_t, uint64_t,
                                   hipStream_t);
template void launch_advance<double>(Film&, double, double, hipStream_t);
template void launch_advance<float>(Film&, double, double, hipStream_t);

template <typename T>
void launch_equilibrium(T* feq, const T* h, const T* ux, const T* uy, T* vsq, double g, int Lx,
                        int Ly, int64_t fs, Enc enc, hipStream_t s) {
  const int64_t N = (int64_t)Lx * Ly;
  hipLaunchKernelGGL(k_equilibrium<T>, grid1d(N), dim3(kBlock1D), 0, s, feq, h, ux, uy, vsq,
                     (T)g, N, fs, enc);
}
template <typename T>
void launch_bgk_and_stream(T* fdst, const T* feq, const T* ftemp, const T* Fx, const T* Fy,
                           double tau, int Lx, int Ly, int64_t fs, Enc enc, hipStream_t s) {
  const double omeg = 1.0 - 1.0 / tau, itau = 1.0 / tau;
  hipLaunchKernelGGL(k_bgk_stream<T>, grid2d(Lx, Ly), dim3(kBX, kBY), 0, s, fdst, feq, ftemp, Fx,
                     Fy, (T)omeg, (T)itau, Lx, Ly, fs, enc);
}
template <typename T>
void launch_moments(T* h, T* ux, T* uy, const T* f, int Lx, int Ly, int64_t fs, Enc enc,
                    hipStream_t s) {
  const int64_t N = (int64_t)Lx * Ly;
  hipLaunchKernelGGL(k_moments<T>, grid1d(N), dim3(kBlock1D), 0, s, h, ux, uy, f, N, fs, enc);
}
template <typename T>
void launch_filmpressure(T* p, const T* h, double gamma, double kappa_scalar, const T* theta,
                         const T* kapf, int n, int m, double hmin, double hcrit, int powmode,
                         int Lx, int Ly, Enc enc, hipStream_t s) {
  hipLaunchKernelGGL(k_filmpressure<T>, grid2d(Lx, Ly), dim3(kBX, kBY), 0, s, p, h, (T)gamma,
                     (T)kappa_scalar, theta, kapf, n, m, (T)hmin, (T)hcrit, powmode, Lx, Ly, enc);
}
template <typename T>
void launch_kappa_field(T* kap, const T* theta, int n, int m, double hmin, int64_t N,
                        hipStream_t s) {
  hipLaunchKernelGGL(k_kappa<T>, grid1d(N), dim3(kBlock1D), 0, s, kap, theta, n, m, hmin, N);
}
template <typename T>
void launch_grad(T* ox, T* oy, const T* f, const T* a, const T* h, int Lx, int Ly, Enc enc,
                 hipStream_t s) {
  hipLaunchKernelGGL(k_grad<T>, grid2d(Lx, Ly), dim3(kBX, kBY), 0, s, ox, oy, f, a, h, Lx, Ly,
                     enc);
}
template <typename T>
void launch_laplacian(T* out, const T* f, double gamma, int Lx, int Ly, hipStream_t s) {
  hipLaunchKernelGGL(k_laplacian<T>, grid2d(Lx, Ly), dim3(kBX, kBY), 0, s, out, f, (T)gamma, Lx,
                     Ly);
}
template <typename T>
void launch_slippage(T* sx, T* sy, const T* h, const T* ux, const T* uy, double delta, double mu,
                     int Lx, int Ly, Enc enc, hipStream_t s) {
  const int64_t N = (int64_t)Lx * Ly;
  hipLaunchKernelGGL(k_slippage<T>, grid1d(N), dim3(kBlock1D), 0, s, sx, sy, h, ux, uy,
                     (T)(6.0 * mu), (T)(6.0 * delta), (T)(3.0 * (delta * delta)), N, enc);
}
template <typename T>
void launch_thermal(T* kx, T* ky, const T* h, double kbt, double mu, double delta, uint64_t seed,
                    uint64_t step, int Lx, int Ly, Enc enc, hipStream_t s) {
  const int64_t N = (int64_t)Lx * Ly;
  hipLaunchKernelGGL(k_thermal<T>, grid1d(N), dim3(kBlock1D), 0, s, kx, ky, h,
                     (T)(((2.0 * kbt) * mu) * 6.0), (T)delta, (T)((3.0 * delta) * delta), seed,
                     step, N, Lx, enc);
}
template <typename T>
void launch_inclination(T* Fx, T* Fy, const T* h, double ax, double ay, double fac, int Lx,
                        int Ly, Enc enc, hipStream_t s) {
  const int64_t N = (int64_t)Lx * Ly;
  hipLaunchKernelGGL(k_inclination<T>, grid1d(N), dim3(kBlock1D), 0, s, Fx, Fy, h, (T)ax, (T)ay,
                     (T)fac, N, enc);
}
template <typename T>
void launch_force_sum(T* Fx, T* Fy, const T* hgpx, const T* hgpy, const T* sx, const T* sy,
                      const T* kx, const T* ky, int64_t N, hipStream_t s) {
  hipLaunchKernelGGL(k_force_sum<T>, grid1d(N), dim3(kBlock1D), 0, s, Fx, Fy, hgpx, hgpy, sx, sy,
                     kx, ky, N);
}
template <typename T>
void launch_fill(T* p, double v, int64_t N, hipStream_t s) {
  hipLaunchKernelGGL(k_fill<T>, grid1d(N), dim3(kBlock1D), 0, s, p, (T)v, N);
}
template <typename T>
void launch_init_random(T* h, int dist, uint64_t seed, double base, double amp, double href,
                        int Lx, int Ly, hipStream_t s) {
  const int64_t N = (int64_t)Lx * Ly;
  hipLaunchKernelGGL(k_init_random<T>, grid1d(N), dim3(kBlock1D), 0, s, h, dist, seed, base, amp,
                     href, N, Lx);
}

#define SW_INSTANTIATE(T)                                                                        \
  template void launch_equilibrium<T>(T*, const T*, const T*, const T*, T*, double, int, int,   \
                                      int64_t, Enc, hipStream_t);                                \
  template void launch_bgk_and_stream<T>(T*, const T*, const T*, const T*, const T*, double, int, \
                                         int, int64_t, Enc, hipStream_t);                        \
  template void launch_moments<T>(T*, T*, T*, const T*, int, int, int64_t, Enc, hipStream_t);    \
  template void launch_filmpressure<T>(T*, const T*, double, double, const T*, const T*, int, int, \
                                       double, double, int, int, int, Enc, hipStream_t);         \
  template void launch_kappa_field<T>(T*, const T*, int, int, double, int64_t, hipStream_t);      \
  template void launch_grad<T>(T*, T*, const T*, const T*, const T*, int, int, Enc, hipStream_t); \
  template void launch_laplacian<T>(T*, const T*, double, int, int, hipStream_t);                 \
  template void launch_slippage<T>(T*, T*, const T*, const T*, const T*, double, double, int, int, \
                                   Enc, hipStream_t);                                            \
  template void launch_thermal<T>(T*, T*, const T*, double, double, double, uint64_t, uint64_t,   \
                                  int, int, Enc, hipStream_t);                                   \
  template void launch_inclination<T>(T*, T*, const T*, double, double, double, int, int, Enc,    \
                                      hipStream_t);                                              \
  template void launch_force_sum<T>(T*, T*, const T*, const T*, const T*, const T*, const T*,     \
                                    const T*, int64_t, hipStream_t);                             \
  template void launch_fill<T>(T*, double, int64_t, hipStream_t);                                \
  template void launch_init_random<T>(T*, int, uint64_t, double, double, double, int, int,        \
                                      hipStream_t);

SW_INSTANTIATE(double)
SW_INSTANTIATE(float)

}  // namespace swalbe
