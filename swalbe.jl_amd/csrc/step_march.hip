// step_march.hip -- the D2Q9 step of a larger film, one wavefront per strip.
//
// A wave owns a strip of 64 columns, one per lane, and marches up a segment of
// rows.  At output row j it loads h(j+3), forms p(j+2) from h(j+1 .. j+3), the
// forces and the nine post-collision populations of row j+1 from p(j .. j+2),
// and streams row j from the populations of rows j-1, j, j+1.  The rows live
// in registers, neighbouring columns in the next lanes (DPP): no LDS, no
// barrier, every quantity computed once per node of the strip.  The three
// stencils cost three columns at each end (58 are written) and three rows of
// start-up per segment.
//
// What bounds it: VALU issue and HBM about evenly.  A step of a 4096 x 4096
// FP32 film that writes the moments only takes 110 us (3.7 TB/s of the 24
// bytes per node, VALU 65 % busy: 160 instructions per node) against 122 with
// the 64 x 16 LDS tiles, whose halo and per-population collisions cost 307;
// FP64 206 against 287 us, with noise 320 against 409; 2500 x 2501 FP64 with
// noise 124 against 161; 2000 x 1500 FP32 21 against 26, FP64 37 against 56.
// A step that also writes f and p is the tiles' (FP64 465 against 670 us at
// 4096 x 4096, 90 against 108 at 2000 x 1500: a strip's 58 columns start on no
// line, nine times per node), so an FP64 loop takes its last step there, with
// the same bits, and τ ≠ 1, which writes them on every step, stays there.  An
// FP32 loop takes every step here, for the same bits however a run is cut into
// loops: its last step costs what the tiles' does wherever a row of the film
// starts on no line either (2501 x 2499 142 against 135 us, 176 with the tiles'
// streaming stores; 4100 x 4100 363 against 381) or the outputs fit the last
// level cache (2000 x 1500 53 against 54).  Two columns per lane (120
// written, on 32-byte sectors) were as fast at 4096 x 4096 (106, 204 us) and
// slower on smaller films (2000 x 1500 FP32 23 us).
#include <math.h>

#include "step_node.h"
#include "swalbe_internal.h"

namespace swalbe {

namespace {

constexpr int kMarchOut = 58;  // columns a strip writes

struct MarchRun {
  int Lx, Ly, nstrips, seg, items, chunk;
  int64_t fstride;
  uint64_t step;
  StepSeries ser;
};

// The value of the lane below / above (DPP wave_shr:1 / wave_shl:1; 0 beyond
// the wave's ends, whose columns are halo and never written).
template <int CTRL>
__device__ __forceinline__ float shift(float v) {
  return __builtin_bit_cast(
      float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true));
}
template <int CTRL>
__device__ __forceinline__ double shift(double v) {
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo =
      (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, CTRL, 0xF, 0xF, true);
  const uint32_t hi =
      (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32), CTRL, 0xF, 0xF, true);
  return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}
template <typename T>
__device__ __forceinline__ T below(T v) {
  return shift<0x138>(v);
}
template <typename T>
__device__ __forceinline__ T above(T v) {
  return shift<0x130>(v);
}

// One row of the strip: this lane's column and its neighbours.
template <typename T>
struct Row {
  T v, m, p;  // at x, x - 1, x + 1
  __device__ __forceinline__ void edges() {
    m = below(v);
    p = above(v);
  }
};

template <typename T>
struct Pops {
  T f[kQ];
};

__device__ __forceinline__ int wrap1(int a, int L) {
  return a < 0 ? a + L : (a >= L ? a - L : a);
}

typedef __attribute__((address_space(1))) char gbytes;
template <typename T>
__device__ __forceinline__ const gbytes* uniform(const T* p) {
  const uint64_t a = (uint64_t)p;
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)a);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(a >> 32));
  return (const gbytes*)(((uint64_t)hi << 32) | lo);
}

template <typename T, bool TH, bool WF, bool GRAV, bool SER>
struct March {
  static constexpr bool F32 = sizeof(T) == 4;
  using R3 = Row<T>;
  using P9 = Pops<T>;
  typedef __attribute__((address_space(1))) T GT;

  const StepIO<T>& io;
  const StepParams& sp;
  const F32K& K32;
  const MarchRun& R;
  int y0, jlast;
  uint32_t gx, off;      // the lane's (wrapped) column and its byte offset in a row
  bool out;              // a column this lane writes
  T nh, nu, nv, nk;      // prefetched rows
  uint32_t w2, w3;       // noise words of the odd row of a pair
  double lmax, lmin;
  unsigned int cnt;

  __device__ __forceinline__ int wy(int j) const { return wrap1(j, R.Ly); }
  __device__ __forceinline__ T get(const T* plane, int64_t row) const {
    return *(const GT*)(uniform(plane + row) + off);
  }
  __device__ __forceinline__ void put(T* plane, int64_t row, T v) const {
    *(GT*)(const_cast<gbytes*>(uniform(plane + row)) + off) = v;
  }

  __device__ __forceinline__ void prefetch(int j) {
    const int64_t r1 = (int64_t)R.Lx * wy(j + 1);
    nh = get(io.h_in, (int64_t)R.Lx * wy(j + 3));
    nu = get(io.ux_in, r1);
    nv = get(io.uy_in, r1);
    if (io.kappa) nk = get(io.kappa, (int64_t)R.Lx * wy(j + 2));
  }

  // from h's rows y - 1, y, y + 1
  __device__ __forceinline__ T pressure(const R3& a, const R3& b, const R3& d, T kap) const {
    const T hip = b.m, him = b.p, hjp = a.v, hjm = d.v, h = b.v;
    const T hipjp = a.m, himjp = a.p, himjm = d.p, hipjm = d.m;
    if constexpr (F32) {
#pragma clang fp contract(fast)
      const float L = (2.0f / 3.0f) * (((hjp + hip) + him) + hjm) +
                      (1.0f / 6.0f) * (((hipjp + himjp) + himjm) + hipjm) - (10.0f / 3.0f) * h;
      return disjoining_f(K32, h, kap, io.kappa != nullptr) - K32.gamma * L;
    } else {
      const T L = (T(2.0 / 3.0) * (((hjp + hip) + him) + hjm) +
                   T(1.0 / 6.0) * (((hipjp + himjp) + himjm) + hipjm)) -
                  T(10.0 / 3.0) * h;
      const T q = Recip<false>(h + sp.hcrit).div(sp.hmin);
      const T p0 = -sp.gamma * (kap * powlaw(q, sp.n, sp.m, sp.powmode));
      return p0 - sp.gamma * L;
    }
  }

  // the nine post-collision populations from p's rows y - 1, y, y + 1
  __device__ __forceinline__ void collide(const R3& a, const R3& b, const R3& d, T h, T u, T v,
                                          uint32_t wa, uint32_t wb, P9& F) const {
    const T fip = b.m, fim = b.p, fjp = a.v, fjm = d.v;
    const T fipjp = a.m, fimjp = a.p, fimjm = d.p, fipjm = d.m;
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
        float z0, z1;
        box_muller_f32(wa, wb, &z0, &z1);
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
      F.f[0] = fe[0];
      F.f[1] = fe[1] + c3 * Fx;
      F.f[2] = fe[2] + c3 * Fy;
      F.f[3] = fe[3] - c3 * Fx;
      F.f[4] = fe[4] - c3 * Fy;
      F.f[5] = fe[5] + c24 * (Fx + Fy);
      F.f[6] = fe[6] + c24 * (Fy - Fx);
      F.f[7] = fe[7] - c24 * (Fx + Fy);
      F.f[8] = fe[8] + c24 * (Fx - Fy);
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
        box_muller(u32(wa), u32(wb), &z0, &z1);
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
        if constexpr (GRAV) f = feq_k<T>(k, h, u, v, usq, c56g, g0);
        else f = feq_k0<T>(k, h, u, v, usq);
        F.f[k] = k > 0 ? f + force_term<T>(k, Fx, Fy) : f;
      }
    }
  }

  // output row j; the rows rotate roles between calls: on entry (hN, h1, h2) = h(j .. j+2),
  // (pN, p0, p1) = p(j-1 .. j+1), (fN, fm, f0) = (free, populations of rows j-1, j)
  __device__ __forceinline__ void row(int j, R3& hN, R3& h1, R3& h2, R3& pN, R3& p0, R3& p1,
                                      P9& fN, P9& fm, P9& f0) {
    if constexpr (SER) {
      if (j >= y0 && out) {
        double hv = (double)hN.v;
        if constexpr (F32) hv = (double)K32.href + hv;
        lmax = hv > lmax ? hv : lmax;
        lmin = hv < lmin ? hv : lmin;
        cnt += hv > sp.wet_thresh ? 1u : 0u;
      }
    }
    hN.v = nh;  // h(j + 3)
    const T u = nu, v = nv, kap = io.kappa ? nk : (F32 ? (T)K32.kap : (T)sp.kappa);
    if (j < jlast) prefetch(j + 1);
    hN.edges();
    pN.v = pressure(h1, h2, hN, kap);  // p(j + 2)
    pN.edges();
    if (j >= y0 - 2) {
      uint32_t wa = 0, wb = 0;
      if constexpr (TH) {
        // one Philox call per vertical node pair (x, 2m), (x, 2m + 1)
        const int rw = wy(j + 1);
        if ((rw & 1) == 0 || j == y0 - 2) {
          uint32_t w[4];
          philox_ctr(sp.seed, R.step, gx + (uint32_t)R.Lx * (uint32_t)(rw >> 1), kTagThermal, w);
          wa = (rw & 1) ? w[2] : w[0];
          wb = (rw & 1) ? w[3] : w[1];
          w2 = w[2];
          w3 = w[3];
        } else {
          wa = w2;
          wb = w3;
        }
      }
      collide(p0, p1, pN, h1.v, u, v, wa, wb, fN);
    }
    if (j >= y0) {
      // pull-stream f_k(x, j) = fo_k(x - c_k) and moments
      T g[kQ];
      g[0] = f0.f[0];
      g[1] = below(f0.f[1]);
      g[2] = fm.f[2];
      g[3] = above(f0.f[3]);
      g[4] = fN.f[4];
      g[5] = below(fm.f[5]);
      g[6] = above(fm.f[6]);
      g[7] = above(fN.f[7]);
      g[8] = below(fN.f[8]);
      if (out) {
        T s = g[0];
#pragma unroll
        for (int k = 1; k < kQ; ++k) s = s + g[k];
        const T mx = ((((g[1] - g[3]) + g[5]) - g[6]) - g[7]) + g[8];
        const T my = ((((g[2] - g[4]) + g[5]) + g[6]) - g[7]) - g[8];
        T un, vn;
        if constexpr (F32) {
          const float ih = __builtin_amdgcn_rcpf(K32.href + s);
          un = mx * ih;
          vn = my * ih;
        } else {
          const Recip<> ih(s);
          un = ih.div(mx);
          vn = ih.div(my);
        }
        const int64_t r = (int64_t)R.Lx * j;
        put(io.h_out, r, s);
        put(io.ux_out, r, un);
        put(io.uy_out, r, vn);
        if constexpr (WF) {
#pragma unroll
          for (int k = 0; k < kQ; ++k) put(io.f_out + k * R.fstride, r, g[k]);
          put(io.p_out, r, p0.v);
        }
      }
    }
  }

  __device__ __forceinline__ void run(int strip, int sg) {
    const int lane = threadIdx.x & 63;
    const int xc = strip * kMarchOut - 3 + lane;  // unwrapped
    y0 = sg * R.seg;
    jlast = min(y0 + R.seg, R.Ly) - 1;
    gx = (uint32_t)wrap1(xc, R.Lx);
    off = (uint32_t)sizeof(T) * gx;
    out = lane >= 3 && lane < 3 + kMarchOut && xc < R.Lx;
    lmax = -__builtin_inf();
    lmin = __builtin_inf();
    cnt = 0;
    R3 hA{}, hB{}, hC{}, pA{}, pB{}, pC{};
    P9 fA{}, fB{}, fC{};
    hB.v = get(io.h_in, (int64_t)R.Lx * wy(y0 - 3));
    hC.v = get(io.h_in, (int64_t)R.Lx * wy(y0 - 2));
    prefetch(y0 - 4);
    hB.edges();
    hC.edges();
    int j = y0 - 4;
#pragma unroll 1
    for (; j + 2 <= jlast; j += 3) {
      row(j, hA, hB, hC, pA, pB, pC, fA, fB, fC);
      row(j + 1, hB, hC, hA, pB, pC, pA, fB, fC, fA);
      row(j + 2, hC, hA, hB, pC, pA, pB, fC, fA, fB);
    }
    if (j <= jlast) row(j, hA, hB, hC, pA, pB, pC, fA, fB, fC);
    if (j + 1 <= jlast) row(j + 1, hB, hC, hA, pB, pC, pA, fB, fC, fA);
    if constexpr (SER) {
      unsigned long long kmax = dkey(lmax), kmin = dkey(lmin);
      for (int o = 32; o > 0; o >>= 1) {
        const unsigned long long a = __shfl_xor(kmax, o), b = __shfl_xor(kmin, o);
        kmax = a > kmax ? a : kmax;
        kmin = b < kmin ? b : kmin;
        cnt += __shfl_xor(cnt, o);
      }
      if (lane == 0) R.ser.add(0, kmax, kmin, cnt);
    }
  }
};

// (Holding the FP64 step with noise to 128 registers, for four waves per SIMD
// instead of three, made it spill: 70 against 63 us at 2000 x 1500.)
template <typename T, bool TH, bool WF, bool GRAV, bool SER>
__global__ __launch_bounds__(64) void k_march(StepIO<T> io, StepParams sp, F32K K32, MarchRun R) {
  // each XCD (blocks go round them) takes a contiguous share of the items,
  // segment-major, so that neighbouring strips share its L2; odd steps take
  // the share backwards
  const int xcd = blockIdx.x & 7, q = blockIdx.x >> 3;
  const int item = xcd * R.chunk + ((R.step & 1) ? R.chunk - 1 - q : q);
  if (item >= R.items) return;
  March<T, TH, WF, GRAV, SER> m{io, sp, K32, R};
  const int sg = item / R.nstrips;
  m.run(item - sg * R.nstrips, sg);
}

}  // namespace

template <typename T>
void launch_march(const StepIO<T>& io, const StepParams& sp, StepSeries ser, uint64_t step,
                  bool write_f, int Lx, int Ly, int64_t fstride, Enc enc, int seg, hipStream_t s) {
  const F32K K32 = make_f32k(sp, enc);
  MarchRun R{Lx, Ly, (Lx - 1) / kMarchOut + 1, seg, 0, 0, fstride, step, ser};
  R.items = R.nstrips * ((Ly - 1) / seg + 1);
  R.chunk = (R.items - 1) / 8 + 1;
  const dim3 grid(8 * R.chunk), block(64);
#define SW_S(TH, WF, GR, SE) \
  hipLaunchKernelGGL((k_march<T, TH, WF, GR, SE>), grid, block, 0, s, io, sp, K32, R)
#define SW_W(TH, WF, GR)               \
  do {                                 \
    if (ser.base) SW_S(TH, WF, GR, true); \
    else SW_S(TH, WF, GR, false);      \
  } while (0)
#define SW_G(TH, WF)                         \
  do {                                       \
    if (sp.g != 0.0) SW_W(TH, WF, true);     \
    else SW_W(TH, WF, false);                \
  } while (0)
  if constexpr (sizeof(T) == 4) {
    if (write_f) {
      if (sp.thermal) SW_G(true, true);
      else SW_G(false, true);
      return;
    }
  }
  if (sp.thermal) SW_G(true, false);
  else SW_G(false, false);
#undef SW_G
#undef SW_W
#undef SW_S
}

constexpr int64_t kMarchShort = 16;

// What a step costs: fixed + row us for each row that a wave computes (its
// segment and `lead` of start-up), times the waves n that share a SIMD, or
// about `alone` while fewer leave it waiting on a row's chain of operations
// (joined smoothly).  Up to six waves n is the fullest SIMD's count, beyond it
// the average and a half.  Fitted to films of 512 x 512 to 4096 x 4096 and
// segments of 3 to 30 rows, 3-6 % rms.  [double, noise]
struct MarchCost {
  double fixed, row, lead, alone;
};
constexpr MarchCost kMarchCost[2][2] = {{{3.5, 0.33, 1.0, 1.7}, {4.5, 0.42, 1.1, 1.5}},
                                        {{2.8, 0.59, 1.7, 1.3}, {4.7, 1.01, 1.7, 1.3}}};

// The segment with the smallest modelled time per step, if that is less than
// the other path's: with several steps per launch the one modelled there
// (without noise, which scales both alike), in tiles that or, with noise,
// 7.5 us and 3.3 us per round of 64 x 8 tiles over the CUs (FP64), 8.6 and
// 1.25, or 5 and 2.3 beyond four, of 64 x 16 (FP32).  Measured, us per step
// without / with noise, other path -> strips: FP64 512² 8.5 -> 9.2 / 12.2 ->
// 13.9, 700 x 640 13.3 -> 11.3 / 20.2 -> 18.8, 850² 20.7 -> 14.0 / 28.8 ->
// 23.3, 1024² 23.5 -> 18.3 / 34.2 -> 30.1; FP32 700 x 640 9.1 -> 7.9 / 10.9 ->
// 9.7, 850² 11.9 -> 9.9 / 13.0 -> 12.2, 1024² 11.9 -> 11.5 / 13.5 -> 15.0 (four
// tiles on every CU), 4000 x 300 15.2 -> 12.1 / 17.1 -> 15.5.
//
// An FP32 film of 4 M nodes and more whose rows start on half a line writes f
// and p in tiles in much less time (us, strips / tiles: 2048² 91 / 68, 16000 x
// 1000 365 / 208, 4096² 368 / 206, 6000² 799 / 477), which a loop makes up for
// after 3 to 16 steps without f and p (2048² 26.8 / 35.6, with noise 36.0 /
// 39.0; 4096² 103 / 116, 123 / 132; 8192² 422 / 448, 442 / 510): loops of up
// to kMarchShort steps stay with the tiles.
//
// Large FP64 films take four waves per SIMD while that gives segments of up to
// 32 rows, and six beyond: 2500 x 2501 77 us with 28 rows (four), 82 with the
// 18 of the model; 4096 x 4096 210 with 48 (six), 214 with 24.
int march_segment(int Lx, int Ly, bool f64, bool noise, int64_t nsteps, const MultiShape& other) {
  if (Lx < 64 || Ly < 8) return 0;
  if (!f64 && nsteps <= kMarchShort && Lx % 16 == 0 && (int64_t)Lx * Ly >= 4000000) return 0;
  const int64_t cus = device_cus(), simds = 4 * cus;
  const int64_t strips = (Lx - 1) / kMarchOut + 1, rows = strips * Ly;
  const int64_t four = (rows - 1) / (4 * simds) + 1, six = (rows - 1) / (6 * simds) + 1;
  if (f64 && four > 16) return (int)(four > 32 ? six : four);
  double least = other.us;
  const bool cn = noise && other.geom < 0;
  if (cn) {
    const int64_t tiles = (int64_t)((Lx - 1) / 64 + 1) * ((Ly - 1) / (f64 ? 8 : 16) + 1);
    const double r = (double)((tiles - 1) / cus + 1);
    least = f64 ? 7.5 + 3.3 * r : r <= 4.0 ? 8.6 + 1.25 * r : 5.0 + 2.3 * r;
  }
  const MarchCost& c = kMarchCost[f64][cn];
  const double a2 = c.alone * c.alone, a4 = a2 * a2;
  int best = 0;
  for (int seg = 3; seg <= 64; ++seg) {
    const int64_t items = strips * ((Ly - 1) / seg + 1);
    const double n = items <= 6 * simds ? (double)((items - 1) / simds + 1)
                                        : (double)items / (double)simds + 0.5;
    const double t = c.fixed + c.row * (seg + c.lead) * sqrt(sqrt(n * n * n * n + a4));
    if (t < least) {
      least = t;
      best = seg;
    }
  }
  return best;
}

template void launch_march<double>(const StepIO<double>&, const StepParams&, StepSeries, uint64_t,
                                   bool, int, int, int64_t, Enc, int, hipStream_t);
template void launch_march<float>(const StepIO<float>&, const StepParams&, StepSeries, uint64_t,
                                  bool, int, int, int64_t, Enc, int, hipStream_t);

}  // namespace swalbe
