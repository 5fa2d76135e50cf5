// nep_math.hpp -- device mathematics shared by the force kernels: cutoff,
// Chebyshev basis, spherical harmonics, the ZBL pair and tanh.
#pragma once

#include <type_traits>

#include "device_common.hpp"

namespace dmgx {

// The angular constants as compile-time values: every use below sits in an
// unrolled loop, so a coefficient is a literal of the instruction (a factor of
// one or a missing power costs nothing, and no register holds the table).
constexpr AngularConstants kAng = derive_angular_constants();

// cosine cutoff (nep_utilities.cuh:317-342).  cos and sin of pi d/rc come
// from the hardware sine/cosine (v_sin_f32 / v_cos_f32), whose argument is in
// revolutions: 0.5 d/rc lies in [0, 0.5), far inside their [-256, 256]
// domain, with absolute errors near 1e-7.
__device__ __forceinline__ void cutoff_fc(float rc, float rcinv, float d, float& fc)
{
  fc = d < rc ? 0.5f * __builtin_amdgcn_cosf(0.5f * d * rcinv) + 0.5f : 0.0f;
}
__device__ __forceinline__ void cutoff_fc_fcp(float rc, float rcinv, float d, float& fc, float& fcp)
{
  if (d < rc) {
    const float rev = 0.5f * d * rcinv;
    const float sn = __builtin_amdgcn_sinf(rev), cs = __builtin_amdgcn_cosf(rev);
    fc = 0.5f * cs + 0.5f;
    fcp = -1.57079633f * sn * rcinv;
  } else {
    fc = 0.0f;
    fcp = 0.0f;
  }
}

// Chebyshev radial basis f_k = (T_k(x)+1)/2 fc, x = 2(d/rc-1)^2-1; entries
// k >= kn are zero
template <int K>
__device__ __forceinline__ void cheb(int kn, float rcinv, float d, float fc, float* f)
{
  const float t = d * rcinv - 1.0f;
  const float x = 2.0f * t * t - 1.0f;
  const float hfc = 0.5f * fc;
  float tm2 = 1.0f, tm1 = x;
  f[0] = fc;
  if (K > 1) f[1] = (x + 1.0f) * hfc;
#pragma unroll
  for (int k = 2; k < K; ++k) {
    const float tk = 2.0f * x * tm1 - tm2;
    tm2 = tm1;
    tm1 = tk;
    f[k] = k < kn ? (tk + 1.0f) * hfc : 0.0f;
  }
}

// scaled polynomials t_k = h T_k(x), h = fc/2: the basis is f_k = t_k + t_0
template <int K>
__device__ __forceinline__ void cheb_scaled(float rcinv, float d, float h, float* t)
{
  const float u = d * rcinv - 1.0f;
  const float x = 2.0f * u * u - 1.0f, x2 = 2.0f * x;
  t[0] = h;
  if (K > 1) t[1] = x * h;
#pragma unroll
  for (int k = 2; k < K; ++k) t[k] = x2 * t[k - 1] - t[k - 2];
}

// basis and d/dd (T_k' = k U_{k-1})
template <int K>
__device__ __forceinline__ void cheb_d(int kn, float rcinv, float d, float fc, float fcp, float* f, float* fp)
{
  const float t = d * rcinv - 1.0f;
  const float x = 2.0f * t * t - 1.0f;
  const float dx = 4.0f * t * rcinv;  // dx/dd
  f[0] = fc;
  fp[0] = fcp;
  float tm2 = 1.0f, tm1 = x, um2 = 1.0f, um1 = 2.0f * x;
  if (K > 1) {
    const float v = 0.5f * (x + 1.0f);
    f[1] = v * fc;
    fp[1] = 0.5f * dx * fc + v * fcp;
  }
#pragma unroll
  for (int k = 2; k < K; ++k) {
    const float tk = 2.0f * x * tm1 - tm2;
    const float v = 0.5f * (tk + 1.0f);
    const float der = 0.5f * k * um1 * dx;  // (T_k'/2) dx/dd, T_k' = k U_{k-1}
    f[k] = k < kn ? v * fc : 0.0f;
    fp[k] = k < kn ? der * fc + v * fcp : 0.0f;
    tm2 = tm1;
    tm1 = tk;
    const float uk = 2.0f * x * um1 - um2;
    um2 = um1;
    um1 = uk;
  }
}

// Z_{L,m}(z) from the powers of z, and its derivative
template <int L, int M, class Pow>
__device__ __forceinline__ float harmonic_z(const Pow& zp)
{
  constexpr int k0 = (L - M) & 1;
  float Z = k0 == 0 ? kAng.zc[L][M][0] : kAng.zc[L][M][1] * zp[1];
#pragma unroll
  for (int k = k0 + 2; k <= L - M; k += 2) Z += kAng.zc[L][M][k] * zp[k];
  return Z;
}
template <int L, int M, class Pow>
__device__ __forceinline__ float harmonic_dz(const Pow& zp)
{
  constexpr int k0 = ((L - M) & 1) ? 1 : 2;
  if (k0 > L - M) return 0.0f;
  float dZ = kAng.zc[L][M][k0] * (float)k0 * zp[k0 - 1];
#pragma unroll
  for (int k = k0 + 2; k <= L - M; k += 2) dZ += kAng.zc[L][M][k] * (float)k * zp[k - 1];
  return dZ;
}

// f(L) for L = first..last with L a compile-time constant
template <int L, int LAST, class F>
__device__ __forceinline__ void static_for(F&& f)
{
  if constexpr (L <= LAST) {
    f(std::integral_constant<int, L>{});
    static_for<L + 1, LAST>(f);
  }
}

// powers of z = u_z and the real and imaginary parts of (u_x + i u_y)^m
template <int LM>
struct DirectionPowers {
  float zp[LM + 1], re[LM + 1], im[LM + 1];
  __device__ __forceinline__ DirectionPowers(float ux, float uy, float uz)
  {
    zp[0] = 1.0f;
    re[0] = 1.0f;
    im[0] = 0.0f;
    zp[1] = uz;
    re[1] = ux;
    im[1] = uy;
#pragma unroll
    for (int k = 2; k <= LM; ++k) {
      zp[k] = zp[k - 1] * uz;
      re[k] = re[k - 1] * ux - im[k - 1] * uy;
      im[k] = re[k - 1] * uy + im[k - 1] * ux;
    }
  }
};

// real solid harmonics Y_{L,m}(u), L=1..LM, packed at L*L-1 (+2m-1 re, +2m im)
template <int LM>
__device__ __forceinline__ void harmonics(float ux, float uy, float uz, float* Y)
{
  const DirectionPowers<LM> p(ux, uy, uz);
  static_for<1, LM>([&](auto l) {
    constexpr int L = decltype(l)::value, b = L * L - 1;
    Y[b] = harmonic_z<L, 0>(p.zp);
    static_for<1, L>([&](auto mm) {
      constexpr int M = decltype(mm)::value;
      const float Z = harmonic_z<L, M>(p.zp);
      Y[b + 2 * M - 1] = Z * p.re[M];
      Y[b + 2 * M] = Z * p.im[M];
    });
  });
}

// x = tanh(v) and s = 1 - tanh(v)^2 from the hardware exp2 and reciprocal, with
// r = 1 / (e^{2|v|} + 1): |x| = 1 - 2 r and s = 4 e^{2|v|} r^2 above |v| = 0.6
// (the second free of the cancellation in 1 - x^2), an odd polynomial (a
// minimax fit of the relative error, below 2 ulp) below it.  No branches.  The
// library's tanh is about twice as long.  The clamp is the minimum that passes
// NaN on (one v_minimum3_f32; fminf would return 20 and make it +-1): a NaN
// descriptor, of two atoms at the same place, stays one in the energy.
__device__ __forceinline__ void tanh_sech2(float v, float& x, float& s)
{
  const float av = __builtin_elementwise_minimum(fabsf(v), 20.0f), z = v * v;
  const float e = __builtin_amdgcn_exp2f(2.88539008f * av), e1 = e + 1.0f;
  float r = __builtin_amdgcn_rcpf(e1);
  r = fmaf(r, fmaf(-e1, r, 1.0f), r);
  float p = -0.00589515547f;
  p = fmaf(p, z, 0.0207959693f);
  p = fmaf(p, z, -0.0537838295f);
  p = fmaf(p, z, 0.133319241f);
  p = fmaf(p, z, -0.333332980f);
  const bool small = av < 0.6f;
  x = small ? fmaf(v * z, p, v) : copysignf(fmaf(-2.0f, r, 1.0f), v);
  s = small ? fmaf(-x, x, 1.0f) : 4.0f * e * r * r;
}

// Screened-Coulomb ZBL pair energy f(d) and df/dd with the cosine switch
// between r_in and r_out (nep_utilities.cuh:347-433); zp is one pair's
// {1/a, Zi Zj K_C, r_in, r_out, (c_k, d_k) x4} record.
__device__ __forceinline__ void zbl_pair(const float* __restrict__ zp, float d, float dinv, float& f, float& fp)
{
  const float x = d * zp[0];
  float phi = 0.0f, dphi = 0.0f;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const float t = zp[4 + 2 * k] * expf(-zp[5 + 2 * k] * x);
    phi += t;
    dphi -= zp[5 + 2 * k] * t;
  }
  const float vv = zp[1] * phi * dinv;
  const float vp = zp[1] * dphi * zp[0] * dinv - vv * dinv;
  const float r1 = zp[2], r2 = zp[3];
  float fc = 0.0f, fcp = 0.0f;
  if (d < r1) {
    fc = 1.0f;
  } else if (d < r2) {
    const float wv = 3.14159265f / (r2 - r1);
    float sn, cs;
    sincosf(wv * (d - r1), &sn, &cs);
    fc = 0.5f * cs + 0.5f;
    fcp = -0.5f * wv * sn;
  }
  f = vv * fc;
  fp = vp * fc + vv * fcp;
}

// Loads the first kp floats of a 16-byte aligned row as float4s into out[0..KP)
// (kp <= KP, both multiples of 4); entries past kp are left as they are.
template <int KP>
__device__ __forceinline__ void load_row4(const float* __restrict__ row, int kp, float* out)
{
  const float4* q = reinterpret_cast<const float4*>(row);
#pragma unroll
  for (int c = 0; c < KP / 4; ++c) {
    if (4 * c < kp) {
      const float4 t = q[c];
      out[4 * c] = t.x;
      out[4 * c + 1] = t.y;
      out[4 * c + 2] = t.z;
      out[4 * c + 3] = t.w;
    }
  }
}

// sum of v over the P consecutive lanes of a lane group (every lane gets the
// same bits: each stage adds two partners that hold each other's value), with
// the lane permutations of the DPP adds (one instruction per stage)
template <int CTRL>
__device__ __forceinline__ float dpp_move(float v)
{
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xf, 0xf, true));
}
template <int CTRL>
__device__ __forceinline__ double dpp_move(double v)
{
  return __hiloint2double(__builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xf, 0xf, true),
                          __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xf, 0xf, true));
}
template <int CTRL>
__device__ __forceinline__ int dpp_move(int v)
{
  return __builtin_amdgcn_mov_dpp(v, CTRL, 0xf, 0xf, true);
}
template <int CTRL>
__device__ __forceinline__ uint64_t dpp_move(uint64_t v)
{
  return (uint64_t)(uint32_t)dpp_move<CTRL>((int)(v >> 32)) << 32 | (uint32_t)dpp_move<CTRL>((int)v);
}
template <int P, class V>
__device__ __forceinline__ V group_sum(V v)
{
  static_assert(P == 1 || P == 4 || P == 8 || P == 16, "lane groups of 4, 8 or 16");
  if (P >= 4) {
    v += dpp_move<0xB1>(v);  // quad_perm [1,0,3,2]
    v += dpp_move<0x4E>(v);  // quad_perm [2,3,0,1]
  }
  if (P >= 8) v += dpp_move<0x141>(v);   // row_half_mirror
  if (P >= 16) v += dpp_move<0x140>(v);  // row_mirror
  return v;
}

// multi-type models with at most this many types keep their coefficient
// blocks (descriptor) and adjoint rows (gather) in LDS
constexpr int kTypesLds = 4;

// orders this wavefront's LDS writes before its later LDS reads (each
// wavefront works in its own LDS region, so no workgroup barrier is needed)
__device__ __forceinline__ void wave_lds_sync()
{
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

}  // namespace dmgx
