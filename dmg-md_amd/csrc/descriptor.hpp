// descriptor.hpp -- the fused descriptor + ANN + adjoint + angular partial
// force kernel of the NEP step and its launches.  The instances are compiled
// in groups (descriptor_instances.hip); descriptor.hip picks one per model.
#pragma once

#include <hip/hip_ext.h>

#include "nep_math.hpp"

namespace dmgx {

// the kernel's workgroup (256: three workgroups per CU by LDS; 512, which
// would allow four wavefronts per SIMD, measured no faster)
constexpr int kDescBlock = 256;

// ANN modes of the descriptor kernel
enum : int { kAnnValu = 0, kAnnMfma32 = 1, kAnnMfmaBf16 = 2, kAnnMfmaSplit = 3 };

// multi-type models with at most this many types run their ANN on the
// matrix cores: every type's weights staged in LDS, one GEMM pass per type
// present in the wavefront, each atom taking the pass of its own type
constexpr int kTypesMfma = 2;

template <int NR, int KR, int NA, int KA, int LM, bool Q222, bool Q1111, bool ONE, bool EXACT, int ANN = kAnnValu,
          bool CL = false>
struct Cfg {
  static constexpr int nr = NR, kr = KR, na = NA, ka = KA, lm = LM, ann = ANN;
  static constexpr bool q222 = Q222, q1111 = Q1111, one = ONE, exact = EXACT;
  static constexpr bool cl = CL && EXACT && !ONE;  // coefficient blocks in LDS (T <= kTypesLds)
  // type pairs of the LDS tables: every pair of up to kMaxTypes types, or
  // the types an LDS-table instance serves (kTypesMfma with the matrix-core
  // ANN, which stages every type's weights too)
  static constexpr int ltypes = !cl ? kMaxTypes : (ANN != kAnnValu ? kTypesMfma : kTypesLds);
  static constexpr int nabc = (LM + 1) * (LM + 1) - 1;
  static constexpr int numl = LM + (Q222 ? 1 : 0) + (Q1111 ? 1 : 0);
  static constexpr int dim = NR + NA * numl;
  // FP32 matrix-core ANN with its operands and results in registers
  // (ann_mfma_rows), where they fit beside the angular moments in the 256
  // registers that leave two wavefronts per SIMD; through LDS (ann_mfma) else
  static constexpr bool ann_rows =
      ANN == kAnnMfma32 && ONE && EXACT && NA * nabc + 4 * ((dim + 3) / 4) + 16 * ((dim + 15) / 16) <= 216;
};

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));

// float -> bfloat16, round to nearest even (inputs are finite)
__device__ __forceinline__ short to_bf16(float x)
{
  unsigned u = __float_as_uint(x);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (short)(u >> 16);
}

// LDS floats per wavefront of the matrix-core ANN: 64 rows of an odd
// stride, then 64 energies
template <int DMAX>
constexpr int ann_lds_floats() { return 64 * (DMAX | 1) + 128; }

// ANN of the 64 atoms of a wavefront on the matrix cores (single-type
// model, H <= 64).  Lane l holds atom l's scaled descriptor q[0..D).
//   GEMM 1: Z^T[h][atom] = sum_d W0[h][d] Q[atom][d]   (A = W0, B = Q^T)
//   x = tanh(Z - b0), E = sum_h w1 x, G = w1 (1 - x^2)
//   GEMM 2: Fp[atom][d] = sum_h G[atom][h] W0[h][d]     (A = G, B = W0)
// With the 16x16 output layout (lane l, register r) -> (row 4(l/16)+r,
// column l%16), the GEMM-1 accumulator of lane l holds atom 16nt + l%16 at
// hidden units 16mt + 4(l/16) + r; ordering GEMM 2's contraction index as
// (mt, r) makes those registers its A operand as they are.  Fp rows and the
// energies go back to their lanes through LDS.  BF16 rounds Q, W0 and G to
// bfloat16 (16x16x16 bf16 MFMA, FP32 accumulation); FP32 uses the 16x16x4
// FP32 MFMA (exact products).
// LDS copy of one type's ANN weights for the matrix-core path: W0 rows
// padded to 64 hidden units with an odd row stride (no bank conflicts), then
// b0 and w1 (zero past H)
template <int DMAX>
constexpr int ann_w_stride() { return DMAX | 1; }
// floats of W0 rows: 64 x WS floats, or with SPLIT three bfloat16 parts of
// 64 x WS shorts each (96 x WS floats); then b0 and w1
template <int DMAX, bool SPLIT = false>
constexpr int ann_w_floats() { return (SPLIT ? 96 : 64) * ann_w_stride<DMAX>() + 128; }

// bfloat16 -> float (exact)
__device__ __forceinline__ float from_bf16(short b) { return __uint_as_float(((unsigned)(unsigned short)b) << 16); }

// x = hi + mid + lo + r with hi = bf16(x), mid = bf16(x - hi),
// lo = bf16(x - hi - mid) (each difference exact in FP32), |r| <= 2^-27 |x|
struct Bf16Split {
  short hi, mid, lo;
};
__device__ __forceinline__ Bf16Split split_bf16(float x)
{
  const short hi = to_bf16(x);
  const float r1 = x - from_bf16(hi);
  const short mid = to_bf16(r1);
  return Bf16Split{hi, mid, to_bf16(r1 - from_bf16(mid))};
}

// SPLIT: W0 is stored as its three bfloat16 parts, shorts [64][WS] each
// (hi, then mid, then lo), in place of the float rows
template <int DMAX, bool SPLIT = false>
__device__ __forceinline__ void stage_ann_weights(const DevModel& m, int D, float* __restrict__ ws, int t = 0)
{
  constexpr int WS = ann_w_stride<DMAX>();
  const int H = m.H;
  const float* __restrict__ w0 = m.w0 + (size_t)t * H * D;
  const float* __restrict__ b0 = m.b0 + (size_t)t * H;
  const float* __restrict__ w1 = m.w1 + (size_t)t * H;
  short* __restrict__ whl = reinterpret_cast<short*>(ws);
  for (int k = threadIdx.x; k < 64 * WS; k += blockDim.x) {
    const int h = k / WS, d = k % WS;
    const float x = (h < H && d < D) ? w0[h * D + d] : 0.0f;
    if (SPLIT) {
      const Bf16Split p = split_bf16(x);
      whl[k] = p.hi;
      whl[64 * WS + k] = p.mid;
      whl[128 * WS + k] = p.lo;
    } else {
      ws[k] = x;
    }
  }
  for (int h = threadIdx.x; h < 64; h += blockDim.x) {
    constexpr int bo = (SPLIT ? 96 : 64) * WS;
    ws[bo + h] = h < H ? b0[h] : 0.0f;
    ws[bo + 64 + h] = h < H ? w1[h] : 0.0f;
  }
}


// MT: multi-type (ti is the lane's type, T the number of types <=
// kTypesMfma, ws holds the types' weight blocks one after another): per
// type present in the wavefront one pass over the hidden tiles whose
// activation gradients and energies count only for atoms of that type.
template <int DMAX, int MODE, bool MT = false>
__device__ __forceinline__ void ann_mfma(const DevModel& m, int D, const float* q, float* Fp, float& E,
                                         float* __restrict__ lds, const float* __restrict__ ws, int ti = 0,
                                         int T = 1)
{
  // MODE kAnnMfma32: FP32 operands (16x16x4 FP32 MFMA, exact products);
  // kAnnMfmaBf16: bfloat16 operands; kAnnMfmaSplit: every operand split
  // into three bfloat16 parts (hi + mid + lo) and each product formed from
  // the six part products of relative size above 2^-24 (hi*hi, hi*mid,
  // mid*hi, mid*mid, hi*lo, lo*hi; 16x16x16 bf16 MFMAs, FP32 accumulation,
  // smallest first): FP32 accuracy from bfloat16 products, the "bf16x6"
  // method of Henry, Tang and Heinecke (ARITH 2019)
  constexpr bool BF16 = MODE == kAnnMfmaBf16;
  constexpr bool X3 = MODE == kAnnMfmaSplit;
  constexpr int DS = DMAX | 1;
  constexpr int DT = (DMAX + 15) / 16;
  const int lane = threadIdx.x & 63, lr = lane & 15, lg = lane >> 4;
  float* Qs = lds;
  float* Es = lds + 64 * DS;
  int* Ts = reinterpret_cast<int*>(lds + 64 * DS + 64);
#pragma unroll
  for (int d = 0; d < DMAX; ++d) Qs[lane * DS + d] = d < D ? q[d] : 0.0f;
  unsigned present = 1u;
  if (MT) {
    Ts[lane] = ti;
    present = 0u;
    for (int t = 0; t < T; ++t)
      if (__any(ti == t)) present |= 1u << t;
  }
  wave_lds_sync();
  const int H = m.H, HT = (H + 15) >> 4;
  constexpr int WS = ann_w_stride<DMAX>();
#pragma unroll 1
  for (int nt = 0; nt < 4; ++nt) {
    const float* qrow = Qs + (16 * nt + lr) * DS;
    // split descriptor operands of this atom tile, reused by every hidden tile
    s16x4 qh[X3 ? DT : 1], qm[X3 ? DT : 1], ql[X3 ? DT : 1];
    if (X3) {
#pragma unroll
      for (int ks = 0; ks < DT; ++ks)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const int d = 16 * ks + 4 * lg + c;
          const Bf16Split p = split_bf16(d < D ? qrow[d] : 0.0f);
          qh[ks][c] = p.hi;
          qm[ks][c] = p.mid;
          ql[ks][c] = p.lo;
        }
    }
    f32x4 facc[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) facc[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    float ep = 0.0f;
    const int at = MT ? Ts[16 * nt + lr] : 0;  // type of this lane's atom in the tile
    // the type loop is unrolled over its compile-time bound: a runtime-bounded
    // loop that skips absent types gave wrong accumulators in GEMM 2 here
    // (forces off by 5% with exact energies), the unrolled form does not
#pragma unroll
    for (int t = 0; t < (MT ? kTypesMfma : 1); ++t) {
      if (t >= T || !((present >> t) & 1u)) continue;
      const bool mine = !MT || at == t;
      // [64][WS] floats (or three [64][WS] bfloat16 parts), zero-padded
      const float* __restrict__ W0 = ws + (size_t)t * ann_w_floats<DMAX, X3>();
      const float* __restrict__ b0 = W0 + (X3 ? 96 : 64) * WS;
      const float* __restrict__ w1 = b0 + 64;
      // one tile of 16 hidden units at a time: GEMM 1, activation, and its
      // share of GEMM 2, so that only one accumulator tile is live
#pragma unroll 1
      for (int mt = 0; mt < HT; ++mt) {
        f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
        const int ha = 16 * mt + lr;
        const short* __restrict__ Wh = reinterpret_cast<const short*>(W0);
        const short* __restrict__ Wm = Wh + 64 * WS;
        const short* __restrict__ Wl = Wh + 128 * WS;
        if (X3) {
#pragma unroll
          for (int ks = 0; ks < DT; ++ks) {
            s16x4 ah, am, al;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
              // columns past the row stride would read the next row or, past
              // the last row, the float biases as bfloat16 pairs (possibly
              // NaN patterns): they hold zeros
              const int d = 16 * ks + 4 * lg + c;
              ah[c] = d < WS ? Wh[ha * WS + d] : (short)0;
              am[c] = d < WS ? Wm[ha * WS + d] : (short)0;
              al[c] = d < WS ? Wl[ha * WS + d] : (short)0;
            }
            acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(al, qh[ks], acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(ah, ql[ks], acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(am, qm[ks], acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(am, qh[ks], acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(ah, qm[ks], acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(ah, qh[ks], acc, 0, 0, 0);
          }
        } else if (!BF16) {
#pragma unroll
          for (int ks = 0; ks < (DMAX + 3) / 4; ++ks) {
            const int d = 4 * ks + lg;
            const float bq = d < D ? qrow[d] : 0.0f;
            const float a = W0[ha * WS + d];
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a, bq, acc, 0, 0, 0);
          }
        } else {
#pragma unroll
          for (int ks = 0; ks < (DMAX + 15) / 16; ++ks) {
            s16x4 bq, a;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
              const int d = 16 * ks + 4 * lg + c;
              bq[c] = to_bf16(d < D ? qrow[d] : 0.0f);
              a[c] = to_bf16(W0[ha * WS + d]);
            }
            acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, bq, acc, 0, 0, 0);
          }
        }
        float G[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int h = 16 * mt + 4 * lg + r;
          G[r] = 0.0f;
          if (h < H && mine) {
            float x, dx;
            tanh_sech2(acc[r] - b0[h], x, dx);
            ep += w1[h] * x;
            G[r] = w1[h] * dx;
          }
        }
        if (X3) {
          s16x4 gh, gm, gl;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const Bf16Split p = split_bf16(G[r]);
            gh[r] = p.hi;
            gm[r] = p.mid;
            gl[r] = p.lo;
          }
#pragma unroll
          for (int dt = 0; dt < DT; ++dt) {
            const int d = 16 * dt + lr;
            s16x4 bh, bm, bl;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
              const int h = 16 * mt + 4 * lg + c;
              bh[c] = d < WS ? Wh[h * WS + d] : (short)0;
              bm[c] = d < WS ? Wm[h * WS + d] : (short)0;
              bl[c] = d < WS ? Wl[h * WS + d] : (short)0;
            }
            facc[dt] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(gl, bh, facc[dt], 0, 0, 0);
            facc[dt] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(gh, bl, facc[dt], 0, 0, 0);
            facc[dt] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(gm, bm, facc[dt], 0, 0, 0);
            facc[dt] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(gm, bh, facc[dt], 0, 0, 0);
            facc[dt] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(gh, bm, facc[dt], 0, 0, 0);
            facc[dt] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(gh, bh, facc[dt], 0, 0, 0);
          }
        } else if (!BF16) {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int h = 16 * mt + 4 * lg + r;
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) {
              const int d = 16 * dt + lr;
              const float bw = W0[h * WS + d];
              facc[dt] = __builtin_amdgcn_mfma_f32_16x16x4f32(G[r], bw, facc[dt], 0, 0, 0);
            }
          }
        } else {
          s16x4 a;
#pragma unroll
          for (int r = 0; r < 4; ++r) a[r] = to_bf16(G[r]);
#pragma unroll
          for (int dt = 0; dt < DT; ++dt) {
            const int d = 16 * dt + lr;
            s16x4 bw;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
              const int h = 16 * mt + 4 * lg + c;
              bw[c] = to_bf16(W0[h * WS + d]);
            }
            facc[dt] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, bw, facc[dt], 0, 0, 0);
          }
        }
      }
    }  // types
    ep += __shfl_xor(ep, 16);
    ep += __shfl_xor(ep, 32);
    if (lg == 0) Es[16 * nt + lr] = ep;
    // this tile's Fp rows replace its (already consumed) Q rows
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int d = 16 * dt + lr;
        if (d < DMAX) Qs[(16 * nt + 4 * lg + r) * DS + d] = facc[dt][r];
      }
  }
  wave_lds_sync();
#pragma unroll
  for (int d = 0; d < DMAX; ++d) Fp[d] = d < D ? Qs[lane * DS + d] : 0.0f;
  E = Es[lane];
}

// 4x4 transposition between four registers and the four 16-lane rows of a
// wavefront: register r of row g becomes register g of row r (four lane-swap
// instructions, no LDS)
__device__ __forceinline__ void swap_rows32(float& a, float& b)
{
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  a = __uint_as_float(r[0]);
  b = __uint_as_float(r[1]);
}
__device__ __forceinline__ void swap_rows16(float& a, float& b)
{
  auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  a = __uint_as_float(r[0]);
  b = __uint_as_float(r[1]);
}
__device__ __forceinline__ void row_transpose(float& a0, float& a1, float& a2, float& a3)
{
  swap_rows32(a0, a2);
  swap_rows32(a1, a3);
  swap_rows16(a0, a1);
  swap_rows16(a2, a3);
}

// The FP32 ANN of a wavefront's 64 atoms on the matrix cores with the
// descriptors and their derivatives in registers (single-type models):
// lane l holds atom l's descriptor q[0..D) and gets its derivatives Fp and
// energy E.  A transposition over the 16-lane rows turns four descriptor
// registers into the operands of the four 16-atom tiles, GEMM 2 is formed
// transposed (Fp^T = W0^T G^T, its operand GEMM 1's accumulator as it is), and
// the same transposition brings its results back, so nothing of an atom goes
// through LDS, and a hidden tile's weights are read from LDS once for all atom
// tiles of a pass (the staged form below keeps 64 (D + 1) floats of LDS per
// wavefront, fences them twice and reads the weights once per atom tile).
// TP atom tiles per pass over the weights: four, or two where the results of
// all four would not fit the registers beside the operands.
template <int D, int TP>
__device__ __forceinline__ void ann_mfma_rows(int H, const float* q, float* Fp, float& E, const float* __restrict__ W0)
{
  constexpr int DK = (D + 3) / 4, DT = (D + 15) / 16, WS = ann_w_stride<D>();
  const int lane = threadIdx.x & 63, lr = lane & 15, lg = lane >> 4;
  const float* __restrict__ b0 = W0 + 64 * WS;
  const float* __restrict__ w1 = b0 + 64;
  float a[4 * DK];
#pragma unroll
  for (int d = 0; d < 4 * DK; ++d) a[d] = d < D ? q[d] : 0.0f;
#pragma unroll
  for (int k = 0; k < DK; ++k) row_transpose(a[4 * k], a[4 * k + 1], a[4 * k + 2], a[4 * k + 3]);
  f32x4 facc[4][DT];
  float e[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    e[t] = 0.0f;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) facc[t][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const int HT = (H + 15) >> 4;
#pragma unroll
  for (int t0 = 0; t0 < 4; t0 += TP) {
#pragma unroll 1
    for (int mt = 0; mt < HT; ++mt) {
      // columns past D meet zero operands (GEMM 1) or give unused rows (GEMM
      // 2); their reads stay inside the weight block
      float wa[DK], wb[4][DT], bias[4], out[4];
#pragma unroll
      for (int k = 0; k < DK; ++k) wa[k] = W0[(16 * mt + lr) * WS + 4 * k + lg];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) wb[r][dt] = W0[(16 * mt + 4 * lg + r) * WS + 16 * dt + lr];
        bias[r] = b0[16 * mt + 4 * lg + r];
        out[r] = w1[16 * mt + 4 * lg + r];
      }
#pragma unroll
      for (int t = t0; t < t0 + TP; ++t) {
        f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < DK; ++k) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(wa[k], a[4 * k + t], acc, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          // hidden units past H have zero weights: no energy, no gradient
          float x, dx;
          tanh_sech2(acc[r] - bias[r], x, dx);
          e[t] += out[r] * x;
          const float g = out[r] * dx;
#pragma unroll
          for (int dt = 0; dt < DT; ++dt)
            facc[t][dt] = __builtin_amdgcn_mfma_f32_16x16x4f32(wb[r][dt], g, facc[t][dt], 0, 0, 0);
        }
      }
    }
  }
  row_transpose(e[0], e[1], e[2], e[3]);
  E = (e[0] + e[1]) + (e[2] + e[3]);
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float f[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) f[t] = facc[t][dt][r];
      row_transpose(f[0], f[1], f[2], f[3]);
#pragma unroll
      for (int t = 0; t < 4; ++t)
        if (16 * dt + 4 * t + r < D) Fp[16 * dt + 4 * t + r] = f[t];
    }
}

// Static LDS of a descriptor instance: pair tables, coefficient blocks, ANN
// weights and the per-wavefront ANN staging.  Instances stay within
// kDescLdsMax per workgroup; where the matrix-core ANN would not, the vector
// ANN runs.
constexpr int kDescLdsMax = 96 * 1024;
template <class C>
constexpr int desc_lds_bytes()
{
  const int pairs = C::ltypes * C::ltypes;
  const int pcut = C::one ? 1 + 2 : 4 * pairs + 4 * pairs;  // float cutoffs, then the FP64 squares
  const int ctab = C::cl ? pairs * (C::nr * C::kr + C::na * C::ka) : 1;
  const int mfma = C::ann != kAnnValu;
  const int annw = mfma ? (C::one ? 1 : kTypesMfma) * ann_w_floats<C::dim, C::ann == kAnnMfmaSplit>() : 1;
  const int annl = mfma && !C::ann_rows ? (kDescBlock / 64) * ann_lds_floats<C::dim>() : 0;
  return 4 * (pcut + ctab + annw + annl);
}

// Wavefronts per SIMD an instance's registers are allocated for.  Two (256
// registers) for the single-type instances with up to kNarrowMoments moments
// (four lanes per atom on 21,952 carbon atoms 63 -> 44 us), and for the
// several-type matrix-core ones whose LDS lets two workgroups share a CU (606
// -> 461 us on 192,000 water atoms, with 84 bytes of spills per lane).  One for
// the wider ones, which would spill hundreds of bytes, for the lane groups of
// several-type models and for the generic instances.
constexpr int kNarrowMoments = 128;
template <class C, int P>
constexpr int desc_waves()
{
  if (!C::exact) return 1;
  if (C::one) return C::na * C::nabc <= kNarrowMoments ? 2 : 1;
  return P == 1 && C::ann == kAnnMfma32 && desc_lds_bytes<C>() <= 80 * 1024 ? 2 : 1;
}

template <int NR, int KR, int NA, int KA, bool Q2, bool Q1, bool ONE, int ANN = kAnnMfma32>
constexpr bool mfma_ann_fits()
{
  // single-type instances reach two wavefronts per SIMD, so they keep two
  // workgroups per CU (64 KiB each); several-type ones hold two wavefronts up to
  // 80 KiB (desc_waves) and, on the matrix cores all the same, one beyond
  return desc_lds_bytes<Cfg<NR, KR, NA, KA, 4, Q2, Q1, ONE, true, ANN, !ONE>>() <=
         (ONE ? 64 * 1024 : kDescLdsMax);
}

// The angular edges' second pass of the generic instance, whose moments (240 or
// 800 a lane) lie in scratch: the basis first and then a function at a time,
// and the adjoint contracted degree by degree, in the order the moments lie
// in.  The form by order of the exact instances, their shared loop for the
// radial terms and their four records in flight cost it registers and code
// without an access less: 110,592 atoms with 10 radial functions 3,040 us
// against 3,876, 32,768 with a basis of 16 1,229 against 1,391, 110,592 at
// order 6 8,031 against 10,471.
template <int NA, int KA>
__device__ __forceinline__ void basis_by_function(int nA, int kA, const float* __restrict__ c, float rcinv, float d,
                                                  float fc, float fcp, float* g, float* gp)
{
  float f[KA], fp[KA];
  cheb_d<KA>(kA, rcinv, d, fc, fcp, f, fp);
#pragma unroll
  for (int n = 0; n < NA; ++n) {
    g[n] = 0.0f;
    gp[n] = 0.0f;
    if (n < nA) {
#pragma unroll
      for (int k = 0; k < KA; ++k)
        if (k < kA) {
          g[n] += c[n * kA + k] * f[k];
          gp[n] += c[n * kA + k] * fp[k];
        }
    }
  }
}
template <int NA, int LM, int NABC>
__device__ __forceinline__ void contract_by_degree(const float (&s)[NA][NABC], const float* g, const float* gp,
                                                   const DirectionPowers<LM>& pw, float& Pr, float& Gx, float& Gy,
                                                   float& Gz)
{
  static_for<1, LM>([&](auto l) {
    constexpr int L = decltype(l)::value, b = L * L - 1;
    float A = 0.0f, B = 0.0f;
#pragma unroll
    for (int n = 0; n < NA; ++n) {
      A += s[n][b] * g[n];
      B += s[n][b] * gp[n];
    }
    Pr += B * harmonic_z<L, 0>(pw.zp);
    Gz += A * harmonic_dz<L, 0>(pw.zp);
    static_for<1, L>([&](auto mm) {
      constexpr int M = decltype(mm)::value, ir = b + 2 * M - 1, ii = ir + 1;
      float Ar = 0.0f, Ai = 0.0f, Br = 0.0f, Bi = 0.0f;
#pragma unroll
      for (int n = 0; n < NA; ++n) {
        Ar += s[n][ir] * g[n];
        Ai += s[n][ii] * g[n];
        Br += s[n][ir] * gp[n];
        Bi += s[n][ii] * gp[n];
      }
      const float Z = harmonic_z<L, M>(pw.zp), dZ = harmonic_dz<L, M>(pw.zp), mz = (float)M * Z;
      Pr += Z * (Br * pw.re[M] + Bi * pw.im[M]);
      Gx += mz * (Ar * pw.re[M - 1] + Ai * pw.im[M - 1]);
      Gy += mz * (Ai * pw.re[M - 1] - Ar * pw.im[M - 1]);
      Gz += dZ * (Ar * pw.re[M] + Ai * pw.im[M]);
    });
  });
}

// What bounds it: vector instruction issue, most of it in the two loops over
// the angular edges (about 240 and 500 instructions per edge and wavefront at
// n_max 4, basis 8, order 4).  The angular coefficients are literals, the
// radial sums take one addition per edge and function (radial_edge below), the
// second loop contracts the adjoint once per order m, and the network's
// activations are branch-free: with the matrix-core ANN above, 228 -> 191 us on
// 256,000 Cu atoms, 713 -> 611 us on 192,000 water atoms and 2.03 -> 1.73 ms on
// a 2.28-million-slot carbon share; with four lanes per atom 45 -> 37 us on
// 4,096 carbon atoms (32 with the registers of two wavefronts, 22 with sixteen
// lanes).  Against 64 bits the other order of the FP32 sums moves the errors by
// a few percent either way (2-norms over six draws of four systems): site
// energies 0.2 to 4% smaller, forces and virials of carbon and Cu 0.2 to 2.7%
// smaller, of BaTiO3 1.5 and 3.6% larger; the short tanh is no part of that (the
// library's in its place: within 1%).  Folding the constant column of c into one
// coefficient would save 16 more additions per edge, but its rounding is common
// to all edges and raised the water model's energy error by a fifth.
//
// CAND: the edges come from the candidate rows (DevWork::split).  edge, vsa
// and eq are w.edge, w.vsa and w.eq, passed as restrict parameters: with
// candidate rows this kernel writes them, and only through them, so the
// model's tables stay provably unmodified (scalar loads).
// P: lanes per atom.  With P > 1 (systems too small to fill the GPU with one
// lane per atom) a group of P lanes shares an atom: each takes every P-th
// edge and every P-th hidden neuron of the (vector-ALU) ANN, and the partial
// sums are combined across the group, so every lane holds the atom's
// descriptor, moments and derivatives.
template <class C, bool CAND, int P = 1>
__global__ __launch_bounds__(kDescBlock, (desc_waves<C, P>())) void k_descriptor(
                                                       DevBox b, DevModel m, int N, int c1, int c2, int nblocks,
                                                       const int* __restrict__ type, double* __restrict__ pe,
                                                       float4* __restrict__ edge, int* __restrict__ vsa,
                                                       short* __restrict__ eq, int accumulate, DevWork w)
{
  constexpr int NR = C::nr, KR = C::kr, NA = C::na, KA = C::ka, LM = C::lm, NABC = C::nabc, DMAX = C::dim;
  static_assert(P == 1 || ((P == 4 || P == 16) && !CAND && C::ann == kAnnValu), "lane groups: the filter's rows, vector ANN");
  const int lr = P == 1 ? 0 : (int)(threadIdx.x & (P - 1));  // lane within the atom's group
  // blocks start at a row tile's first centre, so a wavefront reads whole tiles
  const int i0 = (c1 & ~(kTile - 1)) + xcd_tile(nblocks) * (int)(blockDim.x / P) + (int)(threadIdx.x / P);
  const bool active = i0 >= c1 && i0 < c2;
  // the matrix-core ANN needs every lane of the wavefront: lanes past the
  // range carry an empty row of a valid atom and write nothing
  const int i = active ? i0 : c1;
  // multi-type: per type pair the float cutoffs and their inverses (radial,
  // angular; the FP64 pair mean rounded once) and, with C::cl, the
  // coefficient blocks [pair][n][k] (radial, then angular), staged in LDS
  constexpr int kPairs = C::ltypes * C::ltypes;
  static_assert(desc_lds_bytes<C>() <= kDescLdsMax, "descriptor LDS above its bound per workgroup");
  __shared__ float pcut[C::one ? 1 : 4 * kPairs];
  __shared__ double pcut2[C::one ? 1 : 2 * kPairs];  // FP64 squared pair cutoffs (candidate rows)
  __shared__ float ctab[C::cl ? kPairs * (NR * KR + NA * KA) : 1];
  if (!C::one) {
    const int T = m.T;
    for (int k = threadIdx.x; k < T * T; k += blockDim.x) {
      const int p = k / T, q = k % T;
      const double rrd = (m.rcR[p] + m.rcR[q]) * 0.5, rad = (m.rcA[p] + m.rcA[q]) * 0.5;
      const float rr = (float)rrd, ra = (float)rad;
      pcut[k] = rr;
      pcut[kPairs + k] = 1.0f / rr;
      pcut[2 * kPairs + k] = ra;
      pcut[3 * kPairs + k] = 1.0f / ra;
      pcut2[k] = rrd * rrd;
      pcut2[kPairs + k] = rad * rad;
    }
    if (C::cl) {
      const int nrad = T * T * NR * KR, nang = T * T * NA * KA;
      for (int k = threadIdx.x; k < nrad + nang; k += blockDim.x) ctab[k] = k < nrad ? m.cR[k] : m.cA[k - nrad];
    }
    __syncthreads();
  }
  // candidate rows: the rebuild kernels of this step ran before this launch
  // (the only descriptor launch of the evaluation), which closes the request
  if (CAND && blockIdx.x == 0 && threadIdx.x == 0 && w.flags[kFlagRebuild]) {
    w.flags[kFlagRebuild] = 0;
    w.flags[kFlagRebuildCount] += 1;
  }
  if (C::ann == kAnnValu && !active) return;
  __shared__ float ann_w[C::ann != kAnnValu ? (C::one ? 1 : kTypesMfma) * ann_w_floats<DMAX, C::ann == kAnnMfmaSplit>()
                                           : 1];
  if (C::ann != kAnnValu) {
    // every type's weights (at most kTypesMfma types), staged once per workgroup
    for (int t = 0; t < (C::one ? 1 : m.T); ++t)
      stage_ann_weights<DMAX, C::ann == kAnnMfmaSplit>(
          m, C::exact ? DMAX : m.D, ann_w + t * ann_w_floats<DMAX, C::ann == kAnnMfmaSplit>(), t);
    __syncthreads();
  }
  const int nR = C::exact ? NR : m.nR, nA = C::exact ? NA : m.nA;
  // 3-body order: components L <= Lm, then the 4-/5-body blocks
  const int Lm = C::exact ? LM : m.L;
  const int kR = C::exact ? KR : m.kR, kA = C::exact ? KA : m.kA;
  const bool h222 = C::exact ? C::q222 : (m.has222 != 0);
  const bool h1111 = C::exact ? C::q1111 : (m.has1111 != 0);
  const int D = C::exact ? DMAX : m.D;
  const int T = C::one ? 1 : m.T;
  const int ti = C::one ? 0 : safe_type(type[i], T);
  float rcRf[kMaxTypes], rcAf[kMaxTypes];
  // per-type float cutoffs (the FP64 values rounded once)
  if (C::one) {
    rcRf[0] = (float)m.rcR[0];
    rcAf[0] = (float)m.rcA[0];
  }
  int nr = 0, na = 0;
  if (active && !CAND) {
    nr = w.nr[i];
    na = w.na[i];
  }
  // with candidate rows this kernel writes the angular edges it reads back
  const float4* erow = edge + row_begin(i, w.MR);
  float3* __restrict__ frow = w.f12 + row_begin(i, w.MA);
  float q[DMAX];
#pragma unroll
  for (int d = 0; d < DMAX; ++d) q[d] = 0.0f;

  auto type_of = [&](const float4& r) { return C::one ? 0 : edge_type(w, type, __float_as_int(r.w), T); };

  // ---- radial descriptor: q_n = sum_j sum_k c[ti,tj,n,k] f_k(r_ij),
  // f_k = (T_k(x) + 1) fc / 2.  The scaled polynomials t_k = (fc / 2) T_k are
  // summed per neighbour type (one addition each; f_k = t_k + t_0, so the sums
  // of f_k follow from theirs after the loop) and contracted with the
  // coefficients once per atom (single type: one sum; up to C::ltypes types:
  // one per type); more types contract per edge.
  float Ft[C::cl ? C::ltypes : 1][KR];
#pragma unroll
  for (int t = 0; t < (C::cl ? C::ltypes : 1); ++t)
#pragma unroll
    for (int k = 0; k < KR; ++k) Ft[t][k] = 0.0f;
  // the angular edges' radial terms in the loop over their moments
  constexpr bool kOneLoop = C::exact;
  auto radial_edge = [&](const float d, const int tj) {
    const float rc = C::one ? rcRf[0] : pcut[ti * T + tj];
    const float rcinv = C::one ? 1.0f / rc : pcut[kPairs + ti * T + tj];
    float fc;
    cutoff_fc(rc, rcinv, d, fc);
    if (C::one || C::cl) {
      float f[KR];
      cheb_scaled<KR>(rcinv, d, 0.5f * fc, f);
      if (C::one) {
#pragma unroll
        for (int k = 0; k < KR; ++k) Ft[0][k] += f[k];
      } else {
#pragma unroll
        for (int t = 0; t < C::ltypes; ++t) {
          if (t < T) {
            const float wt = tj == t ? 1.0f : 0.0f;
#pragma unroll
            for (int k = 0; k < KR; ++k) Ft[t][k] = fmaf(wt, f[k], Ft[t][k]);
          }
        }
      }
    } else {
      float f[KR];
      cheb<KR>(kR, rcinv, d, fc, f);
      const float* c = m.cR + (size_t)(ti * T + tj) * nR * kR;
#pragma unroll
      for (int n = 0; n < NR; ++n) {
        if (n < nR) {
          float g = 0.0f;
#pragma unroll
          for (int k = 0; k < KR; ++k)
            if (k < kR) g += c[n * kR + k] * f[k];
          q[n] += g;
        }
      }
    }
  };
  if (!CAND) {
    // radial-only edges, stored from the row's end downward; kAhead records
    // in flight (the work per edge is short).  The angular edges' radial terms
    // are summed in the loop over the angular moments, or here as well.
    constexpr int kAhead = !C::exact ? 8 : P == 1 ? 12 : 3;
    const float4* const first = erow + (size_t)(w.MR - 1) * kTile;
    const int nro = kOneLoop ? nr - na : nr;
    auto record = [&](int e) {
      if (!kOneLoop && e < na) return erow[(size_t)e * kTile];
      return first[-(ptrdiff_t)(kOneLoop ? e : e - na) * kTile];
    };
    float4 ring[kAhead];
#pragma unroll
    for (int u = 0; u < kAhead; ++u)
      ring[u] = u * P + lr < nro ? record(u * P + lr) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    for (int e0 = lr; e0 < nro; e0 += kAhead * P)
#pragma unroll
      for (int u = 0; u < kAhead; ++u) {
        const int e = e0 + u * P;
        if (e >= nro) break;
        const float4 r = ring[u];
        if (e + kAhead * P < nro) ring[u] = record(e + kAhead * P);
        const float d2 = r.x * r.x + r.y * r.y + r.z * r.z;
        radial_edge(d2 * __builtin_amdgcn_rsqf(d2), type_of(r));
      }
  } else {
    // candidate rows: the FP64 minimum-image distance of every candidate
    // (the filter's expressions, so the same edges pass), the radial sum over
    // those within the pair's radial cutoff, and the step's angular edges
    // (in candidate order) with their reverse indices and the candidates'
    // slot status for the gather.  Slot indices are read eight candidates
    // ahead, the packed positions four.
    const int nrc = active ? w.nrc[i] : 0, nac = active ? w.nac[i] : 0;
    const size_t vrow = (size_t)i * w.MV, arow = (size_t)i * w.MA;
    const int* __restrict__ crow = w.cl + vrow;
    float4* ew = edge + row_begin(i, w.MR);
    short* qw = eq + row_begin(i, w.MA);
    const double4 pi = w.xq[i];
    double cr1 = 0.0, ca1 = 0.0;
    if (C::one) {
      const double rr = (m.rcR[0] + m.rcR[0]) * 0.5, ra = (m.rcA[0] + m.rcA[0]) * 0.5;
      cr1 = rr * rr;
      ca1 = ra * ra;
    }
    auto cidx = [&](int e) { return e < nac ? e : w.MV - 1 - (e - nac); };
    constexpr int kSplitAhead = 4;
    int jr[2 * kSplitAhead];
    double4 pr[kSplitAhead];
#pragma unroll
    for (int u = 0; u < 2 * kSplitAhead; ++u) jr[u] = u < nrc ? crow[cidx(u)] : 0;
#pragma unroll
    for (int u = 0; u < kSplitAhead; ++u) pr[u] = u < nrc ? w.xq[jr[u]] : make_double4(0.0, 0.0, 0.0, 0.0);
    int nin = 0;
    for (int e0 = 0; e0 < nrc; e0 += 2 * kSplitAhead)
#pragma unroll
      for (int u = 0; u < 2 * kSplitAhead; ++u) {
        const int e = e0 + u;
        if (e >= nrc) break;
        const int j = jr[u];
        const double4 pj = pr[u % kSplitAhead];
        if (e + kSplitAhead < nrc) pr[u % kSplitAhead] = w.xq[jr[(u + kSplitAhead) % (2 * kSplitAhead)]];
        if (e + 2 * kSplitAhead < nrc) jr[u] = crow[cidx(e + 2 * kSplitAhead)];
        double x = pj.x - pi.x, y = pj.y - pi.y, z = pj.z - pi.z;
        mic(b, x, y, z);
        const double d2 = dist2(x, y, z);
        int tj = 0;
        double cr = cr1, ca = ca1;
        if (!C::one) {
          tj = safe_type((int)__double_as_longlong(pj.w), T);
          cr = pcut2[ti * T + tj];
          ca = pcut2[kPairs + ti * T + tj];
        }
        const bool in_r = d2 < cr;
        const int jo = w.map.owner ? w.map.owner[j] : j;
        const float4 r =
            make_float4((float)x, (float)y, (float)z, __int_as_float(C::one ? jo : edge_word(w.typed, jo, tj)));
        if (e < nac) {
          const bool in_a = in_r && d2 < ca;
          vsa[arow + e] = in_a ? na : -1;
          if (in_a) {
            ew[(size_t)na * kTile] = r;
            qw[(size_t)na * kTile] = (short)w.cq[arow + e];
            ++na;
          }
        }
        if (in_r) {
          ++nin;
          const float rr = r.x * r.x + r.y * r.y + r.z * r.z;
          radial_edge(rr * __builtin_amdgcn_rsqf(rr), tj);
        }
      }
    if (active) {
      w.nr[i] = nin;
      w.na[i] = na;
    }
  }
  // ---- angular moments s[n][lm] = sum_j g_n(r_ij) Y_lm(u_ij), and these
  // edges' radial terms.
  float s[NA][NABC];
#pragma unroll
  for (int n = 0; n < NA; ++n)
#pragma unroll
    for (int a = 0; a < NABC; ++a) s[n][a] = 0.0f;
  float zpe = 0.0f;
  // each lane takes every P-th edge with kRing records in flight: a record
  // comes from beyond L1, and an edge's arithmetic covers a fraction of that
  // (one ahead: 171 us on 256,000 Cu atoms, four: 165)
  constexpr int kRing = P == 1 && C::exact ? 4 : 1;
  auto edge_at = [&](int e) { return erow[(size_t)e * kTile]; };
  float4 ring[kRing];
  auto fill_ring = [&]() {
#pragma unroll
    for (int u = 0; u < kRing; ++u)
      ring[u] = lr + u * P < na ? edge_at(lr + u * P) : make_float4(1.0f, 0.0f, 0.0f, 0.0f);
  };
  fill_ring();
  for (int e0 = lr; e0 < na; e0 += kRing * P)
#pragma unroll
  for (int u = 0; u < kRing; ++u) {
    const int e = e0 + u * P;
    if (e >= na) break;
    const float4 r = ring[u];
    if (e + kRing * P < na) ring[u] = edge_at(e + kRing * P);
    const int tj = type_of(r);
    const float d2 = r.x * r.x + r.y * r.y + r.z * r.z;
    const float dinv = __builtin_amdgcn_rsqf(d2);  // hardware 1/sqrt (1 ulp); edges have d > 0
    const float d = d2 * dinv;
    if (!CAND && kOneLoop) radial_edge(d, tj);
    const float rc = C::one ? rcAf[0] : pcut[2 * kPairs + ti * T + tj];
    const float rcinv = C::one ? 1.0f / rc : pcut[3 * kPairs + ti * T + tj];
    if (m.zbl) {
      // half of each ZBL pair energy belongs to the centre; ZBL pairs are
      // taken from the angular rows, as the reference's ZBL pass does
      float zf, zfp;
      zbl_pair(m.zblp + (size_t)(ti * m.T + tj) * 12, d, dinv, zf, zfp);
      zpe += 0.5f * zf;
    }
    float fc;
    cutoff_fc(rc, rcinv, d, fc);
    float f[KA];
    cheb_scaled<KA>(rcinv, d, 0.5f * fc, f);
#pragma unroll
    for (int k = 1; k < KA; ++k) f[k] += f[0];
    f[0] = fc;
    const float* c = C::cl ? ctab + T * T * NR * KR + (ti * T + tj) * NA * KA
                           : m.cA + (size_t)(ti * T + tj) * nA * kA;
    float g[NA];
#pragma unroll
    for (int n = 0; n < NA; ++n) {
      g[n] = 0.0f;
      if (n < nA) {
#pragma unroll
        for (int k = 0; k < KA; ++k)
          if (k < kA) g[n] += c[n * kA + k] * f[k];
      }
    }
    float Y[NABC];
    harmonics<LM>(r.x * dinv, r.y * dinv, r.z * dinv, Y);
#pragma unroll
    for (int n = 0; n < NA; ++n)
#pragma unroll
      for (int a = 0; a < NABC; ++a) s[n][a] += g[n] * Y[a];
  }
  if (P > 1) {
    // the group's partial moments and ZBL energies
#pragma unroll
    for (int n = 0; n < NA; ++n)
#pragma unroll
      for (int a = 0; a < NABC; ++a) s[n][a] = group_sum<P>(s[n][a]);
    zpe = group_sum<P>(zpe);
  }

  if (P > 1) {
    // the group's partial radial sums
#pragma unroll
    for (int t = 0; t < (C::cl ? C::ltypes : 1); ++t)
#pragma unroll
      for (int k = 0; k < KR; ++k) Ft[t][k] = (C::one || C::cl) ? group_sum<P>(Ft[t][k]) : 0.0f;
    if (!C::one && !C::cl)
#pragma unroll
      for (int n = 0; n < NR; ++n) q[n] = group_sum<P>(q[n]);
  }
  if (C::one || C::cl) {
#pragma unroll
    for (int t = 0; t < (C::cl ? C::ltypes : 1); ++t) {
      const float h = Ft[t][0];
#pragma unroll
      for (int k = 0; k < KR; ++k) Ft[t][k] += h;
    }
#pragma unroll
    for (int n = 0; n < NR; ++n) {
      if (n < nR) {
        float g = 0.0f;
#pragma unroll
        for (int t = 0; t < (C::cl ? C::ltypes : 1); ++t) {
          if (t < T) {
            const float* c = C::cl ? ctab + (ti * T + t) * NR * KR + n * KR : m.cR + n * kR;
#pragma unroll
            for (int k = 0; k < KR; ++k)
              if (k < kR) g += c[k] * Ft[t][k];
          }
        }
        q[n] = g;
      }
    }
  }

  // ---- invariants
#pragma unroll
  for (int n = 0; n < NA; ++n) {
    if (n >= nA) break;
#pragma unroll
    for (int L = 1; L <= LM; ++L) {
      float v = 0.0f;
#pragma unroll
      for (int a = L * L - 1; a < (L + 1) * (L + 1) - 1; ++a) v += kAng.c3[a] * s[n][a] * s[n][a];
      if (L <= Lm) q[nR + (L - 1) * nA + n] = v;
    }
    int li = Lm;
    if (h222) {
      const float* x = &s[n][3];
      q[nR + li * nA + n] = kAng.c4[0] * x[0] * x[0] * x[0] + kAng.c4[1] * x[0] * (x[1] * x[1] + x[2] * x[2]) +
                            kAng.c4[2] * x[0] * (x[3] * x[3] + x[4] * x[4]) +
                            kAng.c4[3] * x[3] * (x[2] * x[2] - x[1] * x[1]) + kAng.c4[4] * x[1] * x[2] * x[4];
      ++li;
    }
    if (h1111) {
      const float r2 = s[n][0] * s[n][0] + s[n][1] * s[n][1] + s[n][2] * s[n][2];
      q[nR + li * nA + n] = kAng.c5 * r2 * r2;
    }
  }

  // ---- ANN (nep_utilities.cuh:209-310): E = sum_h w1 tanh(w0.q - b0) - bias
#pragma unroll
  for (int d = 0; d < DMAX; ++d)
    if (d < D) q[d] *= m.qs[d];
  float Fp[DMAX];
  float E = 0.0f;
  if (C::ann != kAnnValu) {
    if constexpr (C::ann_rows) {
      ann_mfma_rows<DMAX, (DMAX > 32 ? 2 : 4)>(m.H, q, Fp, E, ann_w);
    } else {
      __shared__ float ann_lds[kDescBlock / 64][ann_lds_floats<DMAX>()];
      ann_mfma<DMAX, C::ann, !C::one>(m, D, q, Fp, E, ann_lds[threadIdx.x >> 6], ann_w, ti, T);
    }
  } else {
    const int H = m.H;
    const float* w0 = m.w0 + (size_t)ti * H * D;
    const float* b0 = m.b0 + (size_t)ti * H;
    const float* w1 = m.w1 + (size_t)ti * H;
#pragma unroll
    for (int d = 0; d < DMAX; ++d) Fp[d] = 0.0f;
    for (int h = lr; h < H; h += P) {
      const float* wr = w0 + (size_t)h * D;
      float a = 0.0f;
#pragma unroll
      for (int d = 0; d < DMAX; ++d)
        if (d < D) a += wr[d] * q[d];
      float x, dx;
      tanh_sech2(a - b0[h], x, dx);
      E += w1[h] * x;
      const float gq = w1[h] * dx;
#pragma unroll
      for (int d = 0; d < DMAX; ++d)
        if (d < D) Fp[d] += gq * wr[d];
    }
    if (P > 1) {
      // the group's hidden neurons
      E = group_sum<P>(E);
#pragma unroll
      for (int d = 0; d < DMAX; ++d) Fp[d] = group_sum<P>(Fp[d]);
    }
  }
  E -= m.b1[0];
  if (m.version == 5) E -= m.w1x[ti];
#pragma unroll
  for (int d = 0; d < DMAX; ++d)
    if (d < D) Fp[d] *= m.qs[d];
  const double etot = (double)E + (double)zpe;
  if (active && lr == 0) pe[i] = accumulate ? pe[i] + etot : etot;

  // ---- radial adjoint in basis space: bR[i][t][k] = sum_n Fp_n c[ti,t,n,k]
  for (int t = 0; t < T; ++t) {
    const float* c = C::cl ? ctab + (ti * T + t) * NR * KR : m.cR + (size_t)(ti * T + t) * nR * kR;
    float* out = w.bR + ((size_t)i * T + t) * m.kRp;
    if (!active) break;
#pragma unroll
    for (int k = 0; k < ((KR + 3) & ~3); ++k) {
      float v = 0.0f;
      if (k < kR) {
#pragma unroll
        for (int n = 0; n < NR; ++n)
          if (n < nR) v += Fp[n] * c[n * kR + k];
      }
      if (k < m.kRp && (P == 1 || (k & (P - 1)) == lr)) out[k] = v;
    }
  }

  // ---- angular adjoint a[n][lm] = dE/ds[n][lm], written over s
#pragma unroll
  for (int n = 0; n < NA; ++n) {
    if (n >= nA) break;
    float extra[8];
#pragma unroll
    for (int a = 0; a < 8; ++a) extra[a] = 0.0f;
    int li = Lm;
    if (h222) {
      const float F = Fp[nR + li * nA + n];
      const float* x = &s[n][3];
      extra[3] = F * (3.0f * kAng.c4[0] * x[0] * x[0] + kAng.c4[1] * (x[1] * x[1] + x[2] * x[2]) +
                      kAng.c4[2] * (x[3] * x[3] + x[4] * x[4]));
      extra[4] = F * (2.0f * kAng.c4[1] * x[0] * x[1] - 2.0f * kAng.c4[3] * x[3] * x[1] + kAng.c4[4] * x[2] * x[4]);
      extra[5] = F * (2.0f * kAng.c4[1] * x[0] * x[2] + 2.0f * kAng.c4[3] * x[3] * x[2] + kAng.c4[4] * x[1] * x[4]);
      extra[6] = F * (2.0f * kAng.c4[2] * x[0] * x[3] + kAng.c4[3] * (x[2] * x[2] - x[1] * x[1]));
      extra[7] = F * (2.0f * kAng.c4[2] * x[0] * x[4] + kAng.c4[4] * x[1] * x[2]);
      ++li;
    }
    if (h1111) {
      const float F = Fp[nR + li * nA + n];
      const float r2 = s[n][0] * s[n][0] + s[n][1] * s[n][1] + s[n][2] * s[n][2];
      const float k5 = 4.0f * kAng.c5 * F * r2;
      extra[0] = k5 * s[n][0];
      extra[1] = k5 * s[n][1];
      extra[2] = k5 * s[n][2];
    }
#pragma unroll
    for (int L = 1; L <= LM; ++L) {
      const float F2 = L <= Lm ? 2.0f * Fp[nR + (L - 1) * nA + n] : 0.0f;  // no adjoint above the order
#pragma unroll
      for (int a = L * L - 1; a < (L + 1) * (L + 1) - 1; ++a) {
        float v = F2 * kAng.c3[a] * s[n][a];
        if (a < 8) v += extra[a];
        s[n][a] = v;
      }
    }
  }

  // ---- angular partial forces dE_i/dr_ij (the edges of the moments loop)
  fill_ring();
  for (int e0 = lr; e0 < na; e0 += kRing * P)
#pragma unroll
  for (int u = 0; u < kRing; ++u) {
    const int e = e0 + u * P;
    if (e >= na) break;
    const float4 r = ring[u];
    if (e + kRing * P < na) ring[u] = edge_at(e + kRing * P);
    const int tj = type_of(r);
    const float d2 = r.x * r.x + r.y * r.y + r.z * r.z;
    const float dinv = __builtin_amdgcn_rsqf(d2);  // hardware 1/sqrt (1 ulp); edges have d > 0
    const float d = d2 * dinv;
    const float ux = r.x * dinv, uy = r.y * dinv, uz = r.z * dinv;
    const float rc = C::one ? rcAf[0] : pcut[2 * kPairs + ti * T + tj];
    const float rcinv = C::one ? 1.0f / rc : pcut[3 * kPairs + ti * T + tj];
    float fc, fcp;
    cutoff_fc_fcp(rc, rcinv, d, fc, fcp);
    const float* c = C::cl ? ctab + T * T * NR * KR + (ti * T + tj) * NA * KA
                           : m.cA + (size_t)(ti * T + tj) * nA * kA;
    // with S_n = sum c_nk (T_k(x) + 1) and D_n = sum c_nk T_k'(x):
    // g_n = (fc/2) S_n, g'_n = (fc/2) x' D_n + (fc'/2) S_n
    float g[NA], gp[NA];
    if constexpr (!C::exact) {
      basis_by_function<NA, KA>(nA, kA, c, rcinv, d, fc, fcp, g, gp);
    } else {
      const float t = d * rcinv - 1.0f, x = 2.0f * t * t - 1.0f;
      const float hfc = 0.5f * fc, hfcp = 0.5f * fcp, hx = hfc * (4.0f * t * rcinv);
      float T1 = x, T0 = 1.0f, U1 = 1.0f, U0 = 0.0f;  // U1 = U_{k-1}, T_k' = k U_{k-1}
#pragma unroll
      for (int n = 0; n < NA; ++n) {
        g[n] = n < nA ? 2.0f * c[n * kA] : 0.0f;
        gp[n] = 0.0f;
      }
#pragma unroll
      for (int k = 1; k < KA; ++k) {
        if (k > 1) {
          const float T2 = 2.0f * x * T1 - T0, U2 = 2.0f * x * U1 - U0;
          T0 = T1;
          T1 = T2;
          U0 = U1;
          U1 = U2;
        }
        const float D1 = (float)k * U1;
        const float Tp = T1 + 1.0f;
#pragma unroll
        for (int n = 0; n < NA; ++n)
          if (n < nA && k < kA) {
            g[n] += c[n * kA + k] * Tp;
            gp[n] += c[n * kA + k] * D1;
          }
      }
#pragma unroll
      for (int n = 0; n < NA; ++n) {
        gp[n] = hx * gp[n] + hfcp * g[n];
        g[n] *= hfc;
      }
    }
    // contract the adjoint with the basis, order by order in m: with A = sum_n
    // a g_n and B = sum_n a g'_n of each moment, R + i I = sum_L Z (A_re + i
    // A_im), likewise with dZ/dz and with B; then Pr = sum B Y and G = sum A
    // dY/du (Y = Z(uz) Re/Im (ux + i uy)^m)
    const DirectionPowers<LM> pw(ux, uy, uz);
    float Pr = 0.0f, Gx = 0.0f, Gy = 0.0f, Gz = 0.0f;
    if constexpr (!C::exact) {
      contract_by_degree(s, g, gp, pw, Pr, Gx, Gy, Gz);
    } else {
      static_for<1, LM>([&](auto l) {
        constexpr int L = decltype(l)::value, a = L * L - 1;
        float A = 0.0f, B = 0.0f;
#pragma unroll
        for (int n = 0; n < NA; ++n) {
          A += s[n][a] * g[n];
          B += s[n][a] * gp[n];
        }
        Pr += B * harmonic_z<L, 0>(pw.zp);
        Gz += A * harmonic_dz<L, 0>(pw.zp);
      });
      static_for<1, LM>([&](auto mm) {
        constexpr int M = decltype(mm)::value;
        float R = 0.0f, I = 0.0f, dR = 0.0f, dI = 0.0f, RB = 0.0f, IB = 0.0f;
        static_for<M, LM>([&](auto l) {
          constexpr int L = decltype(l)::value, ir = L * L - 1 + 2 * M - 1, ii = ir + 1;
          float Ar = 0.0f, Ai = 0.0f, Br = 0.0f, Bi = 0.0f;
#pragma unroll
          for (int n = 0; n < NA; ++n) {
            Ar += s[n][ir] * g[n];
            Ai += s[n][ii] * g[n];
            Br += s[n][ir] * gp[n];
            Bi += s[n][ii] * gp[n];
          }
          if constexpr (L == M) {  // Z = 1
            R = Ar;
            I = Ai;
            RB = Br;
            IB = Bi;
          } else {
            const float Z = harmonic_z<L, M>(pw.zp), dZ = harmonic_dz<L, M>(pw.zp);
            R += Z * Ar;
            I += Z * Ai;
            RB += Z * Br;
            IB += Z * Bi;
            dR += dZ * Ar;
            dI += dZ * Ai;
          }
        });
        Pr += RB * pw.re[M] + IB * pw.im[M];
        constexpr float fm = (float)M;
        if constexpr (M == 1) {
          Gx += R;
          Gy += I;
        } else {
          Gx += fm * (R * pw.re[M - 1] + I * pw.im[M - 1]);
          Gy += fm * (I * pw.re[M - 1] - R * pw.im[M - 1]);
        }
        if constexpr (M < LM) Gz += dR * pw.re[M] + dI * pw.im[M];
      });
    }
    const float gu = Gx * ux + Gy * uy + Gz * uz;
    const float3 fo = make_float3(Pr * ux + (Gx - gu * ux) * dinv, Pr * uy + (Gy - gu * uy) * dinv,
                                  Pr * uz + (Gz - gu * uz) * dinv);
    frow[(size_t)e * kTile] = fo;
  }
}

// Arguments of one descriptor launch (launch_descriptor's).
struct DescriptorCall {
  const DevBox& b;
  const DevModel& m;
  int N, c1, c2;
  const int* type;
  double* pe;
  int acc, ann, lanes;
  DevWork& w;
  hipStream_t s;
  hipEvent_t e0, e1;
};

template <class C, bool CAND, int P>
void launch_instance(const DescriptorCall& a)
{
  constexpr int per = kDescBlock / P;
  const int nb = (a.c2 - (a.c1 & ~(kTile - 1)) + per - 1) / per;
  auto k = k_descriptor<C, CAND, P>;
  if (a.e0 || a.e1)
    hipExtLaunchKernelGGL(k, dim3(xcd_grid(nb)), dim3(kDescBlock), 0, a.s, a.e0, a.e1, 0, a.b, a.m, a.N, a.c1, a.c2, nb,
                          a.type, a.pe, a.w.edge, a.w.vsa, a.w.eq, a.acc, a.w);
  else
    k<<<xcd_grid(nb), kDescBlock, 0, a.s>>>(a.b, a.m, a.N, a.c1, a.c2, nb, a.type, a.pe, a.w.edge, a.w.vsa, a.w.eq,
                                           a.acc, a.w);
}

template <class C>
void run_descriptor(const DescriptorCall& a)
{
  if constexpr (C::ann == kAnnValu) {
    if (a.lanes == 4 && !a.w.split) return launch_instance<C, false, 4>(a);
    if (a.lanes == 16 && !a.w.split) return launch_instance<C, false, 16>(a);
  }
  if (a.w.split) launch_instance<C, true, 1>(a);
  else launch_instance<C, false, 1>(a);
}

// An exactly instantiated size with the ANN mode picked at run time: the
// matrix cores for H <= 64 and at most kTypesMfma types, the vector ALUs
// otherwise and for lane groups.
template <int NR, int KR, int NA, int KA, bool Q2, bool Q1, bool ONE>
void run_exact(const DescriptorCall& a)
{
  const bool vector = a.m.H > 64 || (!ONE && a.m.T > kTypesMfma) || (a.lanes != 1 && !a.w.split);
  const int mode = vector ? (int)kAnnValu : a.ann;
  if constexpr (mfma_ann_fits<NR, KR, NA, KA, Q2, Q1, ONE>()) {
    if (mode == kAnnMfma32) return run_descriptor<Cfg<NR, KR, NA, KA, 4, Q2, Q1, ONE, true, kAnnMfma32, !ONE>>(a);
    if (mode == kAnnMfmaBf16) return run_descriptor<Cfg<NR, KR, NA, KA, 4, Q2, Q1, ONE, true, kAnnMfmaBf16, !ONE>>(a);
  }
  if constexpr (mfma_ann_fits<NR, KR, NA, KA, Q2, Q1, ONE, kAnnMfmaSplit>()) {
    if (mode == kAnnMfmaSplit) return run_descriptor<Cfg<NR, KR, NA, KA, 4, Q2, Q1, ONE, true, kAnnMfmaSplit, !ONE>>(a);
  }
  if constexpr (ONE) {
    run_descriptor<Cfg<NR, KR, NA, KA, 4, Q2, Q1, true, true>>(a);
  } else {
    if (a.m.T <= kTypesLds) run_descriptor<Cfg<NR, KR, NA, KA, 4, Q2, Q1, false, true, kAnnValu, true>>(a);
    else run_descriptor<Cfg<NR, KR, NA, KA, 4, Q2, Q1, false, true>>(a);
  }
}

// a single-type size beyond the matrix-core ANN's 64 neurons in use
template <int NR, int KR, int NA, int KA, bool Q2, bool Q1>
void run_vector(const DescriptorCall& a)
{
  run_descriptor<Cfg<NR, KR, NA, KA, 4, Q2, Q1, true, true>>(a);
}

// models beyond the padded sizes: runtime sizes up to the maxima, 3-body
// order up to LM (registers spill)
template <int LM>
void run_generic(const DescriptorCall& a)
{
  run_descriptor<Cfg<kMaxNR, kMaxK, kMaxNA, kMaxK, LM, true, true, false, false>>(a);
}

}  // namespace dmgx
