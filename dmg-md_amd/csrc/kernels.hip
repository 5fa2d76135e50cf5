// kernels.hip -- HIP kernels of the NEP molecular-dynamics step for gfx950.
//
// Design (CDNA4, wave64):
//  * Verlet list with a 1 A skin, rebuilt only when an atom moved more than
//    skin/2 (neighbor.cu:446-582); rows hold slot indices, sorted ascending
//    (or by global id), with a precomputed reverse position per entry.
//  * Every step a filter pass (8, 16 or 32 lanes per centre, ballot compaction) turns
//    each Verlet row into one compact edge row: angular edges first (slots
//    0..na-1, ascending), radial-only edges from the end of the row
//    downward, each edge a float4 (FP64 minimum-image r_ij rounded to float,
//    neighbour slot).  Later kernels stream these rows instead of
//    re-gathering positions.  The edge rows are interleaved by tiles of 64
//    centres (row_begin), the others row-major ([i*M + slot]).
//  * One fused per-atom kernel does descriptor -> ANN -> adjoints -> angular
//    partial forces: the angular moments s[n][lm] stay in registers, are
//    turned in place into the adjoint dE/ds, and each angular edge's
//    dE_i/dr_ij is written at i's slot.
//  * The gather kernel (4, 8 or 16 lanes per atom) forms the radial pair force from
//    both centres' basis-space adjoints, adds the angular partials of both
//    directions (dE_j/dr_ji read from j's row through the reverse index) and
//    ZBL, and writes FP64 force/virial.  No floating-point atomics anywhere:
//    results are deterministic and independent of launch order.
//  * Integrator and thermo in FP64, thermo sums compensated (two-sum).
#include "nep_math.hpp"

#include <cmath>

namespace dmgx {

// ---------------------------------------------------------------------------
// per-step typewise filter (nep.cu:503-561) into compact edge rows
// ---------------------------------------------------------------------------

// kFilterLanes lanes per centre walk its Verlet row kFilterLanes entries per
// round; the kept entries of each round are compacted with a wavefront
// ballot and staged in LDS, from where the workgroup stores whole lines of the
// interleaved rows.  The loads of kFilterBatch rounds (row entries, their reverse positions, then
// the neighbours' packed positions) are issued before any of them is used,
// so a wave waits for two memory latencies per batch instead of two per
// round.  Types were validated when the step's positions were packed; here
// they are only clamped into range.  Pair cutoffs are FP64
// ((rc_i + rc_j) / 2)^2, as the reference's typewise test (nep.cu:503-561).
#ifndef DMGX_FILTER_LANES
#define DMGX_FILTER_LANES 16
#endif
#ifndef DMGX_FILTER_BATCH
#define DMGX_FILTER_BATCH 5
#endif
#ifndef DMGX_GATHER_LANES
#define DMGX_GATHER_LANES 8
#endif
constexpr int kFilterLanes = DMGX_FILTER_LANES;
constexpr int kFilterBatch = DMGX_FILTER_BATCH;
constexpr int kGatherLanes = DMGX_GATHER_LANES;

// CAND: the rebuild-time split of the rows into candidate rows instead (the
// same pass with every cutoff widened by the skin, writing slot indices
// instead of edge records); it runs only when this step rebuilt the rows.
template <bool ONE, bool MAP, int G, int RB, bool CAND = false>
__global__ __launch_bounds__(kBlock) void k_filter(DevBox b, DevModel m, int c1, int c2, int nblocks, int close,
                                                 DevWork w)
{
  constexpr int PER = kBlock / G;
  static_assert(G >= 1 && G <= 32 && (G & (G - 1)) == 0, "filter lanes: a power of two up to 32");
  constexpr unsigned long long gmask = (1ull << G) - 1ull;
  if (CAND && !w.flags[kFlagRebuild]) return;
  __shared__ double cut2[ONE ? 1 : 2 * kMaxTypes * kMaxTypes];  // [ti][tj] radial, then angular
  const int T = m.T;
  const double widen = CAND ? kSkin : 0.0;
  double rr2 = 0.0, ra2 = 0.0;
  if (ONE) {
    const double rr = (m.rcR[0] + m.rcR[0]) * 0.5 + widen, ra = (m.rcA[0] + m.rcA[0]) * 0.5 + widen;
    rr2 = rr * rr;
    ra2 = ra * ra;
  } else {
    for (int k = threadIdx.x; k < T * T; k += blockDim.x) {
      const int p = k / T, q = k % T;
      const double rr = (m.rcR[p] + m.rcR[q]) * 0.5 + widen, ra = (m.rcA[p] + m.rcA[q]) * 0.5 + widen;
      cut2[k] = rr * rr;
      cut2[T * T + k] = ra * ra;
    }
    __syncthreads();
  }
  // the rebuild kernels of this step ran before this one: close the request
  // (one filter launch per evaluation does; the others of a split one skip)
  if (!CAND && close && blockIdx.x == 0 && threadIdx.x == 0 && w.flags[kFlagRebuild]) {
    w.flags[kFlagRebuild] = 0;
    w.flags[kFlagRebuildCount] += 1;
  }
  const int g = threadIdx.x / G, lg = threadIdx.x % G, gw = g % (64 / G);
  const int first = c1 + xcd_tile(nblocks) * PER;  // the workgroup's centres: PER consecutive ones
  const int i = first + g;
  const bool active = i < c2;
  double4 pi = make_double4(0, 0, 0, 0);
  int ti = 0, nv = 0;
  if (active) {
    pi = w.xq[i];
    ti = ONE ? 0 : safe_type((int)__double_as_longlong(pi.w), T);
    nv = min(w.vn[i], w.MV);
  }
  const size_t vrow = (size_t)i * w.MV;
  const unsigned below = (1u << lg) - 1u;
  // The kept edges of a pass of G * RB entries are compacted in LDS (angular
  // ones from the front of a centre's stage, radial-only ones from its end) and
  // stored to the interleaved rows slot by slot: consecutive threads store one
  // slot of the workgroup's consecutive centres, 16 * PER contiguous bytes.
  // (Stored directly, each record is a line access of its own: 154 us against
  // 115 on 256,000 Cu atoms; row-major rows, with shorter loads in the
  // descriptor's way, 122.  One lane per centre, without ballots, reads the
  // neighbours' positions from 64 lines at a time: 204 us.)  The odd record
  // count keeps the store's reads free of bank conflicts.
  constexpr int kStage = G * RB;
  __shared__ float4 stage[CAND ? 1 : PER * (kStage + 1)];
  __shared__ short stage_q[CAND ? 1 : PER * (kStage + 2)];
  __shared__ int4 counts[CAND ? 1 : PER];  // angular / radial-only edges before the pass, and in it
  float4* const st = stage + g * (kStage + 1);
  short* const sq = stage_q + g * (kStage + 2);
  int na = 0, nro = 0;
  // the row's angular bits, assembled a 32-bit word at a time by the
  // group's first lane (a chunk of G consecutive entries never straddles
  // a word) and stored once the word is complete
  unsigned* const mrow = CAND ? nullptr : w.amask + (size_t)i * ((w.MV + 31) >> 5);
  unsigned mword = 0u;
  int mcur = 0;
  for (int p0 = 0; CAND ? __any(p0 < nv) : __syncthreads_or(p0 < nv); p0 += G * RB) {
    int jj[RB], qq[RB], jo[RB];
    double4 pj[RB];
#pragma unroll
    for (int r = 0; r < RB; ++r) {
      const int p = p0 + r * G + lg;
      jj[r] = -1;
      qq[r] = -1;
      if (p < nv) {
        jj[r] = w.vl[vrow + p];
        qq[r] = w.vrev[vrow + p];
      }
    }
    // with an image map an entry stands for its owner in the edge record
    // and the reverse index; its own slot only gives the position
#pragma unroll
    for (int r = 0; r < RB; ++r) {
      pj[r] = jj[r] >= 0 ? w.xq[jj[r]] : make_double4(0, 0, 0, 0);
      jo[r] = (MAP && jj[r] >= 0) ? w.map.owner[jj[r]] : jj[r];
    }
    int pa = 0, pr = 0;  // angular and radial-only edges of this pass
#pragma unroll
    for (int r = 0; r < RB; ++r) {
      const int p = p0 + r * G + lg;
      bool isA = false, isR = false;
      float4 rec = make_float4(0.f, 0.f, 0.f, 0.f);
      if (jj[r] >= 0) {
        double x = pj[r].x - pi.x, y = pj[r].y - pi.y, z = pj[r].z - pi.z;
        mic(b, x, y, z);
        const double d2 = dist2(x, y, z);
        double cr = rr2, ca = ra2;
        int tj = 0;
        if (!ONE) {
          tj = safe_type((int)__double_as_longlong(pj[r].w), T);
          cr = cut2[ti * T + tj];
          ca = cut2[T * T + ti * T + tj];
        }
        if (d2 < cr) {
          isA = d2 < ca;
          isR = !isA;
          rec = make_float4((float)x, (float)y, (float)z, __int_as_float(ONE ? jo[r] : edge_word(w.typed, jo[r], tj)));
        }
      }
      const unsigned gA = (unsigned)((__ballot(isA) >> (gw * G)) & gmask);
      const unsigned gR = (unsigned)((__ballot(isR) >> (gw * G)) & gmask);
      const int a = pa + __popc(gA & below), q = pr + __popc(gR & below);
      if (CAND) {
        // candidate rows hold the slot itself (its position is read every
        // step); the reverse index becomes a candidate slot in k_split_reverse
        if (jj[r] >= 0) w.cpos[vrow + p] = isA ? na + a : -1;
        if (isA) {
          w.cl[vrow + na + a] = jj[r];
          w.cq[vrow + na + a] = qq[r] >= 0 ? jo[r] * w.MV + qq[r] : -1;
        }
        if (isR) w.cl[vrow + w.MV - 1 - (nro + q)] = jj[r];
      } else {
        const int base = p0 + r * G;
        if (lg == 0 && base < nv) {
          if ((base >> 5) != mcur) {
            mrow[mcur] = mword;
            mword = 0u;
            mcur = base >> 5;
          }
          mword |= gA << (base & 31);
        }
        if (isA) {
          st[a] = rec;
          sq[a] = (short)qq[r];
        }
        if (isR) st[kStage - 1 - q] = rec;
      }
      pa += __popc(gA);
      pr += __popc(gR);
    }
    if (!CAND) {
      if (lg == 0) counts[g] = make_int4(na, nro, pa, pr);
      __syncthreads();
      const int c = threadIdx.x % PER;
      const int4 n = counts[c];
      float4* const erow = w.edge + row_begin(first + c, w.MR);
      short* const qrow = w.eq + row_begin(first + c, w.MA);
      for (int k = threadIdx.x / PER; k < n.z; k += G) {
        erow[(size_t)(n.x + k) * kTile] = stage[c * (kStage + 1) + k];
        qrow[(size_t)(n.x + k) * kTile] = stage_q[c * (kStage + 2) + k];
      }
      for (int k = threadIdx.x / PER; k < n.w; k += G)
        erow[(size_t)(w.MR - 1 - (n.y + k)) * kTile] = stage[c * (kStage + 1) + kStage - 1 - k];
      // the next pass's first barrier (the loop condition's) keeps its stage
      // writes behind these reads
    }
    na += pa;
    nro += pr;
  }
  // na + nro <= nv <= MV = MR = MA: the two ends of a row never meet
  if (!CAND && active && lg == 0 && nv > 0) mrow[mcur] = mword;
  if (active && lg == 0) {
    if (CAND) {
      w.nrc[i] = na + nro;
      w.nac[i] = na;
    } else {
      w.nr[i] = na + nro;
      w.na[i] = na;
    }
  }
}

// Rebuild-time reverse of the candidate rows: an angular candidate i->j's
// Verlet reverse index j*MV + q becomes i's angular candidate slot in j's
// row, or -1 where j has no row in [c1, c2) or i is not one of its
// angular candidates.
template <int G>
__global__ __launch_bounds__(kBlock) void k_split_reverse(int c1, int c2, int nblocks, DevWork w)
{
  if (!w.flags[kFlagRebuild]) return;
  constexpr int PER = kBlock / G;
  const int g = threadIdx.x / G, lg = threadIdx.x % G;
  const int i = c1 + xcd_tile(nblocks) * PER + g;
  if (i >= c2) return;
  const int n = w.nac[i];
  const size_t arow = (size_t)i * w.MA;
  for (int a = lg; a < n; a += G) {
    const int q = w.cq[arow + a];
    int v = -1;
    if (q >= 0) {
      const int j = q / w.MV;
      if (j >= c1 && j < c2) {
        const int c = w.cpos[q];
        if (c >= 0) v = c;
      }
    }
    w.cq[arow + a] = v;
  }
}

// ---------------------------------------------------------------------------
// gather: radial pair force, angular partials, ZBL -> FP64 force/virial
// ---------------------------------------------------------------------------

// Radial pair force of one edge: f'_k = (fc/2) x' k U_{k-1} + (fc'/2) (T_k + 1),
// from recurrences scaled by (fc/2) x' and fc'/2; Gi = sum_k b_i f'_k and Gj
// with the neighbour's adjoint.
template <int KR>
__device__ __forceinline__ void radial_pair(float rcinv, float d, float fc, float fcp, const float* bi, const float* bj,
                                            float& Gi, float& Gj)
{
  const float t = d * rcinv - 1.0f, x = 2.0f * t * t - 1.0f, x2 = 2.0f * x;
  const float A = 0.5f * fc * (4.0f * t * rcinv), B = 0.5f * fcp;
  float T0 = B, T1 = x * B, U0 = 0.0f, U1 = A;  // U1 = A U_{k-1}
  Gi = bi[0] * fcp;
  Gj = bj[0] * fcp;
#pragma unroll
  for (int k = 1; k < KR; ++k) {
    const float fp = fmaf((float)k, U1, T1 + B);
    Gi = fmaf(bi[k], fp, Gi);
    Gj = fmaf(bj[k], fp, Gj);
    const float T2 = fmaf(x2, T1, -T0), U2 = fmaf(x2, U1, -U0);
    T0 = T1;
    T1 = T2;
    U0 = U1;
    U1 = U2;
  }
}

// FP64 force and virial sums of a lane, each product formed and added by one
// FP64 FMA (full rate on this chip; an FP32 product, its conversion and an
// addition are three instructions).  A radial pair's virial is symmetric
// (r (x) r): its off-diagonal terms are summed once and added to both at the
// end.
struct PairSums {
  double fx = 0.0, fy = 0.0, fz = 0.0;
  double v[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
  double sxy = 0.0, sxz = 0.0, syz = 0.0;
  // F_i += (Gi + Gj) r/d; virial_i += r (x) dE_j/dr_ji = r (x) (-Gj r/d)
  __device__ __forceinline__ void radial(const float4& q, float dinv, float Gi, float Gj)
  {
    const double x = q.x, y = q.y, z = q.z, sc = (Gi + Gj) * dinv, gj = -Gj * dinv;
    fx = fma(sc, x, fx);
    fy = fma(sc, y, fy);
    fz = fma(sc, z, fz);
    const double wx = gj * x, wy = gj * y, wz = gj * z;
    v[0] = fma(x, wx, v[0]);
    v[1] = fma(y, wy, v[1]);
    v[2] = fma(z, wz, v[2]);
    sxy = fma(x, wy, sxy);
    sxz = fma(x, wz, sxz);
    syz = fma(y, wz, syz);
  }
  __device__ __forceinline__ void angular(const float4& q, float gx, float gy, float gz, float bx, float by, float bz)
  {
    const double x = q.x, y = q.y, z = q.z, wx = bx, wy = by, wz = bz;
    fx += (double)gx;
    fy += (double)gy;
    fz += (double)gz;
    v[0] = fma(x, wx, v[0]);
    v[1] = fma(y, wy, v[1]);
    v[2] = fma(z, wz, v[2]);
    v[3] = fma(x, wy, v[3]);
    v[4] = fma(x, wz, v[4]);
    v[5] = fma(y, wz, v[5]);
    v[6] = fma(y, wx, v[6]);
    v[7] = fma(z, wx, v[7]);
    v[8] = fma(z, wy, v[8]);
  }
  __device__ __forceinline__ void fold()
  {
    v[3] += sxy;
    v[6] += sxy;
    v[4] += sxz;
    v[7] += sxz;
    v[5] += syz;
    v[8] += syz;
  }
};

// G lanes per atom share its edges (interleaved rows: the lanes of
// consecutive atoms read contiguous records); the per-lane FP64 sums are
// combined with a butterfly over the group at the end.  Each lane takes its
// edges a batch at a time: the edge records are loaded, then the neighbours'
// adjoint rows (angular loop: their reverse partials), then all of them are
// used, so the loads of a batch overlap.
// What bounds it: about equal parts of vector issue (60% of the cycles on
// 256,000 Cu atoms) and L1 accesses (three per neighbour row; reading a row's
// chunks with four lanes and passing them on through LDS saved a fifth of the
// accesses for as much more vector work: 128 us against 119).  Scaled
// recurrences (radial_pair), FP64 FMAs (PairSums), DPP sums and, with several
// types, the atom's own rows in LDS take it from 126 to 112 us there and from
// 43 to 36 us on 5,832 atoms with 17 basis functions; HBM reads fell from 614
// to 363 MB with the interleaved edge rows.  One lane per atom takes 141 us.
// CAND: the radial edges come from the candidate rows (DevWork::split).
template <int KR, bool ONE, int G, bool CAND>
__global__ __launch_bounds__(kBlock, 4) void k_gather(DevBox b, DevModel m, int n1, int n2, int nd1, int nd2,
                                                   int nblocks, const int* __restrict__ type, int N,
                                                   double* __restrict__ force, double* __restrict__ virial,
                                                   int accumulate, DevWork w)
{
  constexpr int PER = kBlock / G;
  constexpr int RB = 2, AB = 3;  // radial, angular edges per batch
  static_assert(G >= 1 && G <= 64 && (G & (G - 1)) == 0, "gather lanes: a power of two");
  const int g = threadIdx.x / G, lg = threadIdx.x % G;
  const int i0 = (n1 & ~(kTile - 1)) + xcd_tile(nblocks) * PER + g;
  const bool active = i0 >= n1 && i0 < n2;
  const int i = active ? i0 : n1;
  const int T = ONE ? 1 : m.T;
  int ti = 0, nr = 0, na = 0, nac = 0;
  double4 pi = make_double4(0.0, 0.0, 0.0, 0.0);
  if (active) {
    ti = ONE ? 0 : safe_type(type[i], T);
    na = w.na[i];
    if (CAND) {
      // candidate rows: the radial loop runs over the candidates and keeps
      // those within the pair's radial cutoff (the descriptor's test)
      nr = w.nrc[i];
      nac = w.nac[i];
      pi = w.xq[i];
    } else {
      nr = w.nr[i];
    }
  }
  constexpr int KP = (KR + 3) & ~3;  // padded row: KP/4 float4 loads
  const int kRp = m.kRp;
  const float4* __restrict__ erow = w.edge + row_begin(i, w.MR);
  const float3* __restrict__ frow = w.f12 + row_begin(i, w.MA);
  const short* __restrict__ qrow = w.eq + row_begin(i, w.MA);
  const float* __restrict__ bR = w.bR;
  PairSums sum;
  float bi[KP];
#pragma unroll
  for (int k = 0; k < KP; ++k) bi[k] = 0.0f;
  if (ONE && active) load_row4<KP>(bR + (size_t)i * kRp, kRp, bi);
  const float rcR0 = (float)((m.rcR[0] + m.rcR[0]) * 0.5);
  // radial term of one edge (jj >= 0) with the neighbour's adjoint bj
  constexpr int NC = KP / 4;  // 16-byte chunks of an adjoint row
  // several types: the atom's own rows, one per neighbour type
  __shared__ float4 own[ONE ? 1 : PER][ONE ? 1 : kTypesLds][ONE ? 1 : NC];
  const bool own_lds = !ONE && T <= kTypesLds;
  if (!ONE && own_lds) {
    for (int k = lg; k < T * NC; k += G) {
      const int t = k / NC, c = k % NC;
      if (active && 4 * c < kRp) own[g][t][c] = reinterpret_cast<const float4*>(bR + ((size_t)i * T + t) * kRp)[c];
      else own[g][t][c] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
    wave_lds_sync();  // an atom's lanes lie in one wavefront
  }
  auto radial = [&](const float4& q, float dinv, float d, int tj, const float* bj) {
    const float rc = ONE ? rcR0 : (float)((m.rcR[ti] + m.rcR[tj]) * 0.5);
    const float rcinv = 1.0f / rc;
    float fc, fcp, Gi, Gj;
    cutoff_fc_fcp(rc, rcinv, d, fc, fcp);
    if (ONE) {
      radial_pair<KR>(rcinv, d, fc, fcp, bi, bj, Gi, Gj);
    } else {
      float bo[KP];
      if (own_lds) {
#pragma unroll
        for (int c = 0; c < NC; ++c) reinterpret_cast<float4*>(bo)[c] = own[g][tj][c];
      } else {
#pragma unroll
        for (int k = 0; k < KP; ++k) bo[k] = 0.0f;
        load_row4<KP>(bR + ((size_t)i * T + tj) * kRp, kRp, bo);
      }
      radial_pair<KR>(rcinv, d, fc, fcp, bo, bj, Gi, Gj);
    }
    sum.radial(q, dinv, Gi, Gj);
  };
  auto load_adjoint = [&](int j, float* bj) {
#pragma unroll
    for (int k = 0; k < KP; ++k) bj[k] = 0.0f;
    if (j >= nd1 && j < nd2) load_row4<KP>(bR + ((size_t)j * T + ti) * kRp, kRp, bj);
  };
  // every edge within the radial cutoff: F_i += (G_i + G_j) r_ij/d
  for (int e0 = lg; e0 < nr; e0 += G * RB) {
    float4 rr[RB];
    int jj[RB], tt[RB];
    if (!CAND) {
#pragma unroll
      for (int r = 0; r < RB; ++r) {
        const int e = e0 + r * G;
        jj[r] = -1;
        tt[r] = 0;
        rr[r] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (e < nr) {
          rr[r] = erow[(size_t)(e < na ? e : w.MR - 1 - (e - na)) * kTile];
          jj[r] = __float_as_int(rr[r].w);
          if (!ONE) {
            tt[r] = edge_type(w, type, jj[r], T);
            jj[r] = edge_slot(w.typed, jj[r]);
          }
        }
      }
    } else {
      const int* __restrict__ crow = w.cl + (size_t)i * w.MV;
      int jc[RB];
      double4 pj[RB];
#pragma unroll
      for (int r = 0; r < RB; ++r) {
        const int e = e0 + r * G;
        jc[r] = e < nr ? crow[e < nac ? e : w.MV - 1 - (e - nac)] : -1;
      }
#pragma unroll
      for (int r = 0; r < RB; ++r) pj[r] = jc[r] >= 0 ? w.xq[jc[r]] : make_double4(0.0, 0.0, 0.0, 0.0);
#pragma unroll
      for (int r = 0; r < RB; ++r) {
        rr[r] = make_float4(0.f, 0.f, 0.f, 0.f);
        jj[r] = -1;
        tt[r] = 0;
        if (jc[r] >= 0) {
          double x = pj[r].x - pi.x, y = pj[r].y - pi.y, z = pj[r].z - pi.z;
          mic(b, x, y, z);
          const double d2 = dist2(x, y, z);
          double rc = (m.rcR[0] + m.rcR[0]) * 0.5;
          if (!ONE) {
            tt[r] = safe_type((int)__double_as_longlong(pj[r].w), T);
            rc = (m.rcR[ti] + m.rcR[tt[r]]) * 0.5;
          }
          if (d2 < rc * rc) {
            jj[r] = w.map.owner ? w.map.owner[jc[r]] : jc[r];
            rr[r] = make_float4((float)x, (float)y, (float)z, __int_as_float(jj[r]));
          }
        }
      }
    }
    float bj[RB][KP];
#pragma unroll
    for (int r = 0; r < RB; ++r) load_adjoint(jj[r], bj[r]);
#pragma unroll
    for (int r = 0; r < RB; ++r) {
      const float4 q = rr[r];
      // lanes past the row end carry r = 0: d = 0 and 1/d = 0 there, so every term is zero
      const float d2 = q.x * q.x + q.y * q.y + q.z * q.z;
      const float dinv = jj[r] >= 0 ? __builtin_amdgcn_rsqf(d2) : 0.0f;
      radial(q, dinv, d2 * dinv, tt[r], bj[r]);
    }
  }
  // angular edges: F_i += dE_i/dr_ij - dE_j/dr_ji (the second term is read
  // from j's row at the slot where i sits: Verlet reverse position -> angular
  // slot), and ZBL
  for (int e0 = lg; e0 < na; e0 += G * AB) {
    float4 rr[AB];
    float3 aa[AB], bb[AB];
    int jj[AB], qv[AB], tt[AB];
#pragma unroll
    for (int r = 0; r < AB; ++r) {
      const int e = e0 + r * G;
      rr[r] = make_float4(0.f, 0.f, 0.f, 0.f);
      aa[r] = make_float3(0.f, 0.f, 0.f);
      jj[r] = qv[r] = -1;
      tt[r] = 0;
      if (e < na) {
        rr[r] = erow[(size_t)e * kTile];
        aa[r] = frow[(size_t)e * kTile];
        qv[r] = qrow[(size_t)e * kTile];
        jj[r] = __float_as_int(rr[r].w);
        if (!ONE) {
          tt[r] = edge_type(w, type, jj[r], T);
          jj[r] = edge_slot(w.typed, jj[r]);
        }
      }
    }
#pragma unroll
    for (int r = 0; r < AB; ++r) {
      bb[r] = make_float3(0.f, 0.f, 0.f);
      int e2 = -1;
      const int q = qv[r];
      if (jj[r] >= nd1 && jj[r] < nd2 && q >= 0 && q < w.MV) {
        if (CAND) {
          e2 = w.vsa[(size_t)jj[r] * w.MA + q];
        } else {
          // i's Verlet position q in j's row; its angular slot is the number
          // of angular entries of j's row before it
          const int mw = (w.MV + 31) >> 5;
          const unsigned* mk = w.amask + (size_t)jj[r] * mw;
          if (mw == 4) {
            // rows of up to 128 entries: the row's four words in one load
            const uint4 m4 = *reinterpret_cast<const uint4*>(mk);
            const unsigned wd[4] = {m4.x, m4.y, m4.z, m4.w};
            const int wq = q >> 5;
            const unsigned word = wd[wq];
            if ((word >> (q & 31)) & 1u) {
              int c = __popc(word & ((1u << (q & 31)) - 1u));
              c += (wq > 0 ? __popc(m4.x) : 0) + (wq > 1 ? __popc(m4.y) : 0) + (wq > 2 ? __popc(m4.z) : 0);
              e2 = c;
            }
          } else {
            const unsigned word = mk[q >> 5];
            if ((word >> (q & 31)) & 1u) {
              int c = __popc(word & ((1u << (q & 31)) - 1u));
              for (int k = 0; k < (q >> 5); ++k) c += __popc(mk[k]);
              e2 = c;
            }
          }
        }
      }
      if (e2 >= 0 && e2 < w.MA) bb[r] = w.f12[row_begin(jj[r], w.MA) + (size_t)e2 * kTile];
    }
#pragma unroll
    for (int r = 0; r < AB; ++r) {
      const float4 q = rr[r];
      const bool jdep = jj[r] >= nd1 && jj[r] < nd2;
      float gx = aa[r].x - bb[r].x, gy = aa[r].y - bb[r].y, gz = aa[r].z - bb[r].z;
      float bx = bb[r].x, by = bb[r].y, bz = bb[r].z;
      if (m.zbl && jj[r] >= 0) {
        // each directed pair carries half of the ZBL pair gradient
        // (nep_utilities.cuh:347-433 switch, nep.cu ZBL pass)
        const float d = sqrtf(q.x * q.x + q.y * q.y + q.z * q.z);
        const float dinv = 1.0f / d;
        float zf, zfp;
        zbl_pair(m.zblp + (size_t)(ti * m.T + tt[r]) * 12, d, dinv, zf, zfp);
        const float h = 0.5f * zfp * dinv;  // dE_i/dr_ij = h r_ij
        const float c = jdep ? 2.0f * h : h;
        gx += c * q.x;
        gy += c * q.y;
        gz += c * q.z;
        if (jdep) {  // dE_j/dr_ji = -h r_ij
          bx -= h * q.x;
          by -= h * q.y;
          bz -= h * q.z;
        }
      }
      sum.angular(q, gx, gy, gz, bx, by, bz);
    }
  }
  sum.fold();
  sum.fx = group_sum<G>(sum.fx);
  sum.fy = group_sum<G>(sum.fy);
  sum.fz = group_sum<G>(sum.fz);
#pragma unroll
  for (int c = 0; c < 9; ++c) sum.v[c] = group_sum<G>(sum.v[c]);
  if (!active || lg != 0) return;
  if (accumulate) {
    force[i] += sum.fx;
    force[N + i] += sum.fy;
    force[2 * N + i] += sum.fz;
#pragma unroll
    for (int c = 0; c < 9; ++c) virial[(size_t)c * N + i] += sum.v[c];
  } else {
    force[i] = sum.fx;
    force[N + i] = sum.fy;
    force[2 * N + i] = sum.fz;
#pragma unroll
    for (int c = 0; c < 9; ++c) virial[(size_t)c * N + i] = sum.v[c];
  }
}

// ---------------------------------------------------------------------------
// integrator and thermo (FP64)
// ---------------------------------------------------------------------------

// (the first half also adds the drift to `unwrapped` when given:
// update_unwrapped, runtime.cu:423-440)
__global__ void k_velocity_verlet(int first_half, int N, double dt, const double* __restrict__ mass,
                                  double* __restrict__ pos, double* __restrict__ vel,
                                  const double* __restrict__ force, double* __restrict__ unwrapped)
{
#pragma clang fp contract(off)
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= N) return;
  const double half = dt * 0.5;
  const double im = 1.0 / mass[i];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const double v = vel[c * N + i] + force[c * N + i] * im * half;
    vel[c * N + i] = v;
    if (first_half) {
      const double x0 = pos[c * N + i], x1 = x0 + v * dt;
      pos[c * N + i] = x1;
      if (unwrapped) unwrapped[c * N + i] += x1 - x0;
    }
  }
}

__global__ void k_wrap(DevBox b, int N, double* __restrict__ pos)
{
#pragma clang fp contract(off)
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= N) return;
  const double x = pos[i], y = pos[N + i], z = pos[2 * N + i];
  double s[3] = {b.hi[0] * x + b.hi[1] * y + b.hi[2] * z, b.hi[3] * x + b.hi[4] * y + b.hi[5] * z,
                 b.hi[6] * x + b.hi[7] * y + b.hi[8] * z};
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    if (!b.pbc[d]) continue;
    if (s[d] < 0.0) s[d] += 1.0;
    else if (s[d] > 1.0) s[d] -= 1.0;
  }
  pos[i] = b.h[0] * s[0] + b.h[1] * s[1] + b.h[2] * s[2];
  pos[N + i] = b.h[3] * s[0] + b.h[4] * s[1] + b.h[5] * s[2];
  pos[2 * N + i] = b.h[6] * s[0] + b.h[7] * s[1] + b.h[8] * s[2];
}

// First half of a velocity-Verlet step of the MD loop in one kernel: the
// previous step's pending thermostat factor (v *= f), the half kick and
// drift, the periodic wrap, the step's packed (x, y, z, type) record and the
// displacement test against the last rebuild.  The FP64 expressions are
// those of k_scale_by, k_velocity_verlet, k_wrap and the neighbour pack, in
// that order and without contraction, so the results are bit-identical to
// running them as separate kernels.  KICK: the last step's second half kick
// first (inside a chunk without a thermostat nothing reads the velocities in
// between), one launch a step less: 4,096 carbon atoms 62.6 -> 60.9 us a step.
template <bool KICK>
__global__ __launch_bounds__(kBlock) void k_md_first(DevBox b, int N, int T, double dt,
                                                     const double* __restrict__ mass, double* __restrict__ pos,
                                                     double* __restrict__ vel, const double* __restrict__ force,
                                                     const double* __restrict__ factor,
                                                     const int* __restrict__ type, const double* __restrict__ x0,
                                                     double lim2, int forced, double4* __restrict__ xq,
                                                     int* __restrict__ flags, double* __restrict__ unwrapped)
{
#pragma clang fp contract(off)
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (forced && i == 0) flags[kFlagRebuild] = kRebuildAsked | kRebuildAll;
  bool moved = false, bad = false;
  if (i < N) {
    const double half = dt * 0.5;
    const double im = 1.0 / mass[i];
    double x[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      double v = vel[c * N + i];
      if (factor) v *= factor[0];
      const double f = force[c * N + i];
      if (KICK) v = v + f * im * half;
      v = v + f * im * half;
      vel[c * N + i] = v;
      const double p0 = pos[c * N + i];
      x[c] = p0 + v * dt;
      if (unwrapped) unwrapped[c * N + i] += x[c] - p0;
    }
    double sf[3] = {b.hi[0] * x[0] + b.hi[1] * x[1] + b.hi[2] * x[2], b.hi[3] * x[0] + b.hi[4] * x[1] + b.hi[5] * x[2],
                    b.hi[6] * x[0] + b.hi[7] * x[1] + b.hi[8] * x[2]};
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      if (!b.pbc[d]) continue;
      if (sf[d] < 0.0) sf[d] += 1.0;
      else if (sf[d] > 1.0) sf[d] -= 1.0;
    }
    const double px = b.h[0] * sf[0] + b.h[1] * sf[1] + b.h[2] * sf[2];
    const double py = b.h[3] * sf[0] + b.h[4] * sf[1] + b.h[5] * sf[2];
    const double pz = b.h[6] * sf[0] + b.h[7] * sf[1] + b.h[8] * sf[2];
    pos[i] = px;
    pos[N + i] = py;
    pos[2 * N + i] = pz;
    const int t = type[i];
    bad = t < 0 || t >= T;
    xq[i] = make_double4(px, py, pz, __longlong_as_double((long long)t));
    if (!forced) {
      double dx = px - x0[i], dy = py - x0[N + i], dz = pz - x0[2 * N + i];
      mic(b, dx, dy, dz);
      moved = !(dist2(dx, dy, dz) <= lim2);
    }
  }
  const bool lead = (threadIdx.x & 63) == 0;
  if (__any(moved) && lead) atomicOr(&flags[kFlagRebuild], kRebuildAsked);
  if (__any(bad) && lead) atomicOr(&flags[kFlagBadType], 1);
}

// error-free two-sum accumulation (s, c) += x
struct KSum {
  double s, c;
};
__device__ __forceinline__ void ksum_add(KSum& k, double x)
{
  const double t = k.s + x;
  const double bp = t - k.s;
  const double err = (k.s - (t - bp)) + (x - bp);
  k.s = t;
  k.c += err;
}
__device__ __forceinline__ void ksum_merge(KSum& a, const KSum& b)
{
  ksum_add(a, b.s);
  a.c += b.c;
}

constexpr int kThermoThreads = 256;

int thermo_blocks(int N)
{
  int nb = (N + kThermoThreads - 1) / kThermoThreads;
  return nb < 1 ? 1 : (nb > 512 ? 512 : nb);
}

// compensated reduction of 8 quantities over a 256-thread workgroup: wave
// shuffles, then the 4 wave results through LDS; the total lands in thread 0
__device__ __forceinline__ void block_reduce8(KSum* acc)
{
#pragma unroll
  for (int q = 0; q < 8; ++q)
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      KSum o{__shfl_down(acc[q].s, off), __shfl_down(acc[q].c, off)};
      ksum_merge(acc[q], o);
    }
  __shared__ double sh[kThermoThreads / 64][8][2];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  if (lane == 0)
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      sh[wave][q][0] = acc[q].s;
      sh[wave][q][1] = acc[q].c;
    }
  __syncthreads();
  if (threadIdx.x == 0)
#pragma unroll
    for (int q = 0; q < 8; ++q)
      for (int w = 1; w < kThermoThreads / 64; ++w) ksum_merge(acc[q], KSum{sh[w][q][0], sh[w][q][1]});
}

// velocity factor from this step's normalised temperature, formed where the
// thermo lives (same expressions as Controller::after_force, no contraction)
__device__ __forceinline__ double ensemble_factor(int kind, int N, double coupling, double t_target,
                                                  const double* __restrict__ rand2, double T)
{
#pragma clang fp contract(off)
  double f = 1.0;
  if (kind == 1) {
    f = sqrt(1.0 + coupling * (t_target / T - 1.0));
  } else if (kind == 2) {
    // resamplekin (thermostat_svr.cpp:107-124) with rr and the chi-square sum drawn on the host
    const int ndeg = 3 * N;
    const double kk = T * (ndeg * 8.617343e-5 * 0.5);  // old_KE *= ndeg * K_B * 0.5
    const double sigma = ndeg * 8.617343e-5 * t_target * 0.5;
    const double fac = coupling;  // exp(-1/taut) or 0, formed on the host
    const double rr = rand2[0], sum = rand2[1];
    const double knew = kk + (1.0 - fac) * (sigma * (sum + rr * rr) / ndeg - kk) +
                        2.0 * rr * sqrt(kk * sigma / ndeg * (1.0 - fac) * fac);
    f = sqrt(knew / kk);
  }
  return f;
}

// per-workgroup compensated partial sums of the 8 thermo quantities
// (find_owned_thermo_sums, runtime.cu:442-493)
__global__ __launch_bounds__(kThermoThreads) void k_thermo_partial(int N, const double* __restrict__ mass,
                                                                   const double* __restrict__ pe,
                                                                   const double* __restrict__ vel,
                                                                   const double* __restrict__ vir,
                                                                   double* __restrict__ partial)
{
#pragma clang fp contract(off)
  KSum acc[8];
#pragma unroll
  for (int q = 0; q < 8; ++q) acc[q] = {0.0, 0.0};
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < N; i += gridDim.x * blockDim.x) {
    const double m = mass[i];
    const double vx = vel[i], vy = vel[N + i], vz = vel[2 * N + i];
    ksum_add(acc[0], m * (vx * vx + vy * vy + vz * vz));
    ksum_add(acc[1], pe[i]);
    ksum_add(acc[2], vir[i] + m * vx * vx);
    ksum_add(acc[3], vir[N + i] + m * vy * vy);
    ksum_add(acc[4], vir[2 * N + i] + m * vz * vz);
    ksum_add(acc[5], vir[3 * N + i] + m * vx * vy);
    ksum_add(acc[6], vir[4 * N + i] + m * vx * vz);
    ksum_add(acc[7], vir[5 * N + i] + m * vy * vz);
  }
  block_reduce8(acc);
  if (threadIdx.x == 0)
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      partial[(blockIdx.x * 8 + q) * 2 + 0] = acc[q].s;
      partial[(blockIdx.x * 8 + q) * 2 + 1] = acc[q].c;
    }
}

// Second half kick of the MD step fused with the per-workgroup thermo
// partial sums of the kicked velocities (the sums of k_thermo_partial).
template <bool THERMO>
__global__ __launch_bounds__(kThermoThreads) void k_md_second(int N, double dt, const double* __restrict__ mass,
                                                              double* __restrict__ vel,
                                                              const double* __restrict__ force,
                                                              const double* __restrict__ pe,
                                                              const double* __restrict__ vir,
                                                              double* __restrict__ partial)
{
#pragma clang fp contract(off)
  KSum acc[8];
#pragma unroll
  for (int q = 0; q < 8; ++q) acc[q] = {0.0, 0.0};
  const double half = dt * 0.5;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < N; i += gridDim.x * blockDim.x) {
    const double m = mass[i];
    const double im = 1.0 / m;
    double v3[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const double v = vel[c * N + i] + force[c * N + i] * im * half;
      vel[c * N + i] = v;
      v3[c] = v;
    }
    if (THERMO) {
      const double vx = v3[0], vy = v3[1], vz = v3[2];
      ksum_add(acc[0], m * (vx * vx + vy * vy + vz * vz));
      ksum_add(acc[1], pe[i]);
      ksum_add(acc[2], vir[i] + m * vx * vx);
      ksum_add(acc[3], vir[N + i] + m * vy * vy);
      ksum_add(acc[4], vir[2 * N + i] + m * vz * vz);
      ksum_add(acc[5], vir[3 * N + i] + m * vx * vy);
      ksum_add(acc[6], vir[4 * N + i] + m * vx * vz);
      ksum_add(acc[7], vir[5 * N + i] + m * vy * vz);
    }
  }
  if (THERMO) {
    block_reduce8(acc);
    if (threadIdx.x == 0)
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        partial[(blockIdx.x * 8 + q) * 2 + 0] = acc[q].s;
        partial[(blockIdx.x * 8 + q) * 2 + 1] = acc[q].c;
      }
  }
}

// normalize_global_thermo (runtime_internal.hpp:704-716): T = sum m v^2/(3 N kB), stress/V
// With step_index, the step's target temperature and draws are
// targets[k] and rand2[2k .. 2k+1] for k = *step_index, which the kernel then
// advances: the same launch serves every step of a chunk (a replayed graph).
// Without rand2 the draws are d0 and d1.  With report (pinned host memory)
// the thermo goes there too: a step that the host waits for needs no copy.
__global__ __launch_bounds__(kThermoThreads) void k_thermo_final(int nb, int N, double volume,
                                                                 const double* __restrict__ partial,
                                                                 double* __restrict__ thermo, int kind,
                                                                 double coupling, double t_target,
                                                                 const double* __restrict__ rand2,
                                                                 double* __restrict__ factor,
                                                                 const double* __restrict__ targets,
                                                                 int* __restrict__ step_index, double d0, double d1,
                                                                 double* __restrict__ report)
{
  KSum acc[8];
#pragma unroll
  for (int q = 0; q < 8; ++q) acc[q] = {0.0, 0.0};
  for (int b = threadIdx.x; b < nb; b += blockDim.x)
#pragma unroll
    for (int q = 0; q < 8; ++q) ksum_merge(acc[q], KSum{partial[(b * 8 + q) * 2], partial[(b * 8 + q) * 2 + 1]});
  block_reduce8(acc);
  if (threadIdx.x == 0) {
    if (step_index) {
      const int k = *step_index;
      t_target = targets[k];
      rand2 += 2 * k;
      *step_index = k + 1;
    }
    const double draws[2] = {d0, d1};
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      double v = acc[q].s + acc[q].c;
      if (q == 0) v /= 3.0 * N * 8.617343e-5;
      else if (q >= 2) v /= volume;
      thermo[q] = v;
      if (report) report[q] = v;
      if (q == 0 && factor) factor[0] = ensemble_factor(kind, N, coupling, t_target, rand2 ? rand2 : draws, v);
    }
  }
}

__global__ void k_chunk_start(double* __restrict__ factor, int* __restrict__ step_index)
{
  factor[0] = 1.0;
  *step_index = 0;
}

// Several arrays copied by one launch (a chunk's checkpoint; up to six copies
// of a few microseconds each otherwise).  Bound by memory: 19 doubles an atom
// read and written.
__global__ __launch_bounds__(kBlock) void k_copy_arrays(ArrayCopies c)
{
  const long long t = blockIdx.x * (long long)kBlock + threadIdx.x, stride = (long long)gridDim.x * kBlock;
#pragma unroll
  for (int a = 0; a < kMaxCopies; ++a) {
    const long long pairs = c.n[a] >> 1;
    for (long long k = t; k < pairs; k += stride)
      reinterpret_cast<double2*>(c.to[a])[k] = reinterpret_cast<const double2*>(c.from[a])[k];
    if (t == 0 && (c.n[a] & 1)) c.to[a][c.n[a] - 1] = c.from[a][c.n[a] - 1];
  }
}

__global__ void k_ensemble_factor(int kind, int N, double coupling, double t_target,
                                  const double* __restrict__ rand2, const double* __restrict__ thermo,
                                  double* __restrict__ factor)
{
  factor[0] = ensemble_factor(kind, N, coupling, t_target, rand2, thermo[0]);
}

__global__ void k_scale_by(int n, const double* __restrict__ factor, double* __restrict__ data)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) data[i] *= factor[0];
}

__global__ void k_scale(int n, double factor, double* __restrict__ data)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) data[i] *= factor;
}

__global__ void k_check_scaled(int n, double factor, const double* __restrict__ data, int* __restrict__ flag)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n && !isfinite(data[i] * factor)) atomicOr(flag, 1);
}

// ---------------------------------------------------------------------------
// launch wrappers
// ---------------------------------------------------------------------------

static inline int nblk(int n) { return (n + kBlock - 1) / kBlock; }

// closes a rebuild request as the filter does, for an evaluation whose
// first filter launch has no centres
__global__ void k_close_request(int* __restrict__ flags)
{
  if (flags[kFlagRebuild]) {
    flags[kFlagRebuild] = 0;
    flags[kFlagRebuildCount] += 1;
  }
}

// lanes per centre (8, 16 or 32) and the Verlet entries each lane loads
// per pass (7, 5 or 4)
template <int G, int RB, bool CAND = false>
static void run_filter(const DevBox& b, const DevModel& m, int c1, int c2, int close, DevWork& w, hipStream_t s)
{
  constexpr int per = kBlock / G;
  const int nb = (c2 - c1 + per - 1) / per;
  if (w.map.owner) {
    if (m.T == 1) k_filter<true, true, G, RB, CAND><<<xcd_grid(nb), kBlock, 0, s>>>(b, m, c1, c2, nb, close, w);
    else k_filter<false, true, G, RB, CAND><<<xcd_grid(nb), kBlock, 0, s>>>(b, m, c1, c2, nb, close, w);
  } else {
    if (m.T == 1) k_filter<true, false, G, RB, CAND><<<xcd_grid(nb), kBlock, 0, s>>>(b, m, c1, c2, nb, close, w);
    else k_filter<false, false, G, RB, CAND><<<xcd_grid(nb), kBlock, 0, s>>>(b, m, c1, c2, nb, close, w);
  }
  if (CAND) k_split_reverse<G><<<xcd_grid(nb), kBlock, 0, s>>>(c1, c2, nb, w);
}

hipError_t launch_split(const DevBox& b, const DevModel& m, int c1, int c2, DevWork& w, hipStream_t s, int lanes)
{
  if (!w.split || !w.cl) return hipErrorInvalidValue;
  if (c2 > c1) {
    if (lanes == 8) run_filter<8, 7, true>(b, m, c1, c2, 0, w, s);
    else if (lanes == 32) run_filter<32, 4, true>(b, m, c1, c2, 0, w, s);
    else run_filter<kFilterLanes, kFilterBatch, true>(b, m, c1, c2, 0, w, s);
  } else {
    k_close_request<<<1, 1, 0, s>>>(w.flags);  // no descriptor launch closes it
  }
  return hipGetLastError();
}

hipError_t launch_filter(const DevBox& b, const DevModel& m, int c1, int c2, DevWork& w, hipStream_t s, int lanes,
                         bool close)
{
  if (c2 > c1) {
    const int cl = close ? 1 : 0;
    if (lanes == 8) run_filter<8, 7>(b, m, c1, c2, cl, w, s);
    else if (lanes == 32) run_filter<32, 4>(b, m, c1, c2, cl, w, s);
    else run_filter<kFilterLanes, kFilterBatch>(b, m, c1, c2, cl, w, s);
  } else if (close) {
    k_close_request<<<1, 1, 0, s>>>(w.flags);
  }
  return hipGetLastError();
}

template <int G>
static void run_gather(const DevBox& b, const DevModel& m, int N, int n1, int n2, int nd1, int nd2, const int* type,
                       double* force, double* virial, int a, DevWork& w, hipStream_t s)
{
  constexpr int per = kBlock / G;
  const int nb = (n2 - (n1 & ~(kTile - 1)) + per - 1) / per;
  const int g = xcd_grid(nb);
  auto pick = [&](auto k_rows, auto k_cand) { return w.split ? k_cand : k_rows; };
  decltype(&k_gather<9, true, G, false>) k;
  if (m.T == 1 && m.kR == 9) k = pick(k_gather<9, true, G, false>, k_gather<9, true, G, true>);
  else if (m.T == 1) k = pick(k_gather<kMaxK, true, G, false>, k_gather<kMaxK, true, G, true>);
  else if (m.kR <= 11) k = pick(k_gather<11, false, G, false>, k_gather<11, false, G, true>);
  else k = pick(k_gather<kMaxK, false, G, false>, k_gather<kMaxK, false, G, true>);
  k<<<g, kBlock, 0, s>>>(b, m, n1, n2, nd1, nd2, nb, type, N, force, virial, a, w);
}

hipError_t launch_gather(const DevBox& b, const DevModel& m, int N, int n1, int n2, int nd1, int nd2,
                         const int* type, double* force, double* virial, bool acc, DevWork& w, hipStream_t s,
                         int lanes)
{
  if (n2 <= n1) return hipSuccess;
  const int a = acc ? 1 : 0;
  if (lanes == 4) run_gather<4>(b, m, N, n1, n2, nd1, nd2, type, force, virial, a, w, s);
  else if (lanes == 16) run_gather<16>(b, m, N, n1, n2, nd1, nd2, type, force, virial, a, w, s);
  else run_gather<kGatherLanes>(b, m, N, n1, n2, nd1, nd2, type, force, virial, a, w, s);
  return hipGetLastError();
}

hipError_t launch_velocity_verlet(int first_half, int N, double dt, const double* mass, double* pos,
                                  double* vel, const double* force, hipStream_t s, double* unwrapped)
{
  if (N > 0) k_velocity_verlet<<<nblk(N), kBlock, 0, s>>>(first_half, N, dt, mass, pos, vel, force, unwrapped);
  return hipGetLastError();
}

hipError_t launch_wrap(const DevBox& b, int N, double* pos, hipStream_t s)
{
  if (N > 0) k_wrap<<<nblk(N), kBlock, 0, s>>>(b, N, pos);
  return hipGetLastError();
}

hipError_t launch_thermo(int N, double volume, const double* mass, const double* pe, const double* vel,
                         const double* virial, DevWork& w, hipStream_t s)
{
  const int nb = thermo_blocks(N);
  k_thermo_partial<<<nb, kThermoThreads, 0, s>>>(N, mass, pe, vel, virial, w.partial);
  k_thermo_final<<<1, kThermoThreads, 0, s>>>(nb, N, volume, w.partial, w.thermo, 0, 0.0, 0.0, nullptr, nullptr,
                                              nullptr, nullptr, 0.0, 0.0, nullptr);
  return hipGetLastError();
}

hipError_t launch_scale(int n, double factor, double* data, hipStream_t s)
{
  if (n > 0) k_scale<<<nblk(n), kBlock, 0, s>>>(n, factor, data);
  return hipGetLastError();
}

hipError_t launch_ensemble_scale(int kind, int N, double coupling, double t_target, const double* rand2,
                                 double* factor, const double* thermo, double* vel, hipStream_t s)
{
  k_ensemble_factor<<<1, 1, 0, s>>>(kind, N, coupling, t_target, rand2, thermo, factor);
  k_scale_by<<<nblk(3 * N), kBlock, 0, s>>>(3 * N, factor, vel);
  return hipGetLastError();
}

hipError_t launch_md_first(const DevBox& b, int N, int T, double dt, const double* mass, double* pos, double* vel,
                           const double* force, const double* factor, const int* type, bool forced, DevWork& w,
                           hipStream_t s, double* unwrapped, double half_skin, bool kick)
{
  const double half = half_skin > 0.0 ? half_skin : 0.5 * kSkin;
  if (N > 0)
    (kick ? k_md_first<true> : k_md_first<false>)<<<nblk(N), kBlock, 0, s>>>(
        b, N, T, dt, mass, pos, vel, force, factor, type, w.x0, half * half, forced ? 1 : 0, w.xq, w.flags, unwrapped);
  return hipGetLastError();
}

hipError_t launch_md_second(int N, double dt, const double* mass, double* vel, const double* force, const double* pe,
                            const double* virial, bool thermo, DevWork& tw, hipStream_t s)
{
  if (N <= 0) return hipSuccess;
  const int nb = thermo_blocks(N);
  if (thermo)
    k_md_second<true><<<nb, kThermoThreads, 0, s>>>(N, dt, mass, vel, force, pe, virial, tw.partial);
  else
    k_md_second<false><<<nb, kThermoThreads, 0, s>>>(N, dt, mass, vel, force, pe, virial, tw.partial);
  return hipGetLastError();
}

hipError_t launch_thermo_final(int N, double volume, int kind, double coupling, double t_target,
                               const double* rand2, double* factor, DevWork& tw, hipStream_t s,
                               const double* targets, int* step_index, const double* draws, double* report)
{
  k_thermo_final<<<1, kThermoThreads, 0, s>>>(thermo_blocks(N), N, volume, tw.partial, tw.thermo, kind, coupling,
                                              t_target, rand2, kind ? factor : nullptr, targets, step_index,
                                              draws ? draws[0] : 0.0, draws ? draws[1] : 0.0, report);
  return hipGetLastError();
}

hipError_t launch_copy_arrays(const ArrayCopies& c, hipStream_t s)
{
  long long most = 0;
  for (long long n : c.n) most = std::max(most, n);
  if (most > 0) k_copy_arrays<<<(int)std::min<long long>((most / 2 + kBlock) / kBlock, 4096), kBlock, 0, s>>>(c);
  return hipGetLastError();
}

hipError_t launch_chunk_start(double* factor, int* step_index, hipStream_t s)
{
  k_chunk_start<<<1, 1, 0, s>>>(factor, step_index);
  return hipGetLastError();
}

hipError_t launch_scale_by(int n, const double* factor, double* data, hipStream_t s)
{
  if (n > 0) k_scale_by<<<nblk(n), kBlock, 0, s>>>(n, factor, data);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// small boxes: periodic replicas and the fold of their results
// ---------------------------------------------------------------------------

// Replica k = (ia, ib, ic) of atom i lands at slot k*N + i, shifted by
// ia*a + ib*b + ic*c (the box columns); replica 0 is the original.
__global__ void k_replicate(int N, int r0, int r1, int r2, DevBox b, const double* __restrict__ pos,
                            const int* __restrict__ type, const uint64_t* __restrict__ gid,
                            double* __restrict__ pos2, int* __restrict__ type2, uint64_t* __restrict__ gid2)
{
#pragma clang fp contract(off)
  const int R = r0 * r1 * r2;
  const long long n2 = (long long)N * R;
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n2) return;
  const int k = (int)(t / N), i = (int)(t % N);
  const int ia = k % r0, ib = (k / r0) % r1, ic = k / (r0 * r1);
#pragma unroll
  for (int c = 0; c < 3; ++c)
    pos2[c * n2 + t] = pos[c * N + i] + (ia * b.h[3 * c] + ib * b.h[3 * c + 1] + ic * b.h[3 * c + 2]);
  type2[t] = type[i];
  if (gid) gid2[t] = gid[i];
}

// Copies (or adds) the first N entries of each component of the replicated
// outputs (stride n2) into the caller's arrays (stride N).
__global__ void k_fold(int N, long long n2, int accumulate, const double* __restrict__ pe2,
                       const double* __restrict__ f2, const double* __restrict__ v2, double* __restrict__ pe,
                       double* __restrict__ force, double* __restrict__ virial)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= N) return;
  if (accumulate) {
    pe[i] += pe2[i];
#pragma unroll
    for (int c = 0; c < 3; ++c) force[c * N + i] += f2[c * n2 + i];
#pragma unroll
    for (int c = 0; c < 9; ++c) virial[(size_t)c * N + i] += v2[c * n2 + i];
  } else {
    pe[i] = pe2[i];
#pragma unroll
    for (int c = 0; c < 3; ++c) force[c * N + i] = f2[c * n2 + i];
#pragma unroll
    for (int c = 0; c < 9; ++c) virial[(size_t)c * N + i] = v2[c * n2 + i];
  }
}

hipError_t launch_replicate(int N, const int reps[3], const DevBox& b, const double* pos, const int* type,
                            const uint64_t* gid, double* pos2, int* type2, uint64_t* gid2, hipStream_t s)
{
  const long long n2 = (long long)N * reps[0] * reps[1] * reps[2];
  if (n2 > 0)
    k_replicate<<<(unsigned)((n2 + kBlock - 1) / kBlock), kBlock, 0, s>>>(N, reps[0], reps[1], reps[2], b, pos,
                                                                        type, gid, pos2, type2, gid2);
  return hipGetLastError();
}

hipError_t launch_fold(int N, long long n2, bool accumulate, const double* pe2, const double* f2, const double* v2,
                       double* pe, double* force, double* virial, hipStream_t s)
{
  if (N > 0) k_fold<<<nblk(N), kBlock, 0, s>>>(N, n2, accumulate ? 1 : 0, pe2, f2, v2, pe, force, virial);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// serving loop: masked integrator, ghost refresh, relayout and extraction
// ---------------------------------------------------------------------------

// velocity-Verlet half step of the owned atoms whose request takes an MD
// step this iteration (the FP64 expressions of k_velocity_verlet)
__global__ void k_serve_kick(int first_half, int n, int Nt, const int* __restrict__ atom_req,
                             const int* __restrict__ req_md, const double* __restrict__ req_dt,
                             const double* __restrict__ mass, double* __restrict__ pos, double* __restrict__ vel,
                             const double* __restrict__ force)
{
#pragma clang fp contract(off)
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int r = atom_req[i];
  if (!req_md[r]) return;
  const double dt = req_dt[r];
  const double half = dt * 0.5;
  const double im = 1.0 / mass[i];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const double v = vel[c * Nt + i] + force[c * Nt + i] * im * half;
    vel[c * Nt + i] = v;
    if (first_half) pos[c * Nt + i] += v * dt;
  }
}

// ghost k (slot n_owned + k) = its owner + a box shift
__global__ void k_serve_ghosts(int n_owned, int n_ghost, int Nt, const int* __restrict__ owner,
                               const double* __restrict__ shift, double* __restrict__ pos)
{
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n_ghost) return;
  const int g = n_owned + k, o = owner[k];
#pragma unroll
  for (int c = 0; c < 3; ++c) pos[c * Nt + g] = pos[c * Nt + o] + shift[3 * k + c];
}

// owned atoms of continuing requests move to their new slots (and regions)
// Assembly of a new serving layout, one thread per slot: the slot's request
// is found by binary search over the requests' first slots (both slot ranges
// are in request order and tile [0, n_owned) and [n_owned, Nt)).
__global__ void k_serve_assemble(int R, const ServeSlots* __restrict__ req, ServeLayout from, ServeLayout to,
                                 int* __restrict__ atom_req)
{
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  const int Nt = to.Nt, no = to.n_owned;
  if (s == 0) to.gstart[no] = Nt;
  if (s >= Nt) return;
  const bool owned = s < no;
  int lo = 0, hi = R - 1;
  while (lo < hi) {  // last request whose range starts at or before s
    const int mid = (lo + hi + 1) >> 1;
    if ((owned ? req[mid].new_o : req[mid].new_g) <= s) lo = mid;
    else hi = mid - 1;
  }
  const ServeSlots q = req[lo];
  if (owned) {
    const int k = s - q.new_o;
    atom_req[s] = lo;
    to.owner[s] = s;
    to.image[s] = image_code(0, 0, 0);
    if (q.old_o >= 0) {
      const int src = q.old_o + k;
      to.type[s] = from.type[src];
      to.mass[s] = from.mass[src];
      to.gstart[s] = q.new_g + (from.gstart[src] - q.old_g);
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        to.pos[c * Nt + s] = from.pos[c * from.Nt + src] + q.dtr[c];
        to.vel[c * Nt + s] = from.vel[c * from.Nt + src];
        to.force[c * Nt + s] = from.force[c * from.Nt + src];
        to.home[c * no + s] = from.home[c * from.n_owned + src] + q.dtr[c];
      }
    } else {
      to.type[s] = q.pi[k];
      to.gstart[s] = q.new_g + q.pi[q.n + k];
      to.mass[s] = q.pd[k];
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const double x = q.pd[q.n + 3 * k + c] + q.dtr[c];
        to.pos[c * Nt + s] = x;
        to.home[c * no + s] = x;
        to.vel[c * Nt + s] = q.pd[4 * q.n + 3 * k + c];
        to.force[c * Nt + s] = q.pd[7 * q.n + 3 * k + c];
      }
    }
  } else {
    const int k = s - q.new_g;
    const int g = s - no;
    if (q.old_g >= 0) {
      const int src = q.old_g + k;
      to.owner[s] = q.new_o + (from.owner[src] - q.old_o);
      to.image[s] = from.image[src];
      to.type[s] = from.type[src];
      to.mass[s] = from.mass[src];
#pragma unroll
      for (int c = 0; c < 3; ++c) to.gshift[3 * g + c] = from.gshift[3 * (src - from.n_owned) + c];
    } else {
      const int a = q.pi[2 * q.n + k];
      to.owner[s] = q.new_o + a;
      to.image[s] = q.pi[2 * q.n + q.ng + k];
      to.type[s] = q.pi[a];
      to.mass[s] = q.pd[a];
#pragma unroll
      for (int c = 0; c < 3; ++c) to.gshift[3 * g + c] = q.pd[10 * q.n + 3 * k + c];
    }
  }
}

// the request of slot s among the first R table rows (last whose range starts
// at or before s), by owned or ghost range
__device__ __forceinline__ int serve_request_of(int R, const ServeSlots* __restrict__ req, int s, bool owned)
{
  int lo = 0, hi = R - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if ((owned ? req[mid].new_o : req[mid].new_g) <= s) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

constexpr int kCarryLanes = 16;  // lanes per row in k_serve_carry_rows

__global__ void k_serve_carry_rows(int R, const ServeSlots* __restrict__ req, int old_no, int o_keep,
                                   const int* __restrict__ vl0, const short* __restrict__ vrev0,
                                   const int* __restrict__ vn0, DevWork w)
{
  const int s = blockIdx.x * (blockDim.x / kCarryLanes) + threadIdx.x / kCarryLanes;
  const int lane = threadIdx.x % kCarryLanes;
  if (s >= o_keep) return;
  const ServeSlots t = req[serve_request_of(R, req, s, true)];
  const int so = t.old_o + (s - t.new_o);
  const int n = vn0[so];
  if (lane == 0) w.vn[s] = n;
  const int m = min(n, w.MV);
  const size_t ro = (size_t)so * w.MV, rn = (size_t)s * w.MV;
  // every entry of a request's row is one of its own slots (requests are
  // disjoint in space): owned slots and ghosts each keep their offset
  for (int p = lane; p < m; p += kCarryLanes) {
    const int j = vl0[ro + p];
    w.vl[rn + p] = j < old_no ? t.new_o + (j - t.old_o) : t.new_g + (j - t.old_g);
    w.vrev[rn + p] = vrev0[ro + p];
  }
}

__global__ void k_serve_carry_x0(int R, const ServeSlots* __restrict__ req, int old_nt, int new_no, int new_nt,
                                 int o_keep, int g_keep, const double* __restrict__ x0_0, double* __restrict__ x0)
{
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  const int total = o_keep + (g_keep - new_no);
  if (k >= total) return;
  const bool owned = k < o_keep;
  const int s = owned ? k : new_no + (k - o_keep);
  const ServeSlots t = req[serve_request_of(R, req, s, owned)];
  const int so = owned ? t.old_o + (s - t.new_o) : t.old_g + (s - t.new_g);
#pragma unroll
  for (int c = 0; c < 3; ++c) x0[(size_t)c * new_nt + s] = x0_0[(size_t)c * old_nt + so] + t.dtr[c];
}

__global__ void k_serve_drift(int n_owned, int Nt, const int* __restrict__ atom_req, const double* __restrict__ pos,
                              const double* __restrict__ home, double soft2, double hard2, int* __restrict__ req_flag)
{
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n_owned) return;
  double d2 = 0.0;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const double d = pos[c * Nt + s] - home[c * n_owned + s];
    d2 += d * d;
  }
  if (!(d2 <= soft2)) atomicMax(&req_flag[atom_req[s]], (d2 <= hard2) ? 1 : 2);
}

// finished requests -> their result blocks, one thread per atom; the
// request is found by binary search over the blocks' first atoms
__global__ void k_serve_extract(int R, const ServeOut* __restrict__ req, long long no, int Nt,
                                const double* __restrict__ pos, const double* __restrict__ vel,
                                const double* __restrict__ force, const double* __restrict__ pe,
                                const double* __restrict__ vir, double* __restrict__ out)
{
  const long long k = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= no) return;
  int lo = 0, hi = R - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (req[mid].out / kServeOutDoubles <= k) lo = mid;
    else hi = mid - 1;
  }
  const ServeOut& q = req[lo];
  const int a = (int)(k - q.out / kServeOutDoubles), n = q.n, i = q.slot0 + a;
  double* blk = out + q.out;
  blk[a] = pe[i];
  double x[3], f[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    x[c] = pos[c * Nt + i] - q.trans[c];
    blk[n + c * n + a] = force[c * Nt + i];
    blk[7 * n + c * n + a] = vel[c * Nt + i];
  }
#pragma unroll
  for (int c = 0; c < 9; ++c) blk[10 * n + c * n + a] = vir[(size_t)c * Nt + i];
  // back into the request's box: fractional coordinates, wrapped where periodic
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    f[c] = q.hi[3 * c] * x[0] + q.hi[3 * c + 1] * x[1] + q.hi[3 * c + 2] * x[2];
    if (q.pbc[c]) f[c] -= floor(f[c]);
  }
#pragma unroll
  for (int c = 0; c < 3; ++c) blk[4 * n + c * n + a] = q.h[3 * c] * f[0] + q.h[3 * c + 1] * f[1] + q.h[3 * c + 2] * f[2];
}

hipError_t launch_serve_kick(int first_half, int n, int Nt, const int* atom_req, const int* req_md,
                             const double* req_dt, const double* mass, double* pos, double* vel, const double* force,
                             hipStream_t s)
{
  if (n > 0) k_serve_kick<<<nblk(n), kBlock, 0, s>>>(first_half, n, Nt, atom_req, req_md, req_dt, mass, pos, vel, force);
  return hipGetLastError();
}

hipError_t launch_serve_ghosts(int n_owned, int n_ghost, int Nt, const int* owner, const double* shift, double* pos,
                               hipStream_t s)
{
  if (n_ghost > 0) k_serve_ghosts<<<nblk(n_ghost), kBlock, 0, s>>>(n_owned, n_ghost, Nt, owner, shift, pos);
  return hipGetLastError();
}

hipError_t launch_serve_assemble(int R, const ServeSlots* req, const ServeLayout& from, const ServeLayout& to,
                                 int* atom_req, hipStream_t s)
{
  if (R > 0 && to.Nt > 0) k_serve_assemble<<<nblk(to.Nt), kBlock, 0, s>>>(R, req, from, to, atom_req);
  return hipGetLastError();
}

hipError_t launch_serve_carry_rows(int R_keep, const ServeSlots* req, int old_no, int old_nt, int new_no, int new_nt,
                                   int o_keep, int g_keep, const int* vl0, const short* vrev0, const int* vn0,
                                   const double* x0_0, DevWork& w, hipStream_t s)
{
  if (R_keep <= 0) return hipSuccess;
  if (o_keep > 0) {
    constexpr int per = kBlock / kCarryLanes;
    k_serve_carry_rows<<<(o_keep + per - 1) / per, kBlock, 0, s>>>(R_keep, req, old_no, o_keep, vl0, vrev0, vn0, w);
  }
  const int total = o_keep + (g_keep - new_no);
  if (total > 0)
    k_serve_carry_x0<<<nblk(total), kBlock, 0, s>>>(R_keep, req, old_nt, new_no, new_nt, o_keep, g_keep, x0_0, w.x0);
  return hipGetLastError();
}

hipError_t launch_serve_drift(int n_owned, int Nt, const int* atom_req, const double* pos, const double* home,
                              double soft2, double hard2, int* req_flag, hipStream_t s)
{
  if (n_owned > 0)
    k_serve_drift<<<nblk(n_owned), kBlock, 0, s>>>(n_owned, Nt, atom_req, pos, home, soft2, hard2, req_flag);
  return hipGetLastError();
}

hipError_t launch_serve_extract(int R, const ServeOut* req, long long no, int Nt, const double* pos,
                                const double* vel, const double* force, const double* pe, const double* vir,
                                double* out, hipStream_t s)
{
  if (R > 0 && no > 0)
    k_serve_extract<<<(unsigned)((no + kBlock - 1) / kBlock), kBlock, 0, s>>>(R, req, no, Nt, pos, vel, force, pe,
                                                                             vir, out);
  return hipGetLastError();
}

// largest |v|^2: a wavefront maximum, then one atomicMax per wavefront on
// the bit pattern (non-negative doubles order as their bits)
__global__ void k_max_speed2(int N, const double* __restrict__ vel, unsigned long long* __restrict__ out)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  double v2 = 0.0;
  if (i < N) {
    const double x = vel[i], y = vel[N + i], z = vel[2 * N + i];
    v2 = x * x + y * y + z * z;
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v2 = fmax(v2, __shfl_xor(v2, off, 64));
  if ((threadIdx.x & 63) == 0) atomicMax(out, (unsigned long long)__double_as_longlong(v2));
}

__global__ void k_clear_u64(unsigned long long* p) { *p = 0ull; }

hipError_t launch_max_speed2(int N, const double* vel, unsigned long long* out, hipStream_t s)
{
  k_clear_u64<<<1, 1, 0, s>>>(out);
  if (N > 0) k_max_speed2<<<nblk(N), kBlock, 0, s>>>(N, vel, out);
  return hipGetLastError();
}

hipError_t launch_check_scaled(int n, double factor, const double* data, int* flag, hipStream_t s)
{
  if (n > 0) k_check_scaled<<<nblk(n), kBlock, 0, s>>>(n, factor, data, flag);
  return hipGetLastError();
}

}  // namespace dmgx
