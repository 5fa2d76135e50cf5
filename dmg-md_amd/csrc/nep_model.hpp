// nep_model.hpp -- host representation of a parsed nep.txt and its device
// parameter image.
//
// Grammar and parameter layout follow the reference loader
// NEP::NEP(const char*) (src/gpumd_compat/nep.cu:135-415) and the pointer
// layout of NEP::update_potential (nep.cu:464-496).
#pragma once

#include <cstdint>
#include <numeric>
#include <string>
#include <vector>

namespace dmgx {

constexpr int kMaxTypes = 16;   // per-type device tables
constexpr int kMaxL = 8;        // 3-body angular order supported (nep_utilities.cuh:50, 80 moments)
constexpr int kPadL = 4;        // 3-body order of the bounded instances models are padded to
constexpr int kMaxNA = 10;      // n_max_angular + 1
constexpr int kMaxNR = 16;      // n_max_radial + 1
constexpr int kMaxK = 17;       // basis_size + 1 (nep_utilities.cuh MAX_NUM_N)
constexpr int kMaxDim = 128;
constexpr int kMaxNeurons = 128;

struct NepModel {
  int version = 4;
  int num_types = 0;
  std::vector<std::string> symbols;
  int Z[kMaxTypes] = {};
  bool zbl_enabled = false, zbl_flexible = false, zbl_typewise = false;
  double zbl_rc_inner = 0.0, zbl_rc_outer = 0.0, zbl_factor = 0.0;
  std::vector<double> zbl_para;  // 10 per unordered type pair (flexible ZBL)
  double rcR[kMaxTypes] = {}, rcA[kMaxTypes] = {};
  double rcR_max = 0.0, rcA_max = 0.0;
  int MN_R = 0, MN_A = 0;        // enlarged x1.25 (nep.cu:267-268)
  int nR = 0, nA = 0;            // n_max + 1
  int kR = 0, kA = 0;            // basis_size + 1
  int L_max = 0;
  int has222 = 0, has1111 = 0;
  int num_L = 0, dim = 0, H = 0;
  int num_para_ann = 0, num_para_desc = 0;
  std::vector<double> params;    // ann | descriptor (file order) | q_scaler

  // Parses `path`; throws std::invalid_argument with a message on any error.
  void load(const std::string& path);

  // Flat float image uploaded to the device; offsets in floats.
  struct Image {
    std::vector<float> data;
    int off_w0, off_b0, off_w1, off_w1x, off_b1, off_cR, off_cA, off_qs, off_zbl;
  };
  Image device_image() const;
};

// Closed-form angular constants: weights of s^2 in q_L (factor 2 of m>0
// folded in), integer coefficients of Z_{L,m}(z) = primitive part of
// d^m P_L/dz^m, and the q_222 / q_1111 weights (Wigner-3j couplings).
struct AngularConstants {
  float c3[(kMaxL + 1) * (kMaxL + 1) - 1] = {};
  float zc[kMaxL + 1][kMaxL + 1][kMaxL + 1] = {};
  float c4[5] = {};
  float c5 = 0.0f;
};
constexpr AngularConstants derive_angular_constants()
{
  AngularConstants a{};
  const double pi = 3.14159265358979323846, pi32 = 5.56832799683170784528;  // pi^(3/2)
  auto binom = [](int n, int k) {
    long long r = 1;
    for (int i = 1; i <= k; ++i) r = r * (n - k + i) / i;
    return r;
  };
  for (int L = 1; L <= kMaxL; ++L) {
    // 2^L P_L(z) = sum_k (-1)^k C(L,k) C(2L-2k,L) z^(L-2k)
    long long base[kMaxL + 1] = {};
    for (int k = 0; 2 * k <= L; ++k) {
      const long long val = binom(L, k) * binom(2 * L - 2 * k, L);
      base[L - 2 * k] = (k % 2) ? -val : val;
    }
    double scale = 1.0;  // 2^L
    for (int k = 0; k < L; ++k) scale *= 2.0;
    for (int m = 0; m <= L; ++m) {
      long long d[kMaxL + 1] = {};
      for (int p = m; p <= L; ++p) {
        long long f = 1;
        for (int s = 0; s < m; ++s) f *= (p - s);
        d[p - m] = base[p] * f;
      }
      long long g = 0;
      for (int p = 0; p <= L - m; ++p)
        if (d[p]) g = std::gcd(g, d[p] < 0 ? -d[p] : d[p]);
      for (int p = 0; p <= L - m; ++p) a.zc[L][m][p] = (float)(d[p] / g);
      const double alpha = (double)g / scale;
      double fr = 1.0;
      for (int s = L - m + 1; s <= L + m; ++s) fr /= (double)s;
      const double w = (2.0 * L + 1.0) / (4.0 * pi) * fr * alpha * alpha;
      const int b = L * L - 1;
      if (m == 0) {
        a.c3[b] = (float)w;
      } else {
        a.c3[b + 2 * m - 1] = (float)(2.0 * w);
        a.c3[b + 2 * m] = (float)(2.0 * w);
      }
    }
  }
  // q_222: Wigner-3j (2 2 2; m1 m2 m3) coupling of three l=2 moments, weights
  // k*sqrt(14)/(448 pi^1.5) for s3^3, s3(s4^2+s5^2), s3(s6^2+s7^2),
  // s6(s5^2-s4^2), s4 s5 s7.
  const double u4 = 3.74165738677394138558 / (448.0 * pi32);
  const double k4[5] = {-5.0, -90.0, 45.0, 270.0, -540.0};
  for (int i = 0; i < 5; ++i) a.c4[i] = (float)(k4[i] * u4);
  // q_1111: sum over intermediate L of (1 1 L)(L 1 1) couplings = 21/(80 pi^2) |s_1|^4
  a.c5 = (float)(21.0 / (80.0 * pi * pi));
  return a;
}

}  // namespace dmgx
