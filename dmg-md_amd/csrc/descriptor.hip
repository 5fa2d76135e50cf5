// descriptor.hip -- picks the descriptor instance of a model.
#include "descriptor.hpp"

namespace dmgx {

namespace {
bool model_is(const DevModel& m, int nr, int kr, int na, int ka, int L, bool a, bool b, bool one)
{
  return m.nR == nr && m.kR == kr && m.nA == na && m.kA == ka && m.L == L && (m.has222 != 0) == a &&
         (m.has1111 != 0) == b && (m.T == 1) == one;
}

// sizes of the exactly instantiated configurations (nR, kR, nA, kA, q222,
// q1111, single type); the bounded sizes below come after them
struct ExactCfg {
  int nr, kr, na, ka;
  bool q2, q1, one;
};
constexpr ExactCfg kExact[] = {
    {5, 9, 5, 9, true, true, true},     {7, 9, 5, 9, true, false, true},   {13, 17, 9, 13, true, true, true},
    {7, 11, 7, 11, true, true, false},  {5, 9, 5, 9, true, false, false},  {9, 9, 7, 9, false, false, false},
    {7, 9, 5, 9, true, true, true},     {7, 9, 5, 9, true, true, false},   {9, 13, 7, 13, true, true, true},
    {9, 13, 7, 13, true, true, false}};
constexpr int kBuckets[][4] = {{7, 9, 5, 9}, {9, 13, 7, 13}};
}  // namespace

bool descriptor_bucket(const DevModel& m, int dims[4])
{
  for (const ExactCfg& c : kExact)
    if (model_is(m, c.nr, c.kr, c.na, c.ka, 4, c.q2, c.q1, c.one)) return false;
  if (m.L > 4) return false;
  for (const auto& b : kBuckets)
    if (m.nR <= b[0] && m.kR <= b[1] && m.nA <= b[2] && m.kA <= b[3]) {
      for (int k = 0; k < 4; ++k) dims[k] = b[k];
      return true;
    }
  return false;
}

DescriptorForm descriptor_form(const DevModel& m)
{
  for (const ExactCfg& c : kExact)
    if (model_is(m, c.nr, c.kr, c.na, c.ka, 4, c.q2, c.q1, c.one))
      return c.one && c.na * 24 <= kNarrowMoments ? DescriptorForm::narrow : DescriptorForm::wide;
  return DescriptorForm::generic;
}

// Compiled in descriptor_instances.hip, one group per object file.
extern template void run_exact<5, 9, 5, 9, true, true, true>(const DescriptorCall&);
extern template void run_exact<7, 9, 5, 9, true, false, true>(const DescriptorCall&);
extern template void run_vector<13, 17, 9, 13, true, true>(const DescriptorCall&);
extern template void run_exact<7, 11, 7, 11, true, true, false>(const DescriptorCall&);
extern template void run_exact<5, 9, 5, 9, true, false, false>(const DescriptorCall&);
extern template void run_exact<9, 9, 7, 9, false, false, false>(const DescriptorCall&);
extern template void run_exact<7, 9, 5, 9, true, true, true>(const DescriptorCall&);
extern template void run_exact<7, 9, 5, 9, true, true, false>(const DescriptorCall&);
extern template void run_exact<9, 13, 7, 13, true, true, true>(const DescriptorCall&);
extern template void run_exact<9, 13, 7, 13, true, true, false>(const DescriptorCall&);
extern template void run_generic<kPadL>(const DescriptorCall&);
extern template void run_generic<kMaxL>(const DescriptorCall&);

hipError_t launch_descriptor(const DevBox& b, const DevModel& m, int N, int c1, int c2, const int* type, double* pe,
                             bool acc, int ann, DevWork& w, hipStream_t s, hipEvent_t e0, hipEvent_t e1, int lanes)
{
  if (lanes != 1 && lanes != 4 && lanes != 16) return hipErrorInvalidValue;
  if (c2 <= c1) return hipSuccess;
  const DescriptorCall a{b, m, N, c1, c2, type, pe, acc ? 1 : 0, ann, lanes, w, s, e0, e1};
  auto is = [&](int nr, int kr, int na, int ka, bool q2, bool q1, bool one) {
    return model_is(m, nr, kr, na, ka, 4, q2, q1, one);
  };
  // exact instantiations: the configurations in use, and the bounded sizes
  // that other models are padded to (descriptor_bucket); generic otherwise
  if (is(5, 9, 5, 9, true, true, true)) run_exact<5, 9, 5, 9, true, true, true>(a);
  else if (is(7, 9, 5, 9, true, false, true)) run_exact<7, 9, 5, 9, true, false, true>(a);
  else if (is(13, 17, 9, 13, true, true, true)) run_vector<13, 17, 9, 13, true, true>(a);
  else if (is(7, 11, 7, 11, true, true, false)) run_exact<7, 11, 7, 11, true, true, false>(a);
  else if (is(5, 9, 5, 9, true, false, false)) run_exact<5, 9, 5, 9, true, false, false>(a);
  else if (is(9, 9, 7, 9, false, false, false)) run_exact<9, 9, 7, 9, false, false, false>(a);
  else if (is(7, 9, 5, 9, true, true, true)) run_exact<7, 9, 5, 9, true, true, true>(a);
  else if (is(7, 9, 5, 9, true, true, false)) run_exact<7, 9, 5, 9, true, true, false>(a);
  else if (is(9, 13, 7, 13, true, true, true)) run_exact<9, 13, 7, 13, true, true, true>(a);
  else if (is(9, 13, 7, 13, true, true, false)) run_exact<9, 13, 7, 13, true, true, false>(a);
  else if (m.L > kMaxL || m.nR > kMaxNR || m.kR > kMaxK || m.nA > kMaxNA || m.kA > kMaxK) return hipErrorInvalidValue;
  else if (m.L <= kPadL) run_generic<kPadL>(a);
  // 3-body orders 5..8 (80 angular moments per radial function): the generic
  // instance at order 8, its per-atom arrays partly in scratch
  else run_generic<kMaxL>(a);
  return hipGetLastError();
}

}  // namespace dmgx
