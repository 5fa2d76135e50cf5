// descriptor_instances.hip -- the descriptor instances, one group per
// compilation (DMGX_DESCRIPTOR_GROUP, given by the build; the groups compile
// side by side).
#include "descriptor.hpp"

namespace dmgx {

#if DMGX_DESCRIPTOR_GROUP == 0
template void run_exact<7, 9, 5, 9, true, false, true>(const DescriptorCall&);
#elif DMGX_DESCRIPTOR_GROUP == 1
template void run_exact<5, 9, 5, 9, true, true, true>(const DescriptorCall&);
#elif DMGX_DESCRIPTOR_GROUP == 2
template void run_exact<7, 11, 7, 11, true, true, false>(const DescriptorCall&);
#elif DMGX_DESCRIPTOR_GROUP == 3
template void run_exact<5, 9, 5, 9, true, false, false>(const DescriptorCall&);
#elif DMGX_DESCRIPTOR_GROUP == 4
template void run_exact<9, 9, 7, 9, false, false, false>(const DescriptorCall&);
#elif DMGX_DESCRIPTOR_GROUP == 5
template void run_exact<7, 9, 5, 9, true, true, true>(const DescriptorCall&);
#elif DMGX_DESCRIPTOR_GROUP == 6
template void run_exact<7, 9, 5, 9, true, true, false>(const DescriptorCall&);
#elif DMGX_DESCRIPTOR_GROUP == 7
template void run_exact<9, 13, 7, 13, true, true, true>(const DescriptorCall&);
#elif DMGX_DESCRIPTOR_GROUP == 8
template void run_exact<9, 13, 7, 13, true, true, false>(const DescriptorCall&);
#elif DMGX_DESCRIPTOR_GROUP == 9
template void run_vector<13, 17, 9, 13, true, true>(const DescriptorCall&);
#elif DMGX_DESCRIPTOR_GROUP == 10
template void run_generic<kPadL>(const DescriptorCall&);
#elif DMGX_DESCRIPTOR_GROUP == 11
template void run_generic<kMaxL>(const DescriptorCall&);
#endif

}  // namespace dmgx
