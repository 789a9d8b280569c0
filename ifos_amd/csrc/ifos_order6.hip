// ifos_order6.hip -- time-loop kernels of FDORDER 12.
#include "ifos_resident_kernels.h"
#include "ifos_step_kernels.h"

namespace ifos {

template void vel_n<6>(const StepArgs &a, const StepArgs *da, const LaunchShape &ls, int k, hipStream_t s);
template void str_n<6>(const StepArgs &a, const StepArgs *da, const LaunchShape &ls, int k, hipStream_t s);
template void fused_n<6>(const StepArgs &a, const StepArgs *da, const LaunchShape &ls, int k, hipStream_t s);
template size_t resident_lds<6>(int L, int rows);
template hipError_t resident_n<6>(int L, const ResidentArgs &r, const ResidentPlan &p, hipStream_t s);

}  // namespace ifos
