// Instantiations of the decode-in-registers QMM over K x codebook x row tile.
#include "exl3_launch.hpp"
#include "exl3_wide.hpp"

namespace exl3 {

#define EXL3_WIDE_INST(K, CB)                                      \
  template __global__ void wide_qmm_kernel<K, CB, 4>(WideParams); \
  template __global__ void wide_qmm_kernel<K, CB, 8>(WideParams); \
  template __global__ void wide_qmm_kernel<K, CB, 16>(WideParams);
EXL3_INSTANTIATE(EXL3_WIDE_INST)

#ifndef __HIP_DEVICE_COMPILE__
template <int K, int CB, int R>
static void run_wide(const WideParams& p, dim3 g, hipStream_t s) {
  hipLaunchKernelGGL((wide_qmm_kernel<K, CB, R>), g, dim3(512), 0, s, p);
}
template <int K, int CB>
static void run_wide4(const WideParams& p, dim3 g, hipStream_t s) { run_wide<K, CB, 4>(p, g, s); }
template <int K, int CB>
static void run_wide8(const WideParams& p, dim3 g, hipStream_t s) { run_wide<K, CB, 8>(p, g, s); }
template <int K, int CB>
static void run_wide16(const WideParams& p, dim3 g, hipStream_t s) { run_wide<K, CB, 16>(p, g, s); }
void launch_wide_reduce(const WideParams& p, int R, hipStream_t s) {
  const unsigned units = (unsigned)p.mtiles * p.pairs * R * 2;
  hipLaunchKernelGGL(wide_reduce_kernel, dim3((units + 3) / 4), dim3(256), 0, s, p, R);
}
const WideFn kWide[3][8][3] = {EXL3_TABLE(run_wide4), EXL3_TABLE(run_wide8), EXL3_TABLE(run_wide16)};
#endif

}  // namespace exl3
