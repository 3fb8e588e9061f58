// Instantiations of the decode-in-registers QMM over K x codebook x tile.
#include "exl3_launch.hpp"
#include "exl3_wide.hpp"

namespace exl3 {

#define EXL3_WIDE_INST(K, CB)                                         \
  template __global__ void wide_qmm_kernel<K, CB, 4, 4>(WideParams); \
  template __global__ void wide_qmm_kernel<K, CB, 8, 8>(WideParams); \
  template __global__ void wide_qmm_kernel<K, CB, 16, 8>(WideParams);
EXL3_INSTANTIATE(EXL3_WIDE_INST)

#ifndef __HIP_DEVICE_COMPILE__
template <int K, int CB, int R, int NW>
static void run_wide(const WideParams& p, dim3 g, hipStream_t s) {
  hipLaunchKernelGGL((wide_qmm_kernel<K, CB, R, NW>), g, dim3(64 * NW), 0, s, p);
}
template <int K, int CB>
static void run_wide_4x4(const WideParams& p, dim3 g, hipStream_t s) { run_wide<K, CB, 4, 4>(p, g, s); }
template <int K, int CB>
static void run_wide_8x8(const WideParams& p, dim3 g, hipStream_t s) { run_wide<K, CB, 8, 8>(p, g, s); }
template <int K, int CB>
static void run_wide_16x8(const WideParams& p, dim3 g, hipStream_t s) { run_wide<K, CB, 16, 8>(p, g, s); }
void launch_wide_reduce(const WideParams& p, int NW, hipStream_t s) {
  const unsigned jobs = (unsigned)p.units * ((p.M + 15) / 16) * (NW / 4);
  hipLaunchKernelGGL(wide_reduce_kernel, dim3((jobs + 3) / 4), dim3(256), 0, s, p, NW);
}
const WideFn kWide[3][8][3] = {EXL3_TABLE(run_wide_4x4), EXL3_TABLE(run_wide_8x8),
                               EXL3_TABLE(run_wide_16x8)};
#endif

}  // namespace exl3
