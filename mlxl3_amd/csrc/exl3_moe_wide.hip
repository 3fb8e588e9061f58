// Instantiations of the expert QMMs for many rows per expert over K x codebook.
#include "exl3_launch.hpp"
#include "exl3_moe_wide.hpp"

namespace exl3 {

#define EXL3_MOE_WIDE_INST(K, CB)                                      \
  template __global__ void moe_wide_kernel<K, CB, 2>(MoeMmParams, int, uint16_t*); \
  template __global__ void moe_wide_kernel<K, CB, 1>(MoeMmParams, int, uint16_t*);
// K = 7 is not a SwitchGLU width (switch_glu_layout rejects it).
EXL3_INST_CB(EXL3_MOE_WIDE_INST, 1)
EXL3_INST_CB(EXL3_MOE_WIDE_INST, 2)
EXL3_INST_CB(EXL3_MOE_WIDE_INST, 3)
EXL3_INST_CB(EXL3_MOE_WIDE_INST, 4)
EXL3_INST_CB(EXL3_MOE_WIDE_INST, 5)
EXL3_INST_CB(EXL3_MOE_WIDE_INST, 6)
EXL3_INST_CB(EXL3_MOE_WIDE_INST, 8)
template __global__ void moe_glu_kernel<true>(MoeMmParams, const uint16_t*);
template __global__ void moe_glu_kernel<false>(MoeMmParams, const uint16_t*);
template __global__ void moe_route16_kernel<true>(MoePlanParams, MoeGatherParams);
template __global__ void moe_route16_kernel<false>(MoePlanParams, MoeGatherParams);

#ifndef __HIP_DEVICE_COMPILE__
int moe_wide_rows(int k) { return 16 * (k == 8 ? kMoeWideR<8> : kMoeWideR<4>); }

void launch_moe_route16(const MoePlanParams& pp, const MoeGatherParams& gp, size_t lds,
                        hipStream_t s) {
  const int64_t jobs = (int64_t)((gp.slots + 15) / 16) * 2 * (gp.in / 128);
  const dim3 grid((unsigned)(1 + (jobs + 3) / 4));
  if ((((uintptr_t)gp.x | (uintptr_t)gp.gu_suh | (uintptr_t)gp.xgu) & 15) == 0)
    hipLaunchKernelGGL(moe_route16_kernel<true>, grid, dim3(256), lds, s, pp, gp);
  else
    hipLaunchKernelGGL(moe_route16_kernel<false>, grid, dim3(256), lds, s, pp, gp);
}

template <int K, int CB>
static int run_moe_wide(const MoeMmParams& p, bool gate_up, int blocks, uint16_t* raw,
                        hipStream_t s) {
  if (!gate_up) {
    const int units = p.width / 128;
    hipLaunchKernelGGL((moe_wide_kernel<K, CB, 1>), dim3((unsigned)blocks * units), dim3(256), 0, s,
                       p, units, raw);
    return check_launch("moe down");
  }
  const int units = 2 * (p.width / 128);
  hipLaunchKernelGGL((moe_wide_kernel<K, CB, 2>), dim3((unsigned)blocks * units), dim3(256), 0, s, p,
                     units, raw);
  if (int rc = check_launch("moe gate/up")) return rc;
  if (int rc = launch_gate("moe glu")) return rc;
  const dim3 grid((unsigned)blocks, p.width / 128);
  if (p.gelu)
    hipLaunchKernelGGL(moe_glu_kernel<true>, grid, dim3(256), 0, s, p, raw);
  else
    hipLaunchKernelGGL(moe_glu_kernel<false>, grid, dim3(256), 0, s, p, raw);
  return check_launch("moe glu");
}
#define EXL3_MOE_WIDE_ROW(K) {run_moe_wide<K, 0>, run_moe_wide<K, 1>, run_moe_wide<K, 2>}
const MoeWideFn kMoeWide[8][3] = {
    EXL3_MOE_WIDE_ROW(1), EXL3_MOE_WIDE_ROW(2), EXL3_MOE_WIDE_ROW(3), EXL3_MOE_WIDE_ROW(4),
    EXL3_MOE_WIDE_ROW(5), EXL3_MOE_WIDE_ROW(6), {nullptr, nullptr, nullptr}, EXL3_MOE_WIDE_ROW(8)};
#endif

}  // namespace exl3
