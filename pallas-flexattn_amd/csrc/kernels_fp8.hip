// Instantiations and launches of the fp8 forward and the e4m3 quantiser.
#include "fwd_fp8.h"
#include "launch.h"

namespace fa {

template <int D, bool kMods>
static void run_fwd_fp8(const Fp8FwdArgs& a, bool q16, dim3 grid, hipStream_t s) {
  constexpr int NW = 4;
  if (q16) hipLaunchKernelGGL((fwd_fp8_kernel<D, NW, kMods, true>), grid, dim3(64 * NW), 0, s, a);
  else hipLaunchKernelGGL((fwd_fp8_kernel<D, NW, kMods>), grid, dim3(64 * NW), 0, s, a);
}

int launch_fwd_fp8(const Fp8FwdArgs& a, int D, bool mods, bool q16, hipStream_t s) {
  const dim3 grid((unsigned)fwd_items(a.p, 0, 128));
  if (D == 128) mods ? run_fwd_fp8<128, true>(a, q16, grid, s) : run_fwd_fp8<128, false>(a, q16, grid, s);
  else if (D == 64) mods ? run_fwd_fp8<64, true>(a, q16, grid, s) : run_fwd_fp8<64, false>(a, q16, grid, s);
  else return FA_ERR_UNSUPPORTED;
  return launch_status();
}

int launch_quant_fp8(const QuantArgs& a, hipStream_t s) {
  const unsigned grid = (unsigned)(a.count * a.heads * cdiv(a.S, kFp8ScaleRows));
  switch (a.D) {
    case 32: hipLaunchKernelGGL((quant_fp8_kernel<32>), dim3(grid), dim3(256), 0, s, a); break;
    case 64: hipLaunchKernelGGL((quant_fp8_kernel<64>), dim3(grid), dim3(256), 0, s, a); break;
    case 128: hipLaunchKernelGGL((quant_fp8_kernel<128>), dim3(grid), dim3(256), 0, s, a); break;
    default: return FA_ERR_UNSUPPORTED;
  }
  return launch_status();
}

}  // namespace fa
