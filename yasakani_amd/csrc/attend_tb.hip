// Launches of the decode kernel over trellis-coded rows (attend_tb_device.h).  gfx950.
#include "attend_tb_device.h"

namespace yka {
namespace {

template <int KB, bool MS>
__global__ void __launch_bounds__(256, 2) attend_tb_kernel(TbAttnArgs A) {
  int split = blockIdx.x, kvh = blockIdx.y;
  if (!MS && A.s_short) tb_split_of(A, split + A.S * kvh, split, kvh);
  tbd::attend_tb_body<KB, MS>(A, split, kvh, blockIdx.z, false);
}

}  // namespace

void launch_attend_tb(const TbAttnArgs& A, int kb, hipStream_t st) {
  if (A.rows.pos) {
    const dim3 grid(A.S, A.n_kv, A.M);
    if (kb == 4) hipLaunchKernelGGL((attend_tb_kernel<4, true>), grid, dim3(256), 0, st, A);
    else hipLaunchKernelGGL((attend_tb_kernel<5, true>), grid, dim3(256), 0, st, A);
    return;
  }
  const dim3 grid(A.S, A.n_kv, (A.M + 1) / 2);
  if (kb == 4) hipLaunchKernelGGL((attend_tb_kernel<4, false>), grid, dim3(256), 0, st, A);
  else hipLaunchKernelGGL((attend_tb_kernel<5, false>), grid, dim3(256), 0, st, A);
}

}  // namespace yka
