// Radix-2 transforms of the columns of an array, lanes on adjacent columns:
// the passes of matrix753_kernels.h where every twiddle is the same for all
// columns, so there are no column factors and the first pass has only
// 2^r1 - 1 matrices.  525 columns of 2^12 points, 206 MB: 159 and 194 us (2.6
// and 2.1 TB/s; the second pass reads 2^r1 times as many matrices, and its
// tiles of 525 columns are 3% empty), against 2 x 316 us for the vector
// kernels on rows and 107 for the transpose after them.
#include "columns753.h"

#include "matrix753_kernels.h"

namespace gsn {

template <class F, int KIND, int LOG_R>
__global__ __launch_bounds__(1 << (LOG_R + 3)) __attribute__((amdgpu_waves_per_eu(2))) void col753_kernel(
    const E753 *in, E753 *out, const void *fold, uint32_t log_n, uint32_t log_g, uint32_t cols)
{
    __shared__ uint4 lds[mat_lds_quads(KIND, LOG_R, 5)];
    MatArgs a{};
    a.in = in;
    a.out = out;
    a.fold = fold;
    a.log_n = log_n;
    a.log_g = log_g;
    a.cols = cols;
    a.blk = uniform(xcd_tile(blockIdx.x, gridDim.x));
    MatTile<F, KIND, LOG_R, 5>(a, lds).run();
}

template <class F, int KIND>
static void launch_col(uint32_t log_r, uint32_t grid, const E753 *in, E753 *out, const void *fold, uint32_t log_n,
                       uint32_t log_g, uint32_t cols, hipStream_t st)
{
    const dim3 block(1u << (log_r + 3));
    switch (log_r) {
    case 4:
        hipLaunchKernelGGL((col753_kernel<F, KIND, 4>), dim3(grid), block, 0, st, in, out, fold, log_n, log_g, cols);
        break;
    case 5:
        hipLaunchKernelGGL((col753_kernel<F, KIND, 5>), dim3(grid), block, 0, st, in, out, fold, log_n, log_g, cols);
        break;
    case 6:
        hipLaunchKernelGGL((col753_kernel<F, KIND, 6>), dim3(grid), block, 0, st, in, out, fold, log_n, log_g, cols);
        break;
    default: break;
    }
}

template <class F>
void launch_columns753(const E753 *in, E753 *out, E753 *ws, uint32_t log_n, uint32_t cols, const void *fold1,
                       const void *fold2, hipStream_t st)
{
    uint32_t r1 = 0, r2 = 0;
    columns_split(log_n, r1, r2);
    const uint32_t tiles1 = ((cols << r2) + 31) / 32;
    launch_col<F, COL_FIRST>(r1, tiles1, in, ws, fold1, log_n, 0, cols, st);
    launch_col<F, COL_LAST>(r2, ((cols + 31) / 32) << r1, ws, out, fold2, log_n, r1, cols, st);
}
template void launch_columns753<FMnt4>(const E753 *, E753 *, E753 *, uint32_t, uint32_t, const void *, const void *,
                                       hipStream_t);
template void launch_columns753<FMnt6>(const E753 *, E753 *, E753 *, uint32_t, uint32_t, const void *, const void *,
                                       hipStream_t);

}  // namespace gsn
