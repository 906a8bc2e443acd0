// stage_fast64_3d.hip -- the 3D stage kernels of ModeFast64 (the plain FP64 form).
// Built with -ffp-contract=on: products are fused within an expression, alike in every
// copy of it.  The first planes of a workgroup's chunk and its loop over the others hold
// copies of the k direction's formulas; fused across statements (=fast) they rounded
// differently, and a result depended on the chunk height, which is chosen by timing.
#include "stage_kernels.h"

namespace e4 {

void launch_stage_fast64_3d(const StageArgs& A, dim3 grid, hipStream_t stream, int flux)
{
    launch_stage_dims<ModeFast64, 3>(A, grid, stream, flux);
}

void launch_stage_batch_fast64_3d(const BatchArgs& B, int nwg, bool def, hipStream_t stream, int flux)
{
    launch_stage_batch_dims<ModeFast64, 3>(B, nwg, def, stream, flux);
}

} // namespace e4
