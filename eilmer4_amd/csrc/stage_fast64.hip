// stage_fast64.hip -- instantiations for ModeFast64 (the plain FP64 form): the 2D stage
// kernels, boundary cells and shock detector (the 3D stage kernels: stage_fast64_3d.hip).
// Built with -ffp-contract=fast.
#include "stage_kernels.h"

namespace e4 {

void launch_stage_fast64(const StageArgs& A, dim3 grid, hipStream_t stream, int dims, int flux)
{
    if (dims == 3) launch_stage_fast64_3d(A, grid, stream, flux);
    else launch_stage_dims<ModeFast64, 2>(A, grid, stream, flux);
}

void launch_stage_batch_fast64(const BatchArgs& B, int nwg, bool def, hipStream_t stream, int dims, int flux)
{
    if (dims == 3) launch_stage_batch_fast64_3d(B, nwg, def, stream, flux);
    else launch_stage_batch_dims<ModeFast64, 2>(B, nwg, def, stream, flux);
}

void launch_extrapolate_ghosts_batch_fast64(const BatchArgs& B, int nwg, hipStream_t stream)
{
    launch_extrapolate_ghosts_batch_mode<ModeFast64>(B, nwg, stream);
}

void launch_extrapolate_ghosts_fast64(const StageArgs& A, int faces, hipStream_t stream)
{
    launch_extrapolate_ghosts_mode<ModeFast64>(A, faces, stream);
}

void launch_boundary_cells_batch_fast64(const BatchArgs& B, int nwg, hipStream_t stream, int dims, int flux)
{
    launch_boundary_cells_batch_mode<ModeFast64>(B, nwg, stream, dims, flux);
}

void launch_boundary_cells_fast64(const StageArgs& A, hipStream_t stream, int dims, int flux)
{
    launch_boundary_cells_mode<ModeFast64>(A, stream, dims, flux);
}

void launch_shock_detect_fast64(const StageArgs& A, int dims, hipStream_t stream)
{
    launch_shock_detect_mode<ModeFast64>(A, dims, stream);
}

void launch_shock_detect_batch_fast64(const BatchArgs& B, int nwg, int dims, hipStream_t stream)
{
    launch_shock_detect_batch_mode<ModeFast64>(B, nwg, dims, stream);
}

} // namespace e4
