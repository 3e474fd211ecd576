// stage_tile_vti.hip -- the tile kernel instantiated for the VTI medium.
#include <hip/hip_runtime.h>

#include "stage_tile.h"

namespace cgfdh {

void launch_tile_vti(const LaunchCtx& L, const StageParams& P, int kind, int dx, int dy, int dz)
{
  launch_tile_mt<MEDIUM_VTI>(L, P, kind, dx, dy, dz);
}

}  // namespace cgfdh
