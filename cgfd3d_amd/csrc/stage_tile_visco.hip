// stage_tile_visco.hip -- the tile kernel instantiated for the visco-elastic medium.
#include <hip/hip_runtime.h>

#include "stage_tile.h"

namespace cgfdh {

void launch_tile_visco(const LaunchCtx& L, const StageParams& P, int kind, int dx, int dy, int dz)
{
  launch_tile_mt<MEDIUM_VISCO>(L, P, kind, dx, dy, dz);
}

}  // namespace cgfdh
