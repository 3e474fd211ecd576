// stage_tile_aniso.hip -- the tile kernel instantiated for the general anisotropic medium.
#include <hip/hip_runtime.h>

#include "stage_tile.h"

namespace cgfdh {

void launch_tile_aniso(const LaunchCtx& L, const StageParams& P, int kind, int dx, int dy, int dz)
{
  launch_tile_mt<MEDIUM_ANISO>(L, P, kind, dx, dy, dz);
}

}  // namespace cgfdh
