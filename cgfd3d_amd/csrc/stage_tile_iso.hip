// stage_tile_iso.hip -- the tile kernel instantiated for the isotropic medium.
#include <hip/hip_runtime.h>

#include "stage_tile.h"

namespace cgfdh {

void launch_tile_iso(const LaunchCtx& L, const StageParams& P, int kind, int dx, int dy, int dz)
{
  launch_tile_mt<MEDIUM_ISO>(L, P, kind, dx, dy, dz);
}

}  // namespace cgfdh
