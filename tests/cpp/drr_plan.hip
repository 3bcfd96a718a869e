// Prints how DRR launches march and the key their tuned variants are kept by, one launch per nine
// arguments: storage, layout, geometry, ray distance (voxels), layout bytes (MB), plain voxels (0 / 1),
// tiles, variant (-1, 0, 1) and objects per item. Runs without a GPU.
#include "../../xreg_amd/csrc/xrh_internal.h"

#include <cstdio>
#include <cstdlib>
#include <cstring>

int main(int argc, char** argv)
{
  for (int i = 1; i + 8 < argc; i += 9) {
    xrh::DrrLaunch L;
    std::memset(&L, 0, sizeof(L));
    L.storage = std::atoi(argv[i]);
    L.layout = std::atoi(argv[i + 1]);
    L.geom = std::atoi(argv[i + 2]);
    L.ray_spacing = (float)std::atof(argv[i + 3]);
    L.vol_bytes = (uint64_t)std::atoi(argv[i + 4]) << 20;
    L.plain = std::atoi(argv[i + 5]) != 0;
    const int64_t tiles = std::atoll(argv[i + 6]);
    L.bands = 1;
    L.max_band_tiles = tiles;
    L.reuse = std::atoi(argv[i + 7]);
    L.objs = std::atoi(argv[i + 8]);
    const int64_t plan = xrh::drr_launch_plan(L);
    std::printf("%d %d %d %d %d | %s\n", (int)(plan >> 1 & 7), (int)(plan & 1), (int)(plan >> 10), (int)(plan >> 4 & 63),
                (int)xrh::drr_whole_rays(L), xrh::drr_tune_key(L, 256, 256, tiles).c_str());
  }
  return 0;
}
