// Heat steps in LDS: 3-D tiles, several generations per launch (heat_tile.hip),
// and the plane march of two generations (heat_pair.hip).
#pragma once

namespace mslhip {

int heat_tile_step(float *out, const float *in, int nx, int ny, int nz, float nv, int steps, bool small,
                   float *maxdiff);
long heat_tile_blocks(int nx, int ny, int nz, int steps, bool small);  // workgroups of a heat_tile_step
int heat_pair_step(float *out, const float *in, int nx, int ny, int nz, float nv, float *maxdiff);

}  // namespace mslhip
