// Tile kernel of the mean blur (blur_tile.hip).
#pragma once

namespace mslhip {

struct TileShape {
    int w, m, tile_h;  // LDS columns, rows per thread of the column pass, output rows; w = 0: none fits
    double us;         // modelled time of the launch
};
TileShape tile_shape(int rows, int cols, int r, int steps);
int blur_tile_step(float *out, const float *in, int rows, int cols, int r, float nv, int steps, const TileShape &t);

}  // namespace mslhip
