// conv_plan.h -- which convolution kernel a layer takes: the tile of a block of
// conv3_fwd_kernel (conv3d.hip).  Host arithmetic only, so that tests can ask
// it which kernels their sizes reach.

#ifndef LDW_CONV_PLAN_H
#define LDW_CONV_PLAN_H

#include <stdint.h>

namespace ldw {

constexpr int CONV_BLOCKS = 512;              // two per CU

struct ConvShape { int nt, ty, zt; };

// Output channels per block (16 nt), rows per wave and depth of the tile.
//
// A wave wants 8 rows (a halo row is then read 1.25 times instead of 1.5) as
// long as that makes enough blocks, with up to 32 channels: 8 rows and 48 do
// not fit LDS twice.  80 -> 32 channels on 8 x 64^3: 357 us with (2, 8), 396
// with (2, 4), 459 with (1, 8).  Wider layers take 3 or 4 blocks of 16,
// whichever pads less (32 -> 48 on 8 x 32^3: 32 us with nt = 3, 37 with 2, 36
// with 4), and fewer where the grid would not give each CU two blocks (64 ->
// 64 on 8 x 16^3: 22 us with nt = 4, 17 with 2 or 1).
//
// Multiples of 96 channels take 6 blocks of 16 where that makes enough blocks:
// the halo is staged once instead of twice, and 24 LDS reads serve 72 MFMAs
// (15 serve 36 with nt = 3).  160 -> 96 on 64^3: 198 us with nt = 6, 229 with 3;
// 96 -> 96 on 4 x 33x47x65: 256 us.
//
// Misaligned operands (dma = 0) take 4 rows, which halves the kernels built
// for them.
inline ConvShape conv_shape(int batch, int nx, int ny, int nz, int nb16, bool dma) {
  ConvShape c;
  c.zt = (nz > 8) ? 16 : 8;
  const int cx = 4*16/c.zt;
  auto tiles = [&](int ty) {
    return (int64_t) batch*((nx + cx - 1)/cx)*((ny + ty - 1)/ty)*((nz + c.zt - 1)/c.zt);
  };
  c.ty = 4;
  if (nb16 <= 2) {
    c.nt = nb16;
    if (dma && tiles(8) >= CONV_BLOCKS) c.ty = 8;
  }
  else {
    c.nt = ((nb16 + 3)/4*4 <= (nb16 + 2)/3*3) ? 4 : 3;
  }
  if (nb16 % 6 == 0 && tiles(4)*(nb16/6) >= CONV_BLOCKS) c.nt = 6;
  while (c.nt > 1 && tiles(c.ty)*((nb16 + c.nt - 1)/c.nt) < CONV_BLOCKS) c.nt--;
  return c;
}

}  // namespace ldw

#endif
