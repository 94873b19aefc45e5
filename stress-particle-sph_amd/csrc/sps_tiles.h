// Tile width and window capacities of the tiled pair kernels.
// tune_tiles.py rewrites this file with a candidate it measured, here t256mw4;
// a compiler definition (-DSPS_TILE=... and the others) overrides it.
// Measured (ms per step: FP64 on the 1 M slope; batched ensemble, mixed):
//   t256    (256, 24, 640, 192, 0): 2.2588, 7.9829 (relative 1.0)
//   t256m   (256, 24, 608, 192, 0): 2.2653, 8.0071 (relative 1.003)
//   t256mw4 (256, 24, 608, 192, 4): 2.1751, 7.2848 (relative 0.9374)
//   t256w4  (256, 24, 640, 192, 4): 2.1745, 7.2559 (relative 0.9354)
//   t256s   (256, 24, 576, 160, 0): 2.2665, 8.9566 (relative 1.061)
//   t256sw4 (256, 24, 576, 160, 4): 2.2003, 8.2381 (relative 1.0026)
//   t128    (128, 16, 384, 128, 0): 2.3829, 10.2533 (relative 1.164)
//   t128s   (128, 16, 320, 96, 0): 3.575, 16.1591 (relative 1.7899)
#pragma once
#ifndef SPS_TILE
#define SPS_TILE 256  // receivers per workgroup
#endif
#ifndef SPS_TROWS
#define SPS_TROWS 24  // most window rows staged
#endif
#ifndef SPS_CAP
#define SPS_CAP 608  // staged partners of a main kind per window
#endif
#ifndef SPS_CAP_D
#define SPS_CAP_D 192  // staged dummies per window
#endif
#ifndef SPS_STAGE_WAVES
#define SPS_STAGE_WAVES 4  // waves per SIMD of the stage kernels with STAGE_OCCUPANCY (0: the compiler's choice)
#endif
