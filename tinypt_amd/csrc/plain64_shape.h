// plain64_shape.h -- how the plain FP64 kernel lays pixels over lanes (host arithmetic).
#pragma once

#include <stdint.h>

#include <algorithm>

namespace tpt {

// A pixel's samples follow each other in one random stream, so an image offers only its pixels as
// parallel work, and the kernel (256 VGPRs, 2 waves per SIMD: 2048 waves, 131,072 lanes on the chip)
// is bound by latency and by its divergent lanes.  With four lanes per pixel a leaf's triangles are
// tested side by side and 16 pixels, not 64, share a wave's control flow; fewer lanes in use
// spread few pixels over more waves.
struct Plain64Shape {
  int quads;  // a pixel has four lanes, not one
  int lanes;  // lanes of a wave in use
  int mixed;  // lanes trace shadow rays beside other lanes' extension rays
};

// The shape for n_pix pixels of a scene whose deepest mesh tree has `depth` levels.
//
// Fewer lanes pay while the launch's waves are about as many as are resident; under deep trees, whose
// waves are longer and differ more, up to four times as many.  So the fewest of 16 and 32 lanes with
// at most 512 waves a level (4 to 16 levels), 32 of them up to 49,152 pixels, else 64.  Measured on
// MI355X, ms, one lane per pixel / four with 64, 32 and 16 in use:
//   Cornell box (3 levels)       8,281 px x 16 spp  5.11 /  2.84 /  2.51 /  2.50
//                               16,384              5.42 /  2.90 /  2.95 /  4.08
//                               32,761              5.47 /  3.28 /  4.48 /  6.22
//                               65,536 x 9          3.16 /  3.28 /  4.97 /  7.35
//   mesh of 82 triangles (6)     8,281 x 16         7.62 /  4.68 /  4.11 /  3.79
//                               16,384              7.91 /  4.76 /  4.37 /  4.64
//                               32,761              8.69 /  5.02 /  4.95 /  5.87
//                               65,536 x 9          4.97 /  3.71 /  5.18 /  6.73
//   mesh of 5122 triangles (13)  8,281 x 16        14.65 /  9.53 /  7.73 /  6.22
//                               16,384             16.14 /  9.78 /  7.99 /  7.44
//                               32,761             18.36 / 10.17 /  8.45 /  9.11
//                               46,225 x 12        14.64 /  8.51 /  7.05 /  8.69
//                               65,536 x 9         11.56 /  7.05 /  9.69 / 12.07
//   mesh of 81,922 (17)         16,384 x 16        26.35 / 16.13 / 12.58 / 10.56
//                               32,761             32.38 / 17.43 / 13.59 / 12.66
//                               46,225 x 12        24.82 / 15.08 / 11.41 / 12.41
//                               65,536 x 9         19.01 / 11.94 / 14.55 / 17.41
//                              196,249 x 3          8.22 /  7.36 /  8.96 / 12.09
//                              262,144 x 2          6.25 /  9.81 / 11.24 / 11.77
// One lane per pixel, then, from 32,768 pixels on, with deep trees from 196,608.
// mixed: one ray of any kind per turn keeps more lanes tracing but runs the shading code in every
// turn: 81,922 triangles 5% faster, Cornell box 18% slower.
inline Plain64Shape plain64_shape(int depth, int64_t n_pix) {
  const bool deep = depth >= 6;
  if (n_pix > (deep ? 196608 : 32768)) return Plain64Shape{0, 64, deep};
  const int64_t waves = 512 * std::min(std::max(depth, 4), 16);
  const int lanes = 4 * n_pix <= 16 * waves ? 16 : 4 * n_pix <= 32 * waves && n_pix <= 49152 ? 32 : 64;
  return Plain64Shape{1, lanes, deep};
}

}  // namespace tpt
