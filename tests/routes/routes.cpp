// Prints how the library would run convolutions, without a device.  Input:
// one problem a line, "nx ny nz kx ky kz boundary" (boundary 5: the PSF
// gradient of the periodic convolution); output: its transform
// lengths, whether its forward and its inverse take a whole-plane kernel
// (each 0 or 1) and its workspace bytes.
#include <cstdio>

#include "conv_driver.hpp"

using namespace fcamd;

int main() {
  ConvShape s{};
  int boundary = 0;
  try {
    while (std::scanf("%d %d %d %d %d %d %d", &s.nx, &s.ny, &s.nz, &s.kx, &s.ky, &s.kz,
                      &boundary) == 7) {
      s.cx = s.kx / 2;
      s.cy = s.ky / 2;
      s.cz = s.kz / 2;
      ConvShape e = s;
      if (boundary == kMapPeriodic || boundary == 5) {
        e = with_extension(s, boundary == 5);
      } else {
        const PaddedProblem p = padded_problem(s, boundary);
        // (a padded problem never takes the plane kernels)
        if (!boundary_extension(s, p, boundary, &e)) {
          std::printf("%d %d %d 0 0 %zu\n", p.padded.nx, p.padded.ny, p.padded.nz,
                      workspace_layout(p.padded).total());
          continue;
        }
      }
      std::printf("%d %d %d %d %d %zu\n", e.tx(), e.ty(), e.tz(), (int)plane_path(e, -1),
                  (int)plane_path(e, +1), workspace_layout(e).total());
    }
  } catch (const Error& err) {
    std::fprintf(stderr, "error %d: %s\n", err.code, err.msg.c_str());
    return 1;
  }
  return 0;
}
