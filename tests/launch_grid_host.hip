// Host build of the launch grid's rule (mdtraj_amd/csrc/common.h), for the CPU
// tests.
#include "common.h"

extern "C" void launch_grid_host(long long groups, int threads, unsigned* out) {
    const dim3 g = hr::launch_grid(groups, threads);
    out[0] = g.x;
    out[1] = g.y;
    out[2] = g.z;
}
