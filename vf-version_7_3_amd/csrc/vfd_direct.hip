// vfd_direct.hip -- launches of the direct-convolution form (vfd_direct.hpp).
#include <algorithm>

#include "vfd_direct.hpp"
#include "vfd_launch.h"

namespace vfd {

namespace {

// Columns of a strip.  z: 128 (512-byte rows) against 64: 866 and 878 us for 8
// fields 1024x512x128, 79 and 89 for 301x187x75.
constexpr int kXyTile = 64, kZTile = 128;
constexpr unsigned long kCacheBytes = 256ul << 20;  // last-level cache

int dir_bound_of(int r) {
    int best = kDirMaxR;
#define VFD_B(RB) \
    if (RB >= r && RB < best) best = RB;
    VFD_DIR_RADII(VFD_B)
#undef VFD_B
    return best;
}

int cu_count() {
    static int ncu = 0;
    if (!ncu) {
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || ncu <= 0)
            ncu = 256;
    }
    return ncu;
}

}  // namespace

hipError_t launch_dir_classify(const FieldBatch& fields, int nfields, const DirDims& d, hipStream_t st) {
    hipLaunchKernelGGL(dir_classify_kernel, dim3(3, (unsigned)nfields), dim3(kClassifyThreads), 0, st, fields,
                       d);
    return hipGetLastError();
}

hipError_t launch_dir_xy(const FieldBatch& fields, int nfields, const DirDims& d, hipStream_t st) {
    constexpr int B = dir_batch(kXyTile);
    const int rb = dir_bound_of(d.max_radius);
    const unsigned lds = dir_xy_lds(kXyTile, rb);
    DirDims g = d;
    g.nfields = (unsigned)nfields;
    g.xtiles = (unsigned)((d.nx + kXyTile - 1) / kXyTile);
    // march chunks along y: a chunk pays ceil(2 R / B) batches before its first
    // output, so a plane is cut only while the strips do not fill the card
    const long strips = (long)g.xtiles * d.nz * nfields;
    const long room = (long)cu_count() * std::max(1u, 160u * 1024u / lds);
    const int warm = (2 * dir_r4(rb) + B - 1) / B, rows = (d.ny + B - 1) / B;
    int best = 1;
    double best_cost = 1e300;
    for (int c = 1; c <= rows; ++c) {
        const int per = (rows + c - 1) / c;
        const double cost = std::max(1.0, (double)strips * c / (double)room) * (warm + per);
        if (cost < best_cost * 0.999) {
            best_cost = cost;
            best = c;
        }
    }
    g.yrows = (rows + best - 1) / best * B;
    g.ychunks = (unsigned)((d.ny + g.yrows - 1) / g.yrows);
    const unsigned long groups = (unsigned long)d.nz * g.ychunks * nfields;
    const unsigned long ids = (groups + 7) / 8 * 8 * g.xtiles;
    if (ids > 0x7fffffffu) return hipErrorInvalidConfiguration;
    hipLaunchKernelGGL(dir_xy_kernel<kXyTile>, dim3((unsigned)ids), dim3(kDirThreads), lds, st, fields, g);
    return hipGetLastError();
}

hipError_t launch_dir_z(const FieldBatch& fields, int nfields, const DirDims& d, hipStream_t st, bool vis) {
    const unsigned lds = dir_z_lds(kZTile, dir_bound_of(d.max_radius));
    DirDims g = d;
    g.nfields = (unsigned)nfields;
    const unsigned long np = (unsigned long)d.ny * d.nx;
    const dim3 grid((unsigned)((np + kZTile - 1) / kZTile), (unsigned)nfields);
    // the pass between is read once: past the last-level cache's size it is
    // streamed; a batch that fits is still there from the x-y pass
    if (vis)
        hipLaunchKernelGGL((dir_z_kernel<kZTile, true, kCacheDefault>), grid, dim3(kDirThreads), lds, st, fields, g);
    else if (d.bytes * nfields > kCacheBytes)
        hipLaunchKernelGGL((dir_z_kernel<kZTile, false, kStream>), grid, dim3(kDirThreads), lds, st, fields, g);
    else
        hipLaunchKernelGGL((dir_z_kernel<kZTile, false, kCacheDefault>), grid, dim3(kDirThreads), lds, st, fields, g);
    return hipGetLastError();
}

}  // namespace vfd
