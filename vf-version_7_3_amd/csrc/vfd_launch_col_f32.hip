// Instantiates the col passes for float.
#define VFD_REAL float
#define VFD_COL_TU
#include "vfd_launch_impl.hpp"

namespace vfd {
// classes: bit 0, 1, 2 = the fields of radius class 8, 12, 16.  One launch for
// all of them: a work-group branches on its field's class.
__global__ void __launch_bounds__(64) zdirect_kernel(const FieldBatch fb, ColDesc cd, unsigned classes) {
    const FieldDesc& fd = fb.f[blockIdx.z];
    if (dir_skip(fd)) return;
    const int form = zform_of_table(fd.kspec, cd.kspec_bytes, cd.sep_g);
    if (form == 8 && (classes & 1u)) zdirect_column<8>(fd, cd);
    else if (form == 12 && (classes & 2u)) zdirect_column<12>(fd, cd);
    else if (form == 16 && (classes & 4u)) zdirect_column<16>(fd, cd);
}

hipError_t launch_zdirect(unsigned classes, const FieldBatch& fields, int nfields, const ColDesc& cd, long nplanes,
                          hipStream_t st) {
    dim3 grid((unsigned)((cd.ncols + 63) / 64), (unsigned)nplanes, (unsigned)nfields);
    hipLaunchKernelGGL(zdirect_kernel, grid, dim3(64), 0, st, fields, cd, classes);
    return hipGetLastError();
}
}  // namespace vfd
