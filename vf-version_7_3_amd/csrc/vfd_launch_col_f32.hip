// Instantiates the col passes for float.
#define VFD_REAL float
#define VFD_COL_TU
#include "vfd_launch_impl.hpp"

namespace vfd {
// classes: bit 0, 1, 2 = the fields of radius class 8, 12, 16.  One launch for
// all of them: a wave branches on its field's class.  Launches with records
// walk the fields the FFT form is left with.
__global__ void __launch_bounds__(64) zdirect_kernel(const FieldBatch fb, ColDesc cd, unsigned classes) {
    unsigned id = blockIdx.x, nf = cd.grid_fields, todo = ~0u;
    if (cd.records) {
        todo = fft_fields(fb, (int)nf, cd.rec_off);
        nf = (unsigned)__builtin_popcount(todo);
        if (nf == 0) return;
    }
    const unsigned per = cd.grid_segs * cd.grid_planes;
    for (; id < per * nf; id += gridDim.x) {
        const unsigned bz = id / per, r = id % per;
        const FieldDesc& fd = fb.f[cd.records ? nth_field(todo, bz) : bz];
        const int form = zform_of_table(fd.kspec, cd.kspec_bytes, cd.sep_g);
        const unsigned bx = r % cd.grid_segs, by = r / cd.grid_segs;
        if (form == 8 && (classes & 1u)) zdirect_column<8>(fd, cd, bx, by);
        else if (form == 12 && (classes & 2u)) zdirect_column<12>(fd, cd, bx, by);
        else if (form == 16 && (classes & 4u)) zdirect_column<16>(fd, cd, bx, by);
    }
}

hipError_t launch_zdirect(unsigned classes, const FieldBatch& fields, int nfields, const ColDesc& cd, long nplanes,
                          hipStream_t st) {
    ColDesc g = cd;
    g.grid_segs = (unsigned)((cd.ncols + 63) / 64);
    g.grid_planes = (unsigned)nplanes;
    g.grid_fields = (unsigned)nfields;
    const unsigned long ids = (unsigned long)g.grid_segs * nplanes * nfields;
    if (ids > 0x7fffffffu) return hipErrorInvalidConfiguration;
    const unsigned long cap = 16ul * num_cus();  // resident waves
    hipLaunchKernelGGL(zdirect_kernel, dim3((unsigned)(cd.records == RECORDS_FEW && ids > cap ? cap : ids)), dim3(64), 0, st, fields, g,
                       classes);
    return hipGetLastError();
}
}  // namespace vfd
