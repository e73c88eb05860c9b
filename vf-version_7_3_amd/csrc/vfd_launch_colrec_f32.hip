// Instantiates the col passes of batches with direct-form records (float).
#define VFD_REAL float
#define VFD_COL_TU
#define VFD_COLREC_TU
#include "vfd_launch_impl.hpp"
