// Kernels for 1 to 256 activation rows and weights already decoded to fp16.
#include "sq_mid.h"
namespace sq {
int launch_mid_dense(const MidArgs& a, int nt, int tw, int st, int nw, int grid, hipStream_t s) { return launch_mid_format<0, 0>(a, nt, tw, st, nw, grid, s); }
}
