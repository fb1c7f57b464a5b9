// Kernels for 33 to a few hundred activation rows for 10-bit tags, chunk width 4.
#include "sq_mid.h"
namespace sq {
SQ_MID_FORMAT(10, 4)
}
