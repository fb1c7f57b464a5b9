// Kernels for 33 to a few hundred activation rows for 16-bit tags, chunk width 8.
#include "sq_mid.h"
namespace sq {
SQ_MID_FORMAT(16, 8)
}
