// Kernels of sq_fused.h for 10-bit tags, chunk width 4.
#include "sq_fused.h"
namespace sq {
SQ_FUSED_FORMAT(10, 4)
}
