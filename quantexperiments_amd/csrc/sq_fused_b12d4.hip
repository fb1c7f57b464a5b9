// Kernels of sq_fused.h for 12-bit tags, chunk width 4.
#include "sq_fused.h"
namespace sq {
SQ_FUSED_FORMAT(12, 4)
}
