// Kernels of sq_fused.h for 16-bit tags, chunk width 8.
#include "sq_fused.h"
namespace sq {
SQ_FUSED_FORMAT(16, 8)
}
