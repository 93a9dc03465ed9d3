// i-derivative chunked-path instantiations, group 13 (see ip1_wave.h).
#include "device_common.h"
#include "ip1_wave.h"

namespace mcint {
MCINT_IP1_GROUP13(MCINT_IP1_DEFINE)
}  // namespace mcint
