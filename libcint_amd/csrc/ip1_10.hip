// i-derivative chunked-path instantiations, group 10 (see ip1_wave.h).
#include "device_common.h"
#include "ip1_wave.h"

namespace mcint {
MCINT_IP1_GROUP10(MCINT_IP1_DEFINE)
}  // namespace mcint
