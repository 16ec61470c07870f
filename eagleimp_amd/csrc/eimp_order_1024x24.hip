// eimp_order_1024x24.hip -- the order chain with 1024 threads, up to 24 positions each
#include "eimp_order.h"

namespace eimp {
PbwtVariant variant_1024x24() { return make_variant<1024, 24>(); }
}  // namespace eimp
