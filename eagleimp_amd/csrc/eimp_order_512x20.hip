// eimp_order_512x20.hip -- the order chain with 512 threads, up to 20 positions each
#include "eimp_order.h"

namespace eimp {
PbwtVariant variant_512x20() { return make_variant<512, 20>(); }
}  // namespace eimp
