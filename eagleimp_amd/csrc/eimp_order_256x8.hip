// eimp_order_256x8.hip -- the order chain with 256 threads, up to 8 positions each
#include "eimp_order.h"

namespace eimp {
PbwtVariant variant_256x8() { return make_variant<256, 8>(); }
}  // namespace eimp
