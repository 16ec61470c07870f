// eimp_order_256x16.hip -- the order chain with 256 threads, up to 16 positions each
#include "eimp_order.h"

namespace eimp {
PbwtVariant variant_256x16() { return make_variant<256, 16>(); }
}  // namespace eimp
