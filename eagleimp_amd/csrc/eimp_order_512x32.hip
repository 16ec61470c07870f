// eimp_order_512x32.hip -- the order chain with 512 threads, up to 32 positions each
#include "eimp_order.h"

namespace eimp {
PbwtVariant variant_512x32() { return make_variant<512, 32>(); }
}  // namespace eimp
