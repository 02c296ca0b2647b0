// real FP64 kernels of the folded M2L contraction, orders 11 to 12.
#include "m2l_fold.h"

namespace sumpyhip {
namespace m2l_fold {

SUMPYHIP_FOLD_INSTANCE(f64b, double, false, 11, 12)

}  // namespace m2l_fold
}  // namespace sumpyhip
