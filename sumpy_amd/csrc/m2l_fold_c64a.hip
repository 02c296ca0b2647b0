// complex FP32 kernels of the folded M2L contraction, orders 9 to 10.
#include "m2l_fold.h"

namespace sumpyhip {
namespace m2l_fold {

SUMPYHIP_FOLD_INSTANCE(c64a, float, true, 9, 10)

}  // namespace m2l_fold
}  // namespace sumpyhip
