// real FP32 kernels of the folded M2L contraction, orders 1 to 8.
#include "m2l_fold.h"

namespace sumpyhip {
namespace m2l_fold {

SUMPYHIP_FOLD_INSTANCE(f32, float, false, 1, 8)

}  // namespace m2l_fold
}  // namespace sumpyhip
