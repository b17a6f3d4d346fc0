// The tails of a batch's smaller meshes (batch.hpp).
#include "batch.hpp"

namespace obvhs {

void launch_tail_small(int c, const BatchTail& t) {
    if (c == 0) launch_tail<(int)B_TAIL_SIZES[0]>(t);
    else launch_tail<(int)B_TAIL_SIZES[1]>(t);
}

}  // namespace obvhs
