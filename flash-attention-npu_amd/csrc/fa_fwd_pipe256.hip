// fa_fwd_pipe256.hip -- the pipelined prefill (fa_fwd_pipe.h) at kernel head dim 256.
#include "fa_fwd_pipe.h"

namespace fa {

void launch_prefill_pipe256(const FwdArgs& a, int dtype, int grid, hipStream_t stream) {
    pipe::launch_d<256, 1>(a, dtype, grid, stream);
}

}  // namespace fa
