// fa_fwd_pipe128.hip -- the pipelined prefill (fa_fwd_pipe.h) at kernel head dim 128.
#include "fa_fwd_pipe.h"

namespace fa {

void launch_prefill_pipe128(const FwdArgs& a, int dtype, int grid, hipStream_t stream) {
    if (a.tile_rows == 128) pipe::launch_d<128, 1>(a, dtype, grid, stream);
    else pipe::launch_d<128, 2>(a, dtype, grid, stream);
}

}  // namespace fa
