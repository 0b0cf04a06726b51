// fa_fwd_pipe64.hip -- the pipelined prefill (fa_fwd_pipe.h) at kernel head dim 64.
#include "fa_fwd_pipe.h"

namespace fa {

void launch_prefill_pipe64(const FwdArgs& a, int dtype, int grid, hipStream_t stream) {
    if (a.tile_rows == 128) pipe::launch_d<64, 1>(a, dtype, grid, stream);
    else pipe::launch_d<64, 2>(a, dtype, grid, stream);
}

}  // namespace fa
