// fa_fwd_pipe_fp8.hip -- the pipelined prefill (fa_fwd_pipe.h) on e4m3 inputs at
// kernel head dim 128: tiles stay bytes in LDS, K and V are widened to bf16 between
// their LDS reads and the products. (S^T as e4m3 products of the bytes is exact per
// product, but those MFMAs add with fewer bits: LSE 6e-5 off.) Dense causal B2 S4096
// H32/8: 476 -> 270 us against widening in the staging of fa_fwd.hip.
#include "fa_fwd_pipe.h"

namespace fa {

void launch_prefill_pipe_fp8(const FwdArgs& a, int grid, hipStream_t stream) {
    if (a.tile_rows == 128) pipe::launch_t<DT_FP8, 128, 1>(a, grid, stream);
    else pipe::launch_t<DT_FP8, 128, 2>(a, grid, stream);
}

}  // namespace fa
