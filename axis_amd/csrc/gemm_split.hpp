// fp32 products on the bf16 matrix cores (gemm_split.hip): the larger launches of gemm.hip's family.
//
// Every fp32 operand element is the exact sum of three bf16 values (24 significand bits = 8 + 8 + 8:
// x = hi + mid + lo, each the rounding of what the ones before leave), so a product is the sum of
// nine bf16 products, each exact in fp32.  The six of them above 2^-24 of the whole run on
// v_mfma_f32_16x16x32_bf16, whose rate is sixteen times v_mfma_f32_16x16x4_f32's; mid * lo, lo * mid
// and lo * lo are left out (together about a quarter of one fp32 rounding of the product).
#pragma once

#include "gemm_parts.hpp"

namespace axis {

// Output tiles: 256x128 (eight waves, two LDS stages, one block per CU), 128x128 and 256x64 (four
// waves, one stage, two blocks per CU), 64x64 (four waves of 32x32, two stages, three blocks per CU).
enum class SplitTile { None, Big, Mid, Tall, Small };

struct SplitPlan {
    SplitTile tile = SplitTile::None;
    int rows = 0, cols = 0;
    int64_t splits = 1;
};

// A tile's pace: blocks resident on a CU, microseconds a 32-deep step of a block takes of a full CU, the
// least a step takes (a block with the CU to itself waits on its own latencies), and what a round of
// blocks takes besides (launch, first loads, last stores).
struct TileRate {
    int resident;
    double step_us, alone_us, round_us;
};

// Time of a launch of `blocks` equal blocks of `steps` steps.
double launch_us(int64_t blocks, double steps, const TileRate &rate, int64_t cus);
// Time of writing, reading and summing the slices of a split reduction (5 TB/s and a launch).
double slices_us(int64_t splits, int64_t out_len);

// The tile and slice count of least estimated time, or None when none is below limit_us (the fp32
// kernels' own estimate).
SplitPlan split_plan(int64_t m, int64_t n, int64_t k, int64_t batch, int64_t cus, bool yr, bool aligned, int xmode,
                     double limit_us);

// Launches C = X . Y (operands, epilogue and slices as gemm.hip's kernels take them; p.tiles_m,
// p.tiles_n, p.k_chunk and p.xcd_span set for the plan's tile).  xr / yr: the operand is contiguous
// along the reduction.  aligned: both dense operands take 16-byte aligned vectors.  xmode: dense 0, cols
// mode 2, aligned cols mode 3, buffer rows mode with tap steps in block-major order 4 or without 5.
int split_gemm(axis_device device, const GemmParams &p, SplitTile tile, bool xr, bool yr, bool aligned, int xmode,
               unsigned blocks);

}  // namespace axis
