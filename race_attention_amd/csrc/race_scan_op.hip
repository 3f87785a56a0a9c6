// Instantiations of the fp32 op-path scan kernels (race_op_scan.h), one per bucket tile and padded
// head dim, and their dispatch.
#include "race_launch.h"
#include "race_op_scan.h"

namespace race {

// gpK and gv in one launch wherever both kinds of workgroup have as many waves: 64 buckets and head dim
// 64 (2^20 tokens x 4 streams, linear) 1995 -> 1960 us, 128 buckets (2048 tokens x 16 streams) 54.6 ->
// 51.1, (200003 x 4) 916 -> 927 without the launch between them
template <int ST, int BT, int DP>
constexpr bool op_one_launch = BT == 16 * OpCfg<ST, DP>::DW;

template <int ST, int DP, int ROWS>
static hipError_t launch_v(OpKernel k, const ScanParams &P, dim3 grid, hipStream_t s)
{
    // the bucket kernels of a 128-bucket tile run as two workgroups of 64 buckets: V and gO are
    // read twice, but two or three independent workgroups share a CU instead of one (before the
    // suffixes moved to fp64, 200003 tokens x 4 streams, S = 128, D = 64: gq 565 -> 535, gk 521 ->
    // 508 us; 32 buckets: 785 and 560). Side by side (op_place) against one half of the buckets
    // after the other: totals 182 -> 176, gq 623 -> 615, gk 527 -> 506
    constexpr bool LIN = ROWS != ROWS_BF16;  // (bf16 rows: RACE only, the host asks for nothing else)
    constexpr int BT = ST < 64 ? ST : 64, NWG = ST / BT;
    const dim3 bucket(BT * 4), value(OpCfg<ST, DP>::DW * 64);
    const dim3 bgrid(grid.x * NWG, grid.y, grid.z);
    switch (k) {
    case OP_TOTALS:
        hipLaunchKernelGGL((race_op_totals<BT, DP, NWG, ROWS>), bgrid, bucket, 0, s, P);
        break;
    case OP_READOUT:
        if (P.linear)
            hipLaunchKernelGGL((race_op_out<ST, DP, false, LIN, ROWS>), grid, value, 0, s, P);
        else
            hipLaunchKernelGGL((race_op_out<ST, DP, false, false, ROWS>), grid, value, 0, s, P);
        break;
    case OP_GQ:
        if (P.linear)
            hipLaunchKernelGGL((race_op_gq<BT, DP, NWG, LIN, ROWS>), bgrid, bucket, 0, s, P);
        else
            hipLaunchKernelGGL((race_op_gq<BT, DP, NWG, false, ROWS>), bgrid, bucket, 0, s, P);
        break;
    case OP_GKV:
        if constexpr (op_one_launch<ST, BT, DP>) {
            const dim3 vgrid(grid.x * (NWG + 1), grid.y, grid.z);
            if (P.linear)
                hipLaunchKernelGGL((race_op_gkv<ST, BT, DP, LIN, ROWS>), vgrid, bucket, 0, s, P);
            else
                hipLaunchKernelGGL((race_op_gkv<ST, BT, DP, false, ROWS>), vgrid, bucket, 0, s, P);
        } else if (P.linear) {
            hipLaunchKernelGGL((race_op_gk<BT, DP, NWG, LIN, ROWS>), bgrid, bucket, 0, s, P);
            hipLaunchKernelGGL((race_op_out<ST, DP, true, LIN, ROWS>), grid, value, 0, s, P);
        } else {
            hipLaunchKernelGGL((race_op_gk<BT, DP, NWG, false, ROWS>), bgrid, bucket, 0, s, P);
            hipLaunchKernelGGL((race_op_out<ST, DP, true, false, ROWS>), grid, value, 0, s, P);
        }
        break;
    }
    return hipGetLastError();
}

#define RACE_OP_VARIANTS(X) \
    X(16, 32) X(32, 32) X(64, 32) X(128, 32) \
    X(16, 64) X(32, 64) X(64, 64) X(128, 64) \
    X(16, 128) X(32, 128) X(64, 128) X(128, 128) \
    X(16, 256) X(32, 256) X(64, 256) X(128, 256)

int op_stage_tokens(int DP) { return op_stage(DP); }

hipError_t launch_scan_op(OpKernel k, int ST, int DP, const ScanParams &P, dim3 grid, hipStream_t s)
{
#define X(a, b) if (ST == a && DP == b) \
        return P.rows == ROWS_BF16  ? launch_v<a, b, ROWS_BF16>(k, P, grid, s) \
               : P.rows == ROWS_F32 ? launch_v<a, b, ROWS_F32>(k, P, grid, s) \
                                    : launch_v<a, b, ROWS_ANY>(k, P, grid, s);
    RACE_OP_VARIANTS(X)
#undef X
    return hipErrorInvalidValue;
}

}  // namespace race
