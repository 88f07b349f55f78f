// Prefill EXL3 GEMM (exl3_gemm):
//   C = fp16( H( fp16(H(A * suh)) . W_q ) * svh )
// Replaces the reconstruct branch of orcasaq2/ops.py:50-59 (had_r_128 -> reconstruct ->
// hgemm_recon -> had_r_128), and the fused exl3_gemm of orcasaq2/ops.py:46-49 for 17..144
// rows; the dense W_q is never written to HBM.  Up to KS_MAX_ROWS rows the K-split decode-GEMM
// (gemm_ks.hip); above, one Hadamard pass over A into the workspace (whose first workgroup also
// clears the stream-K launch's tile counters), then the 256-row stream-K kernel of gemm_sk.hip.
// The line lies where the taller tile's decode, paid once for 256 rows, overtakes the K split's
// even load: measured on MI355X (us per call in a HIP graph, K split / stream-K) at 512 rows
// 17408 -> 5120 131 / 156, 5120 -> 17408 135 / 131, 5120 -> 6144 58 / 91, at 256 rows
// 75 / 114, 81 / 105, 39 / 65.
#include "exl3_common.h"
#include "exl3_launch.h"
#include "gemm_sk_plan.h"

namespace exl3 {

size_t gemm_workspace_bytes(int rows, int ic, int oc)
{
    if (rows <= KS_MAX_ROWS) return gemm_ks_shard_bytes(rows, ic, oc);
    return gemm_sk_ah_bytes(rows, ic) + gemm_sk_slot_bytes(rows, oc);
}

int gemm_dispatch(const uint16_t* A, const uint32_t* trellis, uint16_t* C, const uint16_t* suh,
                  const uint16_t* svh, void* workspace, size_t ws_bytes, int rows, int ic, int oc,
                  int K, int cb, hipStream_t stream)
{
    const size_t need = gemm_workspace_bytes(rows, ic, oc);
    if (ws_bytes < need)
        return set_error(EXL3_ERR_WORKSPACE, "exl3_gemm: workspace of %zu bytes, %zu needed", ws_bytes, need);
    if (K < 1 || K > 8) return set_error(EXL3_ERR_ARG, "exl3_gemm: K=%d is not in 1..8", K);
    const GemvShard d{trellis, suh, svh, C, ic, oc, K, cb, (long)oc};
    return gemm_grouped_dispatch(A, &d, 1, rows, static_cast<char*>(workspace), ws_bytes, stream, "exl3_gemm");
}

}  // namespace exl3
