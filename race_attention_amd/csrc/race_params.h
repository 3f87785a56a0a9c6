// Kernel parameter blocks shared by the HIP kernels and the host dispatch code.
#pragma once
#include <stdint.h>

namespace race {

// A [B][H][T][D] tensor view with contiguous last dim (element strides).
struct View {
    const void *p;
    int64_t sb, sh, st;
};

// An output view: like View, plus the element stride between s-tile partials
// (0 when the kernel writes the final tensor) and the element type.
struct OutView {
    void *p;
    int64_t sb, sh, st;
    int64_t tile;   // element offset added per s-tile (partial-sum buffers)
    int f32;        // 1: float32 elements, 0: bfloat16 elements
    // Bucket tiles launched one after another (fused kernels): a non-null acc holds the fp32 sum
    // of the earlier tiles' contributions ([B][H][T][D] with its own element strides), added to
    // this tile's before the store; stage_f32 asks for the kernel variant that stages rows in
    // fp32, so that the sum is rounded once, when the last tile writes it.
    const float *acc;
    int64_t acc_sb, acc_sh, acc_st;
    int stage_f32;
};

// One launch of the chunked causal scan.
//   stream z:  op path   z = n (one of N independent [T,S]/[T,D] streams)
//              qkv mode  z = b * Hkv + hk (one kv head; query heads hk*G .. hk*G+G-1)
//   grid:      (NB blocks along T, n_st bucket tiles, Z streams)
struct ScanParams {
    int T, S, D, L, K, R;  // tokens, buckets S = L*R, head dim, tables, bits, 2^K
    int G, Hkv;            // query heads per kv head, kv heads (qkv mode)
    int CB, NB;            // tokens per block, blocks
    int n_st, S_pad;       // bucket tiles per stream, n_st * tile
    int st_base;           // bucket tile of grid row blockIdx.y = 0 (tiles launched one at a time)
    int DPw;               // padded head dim used by the state workspaces
    float eps, scale, inv_scale;
    // qkv mode (bf16 activations; planes_T fp32 [D][L*K], shared by all heads)
    View q, k, v, go;
    OutView out, dq, dk, dv;
    const float *planes;
    // op path (fp32): probabilities [N][T][S], values/grads rows of D floats (or bf16: ScanParams::rows). Stream z reads its
    // V / gO rows as a [Z / zH][zH][T][D] view: row t of z at (z / zH) sb + (z % zH) sh + t st,
    // strides in v / go (their p unused); contiguous [N][T][D] is zH = 1, sb = T D, st = D
    const float *pK, *pQ, *V, *gO;
    int zH;
    float *gpK, *gpQ;
    // workspaces: block states [Z][NB+1][S_pad][DPw] and [Z][NB+1][S_pad]
    float *wsB, *wsA;    // forward: prefix (A, B) at each block start; slot NB = final
    float *ws2B, *ws2A;  // backward: suffix sums (of W^T go, gA) from each block's start
    // op path and generic bf16 backward kernels: low parts of the same suffix sums (ws2 + ws3 = a double-float)
    float *ws3B, *ws3A;
    // op path, backward: A at every stage start of every block, [Z][NB][NCK][S_pad]
    float *ckA;
    int NCK;
    int rows;  // op path: how the rows of V, gO, out and gV lie (ROWS_* of race_op_scan.h)
    // fused readout of a sequence that is one block: no totals pass and no block scan have run. The
    // state starts at zero, and its final value goes to finB / finA (rows s < finS of stream z at
    // z * finBz / z * finAz; DPw floats per row); with wsB, zeros go to block 0's prefix there.
    int single, finS;
    float *finB, *finA;
    int64_t finBz, finAz;
    // op path only: 1 = unnormalised causal linear attention, W = pQ (no 1/(A+eps), gA = 0)
    int linear;
};

// op path, rows loaded one element at a time: the token that stands in for token t0 + r of a block that ends
// at t_end. Never behind the block's last one, also where the whole stage lies behind it (the look-ahead
// of the last stage), so that every address formed is one of the tensor's rows.
constexpr int op_clamped_row(int t0, int r, int t_end) { return t0 + r < t_end ? t0 + r : t_end - 1; }

}  // namespace race
