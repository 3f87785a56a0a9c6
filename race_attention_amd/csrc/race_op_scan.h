// The fp32 causal scan of the op path (probabilities in HBM): RaceCausalFn and causal linear
// attention. Math and block decomposition as race_scan.h; sub-chunks of 16 tokens.
//
// What bounds it: fp32 MFMA issue (v_mfma_f32_16x16x4_f32, 64 flops per cycle and SIMD) next to
// HBM. So no wave spends MFMA time, LDS traffic or barriers on moving the state: a 16x16
// accumulator tile (lane (n, g): rows 4g + e of column n) is, register by register, the B operand
// (k = 4g + e, n) of a product that sums over its rows, and the matching A operand, row m with
// k = 4g .. 4g + 3, is one 16-byte LDS read of a row-major array. Two splits of the work follow:
//   * bucket kernels (race_op_totals, race_op_gq, race_op_gk): a wave owns 16 buckets and keeps
//     its state transposed, St^T[d][s]. pK, pQ and the gradients of both are read and written as
//     accumulator tiles straight from HBM, the A scan, W and the gA scan stay in registers, and
//     no wave needs another's results: V and go (shared by all waves through LDS, a stage of
//     tokens at a time) and the 16 x 16 products go V^T are all that is exchanged.
//   * value kernel (race_op_out): a wave owns 16 value columns of every bucket, St[s][d], for the
//     products that sum over the buckets. Forward in time it is the readout out = W B; walked in
//     reverse with (pK, W, go) for (W, pK, V) it is gv = pK dS, the same recurrence.
// The backward walks each block in reverse from the suffix behind the block, so the suffixes
// only ever grow, and no sub-chunk is taken back out of a sum. The A prefixes that this needs at
// each stage start are left by race_op_gq, which walks forward, and gA = -gpQ W comes from the
// gpQ that it wrote, instead of a second pass over go St^T with a second copy of the state.
//
// Measured against the kernels with the state in LDS that these replace (us, one MI355X):
//   RACE, 200003 tokens x 4 streams, S = 128, D = 64: totals 189 -> 178, readout 525 -> 355 (and no
//     partial outputs of two bucket tiles to add, 2 x 96), gpQ + totals 707 -> 533, gpK and gv
//     1356 -> 873
//   linear attention, 2^20 tokens x 4 streams, 64 x 64: 421 -> 428, 1205 -> 888, 1687 -> 1334,
//     3185 -> 1864: at 3.2 - 5.0 TB/s of the compulsory reads and writes (a plain copy moves 4.8)
//     with the matrix cores busy 64, 74, 66 and 68 % of the time
//   2047 tokens x 96 streams, bf16 rows, S = 24, D = 128: 35 -> 32, 76 -> 55, 153 -> 110, 337 -> 162
#pragma once
#include <type_traits>

#include "race_scan.h"

namespace race {

// How the rows of V, gO, out and gV lie (ScanParams::rows): fp32 rows of any length and pitch, moved one
// element at a time; fp32 rows that move as 16-byte runs (S % 4 == 0, D % 4 == 0, any address: 200003
// tokens x 4 streams, S = 128, D = 64 at odd addresses, forward and backward 2260 -> 2077 us); bf16 rows that move as 8-byte runs, out and gV rounded to bf16 as they are
// stored. The last are the activations of a bf16 model in their own layout: products, states and
// sums stay fp32 and the results are those of fp32 copies to the bit, but no pass casts and transposes
// V, gO, out and gV (16 x 2047 tokens, 6 heads of 128, S = 24: forward and backward 675 -> 529 us)
enum { ROWS_ANY = 0, ROWS_F32 = 1, ROWS_BF16 = 2 };

// tokens per stage of the bucket kernels (also the spacing of the A checkpoints): as many as leave
// two workgroups' V and go tiles room in LDS (32 tokens at D = 128, S = 32: gq 106 against 100, gk 84
// against 79 us at 32752 tokens x 6 streams)
constexpr int op_stage(int DP) { return DP >= 128 ? 16 : 32; }
// waves per SIMD asked of the register allocator: what the LDS allows of workgroups per CU, as far as
// it does without spills in the main variants (gq at 3: 736 against 630 us, S = 128, D = 64). Without
// it the value kernel's state lands in AGPRs and is copied on every use
constexpr int op_waves_gq(int ST, int DP) { return DP <= 64 || (DP <= 128 && ST > 16) ? 2 : 1; }
constexpr int op_waves_gk(int DP) { return DP <= 64 ? 3 : DP <= 128 ? 2 : 1; }
constexpr int op_waves_value(int ST, int DP) { return DP <= 128 && ST < 128 ? 3 : 2; }

template <int ST, int DP>
struct OpCfg {
    static constexpr int NTS = ST / 16, NTD = DP / 16;
    static constexpr int TS = op_stage(DP);
    // value kernel: waves, column tiles per wave and tokens per stage (its LDS holds the stage's
    // W and pK three times over)
    static constexpr int DW = NTD < 8 ? NTD : 8, TD = NTD / DW;
    static constexpr int DTS = ST >= 32 ? 32 : 64;
    static_assert(DTS % TS == 0, "A checkpoints at every value-kernel stage");
};

RACE_DEV void mma4(f32x4 &c, const f32x4 &a, const f32x4 &b)
{
#pragma unroll
    for (int e = 0; e < 4; ++e)
        c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], b[e], c, 0, 0, 0);
}

// A sum over N reduction steps of 16 in CH chains. One running sum rounds every term at the size of the
// whole; in 4 chains, out of the fp32 layer at 2048 tokens, 128 buckets, is 1.07e-7 off 64 bits (relative
// 2-norm) instead of 1.63e-7, gv 1.23e-7 instead of 1.69e-7, in the same time. The gradients of the
// probabilities, sums over the head dim, take 1 (4 chains: gq 532 -> 579 us at 200003 tokens x 4 streams,
// S = 128, for a tenth of their error), for gpQ of linear attention 2 (1357 -> 1285 us at 2^20 tokens)
template <int N, int C>
struct Chains {
    static constexpr int CH = N < C ? N : C;
    f32x4 c[CH] = {};
    RACE_DEV void add(int i, const f32x4 &a, const f32x4 &b) { mma4(c[i % CH], a, b); }
    RACE_DEV f32x4 sum() const
    {
        f32x4 x = c[0];
        if constexpr (CH == 2)
            x += c[1];
        else if constexpr (CH == 4)
            x = (x + c[1]) + (c[2] + c[3]);
        static_assert(CH == 1 || CH == 2 || CH == 4, "chains are added in pairs");
        return x;
    }
};

RACE_DEV f32x4 ld4(const float *p) { return *reinterpret_cast<const f32x4 *>(p); }
RACE_DEV void st4(float *p, const f32x4 &v) { *reinterpret_cast<f32x4 *>(p) = v; }

// Range-checked access through a buffer descriptor (raw, dword-granular): a lane whose byte offset
// is not below num_records reads zero and stores nothing. One descriptor per stage, ending behind
// the stage's last valid row, therefore replaces every clamp, mask and predicate on rows, and a
// lane without a column takes the offset OP_OOB; addresses are one 32-bit add per access.
typedef __amdgpu_buffer_rsrc_t OpBuf;
constexpr uint32_t OP_OOB = 0x80000000u;
RACE_DEV OpBuf op_buf(const void *p, int64_t floats, int bytes = 4)
{
    // (the same in every lane: stated, so that no loop over the lanes' descriptors is made of it)
    const uint64_t a = reinterpret_cast<uint64_t>(p);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((int)a), hi = __builtin_amdgcn_readfirstlane((int)(a >> 32));
    return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void *>((uint64_t)hi << 32 | lo), 0,
                                             __builtin_amdgcn_readfirstlane((int)(floats * bytes)), 0x00027000);
}
RACE_DEV float buf_ld(OpBuf b, uint32_t off)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(b, off, 0, 0));
}
RACE_DEV f32x4 buf_ld4(OpBuf b, uint32_t off)
{
    return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(b, off, 0, 0));
}
RACE_DEV u32x2 buf_ld2(OpBuf b, uint32_t off)
{
    return __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(b, off, 0, 0));
}
// fp32 of what a load left: fp32, pairs of bf16, or a bf16 in each low half
RACE_DEV f32x4 op_widen(const f32x4 &v) { return v; }
RACE_DEV f32x4 op_widen(const u32x2 &v)
{
    return __builtin_bit_cast(f32x4, u32x4{v[0] << 16, v[0] & 0xffff0000u, v[1] << 16, v[1] & 0xffff0000u});
}
RACE_DEV f32x4 op_widen(const u32x4 &v) { return __builtin_bit_cast(f32x4, v << 16); }
RACE_DEV uint32_t buf_ld_h(OpBuf b, uint32_t off) { return __builtin_amdgcn_raw_buffer_load_b16(b, off, 0, 0); }
RACE_DEV void buf_st_h(OpBuf b, uint32_t off, float v)
{
    __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(unsigned short, (__bf16)v), b, off, 0, 0);
}
RACE_DEV void buf_st(OpBuf b, uint32_t off, float v)
{
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), b, off, 0, 0);
}

// LDS pitches: rows at an odd multiple of 8 words make the 16-row A-fragment reads conflict-free
constexpr int op_pitch(int n) { return n + 8; }

// Position of a workgroup: block, stream, bucket tile.
struct OpCtx {
    int lane, wave, n, g;  // n = lane % 16, g = lane / 16
    int z, blk, s0, S_here;
    int t_begin, t_end;
    int64_t slot;
};

// (tile: this kernel's bucket tile of ST)
template <int ST>
RACE_DEV OpCtx op_ctx(const ScanParams &P, int blk, int tile)
{
    OpCtx c;
    c.lane = threadIdx.x & 63;
    c.wave = threadIdx.x >> 6;
    c.n = c.lane & 15;
    c.g = c.lane >> 4;
    c.blk = blk;
    c.z = blockIdx.z;
    c.s0 = tile * ST;
    c.S_here = min(ST, P.S - c.s0);
    c.t_begin = c.blk * P.CB;
    c.t_end = min(P.T, c.t_begin + P.CB);
    c.slot = (int64_t)c.z * (P.NB + 1) + c.blk;
    return c;
}

// Workgroup w of the NWG that share a block's rows. They are 8 apart in launch order, so they run side
// by side on one XCD (workgroups go round the 8 in turn) and all but the first find the rows in its L2
// or, at worst, in the Infinity Cache. The last NB % 8 blocks form a narrower group.
template <int NWG>
RACE_DEV void op_place(const ScanParams &P, int &blk, int &w)
{
    const int i = blockIdx.x, whole = P.NB & ~7, j = i - whole * NWG;
    if (NWG == 1) {
        w = 0;
        blk = i;
    } else if (j < 0) {
        w = (i >> 3) % NWG;
        blk = (i >> 3) / NWG * 8 + (i & 7);
    } else {
        w = j / (P.NB - whole);
        blk = whole + j % (P.NB - whole);
    }
}

// Rows of V (and go) of one stage into LDS, row-major [TS][DP + 8] and / or transposed
// [DP][TS + 8]. A thread moves 4 rows x 4 columns, so both layouts are written as 16-byte runs.
// Rows beyond the stage and columns >= D read as zeros. bf16 rows wait as they are and are widened on
// their way into LDS. Rows of any length and pitch are loaded one element at a time from clamped addresses, a
// thread's 4 columns DP / 4 apart so that the lanes of a load read consecutive ones, and are masked on
// their way into LDS: masked where they are loaded, the compiler moves each load under its mask and waits
// for it there (200003 tokens x 4 streams, forward and backward: S = 10, D = 64 1724 -> 682 us; S = 128,
// D = 50 3145 -> 2186). The kinds of rows are compiled apart (a branch between the two forms of
// a load makes the compiler wait for it on the spot, 278 -> 200 us for the block totals of 200003
// tokens x 4 streams, S = 128, D = 64). All items wait in registers, fetched a stage ahead.
template <int TS, int DP, int NTH, int NT, int ROWS>
struct RowStage {
    static constexpr int CH = DP / 4, IT = (TS / 4) * CH, N = (NT * IT + NTH - 1) / NTH;
    static constexpr int LDX = op_pitch(DP), LDT = op_pitch(TS);
    static_assert(IT % 64 == 0, "one tensor per wave and item");
    typedef typename std::conditional<ROWS == ROWS_BF16, u32x2, f32x4>::type Raw;
    Raw x[N][4];

    struct Src {  // (p: the address of the stream's first row, whatever its elements)
        const float *p;
        int64_t st;
    };

    // item i of the stage at t0 of a block that ends at t_end (t0 >= t_end: nothing is read, or the
    // block's last row again)
    static RACE_DEV void load(Raw (&v)[4], const Src &s, int i, int t0, int t_end, int D)
    {
        const int r = (i % IT) / CH * 4, c = (i % IT) % CH * 4, nv = min(TS, t_end - t0);
        if constexpr (ROWS == ROWS_BF16) {
            const OpBuf b = op_buf(reinterpret_cast<const __bf16 *>(s.p) + (int64_t)t0 * s.st,
                                   nv > 0 ? (int64_t)(nv - 1) * s.st + D : 0, 2);
            const uint32_t st = (uint32_t)s.st * 2, off = c < D ? r * st + c * 2 : OP_OOB;
#pragma unroll
            for (int j = 0; j < 4; ++j)
                v[j] = buf_ld2(b, off + j * st);
        } else if constexpr (ROWS == ROWS_F32) {
            const OpBuf b = op_buf(s.p + (int64_t)t0 * s.st, nv > 0 ? (int64_t)(nv - 1) * s.st + D : 0);
            const uint32_t st = (uint32_t)s.st * 4, off = c < D ? r * st + c * 4 : OP_OOB;
#pragma unroll
            for (int j = 0; j < 4; ++j)
                v[j] = buf_ld4(b, off + j * st);
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float *row = s.p + (int64_t)op_clamped_row(t0, r + j, t_end) * s.st;
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    v[j][e] = row[min(c / 4 + e * CH, D - 1)];
            }
        }
    }

    static RACE_DEV void store(const Raw (&raw)[4], float *rm, float *tr, int i, int t0, int t_end, int D)
    {
        const int r = (i % IT) / CH * 4, c = (i % IT) % CH * 4;
        f32x4 v[4] = {op_widen(raw[0]), op_widen(raw[1]), op_widen(raw[2]), op_widen(raw[3])};
        if constexpr (ROWS == ROWS_ANY) {
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    v[j][e] = t0 + r + j < t_end && c / 4 + e * CH < D ? v[j][e] : 0.0f;
        }
        if (rm) {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if constexpr (ROWS == ROWS_ANY) {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        rm[(r + j) * LDX + c / 4 + e * CH] = v[j][e];
                } else {
                    st4(rm + (r + j) * LDX + c, v[j]);
                }
        }
        if (tr) {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                st4(tr + (ROWS == ROWS_ANY ? c / 4 + e * CH : c + e) * LDT + r,
                    f32x4{v[0][e], v[1][e], v[2][e], v[3][e]});
        }
    }

    // whether this wave's item k is of tensor a (uniform: IT is a multiple of 64)
    static RACE_DEV bool of_first(int k)
    {
        return NT == 1 || __builtin_amdgcn_readfirstlane(threadIdx.x) + k * NTH < IT;
    }

    // NT = 2: items of tensor a first, then of tensor b
    RACE_DEV void fetch(const Src &a, const Src &b, int t0, int t_end, int D)
    {
#pragma unroll
        for (int k = 0; k < N; ++k) {
            const int i = threadIdx.x + k * NTH;
            if (NT * IT % NTH == 0 || i < NT * IT)
                load(x[k], of_first(k) ? a : b, i, t0, t_end, D);
        }
    }

    RACE_DEV void put(float *rma, float *tra, float *rmb, float *trb, int t0, int t_end, int D)
    {
#pragma unroll
        for (int k = 0; k < N; ++k) {
            const int i = threadIdx.x + k * NTH;
            if (NT * IT % NTH == 0 || i < NT * IT) {
                const bool first = of_first(k);
                store(x[k], first ? rma : rmb, first ? tra : trb, i, t0, t_end, D);
            }
        }
    }
};

// This wave's 16 x 16 tile of an [N][T][S] tensor: rows 4g + e of the sub-chunk at row `row0` of the
// stage. `off` is the byte offset of row 4g in the lane's column (OP_OOB for a padding column), S4
// the row pitch in bytes.
RACE_DEV f32x4 op_tile(OpBuf b, uint32_t off, uint32_t S4, int row0)
{
    f32x4 x;
#pragma unroll
    for (int e = 0; e < 4; ++e)
        x[e] = buf_ld(b, off + (row0 + e) * S4);
    return x;
}
RACE_DEV void op_store_tile(OpBuf b, uint32_t off, uint32_t S4, int row0, const f32x4 &v)
{
#pragma unroll
    for (int e = 0; e < 4; ++e)
        buf_st(b, off + (row0 + e) * S4, v[e]);
}

// Column sums of a tile over its four lane groups: pair = own group + its neighbour (g ^ 1),
// far = the pair of the other half; the column total is pair + far in every lane.
struct GroupSums {
    float near, far, total;
    RACE_DEV explicit GroupSums(float own)
    {
        near = __shfl_xor(own, 16);
        const float pair = own + near;
        far = __shfl_xor(pair, 32);
        total = pair + far;
    }
    // sum over the groups before (after) group g
    RACE_DEV float before(int g) const { return (g & 1 ? near : 0.0f) + (g & 2 ? far : 0.0f); }
    RACE_DEV float after(int g) const { return (g & 1 ? 0.0f : near) + (g & 2 ? 0.0f : far); }
};

// eps of bucket col: 1 for the padding, whose A is zero (eps = 0 is taken, and 0 / 0 of a padding bucket
// would reach every output)
RACE_DEV float op_eps(const ScanParams &P, const OpCtx &c, int col) { return col < c.S_here ? P.eps : 1.0f; }

// inv = 1 / (A + eps) of a sub-chunk tile of pK; a0 (A before the sub-chunk) moves past it
RACE_DEV f32x4 op_inv_a(const f32x4 &pk, float &a0, float eps, int g)
{
    f32x4 c = pk;
#pragma unroll
    for (int e = 1; e < 4; ++e)
        c[e] += c[e - 1];
    const GroupSums gs(c[3]);
    const float base = a0 + gs.before(g);
    a0 += gs.total;
    f32x4 inv;
#pragma unroll
    for (int e = 0; e < 4; ++e)
        inv[e] = frcp(base + c[e] + eps);
    return inv;
}

// M[sub][row][col] = X[row] . Y[col] over K LDS columns for the 16 x 16 diagonal blocks of a stage,
// zero where `upper ? col < row : col > row`; KS waves share a block, each one K / KS range of the
// sum, left as KS partial copies for the reader to add (op_m).
template <int NSUB, int KS, int NW, int K, int LD, int LDM>
RACE_DEV void op_diag(float *sM, const float *X, const float *Y, bool upper, const OpCtx &c)
{
    static_assert(K % (16 * KS) == 0, "whole k steps per share");
#pragma unroll
    for (int j = 0; j < (NSUB * KS + NW - 1) / NW; ++j) {
        const int m = c.wave + j * NW;
        if (m < NSUB * KS) {
            const int sub = m / KS, ks = m % KS;
            const float *px = X + (sub * 16 + c.n) * LD + ks * (K / KS) + 4 * c.g;
            const float *py = Y + (sub * 16 + c.n) * LD + ks * (K / KS) + 4 * c.g;
            f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int k = 0; k < K / KS; k += 16)
                mma4(acc, ld4(px + k), ld4(py + k));
            float *dst = sM + (ks * NSUB + sub) * 16 * LDM;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int row = 4 * c.g + e;
                dst[row * LDM + c.n] = (upper ? c.n < row : c.n > row) ? 0.0f : acc[e];
            }
        }
    }
}

template <int NSUB, int KS, int LDM>
RACE_DEV f32x4 op_m(const float *sM, int sub, const OpCtx &c)
{
    const float *p = sM + (sub * 16 + c.n) * LDM + 4 * c.g;
    f32x4 m = ld4(p);
#pragma unroll
    for (int ks = 1; ks < KS; ++ks)
        m += ld4(p + ks * NSUB * 16 * LDM);
    return m;
}

// waves that share one diagonal block's sum
constexpr int op_shares(int NW, int NSUB, int ksteps)
{
    int ks = 1;
    while (ks < 4 && 2 * ks * NSUB <= NW && ksteps % (2 * ks) == 0)
        ks *= 2;
    return ks;
}

// Whether V and go also lie transposed in LDS, for the products that sum over tokens (their operand is then one
// 16-byte read). One wave to a workgroup and rows of 256 would leave one wave to a CU: 4 single reads
// of the rows instead leave 4 (100003 tokens x 4 streams, S = 16, D = 256: gq 1198 -> 290 us, gk and gv 811 -> 460)
constexpr bool op_transposed(int ST, int DP) { return ST > 16 || DP < 256; }

// rows k (of the transposed tile; columns of the row-major one) x tokens of sub-chunk s
template <bool TR, int LDX, int LDT>
RACE_DEV f32x4 op_tokens(const float *rm, const float *tr, int k, int s, const OpCtx &c)
{
    if constexpr (TR) {
        return ld4(tr + (k * 16 + c.n) * LDT + s * 16 + 4 * c.g);
    } else {
        const float *p = rm + (s * 16 + 4 * c.g) * LDX + k * 16 + c.n;
        return f32x4{p[0], p[LDX], p[2 * LDX], p[3 * LDX]};
    }
}

template <int ROWS>
RACE_DEV const float *op_first_row(const float *p, const View &v, int zH, int z)
{
    if constexpr (ROWS == ROWS_BF16)
        return reinterpret_cast<const float *>(reinterpret_cast<const __bf16 *>(p) + op_row_offset(v.sb, v.sh, zH, z));
    else
        return op_rows(p, v, zH, z);
}
template <class RS, int ROWS>
RACE_DEV typename RS::Src op_src(const float *p, const View &v, int zH, int z)
{
    return typename RS::Src{op_first_row<ROWS>(p, v, zH, z), v.st};
}

// state tiles St^T[d][s] <-> workspace [s][DPw]: a lane owns 4 consecutive d of its bucket
template <int NTD>
RACE_DEV void op_ld_state(f32x4 (&x)[NTD], const float *ws, int DPw, const OpCtx &c)
{
#pragma unroll
    for (int k = 0; k < NTD; ++k)
        x[k] = ld4(ws + (int64_t)(c.wave * 16 + c.n) * DPw + k * 16 + 4 * c.g);
}
template <int NTD>
RACE_DEV void op_st_state(float *ws, const f32x4 (&x)[NTD], int DPw, const OpCtx &c)
{
#pragma unroll
    for (int k = 0; k < NTD; ++k)
        st4(ws + (int64_t)(c.wave * 16 + c.n) * DPw + k * 16 + 4 * c.g, x[k]);
}

// The backward's suffix states (sums of W^T go) are carried in fp64: each sub-chunk's contribution is
// formed in fp32 on the matrix cores and added once. (In fp32 the sum of a block of one-signed terms
// loses more than the products do: gK of causal linear attention over 2^20 tokens 1.6e-7 -> 1.1e-6
// off. The conversions and adds are VALU work beside MFMA-bound waves.) The workspaces hold them as
// (hi, lo) pairs, as the block scan sums them.
struct Suffix {
    double x[4];

    RACE_DEV void load(const float *hi, const float *lo, int64_t o, int64_t pitch)
    {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            x[e] = (double)hi[o + e * pitch] + (double)lo[o + e * pitch];
    }
    RACE_DEV f32x4 value() const { return f32x4{(float)x[0], (float)x[1], (float)x[2], (float)x[3]}; }
    // += A B over 4 x 4 reduction steps
    RACE_DEV void add(const f32x4 &a, const f32x4 &b)
    {
        f32x4 t = {0.f, 0.f, 0.f, 0.f};
        mma4(t, a, b);
#pragma unroll
        for (int e = 0; e < 4; ++e)
            x[e] += (double)t[e];
    }
};

// The forward's prefix state, accumulated in fp32 by the matrix cores (same interface).
struct Prefix {
    f32x4 x;

    RACE_DEV void load(const float *ws, const float *, int64_t o, int64_t pitch)
    {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            x[e] = ws[o + e * pitch];
    }
    RACE_DEV f32x4 value() const { return x; }
    RACE_DEV void add(const f32x4 &a, const f32x4 &b) { mma4(x, a, b); }
};

RACE_DEV void put_hilo(float *hi, float *lo, int64_t o, double v)
{
    const float h = (float)v;
    hi[o] = h;
    lo[o] = (float)(v - (double)h);
}

// ============================================================================ block totals
// sum pK^T v and sum pK of each block -> workspace slot blk
template <int ST, int DP, int NWG, int ROWS>
__global__ __launch_bounds__(ST * 4) void race_op_totals(const ScanParams P)
{
    using CF = OpCfg<ST, DP>;
    constexpr int NTD = CF::NTD, NTH = ST * 4, TS = CF::TS, NSUB = TS / 16;
    using RS = RowStage<TS, DP, NTH, 1, ROWS>;
    __shared__ __align__(16) float sVt[DP * RS::LDT];
    int blk, wg;
    op_place<NWG>(P, blk, wg);
    const OpCtx c = op_ctx<ST>(P, blk, blockIdx.y * NWG + wg);
    const int col = c.wave * 16 + c.n;
    const uint32_t S4 = P.S * 4, off = col < c.S_here ? 4 * c.g * S4 + (c.s0 + col) * 4 : OP_OOB;
    const typename RS::Src src = op_src<RS, ROWS>(P.V, P.v, P.zH, c.z);
    const float *pK = P.pK + (int64_t)c.z * P.T * P.S;

    f32x4 St[NTD], pk[NSUB];
    double a = 0.0;  // (one-signed terms: no rounding of a long sum, beside MFMA-bound waves)
#pragma unroll
    for (int k = 0; k < NTD; ++k)
        St[k] = f32x4{0.f, 0.f, 0.f, 0.f};
    RS rs;
    auto fetch = [&](int t0) {  // (past the block end: nothing is read)
        const int nv = max(min(TS, c.t_end - t0), 0);
        rs.fetch(src, src, t0, c.t_end, P.D);
        const OpBuf bk = op_buf(pK + (int64_t)t0 * P.S, (int64_t)nv * P.S);
#pragma unroll
        for (int s = 0; s < NSUB; ++s)
            pk[s] = op_tile(bk, off, S4, s * 16);
    };
    fetch(c.t_begin);
    for (int t0 = c.t_begin; t0 < c.t_end; t0 += TS) {
        rs.put(nullptr, sVt, nullptr, nullptr, t0, c.t_end, P.D);
        f32x4 p[NSUB];
#pragma unroll
        for (int s = 0; s < NSUB; ++s) {
            p[s] = pk[s];
            a += (double)((p[s][0] + p[s][1]) + (p[s][2] + p[s][3]));
        }
        fetch(t0 + TS);
        __syncthreads();
#pragma unroll
        for (int s = 0; s < NSUB; ++s)
#pragma unroll
            for (int k = 0; k < NTD; ++k) {
                f32x4 t = {0.f, 0.f, 0.f, 0.f};
                mma4(t, ld4(sVt + (k * 16 + c.n) * RS::LDT + s * 16 + 4 * c.g), p[s]);
                St[k] += t;  // (one rounding per sub-chunk at the size of the block's sum)
            }
        __syncthreads();
    }
    op_st_state<NTD>(P.wsB + (c.slot * P.S_pad + c.s0) * P.DPw, St, P.DPw, c);
    a += __shfl_xor(a, 16);
    a += __shfl_xor(a, 32);
    if (c.g == 0)
        P.wsA[c.slot * P.S_pad + c.s0 + col] = P.linear ? 0.0f : (float)a;
}

// ============================================================================ gpQ and suffix totals
// Forward walk: gW = go St^T + tril(go V^T) pK, gpQ = gW / (A + eps), the block totals of W^T go
// and gA = -gpQ W, and A at every stage start for the reverse walks.
template <int ST, int DP, int NWG, bool LIN, int ROWS>
__global__ __launch_bounds__(ST * 4) __attribute__((amdgpu_waves_per_eu(op_waves_gq(ST, DP)))) void race_op_gq(const ScanParams P)
{
    using CF = OpCfg<ST, DP>;
    constexpr int NTD = CF::NTD, NW = ST / 16, NTH = ST * 4, TS = CF::TS, NSUB = TS / 16, LDM = 24;
    constexpr int KS = op_shares(NW, NSUB, DP / 16);
    using RS = RowStage<TS, DP, NTH, 2, ROWS>;
    __shared__ __align__(16) float sV[TS * RS::LDX], sGO[TS * RS::LDX];
    constexpr bool TR = op_transposed(ST, DP);
    __shared__ __align__(16) float sVt[TR ? DP * RS::LDT : 1], sGOt[TR ? DP * RS::LDT : 1];
    __shared__ __align__(16) float sM[KS * NSUB * 16 * LDM];
    int blk, wg;
    op_place<NWG>(P, blk, wg);
    const OpCtx c = op_ctx<ST>(P, blk, blockIdx.y * NWG + wg);
    const int col = c.wave * 16 + c.n;
    const uint32_t S4 = P.S * 4, off = col < c.S_here ? 4 * c.g * S4 + (c.s0 + col) * 4 : OP_OOB;
    const typename RS::Src sv = op_src<RS, ROWS>(P.V, P.v, P.zH, c.z), sg = op_src<RS, ROWS>(P.gO, P.go, P.zH, c.z);
    const float *pK = P.pK + (int64_t)c.z * P.T * P.S, *pQ = P.pQ + (int64_t)c.z * P.T * P.S;
    float *gpQ = P.gpQ + (int64_t)c.z * P.T * P.S;
    float *ck = P.ckA + (((int64_t)c.z * P.NB + c.blk) * P.NCK) * P.S_pad + c.s0 + col;

    f32x4 St[NTD], pk[NSUB], pq[NSUB];
    Suffix Tt[NTD] = {};
    op_ld_state<NTD>(St, P.wsB + (c.slot * P.S_pad + c.s0) * P.DPw, P.DPw, c);
    float a0 = LIN ? 0.0f : P.wsA[c.slot * P.S_pad + c.s0 + col];
    const float eps = op_eps(P, c, col);
    double ga = 0.0;
    RS rs;
    auto fetch = [&](int t0) {
        const int nv = max(min(TS, c.t_end - t0), 0);
        rs.fetch(sv, sg, t0, c.t_end, P.D);
        const OpBuf bk = op_buf(pK + (int64_t)t0 * P.S, (int64_t)nv * P.S);
        const OpBuf bq = op_buf(pQ + (int64_t)t0 * P.S, (int64_t)nv * P.S);
#pragma unroll
        for (int s = 0; s < NSUB; ++s) {
            pk[s] = op_tile(bk, off, S4, s * 16);
            pq[s] = op_tile(bq, off, S4, s * 16);
        }
    };
    fetch(c.t_begin);
    for (int t0 = c.t_begin; t0 < c.t_end; t0 += TS) {
        const int nv = min(TS, c.t_end - t0);
        rs.put(sV, TR ? sVt : nullptr, sGO, TR ? sGOt : nullptr, t0, c.t_end, P.D);
        f32x4 k_[NSUB], q_[NSUB];
#pragma unroll
        for (int s = 0; s < NSUB; ++s) {
            k_[s] = pk[s];
            q_[s] = pq[s];
        }
        fetch(t0 + TS);
        if constexpr (!LIN) {
            if (c.g == 0)
                *ck = a0;
            ck += P.S_pad;
        }
        __syncthreads();
        op_diag<NSUB, KS, NW, DP, RS::LDX, LDM>(sM, sGO, sV, false, c);
        __syncthreads();
        const OpBuf gq = op_buf(gpQ + (int64_t)t0 * P.S, (int64_t)nv * P.S);
#pragma unroll
        for (int s = 0; s < NSUB; ++s) {
            f32x4 inv = {1.f, 1.f, 1.f, 1.f};
            if constexpr (!LIN)
                inv = op_inv_a(k_[s], a0, eps, c.g);
            const f32x4 w = LIN ? q_[s] : q_[s] * inv;
            Chains<NTD, LIN ? 2 : 1> sum;
            sum.add(0, op_m<NSUB, KS, LDM>(sM, s, c), k_[s]);
#pragma unroll
            for (int k = 0; k < NTD; ++k)
                sum.add(k, ld4(sGO + (s * 16 + c.n) * RS::LDX + k * 16 + 4 * c.g), St[k]);
            f32x4 acc = sum.sum();
#pragma unroll
            for (int k = 0; k < NTD; ++k) {
                Tt[k].add(op_tokens<TR, RS::LDX, RS::LDT>(sGO, sGOt, k, s, c), w);
                mma4(St[k], op_tokens<TR, RS::LDX, RS::LDT>(sV, sVt, k, s, c), k_[s]);
            }
            if constexpr (!LIN) {
                acc *= inv;
                const f32x4 gw = acc * w;
                ga -= (double)((gw[0] + gw[1]) + (gw[2] + gw[3]));
            }
            op_store_tile(gq, off, S4, s * 16, acc);
        }
        __syncthreads();
    }
    const int64_t row = c.slot * P.S_pad + c.s0 + col;
#pragma unroll
    for (int k = 0; k < NTD; ++k)
#pragma unroll
        for (int e = 0; e < 4; ++e)
            put_hilo(P.ws2B, P.ws3B, row * P.DPw + k * 16 + 4 * c.g + e, Tt[k].x[e]);
    ga += __shfl_xor(ga, 16);
    ga += __shfl_xor(ga, 32);
    if (c.g == 0)
        put_hilo(P.ws2A, P.ws3A, row, ga);
}

// ============================================================================ gpK
// Reverse walk: gpK = gAhat + V dS^T + triu(V go^T) W, with dS the sum of W^T go and gAhat that of
// gA = -gpQ W over the tokens behind.
template <int ST, int DP>
struct OpGkLds {
    static constexpr int TS = op_stage(DP), NW = ST / 16, NSUB = TS / 16, LDM = 24;
    static constexpr int KS = op_shares(NW, NSUB, DP / 16), LDX = op_pitch(DP), LDT = op_pitch(TS);
    static constexpr bool TR = op_transposed(ST, DP);
    float V[TS * LDX], GO[TS * LDX], GOt[TR ? DP * LDT : 4], M[KS * NSUB * 16 * LDM];
};

template <int ST, int DP, bool LIN, int ROWS>
RACE_DEV void op_gk(const ScanParams &P, const OpCtx &c, OpGkLds<ST, DP> &lds)
{
    using CF = OpCfg<ST, DP>;
    using LD = OpGkLds<ST, DP>;
    constexpr int NTD = CF::NTD, NW = LD::NW, NTH = ST * 4, TS = LD::TS, NSUB = LD::NSUB, LDM = LD::LDM, KS = LD::KS;
    using RS = RowStage<TS, DP, NTH, 2, ROWS>;
    float *const sV = lds.V, *const sGO = lds.GO, *const sGOt = lds.GOt, *const sM = lds.M;
    const int col = c.wave * 16 + c.n;
    const uint32_t S4 = P.S * 4, off = col < c.S_here ? 4 * c.g * S4 + (c.s0 + col) * 4 : OP_OOB;
    const typename RS::Src sv = op_src<RS, ROWS>(P.V, P.v, P.zH, c.z), sg = op_src<RS, ROWS>(P.gO, P.go, P.zH, c.z);
    const int64_t zoff = (int64_t)c.z * P.T * P.S;
    const float *ck = P.ckA + (((int64_t)c.z * P.NB + c.blk) * P.NCK) * P.S_pad + c.s0 + col;

    f32x4 pk[NSUB], pq[NSUB], gq[NSUB];
    Suffix dS[NTD];
    const int64_t row = (c.slot + 1) * P.S_pad + c.s0 + col;
#pragma unroll
    for (int k = 0; k < NTD; ++k)
        dS[k].load(P.ws2B, P.ws3B, row * P.DPw + k * 16 + 4 * c.g, 1);
    double ga = LIN ? 0.0 : (double)P.ws2A[row] + (double)P.ws3A[row];
    const float eps = op_eps(P, c, col);
    float a_next = 0.0f;
    RS rs;
    const int nst = (c.t_end - c.t_begin + TS - 1) / TS;
    auto fetch = [&](int i) {  // stage i (below 0: stage 0 again, not used)
        const int j = max(i, 0), t0 = c.t_begin + j * TS;
        const int nv = min(TS, c.t_end - t0);
        rs.fetch(sv, sg, t0, c.t_end, P.D);
        const int64_t first = zoff + (int64_t)t0 * P.S, floats = (int64_t)nv * P.S;
        const OpBuf bq = op_buf(P.pQ + first, floats);
#pragma unroll
        for (int s = 0; s < NSUB; ++s)
            pq[s] = op_tile(bq, off, S4, s * 16);
        if constexpr (!LIN) {
            const OpBuf bk = op_buf(P.pK + first, floats), bg = op_buf(P.gpQ + first, floats);
#pragma unroll
            for (int s = 0; s < NSUB; ++s) {
                pk[s] = op_tile(bk, off, S4, s * 16);
                gq[s] = op_tile(bg, off, S4, s * 16);
            }
        }
        if constexpr (!LIN)
            a_next = ck[(int64_t)j * P.S_pad];
    };
    fetch(nst - 1);
    for (int i = nst - 1; i >= 0; --i) {
        const int t0 = c.t_begin + i * TS;
        const int nv = min(TS, c.t_end - t0);
        rs.put(sV, nullptr, sGO, LD::TR ? sGOt : nullptr, t0, c.t_end, P.D);
        f32x4 w[NSUB], gA[NSUB];
        float a0 = a_next;
#pragma unroll
        for (int s = 0; s < NSUB; ++s) {
            w[s] = pq[s];
            if constexpr (!LIN) {
                w[s] *= op_inv_a(pk[s], a0, eps, c.g);
                gA[s] = -gq[s] * w[s];
            }
        }
        fetch(i - 1);
        __syncthreads();
        op_diag<NSUB, KS, NW, DP, RS::LDX, LDM>(sM, sV, sGO, true, c);
        __syncthreads();
        const OpBuf out = op_buf(P.gpK + zoff + (int64_t)t0 * P.S, (int64_t)nv * P.S);
#pragma unroll
        for (int s = NSUB - 1; s >= 0; --s) {
            Chains<NTD, 1> sum;
            if constexpr (LIN)
                sum.add(0, op_m<NSUB, KS, LDM>(sM, s, c), w[s]);
#pragma unroll
            for (int k = 0; k < NTD; ++k)
                sum.add(k, ld4(sV + (s * 16 + c.n) * RS::LDX + k * 16 + 4 * c.g), dS[k].value());
            f32x4 acc = sum.sum();
            if constexpr (!LIN)  // (large weights of a sequence's first tokens: last, as in the gv walk)
                mma4(acc, op_m<NSUB, KS, LDM>(sM, s, c), w[s]);
#pragma unroll
            for (int k = 0; k < NTD; ++k)
                dS[k].add(op_tokens<LD::TR, RS::LDX, RS::LDT>(sGO, sGOt, k, s, c), w[s]);
            if constexpr (!LIN) {
                f32x4 q = gA[s];
#pragma unroll
                for (int e = 2; e >= 0; --e)
                    q[e] += q[e + 1];
                const GroupSums gs(q[0]);
                const float behind = (float)ga + gs.after(c.g);
                ga += (double)gs.total;
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    acc[e] += behind + q[e];
            }
            op_store_tile(out, off, S4, s * 16, acc);
        }
        __syncthreads();
    }
}

template <int ST, int DP, int NWG, bool LIN, int ROWS>
__global__ __launch_bounds__(ST * 4) __attribute__((amdgpu_waves_per_eu(op_waves_gk(DP)))) void race_op_gk(const ScanParams P)
{
    __shared__ __align__(16) OpGkLds<ST, DP> lds;
    int blk, wg;
    op_place<NWG>(P, blk, wg);
    op_gk<ST, DP, LIN, ROWS>(P, op_ctx<ST>(P, blk, blockIdx.y * NWG + wg), lds);
}

// ============================================================================ readout / gv
// REV = false: out[t] = sum_s W_t[s] sum_{tau <= t} pK_tau[s] v_tau
// REV = true:  gv[t]  = sum_s pK_t[s] sum_{tau >= t} W_tau[s] go_tau   (blocks and stages in reverse)
// Per stage: W (and pK) of all buckets to LDS, the 16 x 16 products over the buckets, then each
// wave walks the stage on its own with its columns of the state in registers.
template <int ST, int DP>
struct OpValueLds {
    using CF = OpCfg<ST, DP>;
    static constexpr int TS = CF::DTS, NSUB = TS / 16, LDM = 24, LDS_ = op_pitch(ST), LDT = op_pitch(TS);
    static constexpr int KS = op_shares(CF::DW, NSUB, CF::NTS);
    float Q[TS * LDS_], K[TS * LDS_], Kt[ST * LDT], M[KS * NSUB * 16 * LDM];
};

template <int ST, int DP, bool REV, bool LIN, int ROWS>
RACE_DEV void op_value(const ScanParams &P, const OpCtx &c, OpValueLds<ST, DP> &lds)
{
    using CF = OpCfg<ST, DP>;
    using LD = OpValueLds<ST, DP>;
    constexpr int NTS = CF::NTS, NW = CF::DW, TD = CF::TD, TS = LD::TS, NSUB = LD::NSUB, LDM = LD::LDM;
    constexpr int LDS_ = LD::LDS_, LDT = LD::LDT, KS = LD::KS;
    // W: a wave job covers CW buckets of the whole stage, lane (rg, lc): 4 tokens x 4 buckets
    constexpr int CW = 1024 / TS, NJ = ST / CW, JPW = (NJ + NW - 1) / NW, LC = CW / 4, RG = TS / 4;
    static_assert(NJ >= 1 && LC * RG == 64, "one job per 1024 probabilities");
    constexpr bool VEC = ROWS != ROWS_ANY, BF = ROWS == ROWS_BF16;
    float *const sQ = lds.Q, *const sK = lds.K, *const sKt = lds.Kt, *const sM = lds.M;
    const int rg = c.lane / LC, lc = c.lane % LC;
    const int64_t zoff = (int64_t)c.z * P.T * P.S;
    const float *xsrc = REV ? op_first_row<ROWS>(P.gO, P.go, P.zH, c.z) : op_first_row<ROWS>(P.V, P.v, P.zH, c.z);
    const int64_t xst = REV ? P.go.st : P.v.st;

    f32x4 pk[JPW][4], pq[JPW][4], a0[JPW];
    typename std::conditional<BF, u32x4, f32x4>::type xn[TD][NSUB];  // (bf16 in the low halves)
    typename std::conditional<REV, Suffix, Prefix>::type St[TD][NTS];
    {
        const int64_t row = (REV ? c.slot + 1 : c.slot) * P.S_pad + c.s0 + 4 * c.g;
#pragma unroll
        for (int td = 0; td < TD; ++td)
#pragma unroll
            for (int st = 0; st < NTS; ++st)
                St[td][st].load(REV ? P.ws2B : P.wsB, P.ws3B, (row + st * 16) * P.DPw + (c.wave + td * NW) * 16 + c.n,
                                P.DPw);
    }
    const float *ck = P.ckA + (((int64_t)c.z * P.NB + c.blk) * P.NCK) * P.S_pad + c.s0;
    const uint32_t S4 = P.S * 4;
    auto fetch = [&](int i) {  // stage i (past the block's ends: nothing is read, or stage 0 again)
        const int j = max(i, 0), t0 = c.t_begin + j * TS;
        const int nv = max(min(TS, c.t_end - t0), 0);
        const int64_t first = zoff + (int64_t)t0 * P.S, floats = (int64_t)nv * P.S;
        const OpBuf bk = op_buf(P.pK + first, floats), bq = op_buf(P.pQ + first, floats);
#pragma unroll
        for (int jj = 0; jj < JPW; ++jj) {
            const int col = (c.wave + jj * NW) * CW + 4 * lc;
            if (NJ % NW == 0 || c.wave + jj * NW < NJ) {
                const uint32_t off = 4 * rg * S4 + (c.s0 + col) * 4;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    if constexpr (VEC) {  // (S % 4 == 0: 4 buckets are valid or none)
                        const uint32_t o = col < c.S_here ? off + r * S4 : OP_OOB;
                        pk[jj][r] = buf_ld4(bk, o);
                        pq[jj][r] = buf_ld4(bq, o);
                    } else {
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const uint32_t o = col + e < c.S_here ? off + r * S4 + e * 4 : OP_OOB;
                            pk[jj][r][e] = buf_ld(bk, o);
                            pq[jj][r][e] = buf_ld(bq, o);
                        }
                    }
                }
                if constexpr (REV && !LIN)
                    a0[jj] = ld4(ck + (int64_t)j * (TS / CF::TS) * P.S_pad + col);
            }
        }
#pragma unroll
        for (int td = 0; td < TD; ++td) {
            const int d = (c.wave + td * NW) * 16 + c.n;
            if constexpr (BF) {
                const OpBuf bx = op_buf(reinterpret_cast<const __bf16 *>(xsrc) + (int64_t)t0 * xst,
                                        nv > 0 ? (nv - 1) * xst + P.D : 0, 2);
                const uint32_t st = (uint32_t)xst * 2, off = d < P.D ? 4 * c.g * st + d * 2 : OP_OOB;
#pragma unroll
                for (int s = 0; s < NSUB; ++s)
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        xn[td][s][e] = buf_ld_h(bx, off + (s * 16 + e) * st);
            } else if constexpr (VEC) {
                const OpBuf bx = op_buf(xsrc + (int64_t)t0 * xst, nv > 0 ? (nv - 1) * xst + P.D : 0);
                const uint32_t st = (uint32_t)xst * 4, off = d < P.D ? 4 * c.g * st + d * 4 : OP_OOB;
#pragma unroll
                for (int s = 0; s < NSUB; ++s)
                    xn[td][s] = op_tile(bx, off, st, s * 16);
            } else {
#pragma unroll
                for (int s = 0; s < NSUB; ++s)
#pragma unroll
                    for (int e = 0; e < 4; ++e)  // (masked where they are used)
                        xn[td][s][e] = xsrc[(int64_t)op_clamped_row(t0, s * 16 + 4 * c.g + e, c.t_end) * xst +
                                            min(d, P.D - 1)];
            }
        }
    };
    if constexpr (!REV && !LIN) {
#pragma unroll
        for (int jj = 0; jj < JPW; ++jj)
            if (NJ % NW == 0 || c.wave + jj * NW < NJ)
                a0[jj] = ld4(P.wsA + c.slot * P.S_pad + c.s0 + (c.wave + jj * NW) * CW + 4 * lc);
    }
    const int nst = (c.t_end - c.t_begin + TS - 1) / TS;
    fetch(REV ? nst - 1 : 0);
    for (int it = 0; it < nst; ++it) {
        const int i = REV ? nst - 1 - it : it;
        const int t0 = c.t_begin + i * TS;
        const int nv = min(TS, c.t_end - t0);
        // W = pQ / (A + eps) of the stage, with pK, into LDS
#pragma unroll
        for (int jj = 0; jj < JPW; ++jj) {
            if (NJ % NW == 0 || c.wave + jj * NW < NJ) {
                const int col = (c.wave + jj * NW) * CW + 4 * lc;
                f32x4 k_[4], w[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    k_[r] = pk[jj][r];
                    w[r] = pq[jj][r];
                }
                if constexpr (!LIN) {
                    f32x4 p[4];
                    p[0] = k_[0];
#pragma unroll
                    for (int r = 1; r < 4; ++r)
                        p[r] = p[r - 1] + k_[r];
                    f32x4 base;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        // exclusive scan of the 4-token sums over the lane's row groups
                        float x = __shfl_up(p[3][e], LC);
                        x = rg ? x : 0.0f;
#pragma unroll
                        for (int o = 1; o < RG; o *= 2) {
                            const float y = __shfl_up(x, o * LC);
                            x += rg > o ? y : 0.0f;
                        }
                        base[e] = a0[jj][e] + x;
                    }
#pragma unroll
                    for (int r = 0; r < 4; ++r)
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            w[r][e] *= frcp(base[e] + p[r][e] + op_eps(P, c, VEC ? col : col + e));
                    if constexpr (!REV) {
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            a0[jj][e] = __shfl(base[e] + p[3][e], (RG - 1) * LC + lc);
                    }
                }
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    st4(sQ + (4 * rg + r) * LDS_ + col, REV ? k_[r] : w[r]);
                    st4(sK + (4 * rg + r) * LDS_ + col, REV ? w[r] : k_[r]);
                }
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    st4(sKt + (col + e) * LDT + 4 * rg,
                        REV ? f32x4{w[0][e], w[1][e], w[2][e], w[3][e]} : f32x4{k_[0][e], k_[1][e], k_[2][e], k_[3][e]});
            }
        }
        f32x4 x[TD][NSUB];
#pragma unroll
        for (int td = 0; td < TD; ++td)
#pragma unroll
            for (int s = 0; s < NSUB; ++s) {
                x[td][s] = op_widen(xn[td][s]);
                if constexpr (ROWS == ROWS_ANY) {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        x[td][s][e] = s * 16 + 4 * c.g + e < nv && (c.wave + td * NW) * 16 + c.n < P.D ? x[td][s][e] : 0.0f;
                }
            }
        fetch(REV ? i - 1 : i + 1);
        __syncthreads();
        op_diag<NSUB, KS, NW, ST, LDS_, LDM>(sM, sQ, sK, REV, c);
        __syncthreads();
        const OutView &o = REV ? P.dv : P.out;
        // fp32: rows of D floats; bf16 (one bucket tile): rows through the view
        const OpBuf dst = BF ? op_buf(reinterpret_cast<const __bf16 *>(o.p) + op_row_offset(o.sb, o.sh, P.zH, c.z) +
                                          (int64_t)t0 * o.st,
                                      (int64_t)(nv - 1) * o.st + P.D, 2)
                             : op_buf(reinterpret_cast<const float *>(o.p) + (int64_t)blockIdx.y * o.tile +
                                          c.z * o.sb + (int64_t)t0 * P.D,
                                      (int64_t)nv * P.D);
#pragma unroll
        for (int ss = 0; ss < NSUB; ++ss) {
            const int s = REV ? NSUB - 1 - ss : ss;
            Chains<NTS, 4> sum[TD];
            const f32x4 m = op_m<NSUB, KS, LDM>(sM, s, c);
            // the sub-chunk's own tokens first, below the size of the sum; where the weights W of a sequence's
            // first tokens, up to 1 / eps, stand on the other side of m, last: the rest would be rounded
            // at their size (gv of sharp probabilities, 3001 tokens, S = 24, D = 128: 4.5e-7 against 1.3e-7 off)
            constexpr bool OWN_LAST = REV && !LIN;
            if constexpr (!OWN_LAST) {
#pragma unroll
                for (int td = 0; td < TD; ++td)
                    sum[td].add(0, m, x[td][s]);
            }
#pragma unroll
            for (int st = 0; st < NTS; ++st) {
                const f32x4 q = ld4(sQ + (s * 16 + c.n) * LDS_ + st * 16 + 4 * c.g);
                const f32x4 k = ld4(sKt + (st * 16 + c.n) * LDT + s * 16 + 4 * c.g);
#pragma unroll
                for (int td = 0; td < TD; ++td) {
                    sum[td].add(st, q, St[td][st].value());
                    St[td][st].add(k, x[td][s]);
                }
            }
#pragma unroll
            for (int td = 0; td < TD; ++td) {
                f32x4 acc = sum[td].sum();
                if constexpr (OWN_LAST)
                    mma4(acc, m, x[td][s]);
                const int d = (c.wave + td * NW) * 16 + c.n;
                const uint32_t st = BF ? (uint32_t)o.st * 2 : P.D * 4;
                const uint32_t off = d < P.D ? 4 * c.g * st + d * (BF ? 2 : 4) : OP_OOB;
                if constexpr (BF) {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        buf_st_h(dst, off + (s * 16 + e) * st, acc[e]);
                } else {
                    op_store_tile(dst, off, st, s * 16, acc);
                }
            }
        }
        __syncthreads();
    }
}

template <int ST, int DP, bool REV, bool LIN, int ROWS>
__global__ __launch_bounds__((OpCfg<ST, DP>::DW * 64)) __attribute__((amdgpu_waves_per_eu(op_waves_value(ST, DP)))) void race_op_out(const ScanParams P)
{
    __shared__ __align__(16) OpValueLds<ST, DP> lds;
    op_value<ST, DP, REV, LIN, ROWS>(P, op_ctx<ST>(P, blockIdx.x, blockIdx.y), lds);
}

// ============================================================================ gpK and gv in one launch
// The gpK workgroups of a block (ST / BT of them) and its gv workgroup side by side: both walk the block
// in reverse over the same pQ, go, pK and A checkpoints.
template <int ST, int BT, int DP, bool LIN, int ROWS>
__global__ __launch_bounds__(BT * 4) __attribute__((amdgpu_waves_per_eu(op_waves_value(ST, DP)))) void race_op_gkv(const ScanParams P)
{
    static_assert(BT == OpCfg<ST, DP>::DW * 16, "one workgroup size");
    constexpr int NB_ = ST / BT;
    __shared__ __align__(16) union { OpGkLds<BT, DP> k; OpValueLds<ST, DP> v; } lds;
    int blk, wg;
    op_place<NB_ + 1>(P, blk, wg);
    if (wg < NB_)
        op_gk<BT, DP, LIN, ROWS>(P, op_ctx<BT>(P, blk, blockIdx.y * NB_ + wg), lds.k);
    else
        op_value<ST, DP, true, LIN, ROWS>(P, op_ctx<ST>(P, blk, blockIdx.y), lds.v);
}

}  // namespace race
