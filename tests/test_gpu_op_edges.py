"""The fp32 op-path kernels at the edges of their tiles, against the fp64 oracle: sub-chunks of 16
tokens, stages of 16 / 32, bucket tiles of 16 .. 128 (and several), head-dim tiles of 32 .. 256, and
operands whose rows are not 16-byte aligned, and sizes that are no multiple of 4, whose rows move as single floats.

Bars as tests/test_gpu_op.py: forward 2e-5, gradients 1e-4 or twice what the reference formula itself
loses in fp32 (gradProbsK cancels at a sequence's first tokens)."""
import pytest
import torch

from oracle import race_oracle as orc
from race_ref import check, fp32_formula_floor, make_probs, oracle_op

pytestmark = pytest.mark.gpu
EPS = 1e-6


def probs(N, T, S, D, seed):
    pk, pq, v, go = make_probs(N, T, 1, S, D, seed, "raw")
    return pk + 0.05, pq, v, go  # (bounded away from 0: the bars are those of ordinary masses)


@pytest.mark.parametrize("N,T,S,D,block", [
    (1, 15, 15, 30, 0), (2, 16, 16, 32, 0), (2, 17, 17, 33, 0), (3, 31, 32, 64, 16), (1, 33, 33, 65, 0),
    (2, 65, 64, 128, 48), (2, 129, 65, 129, 0), (1, 200, 128, 64, 80), (2, 97, 129, 64, 0), (1, 70, 300, 96, 32),
    (1, 1, 128, 256, 0), (2, 130, 127, 255, 64)])
def test_tile_edges(dev, N, T, S, D, block):
    from race_attention_amd.race_causal_cuda import race_backward, race_fused_fwd
    print(f"edges N={N} T={T} S={S} D={D} block={block}", flush=True)
    pk, pq, v, go = probs(N, T, S, D, seed=T + S + D)
    out_t, gpk_t, gpq_t, gv_t, _, _ = oracle_op(pk, pq, v, go, EPS)
    pkc, pqc, vc, goc = (x.float().to(dev) for x in (pk, pq, v, go))
    check("out", race_fused_fwd(pkc, pqc, vc, EPS, block), out_t, 2e-5)
    floors = fp32_formula_floor(pk, pq, v, go, EPS, (gpk_t, gpq_t, gv_t))
    for name, g, ref, f in zip(("gpK", "gpQ", "gV"), race_backward(pkc, pqc, vc, goc, EPS, block),
                               (gpk_t, gpq_t, gv_t), floors):
        check(name, g, ref, max(1e-4, 2.0 * f))


@pytest.mark.parametrize("S,D", [(20, 32), (32, 64), (40, 64), (128, 64), (129, 64)])
@pytest.mark.parametrize("NB", [1, 7, 8, 9, 16, 27])
def test_block_counts(dev, S, D, NB):
    """Every block of a sequence is visited by all of its workgroups, which sit 8 apart in launch order:
    whole groups of 8 blocks and what is left over, one to three workgroups per block."""
    from race_attention_amd.race_causal_cuda import race_backward, race_fused_fwd
    T = 32 * NB - 5
    pk, pq, v, go = probs(2, T, S, D, seed=S + NB)
    out_t, gpk_t, gpq_t, gv_t, _, _ = oracle_op(pk, pq, v, go, EPS)
    args = [x.float().to(dev) for x in (pk, pq, v, go)]
    check("out", race_fused_fwd(*args[:3], EPS, 32), out_t, 2e-5)
    floors = fp32_formula_floor(pk, pq, v, go, EPS, (gpk_t, gpq_t, gv_t))
    for name, g, ref, f in zip(("gpK", "gpQ", "gV"), race_backward(*args, EPS, 32), (gpk_t, gpq_t, gv_t), floors):
        check(name, g, ref, max(1e-4, 2.0 * f))


@pytest.mark.parametrize("T,E,M", [(15, 15, 31), (16, 16, 32), (33, 17, 64), (65, 64, 65), (100, 129, 128)])
def test_linear_tile_edges(dev, T, E, M):
    from race_attention_amd.linear_attention import causal_linear_attention
    g = torch.Generator().manual_seed(T)
    Q, K, V, G = (torch.randn(2, 1, T, n, generator=g) for n in (E, E, M, M))
    ref_in = [x.double().requires_grad_() for x in (Q, K, V)]
    ref = orc.causal_linear_ref(*ref_in)
    ref.backward(G.double())
    got_in = [x.to(dev).requires_grad_() for x in (Q, K, V)]
    got = causal_linear_attention(*got_in)
    got.backward(G.to(dev))
    # sums of at most T * E products of O(1) terms in fp32
    check("out", got, ref, 2e-5)
    for name, a, b in zip("QKV", got_in, ref_in):
        check("g" + name, a.grad, b.grad, 2e-5)


@pytest.mark.parametrize("S,D", [(24, 64), (128, 128), (64, 256)])
def test_unaligned_rows_equal_aligned_ones(dev, S, D):
    """Rows that start 4 bytes off a 16-byte boundary: the same arithmetic, so the results are bitwise
    those of the aligned operands."""
    from race_attention_amd.race_causal_cuda import race_backward, race_fused_fwd
    args = [x.float().to(dev) for x in probs(2, 150, S, D, seed=S)]

    def shifted(x):
        buf = torch.empty(x.numel() + 1, device=dev)
        y = buf[1:].view(x.shape)
        y.copy_(x)
        assert y.data_ptr() % 16 == 4 and y.is_contiguous()
        return y

    off = [shifted(x) for x in args]
    assert torch.equal(race_fused_fwd(*args[:3], EPS), race_fused_fwd(*off[:3], EPS))
    for name, a, b in zip(("gpK", "gpQ", "gV"), race_backward(*args, EPS), race_backward(*off, EPS)):
        assert torch.equal(a, b), name


@pytest.mark.parametrize("S,D", [(3, 129), (8, 192), (16, 256)])
@pytest.mark.parametrize("T,block", [(1, 0), (17, 0), (100, 48)])
def test_one_wave_of_wide_rows(dev, S, D, T, block):
    """Up to 16 buckets at head dims above 128: a workgroup is one wave, with V and go in LDS as rows only."""
    test_tile_edges(dev, 2, T, S, D, block)


@pytest.mark.parametrize("S", [129, 192, 193, 256, 257, 320])
@pytest.mark.parametrize("D", [40, 128])
def test_several_bucket_tiles(dev, S, D):
    """Both sides of the line between tiles of 64 and of 128 beyond 128 buckets: sums over 2 to 5 tiles."""
    from race_attention_amd.race_causal_cuda import race_backward, race_fused_fwd
    pk, pq, v, go = probs(3, 100, S, D, seed=S)
    out_t, gpk_t, gpq_t, gv_t, _, _ = oracle_op(pk, pq, v, go, EPS)
    a = [x.float().to(dev) for x in (pk, pq, v, go)]
    check("out", race_fused_fwd(*a[:3], EPS), out_t, 2e-5)
    floors = fp32_formula_floor(pk, pq, v, go, EPS, (gpk_t, gpq_t, gv_t))
    for name, g, ref, f in zip(("gpK", "gpQ", "gV"), race_backward(*a, EPS), (gpk_t, gpq_t, gv_t), floors):
        check(name, g, ref, max(1e-4, 2.0 * f))


@pytest.mark.parametrize("S,D", [(6, 30), (18, 62), (24, 126), (10, 250), (66, 65), (130, 33), (3, 3)])
@pytest.mark.parametrize("T,block", [(1, 0), (33, 0), (150, 48)])
def test_odd_sizes_equal_padded_ones(dev, S, D, T, block):
    """Bucket counts or head dims that are no multiple of 4 take the kernels that move single floats; zeros
    behind the buckets and columns make the same call for those that move 16-byte runs. The arithmetic
    is the same, so the results are to the bit."""
    from race_attention_amd.race_causal_cuda import race_backward, race_fused_fwd
    print(f"odd sizes S={S} D={D} T={T} block={block}", flush=True)
    args = [x.float().to(dev) for x in probs(2, T, S, D, seed=S + T)]
    pad = [torch.nn.functional.pad(x, (0, -x.shape[2] % 4)) for x in args]
    assert torch.equal(race_fused_fwd(*args[:3], EPS, block), race_fused_fwd(*pad[:3], EPS, block)[:, :, :D])
    for name, a, b in zip(("gpK", "gpQ", "gV"), race_backward(*args, EPS, block), race_backward(*pad, EPS, block)):
        assert torch.equal(a, b[:, :, :a.shape[2]]), name


def test_values_beyond_a_block_do_not_leak(dev):
    """A non-finite value row reaches the outputs of its own and later tokens only: rows behind a
    block's or a sequence's end are read as zeros, never multiplied by zero probabilities."""
    from race_attention_amd.race_causal_cuda import race_fused_fwd
    pk, pq, v, _ = (x.float().to(dev) for x in probs(2, 96, 24, 64, seed=3))
    clean = race_fused_fwd(pk, pq, v, EPS, 48)
    v[0, 48] = float("nan")  # first row of the second block
    v[1, 0] = float("inf")   # first row of the second stream
    out = race_fused_fwd(pk, pq, v, EPS, 48)
    assert torch.equal(out[0, :48], clean[0, :48])
    assert not torch.isfinite(out[0, 48:]).any()


@pytest.mark.parametrize("T,S,D", [(50, 24, 64), (200, 192, 64), (70, 129, 128), (40, 15, 33)])
def test_eps_zero_with_padding_buckets(dev, T, S, D):
    """eps = 0 is taken: the padding buckets of a tile, whose mass is zero, reach no output."""
    from race_attention_amd.race_causal_cuda import race_backward, race_fused_fwd
    pk, pq, v, go = probs(2, T, S, D, seed=T + S + D)
    out_t, gpk_t, gpq_t, gv_t, _, _ = oracle_op(pk, pq, v, go, 0.0)
    pkc, pqc, vc, goc = (x.float().to(dev) for x in (pk, pq, v, go))
    check("out", race_fused_fwd(pkc, pqc, vc, 0.0, 0), out_t, 2e-5)
    floors = fp32_formula_floor(pk, pq, v, go, 0.0, (gpk_t, gpq_t, gv_t))
    for name, g, ref, f in zip(("gpK", "gpQ", "gV"), race_backward(pkc, pqc, vc, goc, 0.0, 0),
                               (gpk_t, gpq_t, gv_t), floors):
        check(name, g, ref, max(1e-4, 2.0 * f))


@pytest.mark.parametrize("pitch", [1 << 22, (1 << 22) + 4])
def test_value_row_pitch(dev, pitch):
    """Both sides of the row pitch up to which the totals move V in range-checked runs."""
    from race_attention_amd.noncausal import BatchedACE
    T, D = 40, 64
    ace = BatchedACE(D, 3, 3, 1, device=dev, share_planes=True)
    g = torch.Generator().manual_seed(0)
    k, v, q = (torch.randn(1, 1, T, 1, D, generator=g).to(dev) for _ in range(3))
    wide = torch.full((1, 1, T, 1, pitch), float("nan"), device=dev)
    wide[..., :D] = v
    assert torch.equal(ace(k, wide[..., :D], q, EPS), ace(k, v, q, EPS))


def norm_err(got, ref):
    return ((got.double().cpu() - ref).norm() / ref.norm()).item()


def test_rounding_of_the_layer_sums(dev):
    """Errors of the fp32 layer against 64 bits, 128 buckets. The sum over the buckets runs on the matrix
    cores, one rounding per 4 buckets: 32 in a row give u / sqrt(3) * sqrt(32 / 2) = 1.4e-7 (u = 2^-24) of a
    sum of random signs, four chains of 8 half of that or less; the products' own inputs (probabilities, state)
    add 0.8e-7. Measured: out 1.63e-7 in one running sum, 1.07e-7 in four chains; dv 1.69e-7 and 1.23e-7."""
    from race_attention_amd.race_causal_cuda import RaceCausalCuda
    from race_ref import oracle_layer
    B, H, T, D, L, K = 1, 4, 2048, 64, 8, 4
    m = RaceCausalCuda(D, K, L, 1, device=dev, seed=0)
    g = torch.Generator().manual_seed(0)
    q, k, v, go = (torch.randn(B, H, T, D, generator=g) for _ in range(4))
    x = [t.to(dev).requires_grad_() for t in (q, k, v)]
    out = m(*x)
    out.backward(go.to(dev))
    ref, _, _, dv = oracle_layer(q, k, v, m.planes_T.cpu(), L, K, D ** 0.5, m.eps, go)
    errs = norm_err(out.detach(), ref), norm_err(x[2].grad, dv)
    print("out, dv:", ["%.3e" % e for e in errs], flush=True)
    assert errs[0] <= 1.35e-7 and errs[1] <= 1.45e-7, errs


def test_rounding_of_the_linear_sums(dev):
    """As above for causal linear attention on positive features (its sums grow with the sequence), 8 streams of
    3001 tokens: out, dQ, dK, dV 1.21e-7, 2.29e-7, 1.48e-7, 1.14e-7 off in running sums over the head dim and
    a block's tokens, 0.65e-7, 1.71e-7, 1.29e-7, 0.57e-7 in chains and one rounding per sub-chunk; the bars lie
    between the two."""
    from race_attention_amd.linear_attention import causal_linear_attention
    g = torch.Generator().manual_seed(0)
    q, k = (torch.rand(2, 4, 3001, 32, generator=g) for _ in range(2))
    v, go = (torch.randn(2, 4, 3001, 32, generator=g) for _ in range(2))
    ref_in = [t.double().requires_grad_() for t in (q, k, v)]
    ref = orc.causal_linear_ref(*ref_in)
    ref.backward(go.double())
    got_in = [t.to(dev).requires_grad_() for t in (q, k, v)]
    got = causal_linear_attention(*got_in)
    got.backward(go.to(dev))
    errs = [norm_err(a, b) for a, b in zip([got.detach()] + [t.grad for t in got_in],
                                           [ref.detach()] + [t.grad for t in ref_in])]
    print("out, dQ, dK, dV:", ["%.3e" % e for e in errs], flush=True)
    assert all(e <= bar for e, bar in zip(errs, (0.95e-7, 2.0e-7, 1.4e-7, 0.85e-7))), errs
