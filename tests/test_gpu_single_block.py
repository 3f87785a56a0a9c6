"""Sequences of one block (short, or many streams): the fused readout starts from the zero state and
leaves the final one itself, with no totals pass and no block scan. Compared with the same call cut
into blocks of 32 tokens (the general path) and with the fp64 oracle, forward, backward and state."""
import math

import pytest
import torch

from oracle import race_oracle as orc
from race_ref import bf16_planes, check, oracle_layer

pytestmark = pytest.mark.gpu
EPS = 1e-6
BF16 = 2e-2  # the bar of tests/test_gpu_fused.py


@pytest.mark.parametrize("B,Hq,Hkv,T,D,L,K,f32", [
    (1, 1, 1, 1, 64, 8, 4, False), (2, 4, 1, 31, 64, 8, 4, True), (1, 8, 2, 32, 64, 3, 3, False),
    (2, 4, 4, 33, 128, 3, 3, False), (1, 6, 2, 100, 64, 16, 4, False), (2, 8, 1, 128, 64, 8, 4, False),
    (1, 3, 3, 127, 128, 8, 4, True), (1, 2, 2, 96, 64, 20, 2, False), (1, 4, 2, 70, 64, 5, 1, False)])
def test_single_block(dev, B, Hq, Hkv, T, D, L, K, f32):
    from race_attention_amd import build_planes_protos, race_causal_attention, race_causal_attention_with_state
    print(f"single block B={B} Hq={Hq} Hkv={Hkv} T={T} D={D} L={L} K={K} f32={f32}", flush=True)
    g = torch.Generator().manual_seed(T + D)
    q, k, v, go = (torch.randn(B, h, T, D, generator=g).to(torch.bfloat16) for h in (Hq, Hkv, Hkv, Hq))
    planes, protos = build_planes_protos(D, K, L, 1, device=dev, seed=2)
    pl, dt = bf16_planes(planes).cpu(), torch.float32 if f32 else torch.bfloat16
    out, A, Bs = race_causal_attention_with_state(q.to(dev), k.to(dev), v.to(dev), planes, L, K, eps=EPS, out_dtype=dt)
    ref, dq, dk, dv = oracle_layer(q, k, v, pl, L, K, math.sqrt(D), EPS, go)
    check("out", out, ref, BF16)
    pk, _, _, _ = orc.soft_hash_probs(k.double(), k.double(), v.double(), pl.double(), protos.cpu(), L, K, scale=math.sqrt(D))
    check("A", A, pk.sum(1), BF16)
    check("Bs", Bs, pk.transpose(1, 2) @ v.double().reshape(B * Hkv, T, D), BF16)
    grads = {}
    for block in (0, 32):
        x = [t.to(dev).requires_grad_(True) for t in (q, k, v)]
        o = race_causal_attention(*x, planes, L, K, eps=EPS, out_dtype=dt, block=block)
        # the general path forms the same products in the same order within a block of 32 tokens;
        # its block states pass through fp32 sums: bf16 rounding of the results is all that differs
        check(f"out, block {block}", o, out, 2.0 ** -7)
        o.backward(go.to(dev).to(dt))
        grads[block] = [t.grad for t in x]
        # (dk of very short sequences cancels to ~eps: measured against the gradients' common scale)
        top = max(t.abs().max().item() for t in (dq, dk, dv)) if T < 64 else 0.0
        for name, a, r in zip(("dq", "dk", "dv"), grads[block], (dq, dk, dv)):
            check(f"{name}, block {block}", a, r, BF16, abs_floor=max(2e-5, BF16 * top))


def test_prefill_many_streams_leaves_the_state_in_place(dev):
    """256 x 8 streams of 77 tokens: one block each; the decode state's own tensors are written, and a
    reset state prefilled again gives the same bits."""
    from race_attention_amd import RaceDecodeState, build_planes_protos, race_causal_attention_with_state
    B, Hq, Hkv, T, D, L, K = 256, 16, 8, 77, 64, 8, 4
    g = torch.Generator(device=dev).manual_seed(5)
    planes, _ = build_planes_protos(D, K, L, 1, device=dev, seed=0)
    q, k, v = (torch.randn(B, h, T, D, generator=g, device=dev).to(torch.bfloat16) for h in (Hq, Hkv, Hkv))
    st = RaceDecodeState(B, Hq, Hkv, D, L, K, planes, eps=EPS, device=dev)
    where = st.A.data_ptr(), st.Bs.data_ptr()
    out, A, Bs = race_causal_attention_with_state(q, k, v, planes, L, K, eps=EPS)
    for _ in range(2):
        st.reset()
        assert torch.equal(st.prefill(q, k, v), out)
        assert torch.equal(st.A, A) and torch.equal(st.Bs, Bs) and (st.A.data_ptr(), st.Bs.data_ptr()) == where
        assert st.tokens == T
    with pytest.raises(ValueError):
        RaceDecodeState(B // 2, Hq, Hkv, D, L, K, planes, device=dev).prefill(q, k, v)


@pytest.mark.parametrize("T,D,L,K,Hq,Hkv", [(1, 64, 8, 4, 2, 2), (77, 64, 8, 4, 4, 2), (96, 128, 16, 4, 3, 3), (33, 64, 5, 2, 4, 1)])
def test_mass_of_a_single_block_holds_no_eps(dev, T, D, L, K, Hq, Hkv):
    """The state's mass A is a sum of probabilities: whatever eps is (1e4 leaves 2^-11 of a sum that it is part
    of), A has the same bits, and is the sum of the general path's totals."""
    from race_attention_amd import _lib, build_planes_protos, race_causal_attention_with_state
    from race_attention_amd.attention import qkv_shape
    g = torch.Generator().manual_seed(T)
    q, k, v = (torch.randn(1, h, T, D, generator=g).to(torch.bfloat16).to(dev) for h in (Hq, Hkv, Hkv))
    planes, _ = build_planes_protos(D, K, L, 1, device=dev, seed=2)
    scale, S = 0.5, L << K  # (sharp: masses down to 1e-6 of the largest)
    A = [race_causal_attention_with_state(q, k, v, planes, L, K, scale=scale, eps=e)[1] for e in (1e-6, 1e-2, 1e4)]
    assert torch.equal(A[0], A[1]) and torch.equal(A[0], A[2])
    # the general path: the same call in blocks of 32 tokens
    sh, lib = qkv_shape(q, k, L, K, scale, 1e-6, 32), _lib.lib()
    state = _lib.workspace(lib.race_qkv_state_bytes(sh), dev)
    scr = _lib.workspace(lib.race_qkv_scratch_bytes(sh, 0), dev)
    out, A2, B2 = torch.empty_like(q), torch.empty_like(A[0]), torch.empty(Hkv, S, D, device=dev)
    views = [_lib.view4(t)[0] for t in (q, k, v)]
    _lib.check(lib.race_qkv_prefill(sh, *views, _lib.ptr(planes), _lib.out_view4(out), _lib.RACE_BF16, _lib.ptr(A2),
                                    _lib.ptr(B2), _lib.ptr(state), state.numel(), _lib.ptr(scr), scr.numel(),
                                    _lib.stream_of(q)), "race_qkv_prefill")
    # a matrix step adds its 32 tokens to the running sum (or, there, to zero) in at most 8 additions of 4
    # products, each off by up to an ulp of the sum, 2^-23 of it; the sums differ in what they start from
    assert ((A[0] - A2).abs() <= 8 * (T // 32 + 1) * 2.0 ** -23 * A2.abs()).all()


@pytest.mark.parametrize("T", [20, 3000])
def test_prefill_forms(dev, T):
    """One stream's prompt prefills the state of every sequence, and rows of k and v behind the prompt are
    not read; a prompt of another number of streams, or with rows missing, is refused."""
    from race_attention_amd import RaceDecodeState, build_planes_protos, race_causal_attention_with_state
    D, L, K, B, G = 64, 8, 4, 5, 4
    g = torch.Generator().manual_seed(T)
    q, k, v = (torch.randn(1, h, T + 7, D, generator=g).to(torch.bfloat16).to(dev) for h in (G, 1, 1))
    planes, _ = build_planes_protos(D, K, L, 1, device=dev, seed=2)
    out, A, Bs = race_causal_attention_with_state(q[:, :, :T], k[:, :, :T], v[:, :, :T], planes, L, K, eps=EPS)
    st = RaceDecodeState(B, G, 1, D, L, K, planes, eps=EPS, device=dev)
    assert torch.equal(st.prefill(q[:, :, :T], k, v), out)
    assert st.tokens == T and torch.equal(st.A, A.expand_as(st.A)) and torch.equal(st.Bs, Bs.expand_as(st.Bs))
    two = [x.expand(2, -1, -1, -1) for x in (q, k, v)]
    with pytest.raises(ValueError):
        RaceDecodeState(B, G, 1, D, L, K, planes, eps=EPS, device=dev).prefill(*two)
    with pytest.raises(ValueError):
        race_causal_attention_with_state(q, k[:, :, :T], v, planes, L, K, eps=EPS)
