"""The decode kernel at the edges of its variants, against the fp64 oracle: both sides of the workgroup
size rule (512 pairs), projections in several passes, more rows than lane groups, group sizes between
the compiled ones, several passes over the state, and inputs of any alignment."""
import math

import pytest
import torch

from oracle import race_oracle as orc
from race_ref import bf16_planes, check

pytestmark = pytest.mark.gpu
EPS = 1e-6


def oracle_step(A, Bs, q, k, v, planes, L, K):
    """(out, A, Bs) in fp64 of one token: A [Z,S], Bs [Z,S,D], q [Z,G,D], k, v [Z,D]."""
    Z, G, D = q.shape
    _, protos = orc.build_planes_protos(D, K, L)
    rows = torch.cat([k[:, None], q], 1).double()[None]  # [1, Z, G + 1, D]: every row hashed on its own
    p, _, _, _ = orc.soft_hash_probs(rows, rows, rows, planes.double(), protos, L, K, scale=math.sqrt(D))
    p = p.view(Z, G + 1, -1)
    A = A.double() + p[:, 0]
    Bs = Bs.double() + p[:, 0, :, None] * v.double()[:, None]
    return (p[:, 1:] / (A + EPS)[:, None]) @ Bs, A, Bs


@pytest.mark.parametrize("B,Hkv,G,D,L,K,dt", [
    (1, 1, 1, 64, 1, 1, torch.bfloat16), (64, 8, 4, 64, 8, 4, torch.bfloat16), (57, 9, 4, 64, 8, 4, torch.bfloat16),
    (3, 2, 3, 64, 3, 3, torch.float32), (2, 2, 8, 64, 32, 4, torch.float32), (300, 2, 8, 64, 8, 4, torch.float32),
    (2, 1, 8, 128, 32, 4, torch.bfloat16), (520, 1, 2, 128, 5, 2, torch.float32), (9, 3, 5, 128, 16, 4, torch.bfloat16)])
@pytest.mark.parametrize("shift", [0, 1])
def test_decode_edges(dev, B, Hkv, G, D, L, K, dt, shift):
    from race_attention_amd import RaceDecodeState, build_planes_protos
    print(f"decode B={B} Hkv={Hkv} G={G} D={D} L={L} K={K} {dt} shift={shift}", flush=True)
    g = torch.Generator().manual_seed(B + D + L)
    Z, S = B * Hkv, L << K
    planes, _ = build_planes_protos(D, K, L, 1, device=dev, seed=1)
    st = RaceDecodeState(B, Hkv * G, Hkv, D, L, K, planes, eps=EPS, device=dev)
    st.A.copy_(torch.rand(Z, S, generator=g) * 20 + 1)
    st.Bs.copy_(torch.randn(Z, S, D, generator=g))

    def rows(h):  # shifted by one element: rows of any alignment
        buf = torch.randn(B * h * D + shift, generator=g).to(dt).to(dev)
        return buf[shift:].view(B, h, D)

    q, k, v = rows(Hkv * G), rows(Hkv), rows(Hkv)
    pl = bf16_planes(planes) if dt == torch.bfloat16 else planes
    ref = oracle_step(st.A.cpu(), st.Bs.cpu(), q.reshape(Z, G, D).cpu(), k.reshape(Z, D).cpu(), v.reshape(Z, D).cpu(),
                      pl.cpu(), L, K)
    out = st.step(q, k, v)
    # the output's own rounding (2^-9 of its largest value), or fp32 sums of at most 512 buckets
    check("out", out.reshape(Z, G, D), ref[0], 2.0 ** -8 if dt == torch.bfloat16 else 2e-6)
    check("A", st.A, ref[1], 1e-6)
    check("Bs", st.Bs, ref[2], 1e-6)


@pytest.mark.parametrize("B,Hq,Hkv,D,dtype", [(1026, 1, 1, 64, torch.bfloat16), (207, 40, 5, 64, torch.bfloat16), (600, 4, 2, 128, torch.float32),
                                              (260, 32, 8, 64, torch.bfloat16), (173, 18, 6, 128, torch.bfloat16)])
def test_more_pairs_than_run_at_a_time(dev, B, Hq, Hkv, D, dtype):
    """Beyond 1024 (sequence, kv head) pairs a workgroup also reads the inputs of a later one ahead: the same
    step as two halves of the batch, to the bit, over three steps."""
    from race_attention_amd import RaceDecodeState, build_planes_protos
    L, K, n = 4, 3, B // 2
    print(f"pairs B={B} Hq={Hq} Hkv={Hkv} D={D} {dtype}", flush=True)
    planes, _ = build_planes_protos(D, K, L, 1, device=dev, seed=0)
    g = torch.Generator(device=dev).manual_seed(B)
    sizes = (B, n, B - n)
    whole, first, second = (RaceDecodeState(b, Hq, Hkv, D, L, K, planes, device=dev) for b in sizes)
    assert B * Hkv > 1024 and min(n, B - n) * Hkv > 512
    for _ in range(3):
        q, k, v = (torch.randn(B, h, D, generator=g, device=dev).to(dtype) for h in (Hq, Hkv, Hkv))
        out = whole.step(q, k, v)
        assert torch.equal(out, torch.cat([first.step(q[:n], k[:n], v[:n]), second.step(q[n:], k[n:], v[n:])]))
    assert torch.equal(whole.A, torch.cat([first.A, second.A])) and torch.equal(whole.Bs, torch.cat([first.Bs, second.Bs]))
