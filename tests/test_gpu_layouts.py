"""Memory orders of the attention seam: outputs and gradients of race_attend stay in the [B,T,H,D]
order of the activations (no layout copies), with the values of the contiguous [B,H,T,D] call."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
EPS = 1e-6


@pytest.mark.parametrize("B,T,Hq,Hkv,D,L,K", [(2, 100, 4, 2, 64, 8, 4), (1, 513, 3, 3, 128, 3, 3), (2, 33, 6, 1, 64, 16, 4)])
def test_attend_bf16_equals_contiguous_layout(dev, B, T, Hq, Hkv, D, L, K):
    from race_attention_amd import build_planes_protos, race_causal_attention
    from race_attention_amd.nanochat import race_attend
    g = torch.Generator().manual_seed(T)
    planes, _ = build_planes_protos(D, K, L, 1, device=dev, seed=0)
    rows = [torch.randn(B, T, h, D, generator=g).to(torch.bfloat16) for h in (Hq, Hkv, Hkv, Hq)]
    x = [t.to(dev).requires_grad_(True) for t in rows[:3]]
    y = race_attend(*x, planes, L, K, EPS)
    assert y.shape == (B, T, Hq, D) and y.is_contiguous()
    y.backward(rows[3].to(dev))
    z = [t.to(dev).transpose(1, 2).contiguous().requires_grad_(True) for t in rows[:3]]
    o = race_causal_attention(*z, planes, L, K, eps=EPS)
    assert o.is_contiguous()
    o.backward(rows[3].to(dev).transpose(1, 2).contiguous())
    assert torch.equal(y, o.transpose(1, 2))
    for a, b in zip(x, z):
        assert a.grad.is_contiguous() and torch.equal(a.grad, b.grad.transpose(1, 2))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32, torch.float16])
@pytest.mark.parametrize("Hq,Hkv,packed", [(4, 4, False), (4, 2, False), (2, 2, True)])
def test_attend_fp32_equals_the_composed_ops(dev, dtype, Hq, Hkv, packed):
    """race_attend's fp32 path against soft_hash_probs + RaceCausalFn on explicit fp32 copies: the same
    kernels on the same values (bitwise), one rounding to the activations' dtype. `packed`: q, k, v are
    slices of one [B,T,3,H,D] tensor, whose gradient collects all three."""
    from race_attention_amd import RaceCausalFn, build_planes_protos, soft_hash_probs
    from race_attention_amd.nanochat import race_attend
    B, T, D, L, K = 2, 150, 64, 4, 4
    g = torch.Generator().manual_seed(3)
    planes, protos = build_planes_protos(D, K, L, 1, device=dev, seed=0)
    rows = [torch.randn(B, T, h, D, generator=g).to(dtype) for h in (Hq, Hkv, Hkv, Hq)]

    def composed(q, k, v):
        rep = q.shape[2] // k.shape[2]
        f = [t.transpose(1, 2).contiguous().float() for t in (q, k, v)]
        if rep > 1:
            f[1:] = [t.repeat_interleave(rep, 1) for t in f[1:]]
        pK, pQ, V2, _ = soft_hash_probs(*f, planes, protos, L, K, 1, True, scale=math.sqrt(D))
        return RaceCausalFn.apply(pK, pQ, V2, EPS).view(B, Hq, T, D).transpose(1, 2).to(q.dtype)

    res = []
    for fn in (lambda q, k, v: race_attend(q, k, v, planes, L, K, EPS, precision="fp32", protos_T=protos), composed):
        if packed:
            leaves = [torch.stack([t.to(dev) for t in rows[:3]], 2).requires_grad_(True)]
            x = leaves[0].unbind(2)
        else:
            leaves = x = [t.to(dev).requires_grad_(True) for t in rows[:3]]
        y = fn(*x)
        assert y.dtype == dtype and y.shape == (B, T, Hq, D)
        y.backward(rows[3].to(dev))
        res.append([y.detach()] + [t.grad for t in leaves])
    for i, (a, b) in enumerate(zip(*res)):
        if Hq == Hkv or i < 2:
            assert torch.equal(a, b), i
        else:
            # k, v of a group: the heads' fp32 gradients are summed before or behind the (linear)
            # soft-hash backward, then rounded once. dk = J (gp - <p, gp>) cancels: each of a table's 16
            # corner terms carries 2^-24 of |gp|, which is up to ~10 times |dk| at these sizes: 1e-5 of
            # the largest dk; two results so rounded differ by one more ulp of the activations' dtype
            ulp = torch.finfo(dtype).eps  # the spacing of a value's binade, of the value at most
            over = ((a.float() - b.float()).abs() - ulp * b.float().abs() - 1e-5 * b.float().abs().max()).max().item()
            assert over <= 0, (i, over)


@pytest.mark.parametrize("call", ["attend_bf16", "attend_fp32", "attend_fp32_f32_rows", "module_fp32"])
@pytest.mark.parametrize("H", [1, 2])
def test_outputs_change_in_place(dev, call, H):
    """The outputs are no views of a Function's internals: a caller may scale or gate them in place."""
    from race_attention_amd import RaceCausalCuda, build_planes_protos
    from race_attention_amd.nanochat import race_attend
    B, T, D, L, K = 1, 40, 64, 2, 3
    planes, protos = build_planes_protos(D, K, L, 1, device=dev, seed=0)
    mod = RaceCausalCuda(D, K, L, 1, device=dev, seed=0)
    dtype = torch.bfloat16 if call in ("attend_bf16", "attend_fp32") else torch.float32
    g = torch.Generator().manual_seed(1)
    rows = [torch.randn(B, T, H, D, generator=g).to(dtype).to(dev) for _ in range(3)]

    def grads(gate):
        x = [r.clone().requires_grad_(True) for r in rows]
        if call == "module_fp32":
            y = mod(*(t.transpose(1, 2) for t in x))
        else:
            y = race_attend(*x, planes, L, K, EPS, precision="bf16" if call == "attend_bf16" else "fp32", protos_T=protos)
        y = gate(y)
        return (y, *torch.autograd.grad(y, x, torch.ones_like(y)))

    for a, b in zip(grads(lambda y: y.mul_(2)), grads(lambda y: y * 2)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("B,T,H,D,L,K", [(2, 1, 1, 64, 2, 2), (2, 33, 3, 128, 3, 3), (1, 130, 2, 36, 1, 2), (1, 95, 2, 64, 8, 4),
                                         (3, 600, 2, 256, 2, 4), (1, 2100, 6, 32, 4, 4), (1, 40, 2, 20, 5, 3), (1, 90, 2, 256, 2, 2)])
@pytest.mark.parametrize("layout", ["contiguous", "packed", "odd_rows"])
def test_bf16_rows_equal_the_cast_rows(dev, B, T, H, D, L, K, layout):
    """The scan on bf16 rows in place against the same scan on fp32 copies, rounded once: equal to the bit,
    at the edges of stages and tiles, for slices of one [B,T,3,H,D] tensor and for rows that start at odd
    addresses (copied first)."""
    from race_attention_amd import RaceCausalFn, build_planes_protos
    from race_attention_amd.nanochat import race_attend
    from race_attention_amd.race_common import hash_code, hash_fwd
    print(f"bf16 rows B={B} T={T} H={H} D={D} L={L} K={K} {layout}", flush=True)
    g = torch.Generator().manual_seed(T + D)
    planes, protos = build_planes_protos(D, K, L, 1, device=dev, seed=0)
    wide = torch.randn(B, T, 3, H, D + 1, generator=g).to(torch.bfloat16).to(dev)
    if layout == "odd_rows":
        q, k, v = (wide[:, :, i, :, 1:].detach().requires_grad_(True) for i in range(3))
    else:
        x = wide[..., :D].contiguous()
        q, k, v = (t.detach().requires_grad_(True) for t in x.unbind(2)) if layout == "packed" else (
            t.contiguous().detach().requires_grad_(True) for t in x.unbind(2))
    go = torch.randn(B, T, H, D, generator=g).to(torch.bfloat16).to(dev)
    y = race_attend(q, k, v, planes, L, K, EPS, precision="fp32", protos_T=protos)
    dv, = torch.autograd.grad(y, v, go)
    probs = [hash_fwd(t.detach().transpose(1, 2), planes, L, K, 1, False, math.sqrt(D), hash_code(t, fp32_planes=True))[0]
             for t in (k, q)]
    vf = v.detach().transpose(1, 2).float().reshape(B * H, T, D).requires_grad_(True)
    out = RaceCausalFn.apply(*probs, vf, EPS)
    dvf, = torch.autograd.grad(out, vf, go.transpose(1, 2).float().reshape(B * H, T, D))
    assert torch.equal(y, out.detach().view(B, H, T, D).transpose(1, 2).to(torch.bfloat16))
    assert torch.equal(dv, dvf.view(B, H, T, D).transpose(1, 2).to(torch.bfloat16))


@pytest.mark.parametrize("precision", ["fp32", "bf16"])
@pytest.mark.parametrize("T", [1, 70])
def test_rows_at_odd_addresses(dev, precision, T):
    """Contiguous q, k, v and an upstream gradient that start 2 bytes off (a part of a flat buffer): taken, with
    the results of aligned copies."""
    from race_attention_amd import build_planes_protos
    from race_attention_amd.nanochat import race_attend
    B, H, D, L, K = 2, 3, 64, 2, 3
    planes, protos = build_planes_protos(D, K, L, 1, device=dev, seed=0)
    g = torch.Generator().manual_seed(T)
    rows = [torch.randn(B, T, H, D, generator=g).to(torch.bfloat16).to(dev) for _ in range(4)]

    def shifted(x):
        buf = torch.empty(x.numel() + 1, dtype=x.dtype, device=dev)
        y = buf[1:].view(x.shape)
        y.copy_(x)
        assert y.data_ptr() % 8 == 2 and y.is_contiguous()
        return y

    def grads(move):
        x = [move(r).requires_grad_(True) for r in rows[:3]]
        y = race_attend(*x, planes, L, K, EPS, precision=precision, protos_T=protos)
        return (y, *torch.autograd.grad(y, x, move(rows[3])))

    for a, b in zip(grads(shifted), grads(torch.clone)):
        assert torch.equal(a, b)
