"""The fp32 layer as one graph node against its parts (soft_hash_probs and RaceCausalFn), which run
the same kernels on the same values: equal to the bit, over layouts, input dtypes and which inputs
require a gradient."""
import pytest
import torch

from race_attention_amd.race_causal_cuda import RaceCausalCuda, RaceCausalFn
from race_attention_amd.race_common import soft_hash_probs

pytestmark = pytest.mark.gpu


def parts(m, Q, K, V):
    pK, pQ, V2, _ = soft_hash_probs(Q, K, V, m.planes_T, m.protos_T, m.L, m.Kbits, 1, True)
    return RaceCausalFn.apply(pK, pQ, V2, m.eps).view_as(Q)


@pytest.mark.parametrize("dtype,v_dtype", [(torch.float32, torch.float32), (torch.float32, torch.float16),
                                           (torch.bfloat16, torch.bfloat16)])
@pytest.mark.parametrize("B,H,T,D,L,K", [(1, 1, 1, 64, 2, 2), (2, 3, 65, 48, 3, 2), (1, 2, 300, 64, 2, 7)])
@pytest.mark.parametrize("layout", ["bhtd", "bthd", "channel_step"])
@pytest.mark.parametrize("needs", [(True, True, True), (True, False, True), (False, True, False)])
def test_layer_node_equals_its_parts(dtype, v_dtype, B, H, T, D, L, K, layout, needs):
    if dtype == torch.bfloat16 and K <= 4 and D in (64, 128):
        pytest.skip("the fused bf16 path")
    m = RaceCausalCuda(D, K, L, 1, device="cuda", seed=3)
    gen = torch.Generator("cuda").manual_seed(T)
    shape = {"bhtd": (B, H, T, D), "bthd": (B, T, H, D), "channel_step": (B, H, T, 2 * D)}[layout]

    def leaf(need, dtype):
        x = torch.randn(shape, device="cuda", generator=gen).to(dtype).requires_grad_(need)
        return x, x.transpose(1, 2) if layout == "bthd" else x[..., ::2] if layout == "channel_step" else x

    leaves, views = zip(*(leaf(n, t) for n, t in zip(needs, (dtype, dtype, v_dtype))))
    go = torch.randn(B, T, H, D, device="cuda", generator=gen).transpose(1, 2)
    ref, got = parts(m, *views), m(*views)
    assert got.dtype == torch.float32 and torch.equal(got, ref)
    wanted = [x for x in leaves if x.requires_grad]
    for x, a, b in zip(wanted, torch.autograd.grad(got, wanted, go), torch.autograd.grad(ref, wanted, go)):
        assert a.dtype == x.dtype and torch.equal(a, b)


@pytest.mark.parametrize("T,D", [(50, 64), (7, 64), (130, 128)])
@pytest.mark.parametrize("call", ["module", "seam", "temperature"])
def test_overlapping_windows_have_the_gradients_of_their_copies(T, D, call):
    """Inputs whose tokens are windows one element apart (token and channel stride 1, which orders
    torch.empty_like's dims differently): outputs and gradients equal those of contiguous copies."""
    from race_attention_amd.nanochat import race_attend
    from race_attention_amd.noncausal import SoftHashTempFn
    L, K, B, H = 3, 2, 2, 2
    m = RaceCausalCuda(D, K, L, 1, device="cuda", seed=3)
    gen = torch.Generator("cuda").manual_seed(T)
    xs = [torch.randn(B, H, T + D - 1, device="cuda", generator=gen).unfold(2, D, 1) for _ in range(3)]
    go = torch.randn(B, H, T, D, device="cuda", generator=gen)

    def grads(copy):
        x = [(t.contiguous() if copy else t).detach().requires_grad_() for t in xs]
        if call == "module":
            y = m(*x)
        elif call == "seam":
            y = race_attend(*(t.transpose(1, 2) for t in x), m.planes_T, L, K, 1e-6, precision="fp32",
                            protos_T=m.protos_T).transpose(1, 2)
        else:
            y = SoftHashTempFn.apply(x[0], m.planes_T, L, K, 1, False, torch.tensor(4.0, device="cuda"))
            return (y, *torch.autograd.grad(y, x[:1], torch.ones_like(y).cumsum(-1)))
        return (y, *torch.autograd.grad(y, x, go))

    for a, b in zip(grads(False), grads(True)):
        assert torch.equal(a, b)
