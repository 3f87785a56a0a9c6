"""Where the kernels read and write, without a GPU: the library is replaced by one that records the
addresses it was given, and the index arithmetic of the headers is compiled for the host."""
import os
import subprocess

import pytest
import torch

from race_attention_amd import _lib, attention, nanochat, noncausal, race_common


def layouts(B, H, T, D):
    """[B,H,T,D] inputs whose last dim is contiguous, by name."""
    x = torch.randn(B, H, T, D)
    return {
        "bhtd": x,
        "bthd": torch.randn(B, T, H, D).transpose(1, 2),
        "windows_step_1": torch.randn(B, H, T + D - 1).unfold(2, D, 1),  # two dims of stride 1
        "windows_step_8": torch.randn(B, H, 8 * T + D).unfold(2, D, 8)[:, :, :T],
        "one_head_for_all": x[:, :1].expand(B, H, T, D),
        "one_token_for_all": x[:, :, :1].expand(B, H, T, D),
        "fused_qkv": torch.randn(B, T, 3, H, D)[:, :, 1].transpose(1, 2),
        "every_other_row": torch.randn(B, H, 2 * T, D)[:, :, ::2],
    }


class Recorder:
    """Stands in for the library: every call succeeds and its arguments are kept."""

    def __init__(self):
        self.calls = {}

    def __getattr__(self, name):
        def call(*args):
            self.calls[name] = args
            return 16 if name.endswith("_partials") else 0
        return call


@pytest.fixture
def recorder(monkeypatch):
    r = Recorder()
    monkeypatch.setattr(_lib, "lib", lambda: r)
    monkeypatch.setattr(_lib, "stream_of", lambda t: 0)
    monkeypatch.setattr(_lib, "require_device", lambda *t: None)
    return r


def same_rows(view, t):
    assert view.data == t.data_ptr(), "the kernel writes somewhere else than into the result"
    assert (view.stride_b, view.stride_h, view.stride_t, 1) == t.stride()


@pytest.mark.parametrize("B,H,T,D", [(2, 3, 7, 64), (1, 2, 50, 64), (1, 1, 100, 16), (2, 2, 1, 8), (1, 2, 5, 1)])
@pytest.mark.parametrize("layout", sorted(layouts(1, 1, 1, 8)))
def test_soft_hash_gradients_are_written_into_the_result(recorder, B, H, T, D, layout):
    X = layouts(B, H, T, D)[layout]
    L, K = 2, 2
    planes, g = torch.randn(D, L * K), torch.randn(B * H, T, L << K)
    dX = race_common.hash_bwd(X, planes, g, L, K, 1, False, 8.0, _lib.RACE_F32)
    assert dX.shape == X.shape and dX.dtype == X.dtype
    same_rows(recorder.calls["race_soft_hash_bwd"][5], dX)
    X.requires_grad_()
    probs = noncausal.SoftHashTempFn.apply(X, planes, L, K, 1, False, torch.tensor(8.0))
    dX, = torch.autograd.grad(probs, X, g)
    same_rows(recorder.calls["race_soft_hash_bwd_dscale"][6], dX)


def test_a_result_whose_rows_are_scattered_is_refused():
    with pytest.raises(_lib.RaceError, match="rows"):
        _lib.out_view4(torch.empty(1, 2, 64, 7).transpose(2, 3))
    with pytest.raises(_lib.RaceError, match="rows"):
        _lib.out_view4(torch.empty(2, 64, 7))


def odd_rows(B, T, H, D):
    """[B,T,H,D] bf16 rows that the kernels cannot read in place, by name."""
    n = B * T * H * D
    flat = torch.arange(4 * n + 64, dtype=torch.float32).to(torch.bfloat16)
    return {
        "contiguous_at_an_odd_address": flat[1:1 + n].view(B, T, H, D),
        "one_token_with_an_odd_stride": flat.as_strided((B, 1, H, D), (2 * H * D + 8, 3 * H * D + 1, D, 1)),
        "one_token_with_no_stride": flat.as_strided((B, 1, H, D), (H * D, 0, D, 1)),
        "channels_apart": flat[:2 * n].view(B, T, H, 2 * D)[..., ::2],
        "slice_of_wider_rows": flat[:B * T * H * (D + 1)].view(B, T, H, D + 1)[..., 1:],
    }


@pytest.mark.parametrize("B,T,H,D", [(2, 3, 2, 64), (1, 1, 1, 64), (1, 5, 3, 128)])
@pytest.mark.parametrize("layout", sorted(odd_rows(1, 1, 1, 8)))
def test_rows_are_copied_to_where_the_kernels_can_read_them(B, T, H, D, layout):
    x = odd_rows(B, T, H, D)[layout]
    y = nanochat._bf16_rows(x)  # (race_op_fwd_bf16_rows: 8-byte runs, tokens D .. 2^22 elements apart)
    assert torch.equal(y, x.transpose(1, 2)) and y.stride(3) == 1 and y.data_ptr() % 8 == 0
    assert not any(s % 4 for s in y.stride()[:3]) and D <= y.stride(2) <= 1 << 22
    y = attention._bf16_rows(x.transpose(1, 2))  # (race_qkv_fwd: 16-byte runs)
    assert torch.equal(y, x.transpose(1, 2)) and y.stride(3) == 1 and y.data_ptr() % 16 == 0
    assert not any(s % 8 for s in y.stride()[:3])


ROWS = r"""
#include "race_params.h"
#include <cstdio>
int main()
{
    const int stages[] = {16, 32, 64};
    for (int ts : stages)
        for (int T = 1; T <= 3 * 64 + 1; ++T)
            for (int CB = 16; CB <= T + 16; CB += 16)
                for (int t_begin = 0; t_begin < T; t_begin += CB) {
                    const int t_end = t_begin + CB < T ? t_begin + CB : T;
                    for (int t0 = t_begin; t0 < t_end + ts; t0 += ts)  // the stages and one look-ahead
                        for (int r = 0; r < ts; ++r) {
                            const int row = race::op_clamped_row(t0, r, t_end);
                            if (row < t_begin || row >= t_end || (t0 + r < t_end && row != t0 + r)) {
                                std::printf("T=%d CB=%d stage=%d: row %d of [%d,%d) read for %d\n", T, CB, ts, row,
                                            t_begin, t_end, t0 + r);
                                return 1;
                            }
                        }
                }
    return 0;
}
"""


def test_rows_loaded_ahead_stay_inside_the_block(tmp_path):
    """Every row that the element-wise loads of the fp32 scan address, the look-ahead past a block's last
    stage among them, is a row of that block."""
    src, exe = tmp_path / "rows.cpp", tmp_path / "rows"
    src.write_text(ROWS)
    csrc = os.path.join(os.path.dirname(_lib.__file__), "csrc")
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", csrc, str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
