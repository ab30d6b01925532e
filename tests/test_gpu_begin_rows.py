"""The start of a call (residual stream, RoPE table and first norm in one launch) at the edges of its rows and
of the layouts its first projection takes: one layer of the first step's cache rows against float64."""

from __future__ import annotations

import math

import pytest
import torch

from helpers import log

from test_gpu_seq_one import HEADS12, TINY, ULP2, _vm

pytestmark = pytest.mark.gpu

WIDE = dict(HEADS12, hidden_size=2048, num_attention_heads=16)


@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("kw", [HEADS12, TINY, WIDE], ids=["1536", "256", "2048"])
def test_first_layers_cache_rows(kw, dtype):
    vm = _vm(kw, dtype)
    H, nq = kw["hidden_size"], kw["num_attention_heads"]
    _, wqkv, bias, _, _, _, ln_in, _ = vm.params[:8]
    g = torch.Generator(device="cuda")
    g.manual_seed(29)
    ln_in.copy_(1 + 0.1 * torch.randn(H, device="cuda", generator=g))  # read at each call
    for rows, pos in [(1, 0), (31, 7), (32, 4000), (33, 0), (64, 8191), (257, 5), (1100, 3)]:
        ids = torch.randint(0, 999, (rows,), dtype=torch.int32, device="cuda", generator=g)
        x = vm.embed(ids)[None]
        k = torch.zeros((2, 1, pos + rows, 2, 128), dtype=x.dtype, device="cuda")
        v = torch.zeros_like(k)
        log(f"case: {rows} rows at {pos}, hidden {H}, {dtype}")
        vm.forward_cached(x, k, v, torch.tensor(pos, dtype=torch.int32, device="cuda"), pos)
        x64 = x[0].double()
        y = x64 / torch.sqrt((x64 * x64).mean(-1, keepdim=True) + vm.cfg.rms_norm_eps) * ln_in.double()
        y = (y @ wqkv.double().t().contiguous() + bias.double())[:, nq * 128:].view(rows, 4, 128)
        inv = torch.exp(-math.log(vm.cfg.rope_theta) * torch.arange(64, dtype=torch.float64, device="cuda") / 64)
        ang = (pos + torch.arange(rows, device="cuda")).double()[:, None] * inv
        c, s = torch.cos(ang)[:, None], torch.sin(ang)[:, None]
        a, b = y[:, :2, :64], y[:, :2, 64:]
        want_k, want_v = torch.cat([a * c - b * s, b * c + a * s], -1), y[:, 2:]
        # the normalised row is rounded twice, the projection once, the rotation three times: the errors add as
        # their squares, half an ulp each at most (fp32 angles add 8191 x 2^-24 of a turn)
        for got, want in ((k, want_k), (v, want_v)):
            d = got[0, 0, pos:].double() - want
            assert float(d.norm() / want.norm()) < 2 * ULP2[dtype] + 1e-3 * (pos > 1000), (rows, pos)
