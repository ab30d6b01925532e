"""attn_prefill_kernel in its forms (query blocks alone or paired, four or twelve query tiles per workgroup)
against attention in float64 and against the kernel that takes an explicit bias."""

from __future__ import annotations

import pytest
import torch

from helpers import log

from test_gpu_seq_one import HEADS12, TINY, ULP2, _attention64, _vm

from fast_dllm_relax_amd.params import TORCH_DTYPES
from fast_dllm_relax_amd.runtime import build_prefix_block_attention_bias

pytestmark = pytest.mark.gpu

HEADS14 = dict(HEADS12, num_attention_heads=14, hidden_size=1792)  # 14 tiles: the last workgroup has two idle slots


@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("kw,form", [(HEADS12, 0), (HEADS12, 2), (HEADS12, 3), (TINY, 1), (HEADS14, 1)],
                         ids=["12 alone", "12 paired whole", "12 paired", "4", "14"])
def test_prefill_attention_unmasked(monkeypatch, kw, form, dtype):
    """Rows at the edges of query blocks (odd and even counts), keys at the edges of stages and key parts; a
    growing last key makes the softmax renew its reference in the last block."""
    vm = _vm(kw, dtype, monkeypatch, {"FDLLM_SEQ_ATTN": "0", "FDLLM_PREFILL_PAIR": str(form)})
    td, nq, nkv, L = TORCH_DTYPES[dtype], kw["num_attention_heads"], kw["num_key_value_heads"], kw["num_hidden_layers"]
    g = torch.Generator(device="cuda")
    g.manual_seed(11)
    for rows, prefix in [(128, 0), (129, 0), (160, 31), (255, 1), (300, 84), (1056, 33)]:
        cap = prefix + rows
        rnd = lambda *s: torch.randn(s, device="cuda", generator=g).to(td)  # noqa: E731
        q, k, v = rnd(1, rows, nq, 128), rnd(1, rows, nkv, 128), rnd(1, rows, nkv, 128)
        k[:, -1] *= 6
        kc, vc = rnd(L, 1, cap, nkv, 128), rnd(L, 1, cap, nkv, 128)
        log(f"case: {rows} rows at {prefix}, {nq} / {nkv} heads, form {form}, {dtype}")
        _, _, out = vm.attn_inplace(q, k, v, kc, vc, 0, prefix, 0, rows)
        want = _attention64(q[0], kc[0, 0], vc[0, 0])
        d = (out[0].double() - want).abs()
        assert float(d.norm() / want.norm()) < ULP2[dtype], (rows, prefix, float(d.norm() / want.norm()))
        assert float(d.max() / want.abs().max()) < 2 * ULP2[dtype], (rows, prefix)


@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("hpw", [0, 6], ids=["4 tiles", "12 tiles"])
def test_prefill_attention_peaked_rows(monkeypatch, hpw, dtype):
    """Each row's largest probability is exact: it is 2^0 against the running maximum, so its rounding to the model
    dtype for P.V costs nothing.  One key holds all the weight that reaches the output (the other keys' V rows are
    zero) with a score up to 2^12 past the zero scores before it: o = w v, and its only rounding is the output's.
    Half an ulp of the result, and 2 percent of that for the fp32 sums (about 40 roundings of 2^-24 against
    float16's half ulp of at least 2^-12)."""
    vm = _vm(HEADS12, dtype, monkeypatch, {"FDLLM_PREFILL_PAIR": "0", "FDLLM_PREFILL_HPW": str(hpw)})
    td, nq, nkv, L, rows = TORCH_DTYPES[dtype], 12, 2, HEADS12["num_hidden_layers"], 1024
    g = torch.Generator(device="cuda")
    g.manual_seed(14)
    c2 = 1.4426950408889634 / 128 ** 0.5
    for peak in (40, 100, 900, 1023):  # the peak in either key part of the first stage, and of later ones
        lag = torch.rand((1, rows, nq), device="cuda", generator=g) * 12
        q = torch.zeros((1, rows, nq, 128), dtype=td, device="cuda")
        q[..., 5] = (lag / c2 / 8).to(td)
        k, v = (torch.zeros((1, rows, nkv, 128), dtype=td, device="cuda") for _ in range(2))
        k[:, peak, :, 5] = 8
        v[:, peak] = (0.5 + torch.rand((nkv, 128), device="cuda", generator=g)).to(td)
        kc = torch.zeros((L, 1, rows, nkv, 128), dtype=td, device="cuda")
        log(f"case: peak at key {peak} of {rows}, {6 if hpw == 6 else 2} heads per workgroup, {dtype}")
        _, _, out = vm.attn_inplace(q, k, v, kc, torch.zeros_like(kc), 0, 0, 0, rows)
        lead = torch.exp2(q[0, :, :, 5].double() * 8 * c2)
        want = (lead / (lead + (rows - 1)))[..., None] * v[0, peak].double().repeat_interleave(nq // nkv, 0)
        half_ulp = torch.exp2(torch.floor(torch.log2(want)) - (8 if dtype == "bfloat16" else 11))
        worst = float(((out[0].double() - want).abs() / half_ulp).max())
        assert worst < 1.02, (peak, worst)


@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
def test_prefill_attention_block_causal(dtype):
    """The block-causal rule as a key bound against the same rule as an explicit bias (attn_kernel)."""
    vm = _vm(TINY, dtype)
    g = torch.Generator(device="cuda")
    g.manual_seed(12)
    for rows in (128, 129, 192, 353, 1025):
        x = vm.embed(torch.randint(0, 999, (rows,), dtype=torch.int32, device="cuda", generator=g))[None]
        blk = (rows - 1) // 32 * 32
        bias = torch.from_numpy(build_prefix_block_attention_bias(blk, rows - blk, block_size=32)).cuda()
        log(f"case: block-causal {rows} rows, {dtype}")
        a, b = vm.forward_hidden(x, None)[0].double(), vm.forward_hidden(x, bias)[0].double()
        # two layers of rounded tensors: each rounding (about 10 per layer) may flip by an ulp, in any row
        assert float(((a - b).norm(dim=1) / b.norm(dim=1)).max()) < 4 * ULP2[dtype], rows


@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
def test_prefill_stops_at_the_last_layers_cache_rows(dtype):
    """build_prefix_cache leaves out what follows the last layer's K/V rows: the caches of a two-layer model
    are the first two layers' of a three-layer one, bit for bit, on every attention kernel's row counts, with
    and without a bias."""
    from fast_dllm_relax_amd.config import FastDLLMConfig
    from fast_dllm_relax_amd.params import random_params_torch
    from fast_dllm_relax_amd.vm import HipVM

    c3, c2 = FastDLLMConfig(**dict(TINY, num_hidden_layers=3)), FastDLLMConfig(**TINY)
    params = random_params_torch(c3, 5, dtype=dtype)
    vm3, vm2 = HipVM(c3, params, dtype=dtype), HipVM(c2, params[:1 + 14] + params[1 + 21:], dtype=dtype)
    g = torch.Generator(device="cuda")
    g.manual_seed(13)
    for rows in (1, 20, 32, 33, 100, 128, 300):
        x = vm3.embed(torch.randint(0, 999, (rows,), dtype=torch.int32, device="cuda", generator=g))[None]
        full = torch.zeros((1, 1, rows, rows), device="cuda")
        for bias in (None, full):
            log(f"case: build_prefix_cache {rows} rows, bias {bias is not None}, {dtype}")
            caches = []
            for vm, L in ((vm3, 3), (vm2, 2)):
                k = torch.zeros((L, 1, rows + 3, 2, 128), dtype=TORCH_DTYPES[dtype], device="cuda")
                caches.append(vm.build_prefix_cache(x, bias, k, torch.zeros_like(k)))
            for a, b in zip(*caches):
                assert torch.equal(a[:2].view(torch.int16), b.view(torch.int16)), (rows, bias is None)
