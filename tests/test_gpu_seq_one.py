"""One sequence's unmasked attention on attn_seq_kernel (key splits and their merge): calls of 33 to 1023
rows, and shorter ones over more than 5120 keys, against attention in float64 and against the kernels
that take these calls when it is turned off (FDLLM_SEQ_ATTN=0)."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from helpers import TINY, log

from fast_dllm_relax_amd.config import FastDLLMConfig
from fast_dllm_relax_amd.params import TORCH_DTYPES, random_params_torch
from fast_dllm_relax_amd.vm import HipVM

pytestmark = pytest.mark.gpu

HEADS12 = dict(vocab_size=1000, hidden_size=1536, intermediate_size=512, num_hidden_layers=2,
               num_attention_heads=12, num_key_value_heads=2, head_dim=128)
# half an ulp of the output and half an ulp of each probability (the P.V product's operands), relative to
# the output's size: 2 x 2^-9 in bfloat16, 2 x 2^-12 in float16
ULP2 = {"bfloat16": 2.0 ** -8, "float16": 2.0 ** -11}


def _vm(kw, dtype, monkeypatch=None, env=None):
    cfg = FastDLLMConfig(**kw)
    if env:
        for k, v in env.items():
            monkeypatch.setenv(k, v)
    vm = HipVM(cfg, random_params_torch(cfg, 5, dtype=dtype), dtype=dtype)
    if env:
        for k in env:
            monkeypatch.delenv(k)
    return vm


def _attention64(q, k, v):
    rows, nq, hd = q.shape
    grp = nq // k.shape[1]
    out = torch.empty((rows, nq, hd), dtype=torch.float64, device=q.device)
    for h in range(nq):
        s = q[:, h].double() @ k[:, h // grp].double().t().contiguous() / hd ** 0.5
        out[:, h] = torch.softmax(s, -1) @ v[:, h // grp].double().contiguous()
    return out


# rows at the edges of query tiles, tile groups and of the range; keys at the edges of 64-key blocks and key
# parts, of the unsplit calls and of the most splits
@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("kw", [HEADS12, TINY], ids=["12/2", "4/2"])
def test_seq_one_attention(kw, dtype):
    vm = _vm(kw, dtype)
    td, nq, nkv = TORCH_DTYPES[dtype], kw["num_attention_heads"], kw["num_key_value_heads"]
    g = torch.Generator(device="cuda")
    g.manual_seed(7)
    for rows, prefix in [(33, 0), (33, 31), (40, 24), (64, 0), (64, 1), (65, 300), (83, 8192), (127, 129), (128, 0),
                         (200, 513), (301, 84), (1023, 1), (1, 5200), (8, 6001), (32, 5121), (32, 9000)]:
        L, cap = kw["num_hidden_layers"], prefix + rows + 3
        rnd = lambda *s: torch.randn(s, device="cuda", generator=g).to(td)  # noqa: E731
        q, k, v = rnd(1, rows, nq, 128), rnd(1, rows, nkv, 128), rnd(1, rows, nkv, 128)
        kc, vc = rnd(L, 1, cap, nkv, 128), rnd(L, 1, cap, nkv, 128)
        kc[:, :, prefix + rows:] = float("nan")  # rows past the attended ones are not read into any result
        vc[:, :, prefix + rows:] = float("nan")
        log(f"case: {rows} rows at {prefix}, {nq} / {nkv} heads, {dtype}")
        _, _, out = vm.attn_inplace(q, k, v, kc, vc, 1, prefix, 0, rows)
        want = _attention64(q[0], kc[1, 0, :prefix + rows], vc[1, 0, :prefix + rows])
        d = (out[0].double() - want).abs()
        # sums of many rounded probabilities: the errors add as their squares, so twice the bound of one
        assert float(d.norm() / want.norm()) < ULP2[dtype], (rows, prefix, float(d.norm() / want.norm()))
        assert float(d.max() / want.abs().max()) < 2 * ULP2[dtype], (rows, prefix)


@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
def test_seq_one_steps_match_the_other_kernels(monkeypatch, dtype):
    """Cached steps whose attention moved to attn_seq_kernel: the rows written to the caches are the same
    bits in the first layer, and everything else agrees to the rounding of the attention output."""
    vm, ref = _vm(HEADS12, dtype), _vm(HEADS12, dtype, monkeypatch, {"FDLLM_SEQ_ATTN": "0"})
    g = torch.Generator(device="cuda")
    g.manual_seed(9)
    td = TORCH_DTYPES[dtype]
    for rows, prefix, rp in [(32, 5200, None), (8, 8160, 16), (32, 8175, None), (33, 7, None), (83, 640, None),
                             (130, 1000, None), (600, 33, None)]:
        cap = prefix + max(rows, 32)
        kc = torch.randn((2, 1, cap, 2, 128), device="cuda", generator=g).to(td)
        vc = torch.randn((2, 1, cap, 2, 128), device="cuda", generator=g).to(td)
        x = vm.embed(torch.randint(0, 999, (rows,), dtype=torch.int32, device="cuda", generator=g))[None]
        off = torch.tensor(prefix + (rp or 0), dtype=torch.int32, device="cuda")
        log(f"case: step of {rows} rows at {prefix} (rp {rp}), {dtype}")
        res = []
        for m in (vm, ref):
            k, v = kc.clone(), vc.clone()
            h = (m.forward_cached(x, k, v, off, prefix) if rp is None
                 else m._partial(rp, x, k, v, off, prefix))
            res.append((h.float(), k.float(), v.float()))
        (h1, k1, v1), (h2, k2, v2) = res
        for a, b in ((k1, k2), (v1, v2)):
            np.testing.assert_array_equal(a[0].cpu().numpy(), b[0].cpu().numpy())
        # two layers of rounded tensors: each rounding (about 10 per layer) may flip by an ulp
        assert float((h1 - h2).norm() / h2.norm()) < 4 * ULP2[dtype], (rows, prefix)
        assert float((k1 - k2).norm() / k2.norm()) < 4 * ULP2[dtype], (rows, prefix)


def test_noalloc_past_the_chunk_kernels_keys():
    """The allocation-free step over more keys than the chunk kernel takes: forward_cached's bits."""
    from fast_dllm_relax_amd import _lib

    vm = _vm(HEADS12, "bfloat16")
    prefix, rows = 8500, 32
    g = torch.Generator(device="cuda")
    g.manual_seed(3)
    kc = torch.randn((2, 1, prefix + rows, 2, 128), device="cuda", generator=g).bfloat16()
    vc = torch.randn((2, 1, prefix + rows, 2, 128), device="cuda", generator=g).bfloat16()
    x = vm.embed(torch.randint(0, 999, (rows,), dtype=torch.int32, device="cuda", generator=g))[None]
    off = torch.tensor(prefix, dtype=torch.int32, device="cuda")
    k, v = kc.clone(), vc.clone()
    want = vm.forward_cached(x, k, v, off, prefix)
    out = torch.empty_like(want)
    log("case: noalloc 32 rows at 8500")
    _lib.check(vm.lib.fdllm_forward_cached_noalloc(vm.ctx, x.data_ptr(), rows, kc.data_ptr(), vc.data_ptr(), prefix + rows,
                                                   off.data_ptr(), prefix, out.data_ptr(),
                                                   torch.cuda.current_stream().cuda_stream))
    for a, b in ((out, want), (kc, k), (vc, v)):
        np.testing.assert_array_equal(a.float().cpu().numpy(), b.float().cpu().numpy())


@pytest.mark.parametrize("prefix", [0, 57, 2048])
def test_callback_rows_written_by_the_chunk_kernel(prefix):
    """fdllm_attn_inplace on the chunk kernel, which takes the K/V rows from the caller's tensors and writes them
    to the cache: the bytes of the rows (NaN payloads and signed zeros included), nothing beside them, and the
    output of the same call on rows that are not 16-byte aligned (copied first)."""
    vm = _vm(HEADS12, "bfloat16")
    g = torch.Generator(device="cuda")
    g.manual_seed(23)
    for rows in (1, 8, 17, 32):
        cap = prefix + rows + 5
        rnd = lambda *s: torch.randn(s, device="cuda", generator=g).bfloat16()  # noqa: E731
        q, k, v = rnd(1, rows, 12, 128), rnd(1, rows, 2, 128), rnd(1, rows, 2, 128)
        kc, vc = rnd(2, 1, cap, 2, 128), rnd(2, 1, cap, 2, 128)
        log(f"case: callback of {rows} rows at {prefix}")
        res = []
        for shift in (0, 1):
            kk, vv = kc.clone(), vc.clone()
            ks = torch.empty(k.numel() + 8, dtype=k.dtype, device="cuda")[shift:shift + k.numel()].view(k.shape).copy_(k)
            vs = torch.empty(v.numel() + 8, dtype=v.dtype, device="cuda")[shift:shift + v.numel()].view(v.shape).copy_(v)
            out = vm.attn_inplace(q, ks, vs, kk, vv, 1, prefix, 0, rows)[2]
            for got, rows_in, before in ((kk, k, kc), (vv, v, vc)):
                want = before.clone()
                want[1, 0, prefix:prefix + rows] = rows_in[0]
                assert torch.equal(got.view(torch.int16), want.view(torch.int16)), (rows, shift)
            res.append(out)
        assert torch.equal(res[0].view(torch.int16), res[1].view(torch.int16)), rows
        special = k.view(torch.int16).clone()
        special[0, 0, 0, :4] = torch.tensor([0x7FC1, -0x8000, -0x0041, 0x7F80], dtype=torch.int16)
        kk, vv = kc.clone(), vc.clone()
        vm.attn_inplace(q, special.view(torch.bfloat16), v, kk, vv, 0, prefix, 0, rows)
        assert torch.equal(kk[0, 0, prefix:prefix + rows].view(torch.int16), special[0]), rows
