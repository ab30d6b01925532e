"""The projections' kernels of 33 to 3201 rows: the k-grouped register-weight gate_up (33 to 128 rows) and the
block and split choices around it, at the edges of each one's rows."""

from __future__ import annotations

import pytest
import torch

from helpers import WIDE2, log

from test_gpu_seq_one import ULP2, _vm

pytestmark = pytest.mark.gpu

NARROW = dict(vocab_size=1000, hidden_size=640, intermediate_size=1152, num_hidden_layers=2, num_attention_heads=4,
              num_key_value_heads=2, head_dim=128)


@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("kw", [dict(WIDE2, vocab_size=1000), NARROW], ids=["1.5B", "640 x 1152"])
def test_mid_rows_match_the_lds_staged_kernels(monkeypatch, kw, dtype):
    """forward_hidden on the default choice against the LDS-staged kernels with no k split at every row count
    (FDLLM_WR_FFN=0, FDLLM_WR_SMALL=0, FDLLM_WR_OPS=0): the same sums in another order.  Compared row by row and
    16-column tile by tile, so that a wrong remainder is not averaged away."""
    vm = _vm(kw, dtype)
    ref = _vm(kw, dtype, monkeypatch, {"FDLLM_WR_FFN": "0", "FDLLM_WR_SMALL": "0", "FDLLM_WR_OPS": "0", "FDLLM_MM_TARGET_WGS": "1",
                                       "FDLLM_FUSE_OPROJ": "0", "FDLLM_FUSE_DOWN": "0"})
    g = torch.Generator(device="cuda")
    g.manual_seed(17)
    for rows in (33, 48, 63, 64, 65, 96, 97, 127, 128, 129, 224, 225, 320, 321, 400, 401, 417, 640, 641, 672, 673, 896, 897,
                 1024, 1025, 1280, 1281, 1344, 1345, 1537, 2049, 2560, 2561, 2688, 2689, 3201):
        x = vm.embed(torch.randint(0, 999, (rows,), dtype=torch.int32, device="cuda", generator=g))[None]
        log(f"case: forward_hidden {rows} rows, {kw['hidden_size']} x {kw['intermediate_size']}, {dtype}")
        a, b = vm.forward_hidden(x, None)[0].double(), ref.forward_hidden(x, None)[0].double()
        # two layers of rounded tensors: each rounding (about 10 per layer) may flip by an ulp, independently over a
        # row's or a tile's elements as over the matrix
        assert torch.isfinite(a).all()
        d, t = a - b, lambda x: x.view(rows, -1, 16).norm(dim=(0, 2))
        assert float((d.norm(dim=1) / b.norm(dim=1)).max()) < 4 * ULP2[dtype], rows
        assert float((t(d) / t(b)).max()) < 4 * ULP2[dtype], rows
