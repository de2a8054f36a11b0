"""Tiled forward under softmax scales that are not positive: the scale rides in the exponent where it is positive and is applied to
the scores in front of the masks where it is not, in tiles with and without masked elements, against the oracle."""
import pytest
import torch

import fa_oracle as O
from helpers import check_out

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scale", [0.11, -0.09, 0.0])
@pytest.mark.parametrize("opts", [{"causal": True}, {"causal": False}, {"causal": False, "window_size": (70, 9)}])
@pytest.mark.parametrize("d", [64, 128, 256])
def test_scale(d, opts, scale):
    from flash_attn_npu import flash_attn_varlen_func
    lens = [300, 65, 1, 128]
    cu = torch.tensor([sum(lens[:i]) for i in range(len(lens) + 1)], dtype=torch.int32)
    g = torch.Generator().manual_seed(d)
    q = torch.randn(sum(lens), 4, d, generator=g).to(torch.bfloat16)
    k, v = (torch.randn(sum(lens), 2, d, generator=g).to(torch.bfloat16) for _ in range(2))
    out, lse, _ = flash_attn_varlen_func(q.cuda(), k.cuda(), v.cuda(), cu.cuda(), cu.cuda(), 300, 300, softmax_scale=scale,
                                         return_attn_probs=True, **opts)
    torch.cuda.synchronize()
    ref, ref_lse = O.flash_attn_varlen(q, k, v, cu, cu, 300, 300, softmax_scale=scale, mode="fp32", **opts)
    check_out(out, ref, lse, ref_lse, f"d={d} scale={scale}")
