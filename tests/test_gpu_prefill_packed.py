"""Causal packed prompts whose tiles hold the queries of a whole group of heads: lengths around a tile's share of queries
(128 / group), around the 64-key tiles and the tiles that stand side by side, equal and unequal, against the oracle.  Few tokens
are packed or not by the heads that a tile saves; many (`fill`) are packed at every group."""
import pytest
import torch

import fa_oracle as O
from helpers import check_out

pytestmark = pytest.mark.gpu


def ends(lens):
    return torch.tensor([sum(lens[:i]) for i in range(len(lens) + 1)], dtype=torch.int32)


@pytest.mark.parametrize("d,group,hk,dtype,opts", [
    (128, 4, 2, torch.bfloat16, {}),
    (128, 7, 3, torch.float16, {}),
    (64, 2, 10, torch.bfloat16, {"softcap": 15.0}),
    (80, 3, 7, torch.float16, {}),
    (256, 8, 3, torch.bfloat16, {}),
    (128, 16, 2, torch.bfloat16, {"window_size": (40, 0)}),
    (64, 100, 1, torch.float16, {}),
])
@pytest.mark.parametrize("lens_q,lens_k", [
    ([1, 17, 18, 19, 31, 32, 33, 63, 64, 65, 127, 128, 129, 300], None),
    ([257, 3, 258, 2, 256, 1, 255, 4], None),                               # every other sequence is short
    ([160, 160, 160], None),                                                # equal lengths
    ([1, 700, 18, 511, 129, 513, 33, 640] * 3, None),                       # long and short
    ([5, 70, 130, 1], [200, 70, 61, 1]),                                    # more and fewer keys than queries
])
@pytest.mark.parametrize("fill", [False, True])
def test_packed_causal(lens_q, lens_k, d, group, hk, dtype, opts, fill):
    from flash_attn_npu import flash_attn_varlen_func
    lens_k = lens_k or lens_q
    if fill:
        # two rounds of the device in 128-row tiles (two workgroups per compute unit up to D = 128, one at 256): from there on a
        # causal launch packs its heads whatever their tiles save
        rows = 2 * torch.cuda.get_device_properties(0).multi_processor_count * (2 if d <= 128 else 1) * 128
        times = -(-rows // (sum(lens_q) * group * hk))
        lens_q, lens_k = lens_q * times, lens_k * times
        assert sum(lens_q) * group * hk >= rows
    g = torch.Generator().manual_seed(d + group + len(lens_q))
    q = torch.randn(sum(lens_q), group * hk, d, generator=g).to(dtype)
    k, v = (torch.randn(sum(lens_k), hk, d, generator=g).to(dtype) for _ in range(2))
    cu_q, cu_k = ends(lens_q), ends(lens_k)
    out, lse, _ = flash_attn_varlen_func(q.cuda(), k.cuda(), v.cuda(), cu_q.cuda(), cu_k.cuda(), max(lens_q), max(lens_k), causal=True,
                                         return_attn_probs=True, **opts)
    torch.cuda.synchronize()
    ref, ref_lse = O.flash_attn_varlen(q, k, v, cu_q, cu_k, max(lens_q), max(lens_k), causal=True, mode="fp32", **opts)
    check_out(out, ref, lse, ref_lse, f"packed d={d} group={group}")
