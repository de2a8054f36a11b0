"""Tiled forward where the keys that a wave sees end in either half of a 64-key tile, in front of it, or begin behind it: packed
tiles (causal, windows), key ranges over a paged cache, head dimensions below the compiled width, against the oracle."""
import pytest
import torch

import fa_oracle as O
from helpers import check_out, make_paged_case, to_dev

pytestmark = pytest.mark.gpu


def ends(lens):
    return torch.tensor([sum(lens[:i]) for i in range(len(lens) + 1)], dtype=torch.int32)


@pytest.mark.parametrize("d,group", [(128, 4), (64, 7), (256, 2), (80, 4)])
@pytest.mark.parametrize("opts", [{"causal": True}, {"causal": False}, {"causal": True, "window_size": (33, 0)}, {"causal": False, "window_size": (20, 11)}])
def test_packed_blocks(d, group, opts):
    from flash_attn_npu import flash_attn_varlen_func
    lens_k = [1, 31, 32, 33, 63, 64, 65, 95, 96, 97, 128, 200]
    lens_q = [1, 8, 32, 5, 9, 33, 2, 20, 7, 31, 16, 12]
    g = torch.Generator().manual_seed(d)
    q = torch.randn(sum(lens_q), 2 * group, d, generator=g).to(torch.bfloat16)
    k, v = (torch.randn(sum(lens_k), 2, d, generator=g).to(torch.bfloat16) for _ in range(2))
    cu_q, cu_k = ends(lens_q), ends(lens_k)
    out, lse, _ = flash_attn_varlen_func(q.cuda(), k.cuda(), v.cuda(), cu_q.cuda(), cu_k.cuda(), max(lens_q), max(lens_k), return_attn_probs=True, **opts)
    torch.cuda.synchronize()
    ref, ref_lse = O.flash_attn_varlen(q, k, v, cu_q, cu_k, max(lens_q), max(lens_k), mode="fp32", **opts)
    check_out(out, ref, lse, ref_lse, f"d={d} group={group} {opts}")


@pytest.mark.parametrize("page", [32, 64, 256])
@pytest.mark.parametrize("lens", [[2017, 2048, 2049, 1], [2079, 2080, 2081, 33]])
def test_key_ranges(lens, page):
    from flash_attn_npu import flash_attn_with_kvcache
    case = make_paged_case(4, 8, 2, 128, page, lens, seqlen_q=18, seed=page)
    dev = to_dev(case, "cuda:0")
    out, lse = flash_attn_with_kvcache(dev["q"], dev["k_cache"], dev["v_cache"], cache_seqlens=dev["cache_seqlens"], block_table=dev["block_table"],
                                       causal=True, return_softmax_lse=True)
    torch.cuda.synchronize()
    ref, ref_lse = O.flash_attn_with_kvcache(case["q"], case["k_cache"], case["v_cache"], cache_seqlens=case["cache_seqlens"],
                                             block_table=case["block_table"], causal=True, mode="fp32")
    check_out(out, ref, lse, ref_lse, f"page={page}")
