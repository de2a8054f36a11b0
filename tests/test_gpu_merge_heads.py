"""Merge of the key ranges of token-major query blocks where a workgroup takes eight, sixteen or thirty-two heads of a token, with a
last group of heads that is short, so that the waves of a workgroup merge different numbers of heads; against the oracle."""
import pytest
import torch

import fa_oracle as O
from helpers import check_out
from test_gpu_prefill import paged_ragged

pytestmark = pytest.mark.gpu


def heads_per_workgroup(nheads, tokens, num_cus):
    # as many as leave eight workgroups per compute unit
    heads = 4
    while heads < nheads and tokens * -(-nheads // (2 * heads)) >= 8 * num_cus:
        heads *= 2
    return heads


@pytest.mark.parametrize("hq,hk,tokens,heads", [(12, 4, 1023, 4), (12, 2, 1024, 8), (12, 4, 2048, 16), (28, 4, 512, 8), (28, 2, 1024, 16), (40, 8, 410, 8),
                                                (40, 4, 683, 16), (40, 8, 1025, 32)])
@pytest.mark.parametrize("d", [64, 128, 80])
def test_heads_per_workgroup(hq, hk, d, tokens, heads):
    from flash_attn_npu.flash_attn_npu import varlen_fwd
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert heads_per_workgroup(hq, tokens, 256) == heads
    # three ranges, two, none that is asked for (no queries), one, no keys at all
    lens_q, lens_k = [tokens - 330, 300, 0, 29, 1], [700, 400, 513, 256, 0]
    print("merge heads", hq, hk, d, tokens, flush=True)
    case, q, cu_q, cu_k, kl, vl = paged_ragged(lens_q, lens_k, hq, hk, d, 64, seed=hq + d)
    out, lse, _, _ = varlen_fwd(q.cuda(), case["k_cache"].cuda(), case["v_cache"].cuda(), None, cu_q.cuda(), None,
                                case["cache_seqlens"].cuda(), None, case["block_table"].cuda(), None, max(lens_q), max(lens_k),
                                0.0, d ** -0.5, False, False, -1, -1, 0.0, False, None, num_splits=3)
    torch.cuda.synchronize()
    ref, ref_lse = O.flash_attn_varlen(q, kl, vl, cu_q, cu_k, max(lens_q), max(lens_k), causal=False, mode="fp32")
    check_out(out, ref, lse, ref_lse, f"{hq} heads, {tokens} tokens, d={d}")
