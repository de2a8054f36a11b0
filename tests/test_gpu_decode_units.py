"""Short units: one workgroup per (batch row, kv head), its waves' pieces merged through LDS, against the oracle and
against the same call with its units cut over the device."""
import pytest
import torch

import fa_oracle as O
from helpers import check_out, library_env, make_paged_case, rotary_tables, to_dev

pytestmark = pytest.mark.gpu


def call(case, **kw):
    from flash_attn_npu import flash_attn_with_kvcache
    dev = to_dev(case)
    out, lse = flash_attn_with_kvcache(dev["q"], dev["k_cache"], dev["v_cache"], dev["k"], dev["v"], cache_seqlens=dev["cache_seqlens"],
                                       block_table=dev["block_table"], return_softmax_lse=True, **to_dev(kw))
    torch.cuda.synchronize()
    return out.cpu(), lse.cpu(), dev["k_cache"].cpu(), dev["v_cache"].cpu()


# chunks are 32 keys: fewer chunks than waves, one more than a multiple of them, remainders inside a chunk, empty rows
LENS = [0, 1, 31, 33, 127, 128, 129, 257, 511, 900]


@pytest.mark.parametrize("waves", [4, 8])
@pytest.mark.parametrize("d,hq,hk,sq,dtype,opts", [
    (128, 8, 2, 1, torch.bfloat16, {}),
    (128, 4, 1, 4, torch.float16, {}),                                  # 16 rows: a full tile
    (128, 20, 4, 5, torch.bfloat16, {}),                                # 25 rows: two tiles
    (64, 6, 2, 1, torch.float16, {"softcap": 20.0}),
    (64, 16, 1, 2, torch.bfloat16, {"window_size": (100, 0)}),          # 32 rows
    (80, 4, 4, 3, torch.bfloat16, {}),                                  # columns behind the head dimension
    (40, 4, 2, 1, torch.float16, {"window_size": (64, 7), "causal": False}),
    (256, 8, 1, 2, torch.bfloat16, {"softcap": 30.0}),
    (192, 3, 1, 1, torch.float16, {}),
])
def test_units(d, hq, hk, sq, dtype, opts, waves):
    case = make_paged_case(len(LENS), hq, hk, d, 64, LENS, seqlen_q=sq, dtype=dtype, seed=d + sq, extra_table_cols=1)
    kw = {"causal": True, **opts}
    with library_env(FA_ROCM_UNIT_WAVES=waves):
        out, lse, _, _ = call(case, **kw)
    ref, ref_lse = O.flash_attn_with_kvcache(case["q"], case["k_cache"].clone(), case["v_cache"].clone(), cache_seqlens=case["cache_seqlens"],
                                             block_table=case["block_table"], mode="fp32", **kw)
    check_out(out, ref, lse, ref_lse, f"units d={d}")
    with library_env(FA_ROCM_UNIT_WAVES=0):
        cut, cut_lse, _, _ = call(case, **kw)
    check_out(out, cut, lse, cut_lse, f"units against cut units d={d}")


@pytest.mark.parametrize("waves", [0, 4, 8])
@pytest.mark.parametrize("interleaved", [False, True])
@pytest.mark.parametrize("d,hq,hk,sq,new,opts", [
    (128, 8, 2, 1, 1, {}),
    (64, 4, 4, 3, 3, {}),
    (128, 20, 4, 5, 5, {}),
    (256, 4, 2, 2, 2, {}),
    (128, 8, 2, 1, 40, {}),                                  # more new rows than a chunk holds, one query
    (128, 12, 2, 3, 2, {"softcap": 25.0}),
    (64, 8, 2, 4, 2, {"window_size": (50, 0)}),
    (128, 8, 2, 1, 9, {"window_size": (4, 0)}),              # new rows behind the window: written by their own launch
    (96, 4, 1, 2, 3, {"window_size": (70, 5), "causal": False}),
])
def test_units_append(d, hq, hk, sq, new, opts, interleaved, waves):
    """The rows that the waves append are those of the append kernel to the bit, whichever wave owns their chunk."""
    lens = [0, 1, 30, 31, 32, 95, 126, 255, 700]
    case = make_paged_case(len(lens), hq, hk, d, 32, lens, seqlen_q=sq, seqlen_new=new, seed=new)
    cos, sin = rotary_tables(800, d)
    kw = {"causal": True, "rotary_cos": cos, "rotary_sin": sin, "rotary_interleaved": interleaved, **opts}
    with library_env(FA_ROCM_UNIT_WAVES=waves):
        out, lse, kc, vc = call(case, **kw)
    ref_k, ref_v = case["k_cache"].clone(), case["v_cache"].clone()
    ref, ref_lse = O.flash_attn_with_kvcache(case["q"], ref_k, ref_v, case["k"], case["v"], cache_seqlens=case["cache_seqlens"],
                                             block_table=case["block_table"], mode="fp32", **kw)
    check_out(out, ref, lse, ref_lse, f"append d={d}")
    assert torch.equal(kc, ref_k) and torch.equal(vc, ref_v)


def test_units_propagate_nan():
    """A NaN key reaches every row that sees it, and only those, as it does where the units are cut over the device."""
    case = make_paged_case(3, 4, 1, 128, 64, [300, 70, 500], seed=3)
    case["k_cache"][case["block_table"][1, 0], 40, 0, 5] = float("nan")
    got = []
    for waves in (0, 8):
        with library_env(FA_ROCM_UNIT_WAVES=waves):
            got.append(call(case, causal=True)[0].float())
    for out in got:
        assert torch.isfinite(out[[0, 2]]).all() and torch.isnan(out[1]).all()
