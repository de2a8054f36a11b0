"""Latent decode of ragged batches whose units are padded to whole shares, and of batches with too many units for that:
lengths around the 32-key chunk, empty rows, one to many units, against the oracle."""
import pytest
import torch

import fa_oracle as O
from helpers import check_out, library_env
from test_gpu_mla import mla_case, run

pytestmark = pytest.mark.gpu

EDGES = [0, 1, 31, 32, 33, 63, 64, 65, 96, 500, 2049]


@pytest.mark.parametrize("wgs", [0, 13, 40])          # 0: the device's; 13: a worker takes several units; 40: barely enough to align
@pytest.mark.parametrize("lens", [[700, 33], EDGES, [1500, 916, 2489], [40 + 37 * i for i in range(30)]])
def test_ragged_shares(lens, wgs):
    case = mla_case(len(lens), 128, lens, page=64, seed=len(lens) + wgs)
    with library_env(**({"FA_ROCM_DECODE_WGS": wgs} if wgs else {})):
        got, ref, _ = run(case)
    check_out(got[0], ref[0], got[1], ref[1], f"shares {len(lens)} units, {wgs} workers")


@pytest.mark.parametrize("wgs", [0, 2])
@pytest.mark.parametrize("hq,sq,new,window", [(128, 1, 1, -1), (16, 1, 1, 200), (128, 1, 3, -1), (128, 2, 2, -1), (200, 1, 1, -1), (64, 1, 4, 1)])
def test_appended_tokens(hq, sq, new, window, wgs):
    """The quantised rows are the oracle's to the bit whichever workgroup writes them: one that owns the row's chunk, or the
    append kernel where several units read it (several tokens or head groups) or a window hides an appended row."""
    from flash_attn_npu import flash_attn_with_kvcache
    lens = [0, 1, 30, 31, 32, 63, 255, 700]
    case = mla_case(len(lens), hq, [n + new for n in lens], page=32, seed=hq + new)
    g = torch.Generator().manual_seed(new)
    fresh = torch.randn(len(lens), new, 1, 576, generator=g).to(torch.bfloat16)
    fresh[0] = 0                                       # scale 0, codes 0, the only key of its row
    q = torch.randn(len(lens), sq, hq, 576, generator=g).to(torch.bfloat16)
    kw = dict(softmax_scale=192 ** -0.5, causal=True, window_size=(window, -1), return_softmax_lse=True)
    used = torch.tensor(lens, dtype=torch.int32)
    kc, ks = case["k_cache"].cuda(), case["k_scale"].cuda()
    f = fresh.cuda()
    with library_env(**({"FA_ROCM_DECODE_WGS": wgs} if wgs else {})):
        out, lse = flash_attn_with_kvcache(q.cuda(), kc, kc[..., :512], f, f[..., :512], cache_seqlens=used.cuda(),
                                           block_table=case["block_table"].cuda(), k_scale_cache=ks, **kw)
        torch.cuda.synchronize()
    rk, rs = case["k_cache"].clone(), case["k_scale"].clone()
    code, scale = O.quantize_per_token(fresh)
    for b, n in enumerate(lens):
        for t in range(new):
            page, slot = case["block_table"][b, (n + t) // 32], (n + t) % 32
            rk[page, slot], rs[page, slot] = code[b, t], scale[b, t]
    assert torch.equal(kc.cpu(), rk) and torch.equal(ks.cpu().view(rs.shape), rs)
    kw.pop("return_softmax_lse")
    ref, ref_lse = O.flash_attn_with_kvcache(q, rk, rk[..., :512], cache_seqlens=used + new, block_table=case["block_table"], k_scale_cache=rs,
                                             mode="fp32", **kw)
    check_out(out, ref, lse, ref_lse, f"latent append heads {hq} tokens {sq} new {new}")
