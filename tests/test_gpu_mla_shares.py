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
@pytest.mark.parametrize("lens", [[700, 33], EDGES, [1500, 916, 2489], [40 + 37 * i for i in range(30)],
                                  [20] * 40, [1792] * 10, [160 + 37 * i for i in range(30)]])
def test_ragged_shares(lens, wgs):
    case = mla_case(len(lens), 128, lens, page=64, seed=len(lens) + wgs)
    with library_env(**({"FA_ROCM_DECODE_WGS": wgs} if wgs else {})):
        got, ref, _ = run(case)
    check_out(got[0], ref[0], got[1], ref[1], f"shares {len(lens)} units, {wgs} workers")


@pytest.mark.parametrize("lens", [[100], [65, 128, 33], [128, 700, 97, 0, 5000], [128] * 40])
def test_short_units_stay_whole(lens):
    """Units of at most four chunks are written from their fp32 accumulators: values beyond the range of the fp16 partial
    rows that longer units are cut into (65504) reach a bf16 output."""
    magnitude = 1e5
    g = torch.Generator().manual_seed(len(lens))
    case = mla_case(len(lens), 128, lens, page=64, seed=7)
    latent = (torch.randn(*case["k_cache"].shape, generator=g) * magnitude).to(torch.bfloat16)
    case["k_cache"], case["k_scale"] = O.quantize_per_token(latent)
    case["q"] = (case["q"] * 3 / magnitude).to(torch.bfloat16)         # a few keys hold most of the weight
    got, ref, _ = run(case)
    assert ref[0][0].abs().max() > 65504
    out = got[0].float().cpu()
    for b, n in enumerate(lens):
        if 0 < n <= 128:   # weights and results are rounded to bf16, 2^-9 each
            assert ((out[b] - ref[0][b]).norm() / ref[0][b].norm()).item() <= 6e-3, (b, n)
