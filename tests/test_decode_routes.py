"""Which kernel a kvcache call takes (no GPU needed): a workgroup per unit cannot cut a long unit, so the host may choose it
only where no lengths that the table or the window allows make it the slower path."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
pytestmark = pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")

# (units, rows of a unit, head dimension, keys that the table addresses, new keys, route); four heads per kv head, or the rows
CALLS = [
    # one workgroup of eight waves per compute unit, at most four chunks of 32 keys per wave
    (8, 4, 128, 1024, 1, "unit 8"), (256, 4, 128, 1024, 0, "unit 8"), (256, 4, 128, 1056, 1, "cut"), (128, 4, 96, 2048, 1, "cut"),
    (264, 4, 128, 768, 1, "unit 4"), (512, 4, 128, 768, 1, "unit 4"), (264, 4, 128, 800, 1, "cut"), (264, 4, 128, 2048, 1, "cut"),
    (520, 4, 128, 256, 1, "cut"), (1536, 4, 128, 512, 1, "cut"),
    (512, 4, 64, 1024, 1, "unit 8"), (520, 4, 64, 1024, 1, "unit 4"), (1024, 4, 40, 1024, 1, "unit 4"), (1024, 4, 64, 1056, 1, "cut"),
    (1032, 4, 64, 512, 1, "unit 4"), (1032, 4, 64, 544, 1, "cut"), (8192, 4, 64, 512, 1, "unit 4"), (8200, 4, 64, 512, 1, "cut"),
    (256, 4, 256, 512, 1, "unit 4"), (264, 4, 256, 512, 1, "cut"), (256, 4, 192, 2048, 1, "cut"), (64, 4, 256, 544, 1, "cut"),
    # 17-32 rows: the tiled kernel or two tiles per wave on the other side
    (64, 20, 128, 768, 5, "unit 8"), (64, 20, 128, 800, 5, "tiled"), (64, 20, 128, 224, 0, "tiled"), (64, 20, 128, 224, 5, "tiled"), (64, 20, 128, 256, 0, "unit 8"),
    (184, 20, 128, 8000, 5, "tiled"), (192, 20, 128, 8192, 5, "unit 8"), (193, 20, 128, 8192, 5, "tiled"), (248, 20, 128, 8192, 0, "unit 8"), (192, 20, 128, 8224, 5, "tiled"),
    (256, 20, 128, 8000, 5, "cut"), (256, 20, 128, 768, 5, "unit 8"), (264, 20, 128, 768, 5, "unit 4"), (512, 32, 128, 2048, 8, "cut"),
    (64, 32, 128, 768, 8, "tiled"), (64, 24, 128, 768, 6, "unit 8"), (256, 32, 128, 768, 8, "unit 8"), (64, 32, 64, 768, 8, "cut"),
    (256, 20, 64, 1024, 5, "unit 8"), (264, 20, 64, 1024, 5, "unit 4"), (1032, 20, 64, 256, 5, "cut"),
]


def test_decode_routes(tmp_path):
    exe = str(tmp_path / "route_driver")
    r = subprocess.run([HIPCC, "--offload-arch=gfx950", "-O1", "-std=c++17", "-x", "hip", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                        "-Wno-unused-command-line-argument", os.path.join(ROOT, "flash-attention-npu_amd", "csrc", "fa_rocm_api.cpp"),
                        os.path.join(ROOT, "tests", "native", "route_driver.cpp"), "-o", exe], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr[-4000:]

    def routes(calls):
        env = {k: v for k, v in os.environ.items() if not k.startswith("FA_ROCM_")}
        env["HIP_VISIBLE_DEVICES"] = ""                       # 256 compute units are assumed where there is no device
        r = subprocess.run([exe], input="\n".join(" ".join(map(str, c)) for c in calls), capture_output=True, text=True, timeout=60, env=env)
        assert r.returncode == 0, r.stderr
        return r.stdout.split("\n")[:-1]

    def call(units, rows, d, keys, fresh, window=-1):
        heads = 8 if units % 8 == 0 else 1
        sq = rows // 4
        return (units // heads, sq, 4 * heads, heads, d, 32, keys // 32, fresh, window)

    got = routes([call(*c[:5]) for c in CALLS])
    wrong = [(c, g) for c, g in zip(CALLS, got) if c[5] != g]
    assert not wrong and len(got) == len(CALLS), wrong
    # a window bounds the keys as the table does (and one chunk for its place)
    assert routes([call(8, 4, 128, 1 << 20, 1, w) for w in (991, 992)]) == ["unit 8", "cut"]
