"""Which kernel a call takes, and in which order its workgroups walk the tiles (no GPU needed)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
pytestmark = pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")

# A workgroup per unit cannot cut a long unit, so the host may choose it only where no lengths that the table or the window
# allows make it the slower path.
# (units, rows of a unit, head dimension, keys that the table addresses, new keys, route); four heads per kv head, or the rows
CALLS = [
    # one workgroup of eight waves per compute unit, at most four chunks of 32 keys per wave
    (8, 4, 128, 1024, 1, "unit 8"), (256, 4, 128, 1024, 0, "unit 8"), (256, 4, 128, 1056, 1, "cut"), (128, 4, 96, 2048, 1, "cut"),
    (264, 4, 128, 768, 1, "unit 4"), (512, 4, 128, 768, 1, "unit 4"), (264, 4, 128, 800, 1, "cut"), (264, 4, 128, 2048, 1, "cut"),
    (520, 4, 128, 256, 1, "cut"), (1536, 4, 128, 512, 1, "cut"),
    (256, 4, 64, 1024, 1, "unit 8"), (264, 4, 64, 1024, 1, "unit 4"), (520, 4, 64, 1024, 1, "unit 4"), (1024, 4, 40, 1024, 1, "unit 4"), (1024, 4, 64, 1056, 1, "cut"),
    (1032, 4, 64, 512, 1, "unit 4"), (1032, 4, 64, 544, 1, "cut"), (8192, 4, 64, 512, 1, "unit 4"), (8200, 4, 64, 512, 1, "cut"),
    (256, 4, 256, 512, 1, "unit 4"), (264, 4, 256, 512, 1, "cut"), (256, 4, 192, 2048, 1, "cut"), (64, 4, 256, 544, 1, "cut"),
    # 17-32 rows: the tiled kernel or two tiles per wave on the other side
    (64, 20, 128, 768, 5, "unit 8"), (64, 20, 128, 800, 5, "tiled"), (64, 20, 128, 224, 0, "tiled"), (64, 20, 128, 224, 5, "tiled"), (64, 20, 128, 256, 0, "unit 8"),
    (184, 20, 128, 8000, 5, "tiled"), (192, 20, 128, 8192, 5, "unit 8"), (193, 20, 128, 8192, 5, "tiled"), (248, 20, 128, 8192, 0, "unit 8"), (192, 20, 128, 8224, 5, "tiled"),
    (256, 20, 128, 8000, 5, "cut"), (256, 20, 128, 768, 5, "unit 8"), (264, 20, 128, 768, 5, "unit 4"), (512, 32, 128, 2048, 8, "cut"),
    (64, 32, 128, 768, 8, "tiled"), (64, 24, 128, 768, 6, "unit 8"), (256, 32, 128, 768, 8, "unit 8"), (64, 32, 64, 768, 8, "cut"),
    (256, 20, 64, 1024, 5, "unit 8"), (264, 20, 64, 1024, 5, "unit 4"), (1032, 20, 64, 256, 5, "cut"),
]


@pytest.fixture(scope="module")
def ask(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("routes") / "route_driver")
    r = subprocess.run([HIPCC, "--offload-arch=gfx950", "-O1", "-std=c++17", "-x", "hip", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                        "-Wno-unused-command-line-argument", os.path.join(ROOT, "flash-attention-npu_amd", "csrc", "fa_rocm_api.cpp"),
                        os.path.join(ROOT, "tests", "native", "route_driver.cpp"), "-o", exe], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr[-4000:]

    def answers(what, questions):
        env = {k: v for k, v in os.environ.items() if not k.startswith("FA_ROCM_")}
        env["HIP_VISIBLE_DEVICES"] = ""                       # 256 compute units are assumed where there is no device
        lines = "\n".join(what + " " + " ".join(map(str, q)) for q in questions)
        r = subprocess.run([exe], input=lines, capture_output=True, text=True, timeout=60, env=env)
        assert r.returncode == 0, r.stderr
        out = [line.strip() for line in r.stdout.split("\n")[:-1]]
        assert len(out) == len(questions)
        return out

    return answers


def test_decode_routes(ask):
    def call(units, rows, d, keys, fresh, window=-1):
        heads = 8 if units % 8 == 0 else 1
        sq = rows // 4
        return (units // heads, sq, 4 * heads, heads, d, 32, keys // 32, fresh, window)

    got = ask("call", [call(*c[:5]) for c in CALLS])
    wrong = [(c, g) for c, g in zip(CALLS, got) if c[5] != g]
    assert not wrong, wrong
    # a window bounds the keys as the table does (and one chunk for its place)
    assert ask("call", [call(8, 4, 128, 1 << 20, 1, w) for w in (991, 992)]) == ["unit 8", "cut"]


def test_prefill_tiling(ask):
    # (group, heads, longest, tokens, head dimension, compute units, causal) -> heads per tile, tiles side by side, tiles of a unit
    cases = {
        (4, 32, 182, 4043, 128, 256, 1): "4 1 6",         # packed whatever the mask: one by one
        (4, 32, 182, 4043, 128, 256, 0): "4 1 6",
        (4, 32, 4096, 32768, 128, 256, 1): "4 4 128",     # causal, many tiles: packed, the tiles of 128 queries side by side
        (7, 28, 350, 14000, 128, 256, 1): "7 7 20",
        (4, 32, 4096, 32768, 128, 256, 0): "1 1 32",
        (1, 32, 4096, 32768, 128, 256, 1): "1 1 32",
        # two rounds of the device: two workgroups per compute unit up to D = 128, one at 256
        (4, 32, 4096, 4096, 128, 256, 1): "4 4 128", (4, 32, 4096, 4095, 128, 256, 1): "1 1 32",
        (4, 32, 2048, 2048, 256, 256, 1): "4 4 64", (4, 32, 2048, 2047, 256, 256, 1): "1 1 16",
        (4, 32, 2048, 2048, 128, 128, 1): "4 4 64", (4, 32, 4096, 4096, 128, 304, 1): "1 1 32",
    }
    assert dict(zip(cases, ask("tiling", cases))) == cases


@pytest.mark.parametrize("tiles,run,heads", [(t, 1, h) for t in (1, 2, 3, 20) for h in (1, 3)] +
                         [(t, r, 1) for t, r in ((2, 4), (3, 4), (4, 4), (5, 4), (20, 7), (21, 7), (10, 2), (6, 100), (129, 100))])
@pytest.mark.parametrize("units", [8, 24])
def test_prefill_order(ask, tiles, run, heads, units):
    (line,) = ask("order", [(tiles, run, units, heads)])
    places = [tuple(map(int, w.split("/"))) for w in line.split()]
    assert len(set(places)) == len(places) == tiles * units * heads          # every tile of every unit once
    assert set(places) == {(u, t, h) for u in range(units) for t in range(tiles) for h in range(heads)}
    assert all(u % 8 == i % 8 for i, (u, _, _) in enumerate(places))         # a unit stays on its XCD
    if run > 1 and tiles > 2:
        # the tiles of the same 128 queries follow each other on the unit's XCD, the longest sequences' first
        for lane in range(8):
            walk = [(t // run, u) for u, t, _ in places[lane::8]]
            assert walk == sorted(walk, key=lambda w: (-w[0], w[1]))
