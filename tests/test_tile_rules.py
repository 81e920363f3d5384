"""Which tile each launcher's rule picks, asked of the rules themselves (the kernel sources compiled into small libraries
with one query function each), so that the row counts of test_tile_configs_gpu.py cannot drift away from the limits they
are there for. CPU only."""
import concurrent.futures
import ctypes as C
import os
import re
import shutil
import subprocess

import pytest

from tests import test_tile_configs_gpu as G

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "xtagger_amd", "csrc")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
pytestmark = pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not available")

# (source, the expression that calls its rule with a generic lambda f)
RULES = {"res": ("layer.hip", "with_res_cfg(a, b, 1, f)"), "qkv": ("layer.hip", "with_qkv_cfg(a, 1, f)"),
         "fc1": ("layer.hip", "with_fc1_cfg(a, f)"), "pe": ("layer.hip", "with_pe_cfg(a, f)"),
         "px_fc1": ("px.hip", "with_px_fc1_cfg(a, 1, f)"),
         "gemm": ("quant.hip", "with_gemm_cfg<false>(a, b, c, out, f)"),
         "gemm_sp": ("quant.hip", "with_gemm_cfg<true>(a, b, c, out, f)"),
         "res_2": ("layer.hip", "with_res_cfg(a, b, 2, f)"), "qkv_2": ("layer.hip", "with_qkv_cfg(a, 2, f)"),
         "px_fc1_2": ("px.hip", "with_px_fc1_cfg(a, 2, f)")}


@pytest.fixture(scope="module")
def tile(tmp_path_factory):
    """tile(rule, a, b=0, c=0, out=2) -> (BM, BN, waves)"""
    d = tmp_path_factory.mktemp("rules")

    def build(src):
        body = "".join(f'extern "C" int rule_{k}(int a, int b, int c, int out) {{ int t = 0; auto f = [&](auto x) {{ '
                       f'using T = decltype(x); t = (T::BM * 1000 + T::BN) * 1000 + T::NW; }}; {e}; return t; }}\n'
                       for k, (s, e) in RULES.items() if s == src)
        f = d / ("q_" + src)
        f.write_text(f'#include "{os.path.join(CSRC, src)}"\n{body}')
        so = str(f) + ".so"
        r = subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-shared", "-ffp-contract=off",
                            "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-I" + CSRC,
                            "-I" + os.path.join(CSRC, "..", "..", "include"), str(f), "-o", so],
                           capture_output=True, text=True, timeout=600)
        assert r.returncode == 0, r.stderr[-2000:]
        return src, C.CDLL(so)

    with concurrent.futures.ThreadPoolExecutor(3) as ex:
        libs = dict(ex.map(build, sorted({s for s, _ in RULES.values()})))

    def tile(rule, a, b=0, c=0, out=2):
        t = getattr(libs[RULES[rule][0]], "rule_" + rule)(a, b, c, out)
        return t // 1000000, t // 1000 % 1000, t % 1000

    return tile


def _limits(tile, rule, hi, *args):
    """the rows r in 1 .. hi - 1 after which the tile changes"""
    t = [tile(rule, r, *args) for r in range(1, hi + 1)]
    return [r for r in range(1, hi) if t[r - 1] != t[r]]


SML, MID, BIG = (64, 128, 4), (128, 128, 8), (256, 256, 8)


def test_both_sides_of_every_limit(tile):
    """every limit below the tested range's end has a tested row count on either side, without another limit between"""
    def check(limits, rows, end):
        edges = [0, *[x for x in limits if x < end], end]
        for lo, hi in zip(edges[:-1], edges[1:]):
            assert any(lo < r <= hi for r in rows), f"no tested row count in ({lo}, {hi}]"

    assert _limits(tile, "res", 20000, G.HIDP) == _limits(tile, "res", 20000, G.PXH) == [4096, 8192]
    k1024 = _limits(tile, "res", 20000, G.D)
    assert k1024[:3] == [4096, 8447, 16384]
    for limits, rows in ((k1024, G.RES_ROWS), ([4096, 8192], G.RES_ROWS), (k1024[:2], G.PX_ROWS), ([4096, 8192], G.PX_ROWS)):
        check(limits, rows, 16400)
        for x in limits[:2]:
            assert x in rows and x + 1 in rows, x
    assert _limits(tile, "fc1", 20000) == [1408] and {1408, 1409} <= set(G.RES_ROWS)
    wide = (128, 128, 4)
    for rows, want in ((1, wide), (2048, wide), (2049, BIG), (3328, BIG), (3329, wide), (5184, wide), (5377, BIG),
                       (6656, BIG), (6657, wide), (10368, wide), (12288, wide), (12289, BIG), (20736, BIG)):
        assert tile("px_fc1", rows) == want, rows
    assert {tile("px_fc1", r) for r in G.PX_FC1_ROWS} == {wide, BIG}
    assert [tile("qkv", 1025 * nb) for nb in (1, 2, 3, 5, 6, 7, 8, 16, 32)] == [MID, MID, BIG, BIG, MID, BIG, BIG, BIG, BIG]
    assert [tile("pe", r) for r in (1024, 2048, 2049, 3072)] == [(64, 64, 4), (64, 64, 4), MID, MID]


def test_two_lanes(tile):
    """Beside an engine's other lane the tiles that only win alone on the chip (128 x 128 from 4353 rows on, qkv's for a
    short second round, PixAI fc1's) are not taken: batches of 10 to 14 images lost 2 to 5% with them."""
    for k in (G.D, G.HIDP, G.PXH):
        assert _limits(tile, "res_2", 42000, k) == [4096, 4352], k
        assert [tile("res_2", r, k) for r in (4096, 4100, 5125, 16400)] == [SML, MID, BIG, BIG]
    assert _limits(tile, "qkv_2", 42000) == [2688] and tile("qkv_2", 1025) == MID
    assert _limits(tile, "px_fc1_2", 42000) == [] and tile("px_fc1_2", 10368) == BIG
    used = {"engine.cpp": ("xt_qkv", "xt_oproj", "xt_fc2"), "px_engine.cpp": ("xt_px_proj", "xt_px_fc1", "xt_px_fc2")}
    for src, names in used.items():                           # the engines call the launchers that take their lanes
        text = open(os.path.join(CSRC, src)).read()
        for n in names:
            assert n + "(" in text, (src, n)
            assert not re.search(n.replace("xt_px_", "px_k_").replace("xt_", "eva_k_") + r"(_sp)?\(", text), (src, n)


def test_partial_row_tiles_cover_every_tile(tile):
    for k in (G.D, G.HIDP):
        assert [{tile("res", b + t, k) for t in G.TAILS} for b in G.TAIL_BASES[1:]] == [{SML}, {MID}, {BIG}], k
    assert [{tile("fc1", b + t) for t in G.TAILS} for b in G.TAIL_BASES] == [{(128, 256, 16)}, {BIG}, {BIG}, {BIG}]


def test_gemm_shapes_cover_every_tile(tile):
    shapes = next(m for m in G.test_gemm_any_alignment_and_tile.pytestmark if "M,N" in m.args[0]).args[1]
    narrow, wide = {(64, 64, 4), SML, MID}, {(128, 128, 4), BIG}
    for rule in ("gemm", "gemm_sp"):
        got = {0: set(), 1: set(), 2: set()}                  # by what is stored: bf16, fp32, bf16 to an aligned C
        for M, N, K, off, pad in shapes:
            n = (N + 15) // 16 * 16 if rule == "gemm_sp" else N
            out = 2 if (n | n + pad | off) % 8 == 0 else 0
            for o in (out, 1):
                got[o].add(tile(rule, M, n, K, o))
        assert got[1] == narrow | wide, (rule, got[1])
        assert got[2] >= wide and got[0] >= {BIG, MID} and got[0] | got[2] == narrow | wide, (rule, got)
        assert (128, 128, 4) not in got[0]


def test_gemm_limits(tile):
    """both sides of the rule's lines: rounds of 512 blocks (128 x 128) and 256 blocks (256 x 256), and K"""
    wide = (128, 128, 4)
    for args, want in {(3000, 4096, 512): wide, (3000, 4096, 2048): BIG, (3584, 3584, 128): BIG, (4000, 4000, 128): BIG,
                       (4100, 4000, 128): MID, (8100, 3000, 2048): wide, (8200, 3072, 2047): MID, (8200, 3072, 2048): BIG,
                       (2050, 3072, 3072): wide, (8200, 1024, 1024): MID, (3200, 8000, 128): BIG}.items():
        assert tile("gemm", *args) == want, args
    for args, want in {(3000, 4096, 128): wide, (3000, 4096, 2048): MID, (3584, 3584, 128): BIG, (2050, 3072, 128): wide,
                       (2050, 3072, 256): MID, (8200, 3072, 3072): MID}.items():
        assert tile("gemm_sp", *args) == want, args
    assert tile("gemm_sp", 2050, 3072, 896, 1) == wide and tile("gemm_sp", 2050, 3072, 1024, 1) == MID
