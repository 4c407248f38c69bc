"""The tiles that the products of several tokens run on (wick_amd/csrc/gemm_tiles.h): the
shapes of test_model_gpu.py's parity test reach every tile that the rule can give, in each of
the epilogues, so that a change of the rule cannot leave one without a test unnoticed."""
import os
import shutil
import subprocess

import pytest

from test_model_gpu import PRODUCT_CASES

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "wick_amd", "csrc")


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not found")
def test_every_tile_has_a_parity_case(tmp_path):
    exe = str(tmp_path / "gemm_tile_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Werror", "-I", CSRC,
                    os.path.join(HERE, "gemm_tile_check.cpp"), "-o", exe], check=True, timeout=120)

    def tiles(queries):
        text = "".join("%d %d %d %d\n" % q for q in queries)
        out = subprocess.run([exe], input=text, stdout=subprocess.PIPE, text=True, check=True, timeout=120).stdout
        lines = out.splitlines()
        assert len(lines) == len(queries)
        return lines

    covered = set()
    for hidden, ff, heads, kvh, d, vocab, t in PRODUCT_CASES:
        shapes = [("qkv", 0, (heads + 2 * kvh) * d, hidden), ("resid", 0, hidden, heads * d), ("resid", 0, hidden, ff),
                  ("gate/up", 1, ff, hidden), ("store", 0, vocab, hidden)]
        covered |= set(zip([s[0] for s in shapes], tiles([(s[1], s[2], s[3], t) for s in shapes])))
    sizes = [(rows, cols, t) for rows in list(range(16, 4200, 92)) + [5632, 8960, 14336, 32000, 49152, 151936]
             for cols in (16, 64, 100, 164, 260, 576, 580, 896, 1024, 1536, 2048, 2052, 4096, 5632, 14336)
             for t in (2, 3, 4, 15, 16, 17, 32, 33, 64, 65, 100, 130, 192, 200, 251, 256, 257, 512, 1000, 4000)]
    plain, gate_up = (set(tiles([(g, *s) for s in sizes])) for g in (0, 1))
    want = {(kind, tile) for kind in ("qkv", "resid", "store") for tile in plain} | {("gate/up", x) for x in gate_up}
    assert covered >= want, sorted(want - covered)
    assert len(plain) == 9 and len(gate_up) == 4  # as many as gemm_epi (model.hip) launches
