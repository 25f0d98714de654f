"""What bench.py says a launch moves: each input once, each output once, for every algorithm."""
import importlib.util
import os

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


# read: partials, delivered rows of the stage, residual, gamma; written: residual_out, summed rows of the stage, outputs
@pytest.mark.parametrize("n,tokens,hidden,elem,out,algo,read,written", [
    (8, 2048, 8192, 2, 2048 * 8192 + 4 * 2048, "auto", (8 + 1) * 2048 * 16384 + 16384, 2048 * (16384 + 8192 + 4)),
    (8, 2048, 8192, 2, 2048 * 8192 + 4 * 2048, "staged", (8 + 1) * 2048 * 16384 + 16384, 2048 * (16384 + 16384 + 8192 + 4)),
    (8, 2048, 8192, 2, 2048 * 8192 + 4 * 2048, "staged_owned", (256 * 8 + 1792 + 2048 + 1) * 16384, 2048 * (16384 + 8192 + 4) + 256 * 16384),
    (4, 10, 64, 4, 10 * 256, "staged_owned", (3 * 4 + 7 + 10 + 1) * 256, (10 + 10 + 3) * 256),
])
def test_moved_bytes(n, tokens, hidden, elem, out, algo, read, written):
    spec = importlib.util.spec_from_file_location("tde_bench", os.path.join(ROOT, "bench.py"))
    bench = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(bench)
    row = hidden * elem
    fused = (n + 1) * tokens * row + row + tokens * row + out
    assert bench.moved_bytes(fused, n, tokens, hidden, elem, algo) == (read, written)
