"""bench.py's roofs bound what was measured: the FP16 tiles are rated against the
whole dense 16-bit peak, the split BF16 against a third of it."""
import importlib.util
import os

import pytest

from conftest import ROOT


# dim, points, pairs evaluated, kernel ms, operands: measured launches
@pytest.mark.parametrize("dim, n, evals, ms, operands", [
    (18, 2_000_000, 1.35e12, 66.6, "f16"), (90, 1_000_000, 5.0e11, 66.3, "f16"),
    (18, 2_000_000, 2.7e12, 488.5, "bf16"), (90, 1_000_000, 1.0e12, 701.0, "bf16")])
def test_mfma_roof_is_not_passed(dim, n, evals, ms, operands):
    spec = importlib.util.spec_from_file_location("bench", os.path.join(ROOT, "bench.py"))
    bench = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(bench)
    roof, _ = bench.rooflines(n, dim, 1000, 30 * n, evals, ms, "mfma", operands)
    assert roof["bound"] == "mfma" and 0.1 < roof["frac"] < 1.0 and roof["roof_ms"] < ms
    assert roof["peak"] == pytest.approx(2500.0 / (3 if operands == "bf16" else 1))
