"""Rule sets beyond the sliced form's limits are generated without it, and in the time
that the rest of the program takes."""
import time

import pytest

import sandengine_amd as S


def probabilities(n):
    rules = "".join(f"  r{i}:\n    if: rand.y < {(i + 1) / (n + 2):.4f} and isType_EMPTY(DOWN)\n    do: SWAP SELF DOWN\n"
                    for i in range(n))
    return ("rules:\n" + rules + "types:\n  base:\n    base_rules: [" + ", ".join(f"r{i}" for i in range(n)) +
            "]\nmaterials:\n  sand:\n    type: base\n    color: [0.5, 0.5, 0.5]\n    density: 1.5\n")


# the mirror's hash plane is one of eight
@pytest.mark.parametrize("n,sliced", [(1, True), (7, True), (8, False), (9, False), (24, False), (30, False), (33, False)])
def test_many_probabilities(n, sliced):
    t = time.perf_counter()
    src = S.emit_hip(probabilities(n))
    assert ("// ---- sliced form" in src) == sliced
    assert time.perf_counter() - t < 5.0  # hundredths of a second; the class words of 24 take more than one, of 30 minutes
