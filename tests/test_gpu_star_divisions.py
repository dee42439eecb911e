"""Dana-Star's vector path divides by a short sequence while every |g|, |m| and
sqrt(v) + epsilon of the four elements lies in its range, by the IEEE sequence
otherwise: parity with the oracle (bit-exact state) for gradients on both sides
of each bound, alone and mixed within a group of four, and the short sequence
against the IEEE quotient over its declared range."""
import numpy as np
import pytest
import torch

from test_gpu_mathcheck import _run
from test_gpu_parity import Pair

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a ROCm GPU")]


def test_div_short_over_its_range():
    """div_short(a, b) == a / b for every mantissa of b, each against 512
    mantissas of a, with exponents over b in [2^-66, 2^21], a in [2^-98, 2^86],
    a / b below 2^110, and a == 0."""
    print("case: div_short", flush=True)
    bad, first = _run(7, 0, 0xFFFFFFFF)
    assert bad == 0, f"{bad} mismatches, first pattern {first:#010x}"


def _edges(rng, n, zeros):
    """Magnitudes at, next to and well inside both bounds: groups of four that are
    all inside, all outside, and mixed."""
    lo, hi = np.float32(2.0 ** -66), np.float32(2.0 ** 20)
    pool = np.array([lo, np.nextafter(lo, np.float32(0)), np.nextafter(lo, hi), 2.0 ** -70, 2.0 ** -60, 1e-3, 1.0,
                     hi, np.nextafter(hi, lo), np.nextafter(hi, np.float32(np.inf)), 2.0 ** 24,
                     0.0 if zeros else 2.0 ** -40], np.float32)
    g = rng.choice(pool, n)
    inside = np.repeat(rng.random(n // 4 + 1) < 0.5, 4)[:n]
    g[inside] = (2.0 ** rng.uniform(-65, 19, n)).astype(np.float32)[inside]
    return (g * rng.choice(np.array([-1, 1], np.float32), n)).astype(np.float32)


@pytest.mark.parametrize("foreach", [False, True])
@pytest.mark.parametrize("epsilon", [1e-8, 1.3e-20, 0.0])    # 2^-66 = 1.36e-20
def test_star_step_at_the_bounds(oracle_mod, epsilon, foreach):
    print("case: star divisions", epsilon, foreach, flush=True)
    rng = np.random.default_rng(7)
    sizes = [4099, 16 * 1024, 3]
    pair = Pair(oracle_mod, True, [([rng.normal(0, 0.02, n).astype(np.float32) for n in sizes], {})], lr=1e-3,
                delta=8.0, kappa=0.85, epsilon=epsilon, weight_decay=0.1, clipsnr=2.0, foreach=foreach)
    for t in range(3):
        pair.step([[_edges(rng, n, zeros=epsilon > 0) for n in sizes]])
        pair.compare(where=f"eps {epsilon} t={t}", check_diag=False)
