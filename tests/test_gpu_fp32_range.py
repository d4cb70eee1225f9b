"""FP32 gradients of families whose reverse sweep comes close to the ends of
FP32: clades that enter a branch at 2^-100 of their later value, so that a
split's coefficient and the adjoint of its owner are each near 2^100 and only
the coefficient times the other part's value is near 1."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_gradient_near_the_fp32_range(w):
    from whale_jl_amd import synth
    nw = synth.species_tree(1001, 50, 4)
    texts, _ = synth.families(nw, 78, 2746, ("lognormal", 20, 0.9, 4, 200), 200, 2000, 1000000, nthreads=8)
    texts = [texts[i] for i in (2487, 2745)]
    rng = np.random.default_rng([1, 1])
    rng.permutation(12500)
    n = 2 * 50 - 1
    λ = math.log(0.2) + 0.5 * rng.standard_normal(n)
    μ = math.log(0.15) + 0.5 * rng.standard_normal(n)
    m = w.WhaleModel(w.DLWGD(λ=list(λ), μ=list(μ), q=list(rng.uniform(0.1, 0.6, 4)), η=0.9), w.readnw(nw), 0.01)
    for t in texts:
        c = w.ccds_from_texts([t], m)
        v, g, _ = w.gradient(m, c, mode="fp64s")
        v32, g32, _ = w.gradient(m, c, mode="fp32")
        assert np.isfinite(g32).all()
        # the tolerances of every FP32 comparison here
        assert abs(v32 - v) <= 1e-6 * abs(v)
        assert np.max(np.abs(g32 - g)) <= 1e-5 * np.max(np.abs(g))
