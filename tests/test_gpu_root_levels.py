"""The reverse sweep's root levels with terms read from memory (families whose
stages lie in global memory take them so in every form) against the CPU oracle:
families of two genes, levels within one chunk of 64 slots, levels wider than a
team's chunks and lanes of more than four terms, odd and even level counts."""
import numpy as np
import pytest

from oracle.oracle import OracleModel, ConstantDLWGD as OConst

pytestmark = pytest.mark.gpu

# genes per family (on 3 taxa with one WGD), gene trees per family, number of families
SIZES = {"two genes": (2, 2, 5, 3), "few": (3, 8, 60, 6), "one chunk": (18, 30, 60, 4), "wide": (120, 140, 1500, 1)}


@pytest.mark.parametrize("memory", [False, True])
@pytest.mark.parametrize("size", list(SIZES))
def test_root_levels_vs_oracle(w, size, memory):
    from whale_jl_amd import synth
    lo, hi, trees, k = SIZES[size]
    seed = synth.SEED + 911
    nw = synth.species_tree(seed, 3, 1)
    texts = synth.families(nw, seed + hi, k, ("uniform", 0, 0, lo, hi), trees, 100000, 1000000, nthreads=8)[0]
    om = OracleModel(nw, [], 0.05)
    ov, og = om.gradient(om.ccds(texts), OConst(0.3, 0.2, [0.25], 0.8), nthreads=8)
    m = w.WhaleModel(w.ConstantDLWGD(λ=0.3, μ=0.2, q=[0.25], η=0.8), w.readnw(nw), 0.05)
    c = w.ccds_from_texts(texts, m)
    if memory:
        w.device_batch(m, c).set_lds_limit(1)
    # the tolerances of every comparison of the device paths with the oracle
    for mode, tv, tg in (("fp32", 1e-6, 1e-5), ("fp64s", 1e-12, 1e-10)):
        v, g, _ = w.gradient(m, c, mode=mode)
        assert abs(v - ov) <= tv * abs(ov)
        assert np.max(np.abs(g - og)) <= tg * np.max(np.abs(og))
