"""Species trees around the boundaries of the table and gradient kernels, and
batches around those of the results' way to the host, against the CPU oracle:
as many nodes as a workgroup has lanes (1023, 1025), trees whose table
workspace leaves LDS (128 KB) and whose gradient workspace does (1537 nodes
and more), one and several workgroups that hand over the families' values."""
import numpy as np
import pytest

from oracle.oracle import OracleModel, ConstantDLWGD as OConst

pytestmark = pytest.mark.gpu

# taxa, slice length, families
SIZES = {"1023 nodes": (512, 0.05, 6), "1025 nodes": (513, 0.05, 6), "tables in memory": (400, 0.005, 6),
         "1559 nodes": (780, 0.05, 6), "one copy group": (3, 0.05, 2048), "two copy groups": (3, 0.05, 2049),
         "one family": (3, 0.05, 1)}


@pytest.mark.parametrize("size", list(SIZES))
def test_sizes_vs_oracle(w, size):
    from whale_jl_amd import synth
    taxa, dt, n = SIZES[size]
    seed = synth.SEED + 733
    nw = synth.species_tree(seed, taxa, 1)
    texts = synth.families(nw, seed + taxa, n, ("uniform", 0, 0, 3, 8), 20, 1000, 1000000, nthreads=8)[0]
    om = OracleModel(nw, [], dt)
    oc = om.ccds(texts)
    orr = OConst(0.3, 0.2, [0.25], 0.8)
    m = w.WhaleModel(w.ConstantDLWGD(λ=0.3, μ=0.2, q=[0.25], η=0.8), w.readnw(nw), dt)
    c = w.ccds_from_texts(texts, m)
    ref = om.logpdf(oc, orr, per_family=True, precision="long")
    ov, og = om.gradient(oc, orr, nthreads=8)
    # the tolerances of every comparison of the device paths with the oracle
    for mode, tv, tg in (("fp64s", 1e-12, 1e-10), ("fp64", 1e-12, 1e-10)):
        got = w.logpdf_families(m, c, mode=mode)
        assert np.max(np.abs(got - ref) / np.abs(ref)) <= tv
        v, g, fam = w.gradient(m, c, mode=mode)
        assert np.max(np.abs(fam - ref) / np.abs(ref)) <= tv
        assert abs(v - ov) <= tv * abs(ov)
        err = np.max(np.abs(g - og)) / np.max(np.abs(og))
        print(size, mode, "gradient error", err)
        assert err <= tg
