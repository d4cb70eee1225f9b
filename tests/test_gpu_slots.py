"""Families around the boundaries of the kernels' slot layout against the
CPU oracle: stages that fit one chunk of 64 slots, fill a team's registers and
overflow them (more than 12 chunks), items with no split, with more than one
lane's terms and with more than 16 lanes hold, one-wave and team launches,
families narrower than their launch's team."""
import numpy as np
import pytest

from oracle.oracle import OracleModel, ConstantDLWGD as OConst

pytestmark = pytest.mark.gpu

# genes per family (on 3 taxa with one WGD), gene trees per family, number of families
SIZES = {"one chunk": [(2, 8, 60, 6)], "two chunks": [(18, 30, 60, 4)],
         "teams": [(60, 70, 60, 2), (130, 150, 60, 2)], "past the registers": [(230, 250, 2000, 1)],
         "mixed": [(2, 8, 60, 3), (18, 30, 60, 2), (130, 150, 60, 1), (230, 250, 2000, 1)]}


@pytest.mark.parametrize("size", list(SIZES))
def test_slot_layout_vs_oracle(w, size):
    from whale_jl_amd import synth
    seed = synth.SEED + 501
    nw = synth.species_tree(seed, 3, 1)
    texts = []
    for lo, hi, trees, k in SIZES[size]:
        texts += synth.families(nw, seed + hi, k, ("uniform", 0, 0, lo, hi), trees, 100000, 1000000, nthreads=8)[0]
    om = OracleModel(nw, [], 0.05)
    oc = om.ccds(texts)
    orr = OConst(0.3, 0.2, [0.25], 0.8)
    m = w.WhaleModel(w.ConstantDLWGD(λ=0.3, μ=0.2, q=[0.25], η=0.8), w.readnw(nw), 0.05)
    c = w.ccds_from_texts(texts, m)
    ref = om.logpdf(oc, orr, per_family=True, precision="long")
    ov, og = om.gradient(oc, orr, nthreads=8)
    # the tolerances every comparison of the device paths with the oracle uses:
    # FP64 rounding over a few hundred rows, FP32 rounding likewise
    for mode, tv, tg in (("fp64s", 1e-12, 1e-10), ("fp64", 1e-12, 1e-10), ("fp32", 1e-6, 1e-5)):
        got = w.logpdf_families(m, c, mode=mode)
        ok = np.isfinite(got) if mode == "fp64" else np.isfinite(ref)  # the plain form underflows on large families
        assert np.array_equal(np.isfinite(got), ok)
        assert np.max(np.abs(got[ok] - ref[ok]) / np.abs(ref[ok]), initial=0.0) <= tv
        if not ok.all():
            continue
        v, g, _ = w.gradient(m, c, mode=mode)
        err = np.max(np.abs(g - og)) / np.max(np.abs(og))
        print(size, mode, "clades", [len(x.size) for x in c], "gradient error", err)
        assert abs(v - ov) <= tv * abs(ov)
        assert err <= tg
