"""The backtracking kernel where its layout has edges, against the oracle's
sampler (same uniform numbers, so the same trees): walks with more pending
states than the stack in LDS holds, branches of more rows and clades of more
splits than a wave has lanes, a species tree whose branches do not fit LDS."""
from collections import defaultdict

import numpy as np
import pytest

from ale_util import ale_from_tree
from oracle.oracle import OracleModel, ConstantDLWGD as OConst

pytestmark = pytest.mark.gpu


def caterpillar(k):
    """k genes of A and one of B on a spine; from the B end every split lists
    the rest of the spine first, so a walk leaves one pending gene per split."""
    adj, names = defaultdict(list), {}
    for i in range(k - 1):
        adj[i] = [i + 1 if i < k - 2 else "last", f"g{i}", i - 1 if i else "b"]
        adj[f"g{i}"] = [i]
        names[f"g{i}"] = f"A_{i}"
    adj["last"] = [k - 2]
    names["last"] = f"A_{k}"
    adj["b"] = [0]
    names["b"] = "B_1"
    return ale_from_tree(adj={str(u): [str(v) for v in x] for u, x in adj.items()},
                         names={str(u): n for u, n in names.items()})


def synthetic(k, genes, trees, taxa=4):
    def make(synth):
        nw = synth.species_tree(synth.SEED + 9, taxa, 1)
        return nw, synth.families(nw, synth.SEED + genes, k, ("uniform", 0, 0, genes, genes + 8), trees, 100000, 1000000)[0]
    return make


CASES = {"deep stack": (lambda synth: ("(A:1.0,B:1.0);", [caterpillar(180)]), 0.05, 4),
         "long branches": (synthetic(3, 8, 100), 0.005, 20),
         "many splits": (synthetic(2, 60, 3000), 0.1, 20),
         "large species tree": (synthetic(2, 40, 100, 300), 0.1, 5)}


@pytest.mark.parametrize("case", list(CASES))
def test_walks_equal_oracle(w, case):
    from whale_jl_amd import synth
    make, dt, n = CASES[case]
    nw, texts = make(synth)
    q = [0.3] if case != "deep stack" else []
    om = OracleModel(nw, [], dt)
    oc = om.ccds(texts)
    m = w.WhaleModel(w.ConstantDLWGD(λ=0.4, μ=0.3, q=q, η=0.8), w.readnw(nw), dt)
    c = w.ccds_from_texts(texts, m)
    for mode in ("fp64", "fp64s"):
        if not np.isfinite(w.logpdf_(m, c, mode=mode)):
            assert mode == "fp64"  # the plain form underflows on a large family
            continue
        for fam, ts in enumerate(w.backtrack(m, c, n=n, seed=12)):
            ref = om.backtrack(oc, fam, OConst(0.4, 0.3, q, 0.8), seed=12, n_samples=n)
            assert all(np.array_equal(t.nodes, x) for t, x in zip(ts, ref))
