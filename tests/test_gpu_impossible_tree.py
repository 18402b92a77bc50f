"""A displayed tree that gives a site a likelihood of exactly zero has weight
zero in the mixture, and its roots seed nothing into the reverse sweep: the
gradient is the one without that tree, and finite.

Two tips under a reticulation lie at distance zero in the first tree.  G and T
are the only states that exchange with each other (A and C likewise), with
frequencies for which the rate matrix's eigenvectors make P(0) exactly the
identity, so sites where the two tips differ are impossible there."""
import math

import numpy as np
import pytest

from netrax_amd import AnnotatedNetwork, LikelihoodVariant, NetraxOptions, Precision
from netrax_amd.network import parse_newick
from netrax_amd.simulate import Model, Partition
from oracle import oracle as O

pytestmark = pytest.mark.gpu

NEWICK = "((A:0,(B:0)#H1:0::0.4):0.1,(#H1:0.3::0.6,(C:0.2,D:0.15):0.1):0.05);"
G, T = 4, 8


@pytest.mark.parametrize("variant", [0, 1])
@pytest.mark.parametrize("precision", [Precision.FP64, Precision.FP32])
@pytest.mark.parametrize("ncat", [1, 4])
def test_gradient_with_an_impossible_tree(precision, variant, ncat):
    print("impossible tree", precision, variant, ncat, flush=True)
    net = parse_newick(NEWICK)
    net.brlen = np.where(net.brlen <= 1e-6, 0.0, net.brlen)  # (the reader's lower limit)
    assert (net.brlen == 0.0).sum() == 3
    rng = np.random.default_rng(5)
    masks = np.where(rng.integers(0, 2, (4, 90)) == 1, G, T).astype(np.uint32)
    a, b = (net.tip_labels.index(x) for x in "AB")
    assert (masks[a] != masks[b]).sum() > 2
    parts = [Partition(Model(4, np.array([1.0, 0, 0, 0, 0, 1.0]), np.array([0.5, 0.25, 0.125, 0.125]), 0.8, ncat),
                       masks, np.ones(90, np.uint32))]
    opt = dict(likelihood_variant=LikelihoodVariant(variant), precision=precision, brlen_min=0.0)
    ann = AnnotatedNetwork(net.copy(), parts, NetraxOptions(**opt))
    lnl, db, dp = ann.gradient()
    trees, _ = ann.tree_logls()
    assert np.isneginf(trees).sum() == 1  # the first tree
    want, g, gp = O.gradient(net, parts, variant, min_tree_logprob=math.log(0.5))  # the second tree alone
    tol = 1e-9 if precision == Precision.FP64 else 1e-6
    assert abs(lnl - want) <= tol * abs(want)
    tol = 1e-8 if precision == Precision.FP64 else 1e-4
    np.testing.assert_allclose(db, g, rtol=0, atol=tol * max(1.0, np.abs(g).max()))
    np.testing.assert_allclose(dp, gp, rtol=0, atol=tol * max(1.0, np.abs(gp).max()))
    if precision == Precision.FP64:
        _, m = ann.model_gradient()
        assert all(np.isfinite(x).all() for x in m[0].values())
    ann.close()
