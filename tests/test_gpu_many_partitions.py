"""Engines of many partitions, past the limits up to which the P kernels read
the lengths in the host's memory (4,096 waves of P entries) and the last
kernels write the results there (16,384 doubles): both precisions, eager and
from graphs, replayed with the lengths moved, against the oracle."""
import numpy as np
import pytest

from netrax_amd import AnnotatedNetwork, NetraxOptions, Precision
from netrax_amd.network import random_network
from netrax_amd.simulate import Partition, random_dna_model
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def case(taxa, retic, n_parts, ncat, seed):
    rng = np.random.default_rng(seed)
    net = random_network(taxa, retic, rng)
    parts = []
    for _ in range(n_parts):
        n = int(rng.integers(1, 24))
        masks = np.uint32(1) << rng.integers(0, 4, (taxa, n)).astype(np.uint32)
        parts.append(Partition(random_dna_model(rng, ncat), masks, rng.integers(1, 4, n).astype(np.uint32)))
    return net, parts


# (100 taxa, 4 reticulations: 214 edges, 16 trees: 20,000 results)
@pytest.mark.parametrize("taxa,retic", [(38, 1), (100, 4)])
@pytest.mark.parametrize("precision,use_graph", [(Precision.FP64, False), (Precision.FP32, False), (Precision.FP32, True)])
def test_many_partitions(taxa, retic, precision, use_graph):
    print("many partitions", taxa, retic, precision, use_graph, flush=True)
    net, parts = case(taxa, retic, 64, 4, seed=taxa)
    assert 64 * net.n_edges * 4 * 16 > 64 * 4096
    opt = NetraxOptions(precision=precision, use_graph=use_graph, min_interesting_tree_logprob=-1e9)
    ann = AnnotatedNetwork(net.copy(), parts, opt)
    tol = 1e-9 if precision == Precision.FP64 else 1e-6
    for step in range(4):  # (graphs: replays with the program's own work between them)
        b = net.brlen * (1.0 + 0.2 * step)
        ann.set_branch_lengths(b)
        want, per = O.loglikelihood(net, parts, brlen=b, min_tree_logprob=-1e9)
        if step % 2:
            lnl = ann.loglikelihood(0)
        else:
            lnl, db, dp, pdb = ann.gradient(per_partition=True)
            _, g, gp, pg = O.gradient(net, parts, brlen=b, min_tree_logprob=-1e9, per_partition=True)
            gtol = (1e-7 if precision == Precision.FP64 else 1e-4) * max(1.0, np.abs(g).max())
            for x, y in ((db, g), (dp, gp), (pdb, pg)):
                np.testing.assert_allclose(x, y, rtol=0, atol=gtol)
            lnl2 = ann.loglikelihood(0)
            assert abs(lnl2 - lnl) <= 1e-12 * abs(lnl)
        assert abs(lnl - want) <= tol * abs(want), (step, lnl, want)
        np.testing.assert_allclose(ann.partition_loglh, per, rtol=10 * tol, atol=1e-6)
    ann.close()


@pytest.mark.parametrize("retic", [0, 1, 2, 3, 5, 7])
@pytest.mark.parametrize("n_parts", [1, 3, 64])
@pytest.mark.parametrize("variant", [0, 1])
def test_mixture_shapes(n_parts, retic, variant):
    """The mixture's groups of lanes: 1 to 64 partitions of 1 to 128 trees, root
    sums formed in its workgroup (few rows and partials) and before it."""
    print("mixture", n_parts, retic, variant, flush=True)
    net, parts = case(9, retic, n_parts, 2, seed=100 + retic)
    ann = AnnotatedNetwork(net.copy(), parts, NetraxOptions(min_interesting_tree_logprob=-1e9))
    lnl = ann.loglikelihood(0, variant=variant)
    want, per, trees, _ = O.loglikelihood(net, parts, variant, min_tree_logprob=-1e9, tree_logls=True)
    assert abs(lnl - want) <= 1e-9 * abs(want)
    np.testing.assert_allclose(ann.partition_loglh, per, rtol=1e-9, atol=1e-9)
    got, _ = ann.tree_logls()
    np.testing.assert_allclose(np.sort(got, axis=1), np.sort(trees, axis=1), rtol=1e-9, atol=1e-9)
    _, db, dp = ann.gradient(variant=variant)
    _, g, gp = O.gradient(net, parts, variant, min_tree_logprob=-1e9)
    np.testing.assert_allclose(db, g, rtol=0, atol=1e-7 * max(1.0, np.abs(g).max()))
    np.testing.assert_allclose(dp, gp, rtol=0, atol=1e-7 * max(1.0, np.abs(gp).max(initial=0.0)))
    ann.close()
