"""The 4-state walks at the edges of their shapes: 1, 2, 4 and 8 rate
categories, few and many sites (one, two and four granules per wave in FP64,
one and two row blocks in FP32), ragged partitions, and rescaled sites (a
deep network with long branches: every site likelihood is below 2^-256).
lnL and gradient against the oracle in both variants; 1e-9 of the value and
1e-7 of the largest derivative in FP64, 1e-6 and 1e-4 in FP32, the bars of the
parity tests."""
import sys

import numpy as np
import pytest

from netrax_amd import AnnotatedNetwork, LikelihoodVariant, NetraxOptions, NetworkBatch, Precision
from netrax_amd.network import random_network
from netrax_amd.simulate import Model, Partition
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _parts(net, ncat, sizes, rng):
    parts = []
    for n in sizes:
        model = Model(4, rng.dirichlet(np.full(6, 2.0)) * 6, rng.dirichlet(np.full(4, 5.0)), 0.7, ncat)
        masks = np.uint32(1) << rng.integers(0, 4, (net.n_tips, n)).astype(np.uint32)
        masks[rng.random(masks.shape) < 0.05] = 15
        parts.append(Partition(model, masks, rng.integers(1, 4, n).astype(np.uint32)))
    return parts


def _against_oracle(net, parts, variant, shape=None):
    ann = AnnotatedNetwork(net, parts, NetraxOptions(likelihood_variant=LikelihoodVariant(variant),
                                                     precision=Precision.FP32 if shape else Precision.FP64))
    if shape:
        ann.set_tuning(*shape)
    tol, gtol = (1e-6, 1e-4) if shape else (1e-9, 1e-7)
    lnl, db, dp = ann.gradient()
    ol, odb, odp = O.gradient(net, parts, variant)
    assert abs(lnl - ol) <= tol * abs(ol), (lnl, ol)
    assert abs(ann.loglikelihood() - ol) <= tol * abs(ol)
    np.testing.assert_allclose(db, odb, rtol=0, atol=gtol * np.abs(odb).max())
    np.testing.assert_allclose(dp, odp, rtol=0, atol=gtol * max(1.0, np.abs(odp).max(initial=0.0)))
    ann.close()


@pytest.mark.parametrize("ncat,sizes", [(1, (1, 63)), (1, (30000, 36001)), (2, (65, 129)), (2, (33000,)), (4, (5, 64)),
                                        (4, (8300,)), (4, (16500, 77)), (8, (3, 130)), (8, (4200,))])
@pytest.mark.parametrize("variant", [0, 1])
def test_walk_shapes(ncat, sizes, variant):
    print("walk", ncat, sizes, variant, flush=True)
    sys.stdout.flush()
    rng = np.random.default_rng(1000 * ncat + len(sizes))
    net = random_network(9, 2, rng)
    net.brlen = rng.exponential(0.1, net.n_edges) + 1e-6
    net.retic_prob = rng.uniform(0.2, 0.8, net.n_retic)
    _against_oracle(net, _parts(net, ncat, sizes, rng), variant)


@pytest.mark.parametrize("ncat,n", [(1, 66000), (2, 33000), (4, 100), (4, 16500), (8, 4200)])
def test_walk_rescales(ncat, n):
    print("rescale", ncat, n, flush=True)
    rng = np.random.default_rng(ncat)
    net = random_network(200, 1, rng)
    net.brlen = rng.uniform(0.5, 5.0, net.n_edges)
    net.retic_prob = np.array([0.4])
    parts = _parts(net, ncat, (n,), rng)
    for p in parts:  # a few patterns repeated: the oracle's cost is in the patterns
        p.masks[:, 300:] = p.masks[:, rng.integers(0, min(300, n), max(0, n - 300))]
    _against_oracle(net, parts, 0)


@pytest.mark.parametrize("ncat,sizes", [(1, (1, 63)), (2, (65, 129)), (4, (5, 64, 1300)), (8, (3, 130))])
@pytest.mark.parametrize("shape", [(2, 64, 1), (3, 64, 1)])
@pytest.mark.parametrize("variant", [0, 1])
def test_fp32_walk_shapes(ncat, sizes, shape, variant):
    print("fp32 walk", ncat, sizes, shape, variant, flush=True)
    rng = np.random.default_rng(2000 * ncat)
    net = random_network(9, 2, rng)
    net.brlen = rng.exponential(0.1, net.n_edges) + 1e-6
    net.retic_prob = rng.uniform(0.2, 0.8, net.n_retic)
    _against_oracle(net, _parts(net, ncat, sizes, rng), variant, shape)


@pytest.mark.parametrize("ncat", [1, 2, 4, 8])
@pytest.mark.parametrize("shape", [(2, 64, 1), (3, 64, 1)])
def test_fp32_walk_underflow(ncat, shape):
    print("fp32 underflow", ncat, shape, flush=True)
    rng = np.random.default_rng(30 + ncat)
    net = random_network(50 if ncat == 8 else 100, 1, rng)
    net.brlen = rng.uniform(0.5, 5.0, net.n_edges)
    net.retic_prob = np.array([0.4])
    _against_oracle(net, _parts(net, ncat, (200,), rng), 0, shape)


def test_batch_changes_the_wave_shape_of_its_engines():
    """A batch that fills the GPU takes two row blocks per wave, its engines
    alone one: scored alone, in the batch, and alone again after one branch
    moved (an incremental evaluation), against the oracle."""
    rng = np.random.default_rng(9)
    nets, anns = [], []
    for n in (30000, 36500):
        net = random_network(8, 2, rng)
        net.brlen = rng.exponential(0.1, net.n_edges) + 1e-6
        net.retic_prob = rng.uniform(0.2, 0.8, net.n_retic)
        nets.append((net, _parts(net, 4, (n,), rng)))
        anns.append(AnnotatedNetwork(*nets[-1], NetraxOptions(precision=Precision.FP32)))
    alone = [a.gradient() for a in anns]
    batch = NetworkBatch(anns)
    lnl, dbs, _, _ = batch.evaluate(0)
    for (net, parts), a, one, l, db in zip(nets, anns, alone, lnl, dbs):
        ol, odb, _ = O.gradient(net, parts, 0)
        assert abs(l - ol) <= 1e-6 * abs(ol) and abs(one[0] - ol) <= 1e-6 * abs(ol), (l, one[0], ol)
        np.testing.assert_allclose(db, odb, rtol=0, atol=1e-4 * np.abs(odb).max())
        b = a.branch_lengths()
        b[3] *= 1.7
        a.set_branch_length(3, b[3])
        om = O.loglikelihood(net, parts, 0, brlen=b)[0]
        assert abs(a.loglikelihood() - om) <= 1e-6 * abs(om)
    batch.close()
