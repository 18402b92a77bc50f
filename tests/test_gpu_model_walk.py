"""The model gradient's sums formed inside the reverse walk, at the edges of
the walk's shapes: 1, 2, 4 and 8 rate categories, one, two and four granules
per wave, ragged partitions.  Per partition: the central difference of the
oracle's lnL in one exchangeability and one frequency (2e-6 of the largest
entry, the bar of the model gradient tests); per network: scaling all category
rates equals scaling all branch lengths, to 1e-8."""
import dataclasses

import numpy as np
import pytest

from netrax_amd import AnnotatedNetwork, LikelihoodVariant, NetraxOptions
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


def _difference(net, parts, variant, p, field, i):
    h, vals = 1e-5, []
    for sign in (1, -1):
        m = dataclasses.replace(parts[p].model, subst_rates=parts[p].model.subst_rates.copy(),
                                freqs=parts[p].model.freqs.copy())
        getattr(m, field)[i] += sign * h
        ps = [dataclasses.replace(q, model=m) if k == p else q for k, q in enumerate(parts)]
        vals.append(O.loglikelihood(net, ps, variant)[0])
    return (vals[0] - vals[1]) / (2 * h)


@pytest.mark.parametrize("ncat,sizes", [(1, (1, 63)), (1, (33000, 33001)), (2, (65, 129)), (2, (33000,)), (4, (5, 64)),
                                        (4, (8300,)), (4, (16500, 77)), (8, (3, 130)), (8, (4200,))])
@pytest.mark.parametrize("variant", [0, 1])
def test_model_gradient_shapes(ncat, sizes, variant):
    print("model walk", ncat, sizes, variant, flush=True)
    rng = np.random.default_rng(4000 * ncat + len(sizes))
    net = random_network(7, 1, rng)
    net.brlen = rng.exponential(0.1, net.n_edges) + 1e-3
    net.retic_prob = rng.uniform(0.3, 0.7, net.n_retic)
    parts = _parts(net, ncat, sizes, rng)
    ann = AnnotatedNetwork(net, parts, NetraxOptions(likelihood_variant=LikelihoodVariant(variant)))
    lnl, grads = ann.model_gradient()
    want, db, _ = O.gradient(net, parts, variant)
    assert abs(lnl - want) <= 1e-9 * abs(want)
    by_rates = sum(float(np.dot(O.gamma_rates(q.model.alpha, ncat), g["rates"])) for q, g in zip(parts, grads))
    by_lengths = float(np.dot(net.brlen, db))
    assert abs(by_rates - by_lengths) <= 1e-8 * max(1.0, abs(by_lengths)), (by_rates, by_lengths)
    for p, g in enumerate(grads):
        for field, key, i in (("subst_rates", "subst", 1), ("freqs", "freqs", 2)):
            fd = _difference(net, parts, variant, p, field, i)
            assert abs(g[key][i] - fd) <= 2e-6 * max(1.0, np.abs(g[key]).max()), (p, field, g[key][i], fd)
    ann.close()
