"""Branch derivatives of both kinds (sumtables, and the variant without
allocations, which walks the paths anew) against the oracle at the edges of
their kernels: 4 and 20 states, 1, 2, 4 and 8 rate categories, partitions of
one site to a little more than a tile, ambiguous tips, and a network so deep
that sites are rescaled on the paths."""
import ctypes as C

import numpy as np
import pytest

from netrax_amd import AnnotatedNetwork, NetraxOptions, Precision, _lib
from netrax_amd.network import random_network
from netrax_amd.simulate import Partition, random_dna_model, random_protein_model
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def case(states, ncat, taxa, sizes, mean_length, seed):
    rng = np.random.default_rng(seed)
    net = random_network(taxa, 1, rng)
    net.brlen = rng.exponential(mean_length, net.n_edges) + 1e-3
    net.retic_prob = np.array([0.4])
    parts = []
    for n in sizes:
        masks = np.uint32(1) << rng.integers(0, states, (taxa, n)).astype(np.uint32)
        masks[rng.random(masks.shape) < 0.05] = (1 << states) - 1
        model = (random_dna_model if states == 4 else random_protein_model)(rng, ncat)
        parts.append(Partition(model, masks, rng.integers(1, 4, n).astype(np.uint32)))
    return net, parts


def check(ann, net, parts, edges, tol):
    lib = _lib.load()
    P = len(parts)
    ann.loglikelihood()
    for e in edges:
        b = float(net.brlen[e]) * 1.25
        d1, d2, p1, p2 = C.c_double(), C.c_double(), np.zeros(P), np.zeros(P)
        ptr = lambda x: x.ctypes.data_as(C.POINTER(C.c_double))
        lengths = net.brlen.copy()
        lengths[e] = b
        # each tree's share at the moved length, normalised at the present one
        want = O.brlen_derivatives(net, parts, e, 0, 1, brlen=lengths)
        for call in (lib.nrx_brlen_derivatives_noalloc, lib.nrx_brlen_derivatives):
            rc = call(ann.handle, 0, int(e), 1, C.c_double(b), C.byref(d1), C.byref(d2), ptr(p1), ptr(p2))
            assert rc == _lib.NRX_OK, lib.nrx_last_error()
            for got, w in ((d1.value, want[0]), (d2.value, want[1])):
                assert abs(got - w) <= tol * max(1.0, abs(w)), (e, got, w)
            np.testing.assert_allclose(p1, want[2], rtol=tol, atol=tol)
            np.testing.assert_allclose(p2, want[3], rtol=tol, atol=tol)


@pytest.mark.parametrize("ncat", [1, 2, 4, 8])
@pytest.mark.parametrize("states,precision", [(4, Precision.FP64), (4, Precision.FP32), (20, Precision.FP64)])
def test_shapes(states, precision, ncat):
    print("branch walks", states, precision, ncat, flush=True)
    net, parts = case(states, ncat, 9, (1, 17, 64, 131), 0.1, 70 + ncat)
    ann = AnnotatedNetwork(net.copy(), parts, NetraxOptions(precision=precision))
    check(ann, net, parts, range(0, net.n_edges, 3), 1e-8 if precision == Precision.FP64 else 2e-4)
    ann.close()


@pytest.mark.parametrize("ncat", [1, 2, 4, 8])
@pytest.mark.parametrize("states,taxa", [(4, 150), (20, 70)])
def test_rescaled_sites_on_the_path(states, taxa, ncat):
    print("rescaled branch walks", states, ncat, flush=True)
    net, parts = case(states, ncat, taxa, (70,), 1.0, 80 + ncat)
    ann = AnnotatedNetwork(net.copy(), parts, NetraxOptions())
    total = float(parts[0].weights.sum())
    assert ann.loglikelihood() / total < -256 * np.log(2.0)  # a site takes a rescaling on average
    check(ann, net, parts, range(0, net.n_edges, 23), 1e-8)
    ann.close()
