"""FP32 walks of one and of two 64-row blocks per wave form the same gradient:
each block's shares are summed in FP32 over its 64 rows, and from there on in
FP64, so that the number of blocks (chosen by the size of the launch) changes
the order of an FP64 sum only."""
import numpy as np
import pytest

from netrax_amd import AnnotatedNetwork, NetraxOptions, Precision
from netrax_amd.network import random_network
from netrax_amd.simulate import Partition, random_dna_model, simulate_states, states_to_masks

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sites", [[64], [45, 130, 1001]])
@pytest.mark.parametrize("ncat", [2, 4, 8])
def test_gradient_does_not_depend_on_the_blocks_of_a_wave(ncat, sites):
    print("blocks", ncat, sites, flush=True)
    rng = np.random.default_rng(17 + ncat)
    net = random_network(14, 0, rng)  # a tree: the mixture's weights are exactly one
    parts = []
    for n in sites:
        model = random_dna_model(rng, ncat)
        parts.append(Partition(model, states_to_masks(simulate_states(net, model, n, rng)),
                               rng.integers(1, 9, n).astype(np.uint32)))
    ann = AnnotatedNetwork(net, parts, NetraxOptions(precision=Precision.FP32))
    got = {}
    for shape in ((3, 64, 1), (2, 64, 1)):
        ann.set_tuning(*shape)
        got[shape[0]] = ann.gradient(per_partition=True)
    one, two = got[3], got[2]
    assert abs(one[0] - two[0]) <= 1e-13 * abs(one[0])
    # FP64 sums of at most 2,000 terms: 2,000 x 2^-53 of the sum of their sizes,
    # which is within 100 of the largest derivative here
    for a, b in ((one[1], two[1]), (one[3], two[3])):
        np.testing.assert_allclose(a, b, rtol=0, atol=2000 * 2.0**-53 * 100 * np.abs(a).max())
    ann.close()
