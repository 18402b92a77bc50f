"""The model gradient takes no memory that grows with the alignment beyond
what a gradient takes: its sums over sites stand in adjoint rows that the walk
is done with."""
import numpy as np
import pytest
import torch

from netrax_amd import AnnotatedNetwork, NetraxOptions
from netrax_amd.network import random_network
from netrax_amd.simulate import Partition, random_dna_model

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ncat,sites", [(1, 60000), (2, 30000), (4, 6000), (4, 30000), (8, 30000)])
def test_model_gradient_memory(ncat, sites):
    print("model memory", ncat, sites, flush=True)
    rng = np.random.default_rng(9)
    net = random_network(30, 2, rng)
    masks = np.uint32(1) << rng.integers(0, 4, (net.n_tips, sites)).astype(np.uint32)
    ann = AnnotatedNetwork(net, [Partition(random_dna_model(rng, ncat), masks, np.ones(sites, np.uint32))],
                           NetraxOptions())
    _, db, _ = ann.gradient()
    held = ann.stats().clv_bytes
    free = torch.cuda.mem_get_info()[0]
    ann.model_gradient()
    taken = free - torch.cuda.mem_get_info()[0]
    print("held", held, "taken", taken, flush=True)
    # its workspaces: 8 slices of 64 (128) sums per use, a few hundred uses, in
    # pieces of 2 MiB; the CLVs and adjoints are hundreds of MB
    assert taken <= 12 << 20
    # the adjoint rows serve the next gradient again
    np.testing.assert_array_equal(ann.gradient()[1], db)
    ann.close()
