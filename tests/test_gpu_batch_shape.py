"""A batch's launch has a wave shape of its own (two row blocks per wave and
fewer LDS slots than its engines alone): the engines keep theirs, so that an
engine alone computes and is counted as before the batch, while the batch
lives and after it, and each side can go on from the CLVs and root sums that
the other left."""
import numpy as np
import pytest

from netrax_amd import AnnotatedNetwork, NetraxOptions, NetworkBatch, Precision, _lib
from netrax_amd.network import random_network
from netrax_amd.simulate import Partition, random_dna_model

pytestmark = pytest.mark.gpu


def engines(sizes, ncat=4, use_graph=False):
    out = []
    for i, n in enumerate(sizes):
        rng = np.random.default_rng(31 + i)
        net = random_network(24 + 3 * i, 2, rng)
        masks = np.uint32(1) << rng.integers(0, 4, (net.n_tips, n)).astype(np.uint32)
        out.append(AnnotatedNetwork(net, [Partition(random_dna_model(rng, ncat), masks, np.ones(n, np.uint32))],
                                    NetraxOptions(precision=Precision.FP32, use_graph=use_graph)))
    return out


@pytest.mark.parametrize("use_graph", [False, True])
@pytest.mark.parametrize("ncat,size", [(2, 48000), (4, 24000), (8, 12000)])
def test_engines_keep_their_shape(ncat, size, use_graph):
    print("batch shape", ncat, size, use_graph, flush=True)
    anns = engines([size, size - 77, size + 130], ncat, use_graph)  # 4,500 blocks: two per wave, alone one
    solo = [a.gradient(per_partition=True) for a in anns]
    handoffs = [a.stats().n_lds_handoffs for a in anns]
    batch = NetworkBatch(anns)
    lnl, dbs, _, _ = batch.evaluate(0)
    for again in range(2):
        for i, a in enumerate(anns):
            # alone on the CLVs and root sums that the batch left
            assert a.loglikelihood() == solo[i][0] == lnl[i]
            np.testing.assert_allclose(dbs[i], solo[i][1], rtol=0, atol=1e-6 * np.abs(solo[i][1]).max())
            got = a.gradient(per_partition=True)
            for x, y in zip(got, solo[i]):
                np.testing.assert_array_equal(x, y)
            # a part of the CLVs recomputed on the batch's, and the batch again
            e = int(a.network.n_edges // 2)
            b = a.network.brlen.copy()
            a.set_branch_length(e, 1.5 * b[e])
            moved = a.loglikelihood()
            assert moved == a.loglikelihood(0)
            a.set_branch_lengths(b)
        if not again:
            lnl, dbs, _, _ = batch.evaluate(0)
            assert [a.stats().n_lds_handoffs for a in anns] <= handoffs
            batch.close()
    assert [a.stats().n_lds_handoffs for a in anns] == handoffs
    for a in anns:
        a.close()


def test_two_batches_share_an_engine():
    print("two batches", flush=True)
    anns = engines([24000, 23000, 25000, 700])
    big, small = NetworkBatch(anns[:3]), NetworkBatch([anns[0], anns[3]])
    l0, g0, _, _ = big.evaluate(0)
    l1, g1, _, _ = small.evaluate(0)
    for _ in range(2):
        la, ga, _, _ = big.evaluate(0)
        lb, gb, _, _ = small.evaluate(0)
        np.testing.assert_array_equal(la, l0)
        np.testing.assert_array_equal(lb, l1)
        for x, y in zip(ga + gb, g0 + g1):
            np.testing.assert_array_equal(x, y)
    assert l0[0] == l1[0] == anns[0].loglikelihood(0)
    anns[0].close()  # an engine may go first; its batches are not used again
    small.close()
    big.close()
    for a in anns[1:]:
        a.close()


def test_refused_batch_leaves_the_engines_their_changes():
    """A batch that is refused (its engines' shapes differ by now) has not
    taken over the lengths set before: the engines alone evaluate at them."""
    print("refused batch", flush=True)
    anns = engines([300, 500])
    batch = NetworkBatch(anns)
    batch.evaluate(0)
    for a in anns:
        a.set_branch_lengths(a.network.brlen * 1.7)
    anns[1].set_tuning(3, 64, 1)
    with pytest.raises(_lib.NrxError):
        batch.evaluate(0)
    fresh = engines([300, 500])
    for a, f in zip(anns, fresh):
        f.set_branch_lengths(a.network.brlen)
        assert a.loglikelihood() == f.loglikelihood(0)
    # with one shape again it takes them
    anns[1].set_tuning(4, 64, 1)
    lnl, _, _, _ = batch.evaluate(0)
    assert [f.loglikelihood(0) for f in fresh] == list(lnl)
    batch.close()
    for a in anns + fresh:
        a.close()
