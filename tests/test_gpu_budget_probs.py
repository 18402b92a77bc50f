"""Reticulation probabilities that make more displayed trees count than the
memory budget has rows for are refused, and the refusal changes nothing: the
engine goes on with the probabilities and the plan that it had."""
import math
import re

import numpy as np
import pytest

from netrax_amd import AnnotatedNetwork, NetraxOptions, Precision, _lib
from netrax_amd.simulate import make_workload

pytestmark = pytest.mark.gpu


def test_refused_probabilities_change_nothing():
    w = make_workload("budget", 12, 2, [300], seed=5)
    few, many = np.full(2, 0.9), np.full(2, 0.5)
    anns = [AnnotatedNetwork(w.network.copy(), w.partitions,
                             NetraxOptions(precision=Precision.FP64, min_interesting_tree_logprob=math.log(0.2)))
            for _ in range(2)]
    smallest = []
    for probs in (many, few):  # 4 trees of 0.25 count; of 0.81, 0.09, 0.09 and 0.01 the first
        anns[0].set_reticulation_probs(probs)
        with pytest.raises(_lib.NrxError) as ex:
            anns[0].set_memory_budget(1)
        smallest.append(int(re.search(r"\((\d+) bytes\)", str(ex.value)).group(1)))
    assert smallest[1] < smallest[0]
    a, ref = anns
    ref.set_reticulation_probs(few)
    a.set_memory_budget(smallest[1])
    plan = a.memory_plan()
    assert plan["segments"] >= 2
    for fresh in (True, False):  # refused before and after an evaluation
        with pytest.raises(_lib.NrxError) as ex:
            a.set_reticulation_probs(many)
        assert ex.value.code == _lib.NRX_ERR_ARG
        assert a.memory_plan() == plan
        print("refused", fresh, flush=True)
        lnl, db, dp = a.gradient()
        want, db_want, dp_want = ref.gradient()
        assert lnl == want and a.loglikelihood() == want
        np.testing.assert_array_equal(db, db_want)
        np.testing.assert_array_equal(dp, dp_want)
    # and the next ones are taken
    a.set_memory_budget(0)
    for e in (a, ref):
        e.set_reticulation_probs(many)
    assert a.loglikelihood() == ref.loglikelihood()
    for e in anns:
        e.close()
