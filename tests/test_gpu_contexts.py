"""Several contexts on one device: their persistent launches take turns."""
import threading

import numpy as np
import pytest

from mongoose_amd import configs
from mongoose_amd import engine as E
from tests import helpers as H

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    eng = E.NewHIP(0)
    assert eng is not None, "no HIP device"
    return eng


@pytest.mark.parametrize("per_launch", [64, 1])
def test_contexts_take_turns(hip, per_launch):
    """Three contexts, all through the persistent launch (runs of tokens in a launch; graph replays of one token): what each
    generates alone it also generates between the others' calls and from threads of their own."""
    s = H.with_layers(configs.TOY, 2)
    ms = [H.Model(s, seed=50 + i, maxSeq=80, eng=hip, oracle=False) for i in range(3)]
    prompts = [m.prompt(5) for m in ms]
    for m in ms:
        assert m.hip.SetTokensPerLaunch(per_launch) == 0
    alone = []
    for m, p in zip(ms, prompts):
        rc, t = m.hip.Generate(p, 60, useGraph=True)
        assert rc == 0, E.last_error()
        assert m.hip.FlowTailInUse()
        alone.append(t.copy())
    for _ in range(4):
        for m, p, a in zip(ms, prompts, alone):
            rc, t = m.hip.Generate(p, 60, useGraph=True)
            assert rc == 0 and (t == a).all(), E.last_error()
    got = [[] for _ in ms]

    def work(i):
        for _ in range(6):
            got[i].append(ms[i].hip.Generate(prompts[i], 60, useGraph=True))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for g, a in zip(got, alone):
        assert len(g) == 6
        for rc, t in g:
            assert rc == 0 and (t == a).all()
    assert all(m.hip.FlowTailInUse() for m in ms) and [m.hip.FlowInUse() for m in ms] == [True, False, False]
    ms[1].close()                                            # one leaves, the others go on
    rc, t = ms[0].hip.Generate(prompts[0], 60, useGraph=True)
    assert rc == 0 and (np.asarray(t) == alone[0]).all()
    ms[0].close()
    ms[2].close()
