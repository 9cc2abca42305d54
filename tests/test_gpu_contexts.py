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


def _eager_and_graphs(h, s, prompt, hidden):
    """What a context gives through eager layers, a captured layer range, the token graph and one run of tokens."""
    out = np.empty(s.dim, np.float32)
    assert h.ResetKV() == 0
    rc, t = h.Generate(prompt, 12, useGraph=True)
    assert rc == 0, E.last_error()
    assert h.PartialStep(hidden, 3, 0, 1, out, None) == 0, E.last_error()
    assert h.CaptureTokenGraph() == 0, E.last_error()
    rc, nxt = h.GraphLaunch(int(t[-1]), len(prompt) + 11)
    assert rc == 0, E.last_error()
    g = h.CaptureGraph(E.GraphCaptureConfig(LayerStart=0, LayerEnd=s.nLayers), 0)
    assert g is not None, E.last_error()
    assert h.UploadHidden(hidden) == 0 and g.Launch(5) == 0, E.last_error()
    deep = h.ReadHidden()
    assert deep is not None, E.last_error()
    g.Destroy()
    return t.tolist() + [nxt], out, deep.copy()


def _same(a, b):
    return a[0] == b[0] and np.array_equal(a[1], b[1]) and np.array_equal(a[2], b[2])


def test_steps_captures_and_mode_changes_between_turns(hip):
    """Two contexts in turn through every kind of call, one of them leaving the launch (mode 1) and coming back: each gives
    what it gave alone in that mode."""
    s = H.with_layers(configs.TOY, 2)
    a, b = (H.Model(s, seed=70 + i, maxSeq=64, eng=hip, oracle=False) for i in range(2))
    pa, pb, hid = a.prompt(6), b.prompt(7), E.synth_normal(70, 1, 1.0, (s.dim,))
    want = {}
    for mode in (1, 3):
        assert a.hip.SetExecMode(mode) == 0
        want[mode] = _eager_and_graphs(a.hip, s, pa, hid)
    wb = _eager_and_graphs(b.hip, s, pb, hid)
    for mode in (3, 1, 1, 3, 3):
        assert a.hip.SetExecMode(mode) == 0
        assert _same(_eager_and_graphs(a.hip, s, pa, hid), want[mode])
        assert _same(_eager_and_graphs(b.hip, s, pb, hid), wb)
    a.close()
    b.close()


def test_a_context_that_left_the_launch_captures_while_another_takes_the_turn(hip):
    """One context launches last, changes to mode 1 and captures graphs while another one's thread decodes: the other's turn
    is not to reach into the capture, on either side."""
    s = H.with_layers(configs.TOY, 2)
    a, b = (H.Model(s, seed=80 + i, maxSeq=64, eng=hip, oracle=False) for i in range(2))
    pa, pb, hid = a.prompt(6), b.prompt(7), E.synth_normal(80, 1, 1.0, (s.dim,))
    assert a.hip.SetExecMode(1) == 0
    want = _eager_and_graphs(a.hip, s, pa, hid)
    rc, wb = b.hip.Generate(pb, 20)
    assert rc == 0, E.last_error()
    stop, bad = threading.Event(), []

    def decode():
        while not stop.is_set():
            rc, t = b.hip.Generate(pb, 20)
            if rc != 0 or t.tolist() != wb.tolist():
                bad.append((rc, E.last_error()))
                return

    th = threading.Thread(target=decode)
    th.start()
    try:
        for _ in range(15):
            assert a.hip.SetExecMode(3) == 0
            rc, _ = a.hip.DecodeToken(int(pa[0]), 0)          # the launch's last user for now
            assert rc == 0, E.last_error()
            assert a.hip.SetExecMode(1) == 0
            assert _same(_eager_and_graphs(a.hip, s, pa, hid), want)
    finally:
        stop.set()
        th.join()
    assert not bad, bad
    a.close()
    b.close()
