"""Device blocks kept between handles (awk_mem.hip): a handle made on another's
released blocks, whatever they hold, gives the results of the first one, on one thread
and on several with streams of their own."""
import threading

import numpy as np
import pytest

from atlaswerks_amd import synth

pytestmark = pytest.mark.gpu


def _pair(shape, seed):
    import torch
    t, _, _ = synth.pair(shape, seed=seed)
    s, _, _ = synth.pair(shape, seed=seed + 100)
    return torch.from_numpy(t).cuda(), torch.from_numpy(s).cuda()


def _greedy(I0, I1):
    import torch
    from atlaswerks_amd.greedy import GreedyWarp
    w = GreedyWarp(I0, I1, scale_levels=[(2, 4), (1, 3)])
    d = w.RunWarp(torch.cuda.current_stream())
    return np.concatenate([d.Def1To0.cpu().numpy().ravel(), np.concatenate(w.energy_history), w.step_history])


def _ldmm(I0, I1):
    from atlaswerks_amd.ldmm import LDMMWarp
    w = LDMMWarp(I0, I1, n_time_steps=3, n_iter=2)
    d = w.RunWarp()
    return np.concatenate([d.v.cpu().numpy().ravel(), d.energies().ravel()])


@pytest.mark.filterwarnings("ignore::RuntimeWarning")
@pytest.mark.parametrize("shape", [(20, 24, 28), (34, 31, 37)])
@pytest.mark.parametrize("kind", ["greedy", "ldmm"])
def test_handles_on_used_blocks(kind, shape):
    from atlaswerks_amd import _lib
    print("mem", kind, shape, flush=True)
    f = _greedy if kind == "greedy" else _ldmm
    I0, I1 = _pair(shape, 1)
    first = f(I0, I1)
    bad = I0.clone()
    bad[:] = float("nan")  # every buffer of these handles ends up with NaN
    try:
        f(bad, bad)
    except _lib.NumericalError:
        pass
    np.testing.assert_array_equal(f(I0, I1), first)


def test_threads_and_streams():
    import torch
    print("mem threads", flush=True)
    shapes = [(20, 24, 28), (24, 24, 24), (20, 24, 28), (18, 30, 26)]
    pairs = [_pair(s, k) for k, s in enumerate(shapes)]
    ref = [_greedy(*p) for p in pairs]
    torch.cuda.synchronize()
    got = [[] for _ in shapes]

    def work(k):
        st = torch.cuda.Stream()
        with torch.cuda.stream(st):
            for _ in range(4):
                got[k].append(_greedy(*pairs[k]))

    ts = [threading.Thread(target=work, args=(k,)) for k in range(len(shapes))]
    [t.start() for t in ts]
    [t.join(60) for t in ts]
    for k in range(len(shapes)):
        assert len(got[k]) == 4
        for g in got[k]:
            np.testing.assert_array_equal(g, ref[k])
