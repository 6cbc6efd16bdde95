"""Sequences replayed as launches (few kernels) and as graphs: the same results,
later input values seen, and whole sequences kept in order between threads."""
import threading

import pytest

pytestmark = pytest.mark.gpu


def _chain(tmc, rt, torch, steps, n=4096):
    """y = 2^steps x by `steps` element-wise additions."""
    bufs = [torch.zeros(n, dtype=torch.float32, device="cuda") for _ in range(steps + 1)]
    key = rt.resolve(f"add?count={n}&dtype=f32")
    w = [rt.wrap(b) for b in bufs]
    twin = [rt.wrap(b) for b in bufs]
    execs = [rt.prepare(key, [w[i], twin[i]], [w[i + 1]]) for i in range(steps)]
    torch.cuda.synchronize()
    return bufs, rt.sequence(execs), execs


@pytest.mark.parametrize("steps", [1, 6, 7, 20])
def test_replays_see_later_inputs(tmc, steps):
    import torch
    rt = tmc.Runtime()
    bufs, seq, _ = _chain(tmc, rt, torch, steps)
    for value in (1.0, -3.0, 0.5):
        bufs[0].fill_(value)
        torch.cuda.synchronize()
        seq.launch()
        seq.run()
        torch.cuda.synchronize()
        assert bool((bufs[-1] == value * 2.0 ** steps).all())


def test_sequences_of_two_threads_do_not_interleave(tmc):
    """Two sequences through one scratch buffer, launched from two threads on
    one runtime: each output comes from its own input."""
    import torch
    rt = tmc.Runtime()
    n = 1 << 16
    make = lambda v: torch.full((n,), v, dtype=torch.float32, device="cuda")  # noqa: E731
    a, b, scratch, oa, ob = make(1.0), make(100.0), make(0.0), make(0.0), make(0.0)
    key = rt.resolve(f"add?count={n}&dtype=f32")
    wrap = {id(t): rt.wrap(t) for t in (a, b, scratch, oa, ob)}
    zero = rt.wrap(make(0.0))
    w = lambda t: wrap[id(t)]  # noqa: E731
    seqs = []
    for src, dst in ((a, oa), (b, ob)):
        seqs.append(rt.sequence([rt.prepare(key, [w(src), zero], [w(scratch)]),
                                 rt.prepare(key, [w(scratch), zero], [w(dst)])]))
    torch.cuda.synchronize()
    bad = []

    def work(i):
        for _ in range(300):
            seqs[i].launch()

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    if not bool((oa == 1.0).all()):
        bad.append("first")
    if not bool((ob == 100.0).all()):
        bad.append("second")
    assert not bad
