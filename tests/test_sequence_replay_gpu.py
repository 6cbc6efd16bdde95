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
    n, replays = 1 << 14, 200
    make = lambda v: torch.full((n,), v, dtype=torch.float32, device="cuda")  # noqa: E731
    key = rt.resolve(f"add?count={n}&dtype=f32")
    zero, scratch = rt.wrap(make(0.0)), rt.wrap(make(0.0))
    # every replay has an output of its own, so a wrong one stays to be seen
    outs = torch.zeros((2, replays, n), dtype=torch.float32, device="cuda")
    seqs = []
    for i, value in enumerate((1.0, 100.0)):
        first = rt.prepare(key, [rt.wrap(make(value)), zero], [scratch])
        seqs.append([rt.sequence([first, rt.prepare(key, [scratch, zero], [rt.wrap(o)])])
                     for o in outs[i]])
    torch.cuda.synchronize()
    start = threading.Barrier(2)

    def work(i):
        start.wait()
        for seq in seqs[i]:
            seq.launch()

    _run_threads([lambda i=i: work(i) for i in range(2)])
    torch.cuda.synchronize()
    assert bool((outs[0] == 1.0).all()), "the second thread's scratch reached the first's outputs"
    assert bool((outs[1] == 100.0).all()), "the first thread's scratch reached the second's outputs"


def _two_writes(tmc, rt, torch, pairs, n=1 << 14):
    """A sequence of `pairs` times a kernel that stores 2 and one that stores
    100 into one buffer, which holds 100 before and after a replay."""
    make = lambda v: torch.full((n,), v, dtype=torch.float32, device="cuda")  # noqa: E731
    key = rt.resolve(f"add?count={n}&dtype=f32")
    zero, out = rt.wrap(make(0.0)), make(100.0)
    buf = rt.wrap(out)
    steps = [rt.prepare(key, [rt.wrap(make(v)), zero], [buf]) for v in (2.0, 100.0)]
    torch.cuda.synchronize()
    return buf, rt.sequence(steps * pairs)


def _run_threads(bodies):
    threads = [threading.Thread(target=b) for b in bodies]
    for t in threads:
        t.start()
    for t in threads:
        t.join()


@pytest.mark.parametrize("steps", [1, 2, 6, 7])
def test_an_unread_error_of_the_thread_is_not_the_replays(tmc, steps):
    """A HIP call that the program itself made and that failed (a device that
    does not exist), its error not yet read, does not stop a replay."""
    import ctypes
    import torch
    rt = tmc.Runtime()
    bufs, seq, _ = _chain(tmc, rt, torch, steps)
    path = next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line)
    hip = ctypes.CDLL(path)
    bufs[0].fill_(1.5)
    torch.cuda.synchronize()
    try:
        assert hip.hipSetDevice(9999) != 0
        seq.launch()
    finally:
        hip.hipGetLastError()
    torch.cuda.synchronize()
    rt_done = rt.wrap(bufs[-1]).read()  # after the replay, on its stream
    assert bool((rt_done == 1.5 * 2.0 ** steps).all())


@pytest.mark.parametrize("pairs", [1, 3, 5])
def test_a_read_sees_whole_replays(tmc, pairs):
    """A buffer read from another thread falls before or after a replay."""
    import torch
    rt = tmc.Runtime()
    buf, seq = _two_writes(tmc, rt, torch, pairs)
    done, seen = threading.Event(), set()

    def launch():
        for _ in range(3000):
            seq.launch()
        done.set()

    def read():
        while not done.is_set():
            seen.update(set(buf.read_raw().tolist()))

    _run_threads([launch, read])
    torch.cuda.synchronize()
    assert seen == {100.0}, seen
