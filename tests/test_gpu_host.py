"""The native twins of the small calls' entries (csrc/vq2_host.cpp) against
the Python entries they stand in for: the same launch, so bit-identical results
(given outputs take the Python entry), over types, strides of the batch and
one to four matrices; calls they decline raise what the Python entry raises;
each stream has its own workspace."""
import threading
import time

import pytest
import torch

from compressai_amd import _lib, kernels as K, synth
from compressai_amd.graph import DecodeStepGraph
from compressai_amd.kernels import Vq2Error
from compressai_amd.moe import ResidentMoEExperts

pytestmark = pytest.mark.gpu


def _mats(dev, seed, n, rows, bpw):
    ms = [synth.vq_matrix(seed + i, r, n, bpw=bpw) for i, r in enumerate(rows)]
    cb0 = synth.codebook(seed + 50).to(dev)
    cb1 = {2: None, 3: synth.codebook(seed + 51, rows=256), 4: synth.codebook(seed + 51)}[bpw]
    return ms, cb0, None if cb1 is None else cb1.to(dev)


def _tables(dev, n):
    return synth.permutation(8810, n).to(dev), synth.signs(8811, n).to(dev)


@pytest.mark.parametrize("n,rows,bpw,x_dtype,y_dtype", [
    (2048, (2048,), 2, torch.float16, torch.float16),           # one slice
    (2048, (6144, 6144), 4, torch.bfloat16, torch.bfloat16),    # slices: the stream's workspace
    (512, (96, 17, 1, 33), 3, torch.float32, torch.float32),
])
def test_sorted_gemv(dev, n, rows, bpw, x_dtype, y_dtype):
    ms, cb0, cb1 = _mats(dev, 8800, n, rows, bpw)
    mats = [(K.SortedPlanes(m["idx0"], m["idx1"], r, n, device=dev), m["scale"].to(dev)) for m, r in zip(ms, rows)]
    perm, sign = _tables(dev, n)
    x = synth.activations(8820, n, dtype=x_dtype).to(dev)
    for kw in (dict(hb=min(n, 2048)), dict(hb=0, rs=0.5), dict(hb=64, rht_scale=0.25)):
        p, s = (perm, sign) if kw["hb"] else (None, None)
        ref = K.vq_sorted_gemv(x, mats, cb0, cb1, n, p, s, ys=[torch.empty(r, dtype=y_dtype, device=dev) for r in rows], **kw)
        side = torch.cuda.Stream(dev)
        side.wait_stream(torch.cuda.current_stream(dev))
        with torch.cuda.stream(side):
            got = K.vq_sorted_gemv(x, mats, cb0, cb1, n, p, s, out_dtype=y_dtype, **kw)
        torch.cuda.synchronize(dev)
        assert len(got) == len(ref) and all(torch.equal(a, b) and a.dtype == y_dtype for a, b in zip(got, ref))


@pytest.mark.parametrize("fn,B", [("vq_gemv_rht", 1), ("vq_gemv_rht", 2), ("vq_rows_gemm", 3), ("vq_rows_gemm", 70)])
@pytest.mark.parametrize("bpw", [2, 3, 4])
def test_rotated_products(dev, fn, B, bpw):
    n, rows = 1024, (300, 77)
    ms, cb0, cb1 = _mats(dev, 8830, n, rows, bpw)
    mats = [(m["idx0"].to(dev), None if m["idx1"] is None else m["idx1"].to(dev), m["scale"].to(dev), r)
            for m, r in zip(ms, rows)]
    perm, sign = _tables(dev, n)
    x = synth.activations(8840, (B, n), dtype=torch.bfloat16).to(dev)
    call = getattr(K, fn)
    got = call(x, mats, cb0, cb1, n, perm, sign, 1024, out_dtype=torch.bfloat16)
    ref = call(x, mats, cb0, cb1, n, perm, sign, 1024,
               ys=[torch.empty(B, r, dtype=torch.bfloat16, device=dev) for r in rows])
    assert all(torch.equal(a, b) and a.shape == b.shape for a, b in zip(got, ref))


@pytest.mark.parametrize("T", [1, 5, 20])
def test_sorted_moe(dev, T):
    E, P = 12, 3
    gu, dn = synth.indices16(8850, (E, 1024, 256)).to(dev), synth.indices16(8851, (E, 2048, 64)).to(dev)
    gus, dns = synth.scales(8852, (E, 1024)).to(dev), synth.scales(8853, (E, 2048)).to(dev)
    mod = ResidentMoEExperts.from_pools(gu, gus, dn, dns, synth.codebook(8854).to(dev), sorted_layout=True)
    h = synth.activations(8855, (T, 2048)).to(dev)
    ids = torch.randint(0, E, (T, P), generator=synth.gen(8856)).to(dev)
    w = torch.rand(T, P, generator=synth.gen(8857)).to(dev)
    rh, ri = mod._rots()
    args = (h, mod.sorted_gu, gus, mod.sorted_dn, dns, mod.cb16, rh, ri)
    ref = K.vq_sorted_moe(*args, ids=ids, w=w, out=torch.empty(T, 2048, device=dev))
    assert torch.equal(K.vq_sorted_moe(*args, ids=ids, w=w), ref)
    lg = synth.activations(8858, (T, E - 1), dtype=torch.float32).to(dev)
    kw = dict(logits=lg, top_k=2, shared_id=E - 1, shared_gate=synth.activations(8859, 2048).to(dev))
    ref = K.vq_sorted_moe(*args, out=torch.empty(T, 2048, device=dev), **kw)
    assert all(torch.equal(a, b) for a, b in zip(K.vq_sorted_moe(*args, **kw), ref))


def test_other_threads_run_while_a_launch_waits(dev):
    """A launch waits while the GPU's queue is full; other Python threads go
    on meanwhile, as they do behind the Python entry's launch (the longest
    pause of a ticking thread against the longest launch: 605 of 600 ms with
    the interpreter lock held, 1 without)."""
    n, rows = 2048, 64
    ms, cb0, _ = _mats(dev, 8860, n, (rows,), 2)
    mats = [(ms[0]["idx0"].to(dev), None, ms[0]["scale"].to(dev), rows)]
    x = torch.zeros(1, n, dtype=torch.float16, device=dev)
    a = torch.zeros(8192, 8192, dtype=torch.bfloat16, device=dev)
    K.vq_gemv_rht(x, mats, cb0, None, n)
    torch.cuda.synchronize(dev)
    pause, stop = [0.0], threading.Event()

    def tick():
        last = time.perf_counter()
        while not stop.is_set():
            time.sleep(0.001)
            now = time.perf_counter()
            pause[0] = max(pause[0], now - last)
            last = now

    t = threading.Thread(target=tick)
    t.start()
    try:
        for _ in range(800):  # ~0.6 s of work, then more launches than the queue holds
            torch.mm(a, a)
        longest = 0.0
        for _ in range(20000):
            t0 = time.perf_counter()
            K.vq_gemv_rht(x, mats, cb0, None, n)
            longest = max(longest, time.perf_counter() - t0)
    finally:
        stop.set()
        t.join()
    torch.cuda.synchronize(dev)
    assert pause[0] < max(0.1, longest / 4), (pause[0], longest)


def test_declined_calls(dev):
    """What the native checks decline, the Python entry refuses or handles."""
    n = 512
    ms, cb0, _ = _mats(dev, 8870, n, (64,), 2)
    i0, sc = ms[0]["idx0"].to(dev), ms[0]["scale"].to(dev)
    x = torch.zeros(2, n, dtype=torch.float16, device=dev)
    sp = K.SortedPlanes(ms[0]["idx0"], None, 64, n, device=dev)
    host = _lib.host()
    bad = [dict(x=x.cpu()), dict(x=x[:, ::2]), dict(cb0=cb0[:100]), dict(perm=torch.zeros(n, dtype=torch.int64, device=dev)),
           dict(mats=[(i0, None, sc[:3], 64)]), dict(mats=[(i0, None, sc.cpu(), 64)]), dict(mats=[])]
    for b in bad:
        a = dict(x=x, mats=[(i0, None, sc, 64)], cb0=cb0, perm=None)
        a.update(b)
        args = (a["x"], a["mats"], a["cb0"], None, n, a["perm"], None, n)
        assert host.gemv_rht(*args, None, 1.0, torch.float32) is None, b
        assert host.rows_gemm(*args, None, 1.0, torch.float32, torch.float32) is None, b
        with pytest.raises(Vq2Error):
            K.vq_gemv_rht(*args)
        with pytest.raises(Vq2Error):
            K.vq_rows_gemm(*args)
    with pytest.raises(Vq2Error):
        K.vq_sorted_gemv(x[0], [(sp, sc)], cb0.float(), None, n, hb=0)
    with pytest.raises(Vq2Error):
        K.vq_sorted_gemv(x, [(sp, sc)], cb0, None, n, hb=0)
    # uint16 planes: handled by the Python entry
    (y,) = K.vq_gemv_rht(x, [(i0.view(torch.uint16), None, sc, 64)], cb0, None, n, hb=n)
    assert torch.equal(y, K.vq_gemv_rht(x, [(i0, None, sc, 64)], cb0, None, n, hb=n)[0])


def test_every_graph_clears_the_counters_it_uses(dev):
    """Graphs captured on one stream without an eager call before: each takes
    a workspace of its own and clears it, so they may be replayed in any order
    and their results are the eager ones.  A DecodeStepGraph keeps the
    workspace its warm-up cleared, apart from its stream's later calls."""
    n, rows = 2048, (6144, 6144)  # slices: counters of the workspace
    ms, cb0, cb1 = _mats(dev, 8890, n, rows, 4)
    mats = [(K.SortedPlanes(m["idx0"], m["idx1"], r, n, device=dev), m["scale"].to(dev)) for m, r in zip(ms, rows)]
    xs = [synth.activations(8895 + i, n, dtype=torch.float16).to(dev) for i in range(3)]
    refs = [K.vq_sorted_gemv(x, mats, cb0, cb1, n) for x in xs]
    stream, used = torch.cuda.Stream(dev), []
    K.take_workspaces(stream)  # (a pooled stream: an earlier user's)
    torch.cuda.synchronize(dev)

    def capture(x):
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=stream):
            for _ in range(2):
                ys = K.vq_sorted_gemv(x, mats, cb0, cb1, n)
            used.append(K._workspace(dev, 1 << 16, sorted_kind=True).data_ptr())
        return g, ys

    graphs = [capture(x) for x in xs]
    assert len(set(used)) == 3
    for i in (2, 0, 1, 2, 2, 0):
        graphs[i][0].replay()
        torch.cuda.synchronize(dev)
        assert all(torch.equal(a, b) for a, b in zip(graphs[i][1], refs[i])), i
        with torch.cuda.stream(stream):  # the stream's eager calls have their own
            assert all(torch.equal(a, b) for a, b in zip(K.vq_sorted_gemv(xs[1], mats, cb0, cb1, n), refs[1]))
        torch.cuda.synchronize(dev)
    steps = [DecodeStepGraph(lambda x: K.vq_sorted_gemv(x, mats, cb0, cb1, n), [x]) for x in xs[:2]]
    own = [w.data_ptr() for s in steps for w in s._workspaces]
    assert len(set(own)) == len(own) >= 2 and not set(own) & {w.data_ptr() for w in K._WS.values()}
    for i in (1, 0, 2, 1):
        assert all(torch.equal(a, b) for a, b in zip(steps[i % 2](xs[i]), refs[i]))
