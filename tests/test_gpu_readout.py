"""Results read back from the device: whole blocks below, at and above one
pinned slot (2^17 words), through one and through several host threads, and
from several threads of the caller at once.  Everything bit for bit: the fields
against what was set, node values against the host expressions on them,
markers against what was loaded."""
import os
import subprocess
import sys
import threading

import numpy as np
import pytest

import mandor3_amd as ma
from mandor3_amd.workloads import courant_tau

pytestmark = pytest.mark.gpu
H = (0.05, 0.04, 0.06)
SLOT = 1 << 17


def make(n, prec, markers=0, seed=1):
    rng = np.random.default_rng(seed)
    M = np.zeros(markers, dtype=ma.MARKER_DTYPE)
    for a, c in enumerate("xyz"):
        M[c] = rng.uniform(0.01, n[a] * H[a] - 0.01, markers)
        M["v" + c] = rng.normal(0, 0.5, markers)
    M["rho"] = rng.normal(0, 1, markers)
    M["qDivM"] = rng.choice([-1.0, 0.25], markers)
    M["id"] = np.arange(1, markers + 1)
    nodes = 3 * int(np.prod([v + 1 for v in n]))
    E, F = rng.normal(0, 1, nodes), rng.normal(0, 1, nodes)
    if prec == ma.FP32_SPLIT:
        E, F = E.astype(np.float32).astype(float), F.astype(np.float32).astype(float)
    r = ma.Run(n, H, tuple(v * h for v, h in zip(n, H)), courant_tau(H), (0,) * 6, 0.0,
               precision=prec, max_markers=max(markers, 1))
    r.set_fields(E, F)
    r.load_markers(M)
    return r, E, F, M


# words of E and H together: below one slot, E alone below, E just above, many slots
@pytest.mark.parametrize("prec", [ma.FP64, ma.FP32_SPLIT])
@pytest.mark.parametrize("n", [(7, 9, 12), (26, 26, 28), (33, 34, 35), (40, 30, 33), (110, 90, 100)])
def test_fields_and_node_values(n, prec):
    r, E, F, _ = make(n, prec)
    for x, y in zip(r.fields(), (E, F)):
        assert np.array_equal(x, y)
    r.close()
    # node values, away from the ghost layer
    r, E, F, _ = make(n, prec)
    r.init()
    e, h = (v.reshape([a + 1 for a in n] + [3]) for v in (E, F))
    got = [r.node_fields(q).reshape([a + 1 for a in n] + [3])[:-1, :-1, :-1] for q in (0, 1)]
    want = np.stack([0.5 * (e[:-1, :-1, :-1, 0] + e[1:, :-1, :-1, 0]),
                     0.5 * (e[:-1, :-1, :-1, 1] + e[:-1, 1:, :-1, 1]),
                     0.5 * (e[:-1, :-1, :-1, 2] + e[:-1, :-1, 1:, 2])], -1)
    inner = (slice(1, -1),) * 3
    assert np.array_equal(got[0][inner], want[inner])
    o = h[:-1, :-1, :-1]
    want = np.stack([0.25 * (o[..., 0] + h[:-1, 1:, :-1, 0] + h[:-1, :-1, 1:, 0] + h[:-1, 1:, 1:, 0]),
                     0.25 * (o[..., 1] + h[1:, :-1, :-1, 1] + h[:-1, :-1, 1:, 1] + h[1:, :-1, 1:, 1]),
                     0.25 * (o[..., 2] + h[1:, :-1, :-1, 2] + h[:-1, 1:, :-1, 2] + h[1:, 1:, :-1, 2])], -1)
    assert np.array_equal(got[1][inner], want[inner])
    r.close()


@pytest.mark.parametrize("recsize", [64, 56])
@pytest.mark.parametrize("prec", [ma.FP64, ma.FP32_SPLIT])
@pytest.mark.parametrize("count", [0, 1, SLOT // 8, SLOT // 8 + 1, 300001])
def test_markers(count, prec, recsize):
    n = (20, 21, 23)
    r, _, _, M = make(n, prec, count)
    r.init()
    S = r.markers(recsize)
    assert S.size == count
    # 56-byte records carry no id: match by the (distinct) momenta
    key = "id" if recsize == 64 else "vx"
    want = M["vx"].astype(np.float32).astype(float) if prec == ma.FP32_SPLIT else M["vx"]
    a = S[np.argsort(S[key], kind="stable")]
    b = M[np.argsort(M["id"] if recsize == 64 else want, kind="stable")]
    if recsize == 56 and prec == ma.FP32_SPLIT:      # equal FP32 momenta: compare as sets per column
        assert np.array_equal(np.sort(S["vx"]), np.sort(want))
        r.close()
        return
    for q, c in enumerate("xyz"):
        if prec == ma.FP64:
            assert np.array_equal(a[c], b[c])
        else:                                        # cell + FP32 offset, then times h
            s = b[c] / H[q]
            cell = (s + 128.0).astype(np.int64) - 128
            assert np.array_equal(a[c], (cell + (s - cell).astype(np.float32).astype(float)) * H[q])
        v = b["v" + c]
        assert np.array_equal(a["v" + c], v if prec == ma.FP64 else v.astype(np.float32).astype(float))
    assert np.array_equal(a["rho"], b["rho"]) and np.array_equal(a["qDivM"], b["qDivM"])
    with pytest.raises(ma.MpicError):                # a buffer too small is refused
        if count == 0:
            raise ma.MpicError("nothing to refuse")
        import ctypes
        cap = ctypes.c_long(count - 1)
        buf = np.zeros(count * 64, dtype=np.uint8)
        ma._check(ma.lib().mpic_markers_save(r.handle, ma._ptr(buf), ctypes.byref(cap), recsize), "save")
    r.close()


def test_several_threads_at_once():
    runs = [make((50 + 5 * q, 40, 45), ma.FP64, seed=q) for q in range(4)]
    bad = []

    def read(q):
        r, E, F, _ = runs[q]
        for _ in range(5):
            e, f = r.fields()
            if not (np.array_equal(e, E) and np.array_equal(f, F)):
                bad.append(q)

    th = [threading.Thread(target=read, args=(q,)) for q in range(4)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad
    for r in runs:
        r[0].close()


def test_process_ends_with_a_run_still_open():
    """The helper threads of a large read-out do not keep the process."""
    code = ("import numpy as np, os, mandor3_amd as ma\n"
            "r = ma.Run((60, 60, 60), (.05,) * 3, (3.,) * 3, .012, (0,) * 6)\n"
            "z = np.ones(3 * r.nodes)\n"
            "r.set_fields(z, z)\n"
            "assert r.fields()[0].sum() == z.size\n"
            "keep = [r]; keep.append(keep); ma.Run.__del__ = lambda self: None\n")
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    p = subprocess.run([sys.executable, "-c", code], cwd=root, timeout=60)
    assert p.returncode == 0
