"""Launch shapes of the FP32 push beside those of test_gpu_modes.py: 1 and 8
wavefronts per workgroup (8 is the rule's choice on small boxes), and the
kinetic sums, which every wavefront adds to one of 256 slots.  Bars: the split
form's own."""
import numpy as np
import pytest

import mandor3_amd as ma
from mandor3_amd import workloads
from test_gpu_modes import _split_twenty_steps
from test_gpu_parity import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("items", [None, "64"])
@pytest.mark.parametrize("waves", ["1", "8"])
@pytest.mark.parametrize("case", ["periodic", "mixed"])
def test_one_and_eight_wavefronts_per_tile(case, waves, items, monkeypatch):
    monkeypatch.setenv("MPIC_TILE_WAVES", waves)
    if items:
        monkeypatch.setenv("MPIC_ITEM_MARKERS", items)
    _split_twenty_steps(case, "%s wavefronts, items %s" % (waves, items))


@pytest.mark.parametrize("prec", [ma.FP64, ma.FP32_SPLIT])
@pytest.mark.parametrize("n", [8, 33])
def test_kinetic_sums(n, prec):
    """The first push of the two-stream box starts from E = H = 0, so its sums
    are sum (gamma - 1) w u_a^2 / u^2 h^3 m/q over the loaded momenta: 8^3 has
    fewer wavefronts than slots, 33^3 several per slot."""
    st = workloads.two_stream_box(n)
    M = st["markers"]
    r = ma.Run(st["n"], st["h"], st["L"], st["tau"], st["bc"], 0.0, precision=prec,
               max_markers=M.size)
    z = np.zeros(3 * r.nodes)
    r.set_fields(z, z)
    r.load_markers(M)
    r.init()
    u = np.stack([M["vx"], M["vy"], M["vz"]])
    u2 = (u * u).sum(0)
    # (gamma - 1) / u^2 = 1 / (gamma + 1): no cancellation for slow markers
    w = M["rho"].astype(float) / M["qDivM"] / (np.sqrt(1 + u2) + 1) * 0.05 ** 3
    want = (w * u * u).sum(1)
    r.stage("em_h_half")
    r.stage("push_deposit")
    got = r.temperature()
    # FP32: momenta and each term rounded to 2^-24, all terms of one sign
    np.testing.assert_allclose(got, want, rtol=1e-11 if prec == ma.FP64 else 1e-6)
    r.close()


@pytest.mark.parametrize("prec", [ma.FP64, ma.FP32_SPLIT])
@pytest.mark.parametrize("n", [(7, 7, 7), (16, 16, 16), (16, 16, 17), (128, 64, 65)])
def test_field_energy_sums(n, prec):
    """Two, 16, 17 and 2048 (the most: a thread then sums several nodes)
    workgroups, against the sums over em.c:226-252's points in longdouble."""
    rng = np.random.default_rng(7)
    h = (0.1, 0.2, 0.05)
    r = ma.Run(n, h, tuple(a * b for a, b in zip(n, h)), 0.01, [0] * 6, 0.0, precision=prec)
    d = tuple(a + 1 for a in n)
    E, H = (rng.standard_normal(d + (3,)) for _ in range(2))
    if prec == ma.FP32_SPLIT:
        E, H = (F.astype(np.float32).astype(float) for F in (E, H))
    r.set_fields(E.ravel(), H.ravel())

    def total(F, off):
        s = np.longdouble(0)
        for c in range(3):
            sl = tuple(slice(off[c][a], off[c][a] + n[a]) for a in range(3))
            s += (F[sl + (c,)].astype(np.longdouble) ** 2).sum()
        return float(s * 0.5 * h[0] * h[1] * h[2])

    want = (total(E, ((1, 0, 0), (0, 1, 0), (0, 0, 1))),
            total(H, ((0, 1, 1), (1, 0, 1), (1, 1, 0))))
    # a thread adds at most 2 nodes of 3 squares, then 8 tree levels and 2048
    # partial sums, all positive: (6 + 8 + 2048) 2^-53 < 3e-13
    np.testing.assert_allclose(r.energy(), want, rtol=3e-13)
    r.close()


@pytest.mark.parametrize("prec,tol", [(ma.FP64, 1e-12), (ma.FP32_SPLIT, 2e-5)])
def test_fused_runs_with_fewer_workgroups_than_tiles(prec, tol):
    """Fused launches share workgroups out by markers: the 32^3 box with a
    sixteenth of the markers beside the full one gets fewer than its 512 tiles
    (241 FP32 in two runs, 128 FP64 in six, on 256 CUs): a workgroup takes
    several; the results are those of the run alone, to the order of the J sums (the serving
    loop's bar)."""
    st = workloads.two_stream_box(32)

    def make(M):
        r = ma.Run(st["n"], st["h"], st["L"], st["tau"], st["bc"], 0.0, precision=prec,
                   max_markers=M.size)
        z = np.zeros(3 * r.nodes)
        r.set_fields(z, z)
        r.load_markers(M)
        r.init()
        return r

    thin, full = st["markers"][::16], st["markers"]
    alone = make(thin)
    runs = [make(thin)] + [make(full) for _ in range(5 if prec == ma.FP64 else 1)]
    alone.advance(6)
    ma.batch_advance(runs, 6)
    for a, b in zip(alone.fields(), runs[0].fields()):
        assert np.linalg.norm(a) > 0 and rel_l2(b, a) <= tol
    assert alone.marker_count() == runs[0].marker_count() == thin.size
    for r in [alone] + runs:
        r.close()


@pytest.mark.parametrize("prec", [ma.FP64, ma.FP32_SPLIT])
@pytest.mark.parametrize("count", [1, 63, 64, 65, 700])
def test_charge_density_by_runs(count, prec):
    """A wavefront's markers are summed by runs of one cell: runs that end at,
    before and past a row of 16 lanes, a wavefront and a workgroup (markers in
    three cells), against the CIC sum in numpy."""
    n, h = (9, 10, 11), (0.1, 0.2, 0.05)
    rng = np.random.default_rng(count)
    M = np.zeros(count, dtype=ma.MARKER_DTYPE)
    c0 = np.array([(3, 4, 5), (3, 4, 6), (6, 3, 2)])[np.arange(count) * 3 // count]
    for a, c in enumerate("xyz"):
        M[c] = (c0[:, a] + rng.uniform(0.01, 0.99, count)) * h[a]
    M["rho"] = rng.uniform(-1, 1, count).astype(np.float32)
    M["qDivM"], M["id"] = -1.0, np.arange(1, count + 1)
    r = ma.Run(n, h, tuple(a * b for a, b in zip(n, h)), 0.01, [ma.BC_OPEN] * 6, 0.0,
               precision=prec, max_markers=count)
    z = np.zeros(3 * r.nodes)
    r.set_fields(z, z)
    r.load_markers(M)
    r.init()
    # nodes [0, n]: the fold at the walls mirrors inner nodes onto the ghosts (plasma_rho.c:23-96)
    own = (slice(2, -2),) * 3
    got = r.rho().reshape([v + 5 for v in n])[own]
    P = r.markers()
    assert P.size == count
    want = np.zeros([v + 5 for v in n])
    s = [P[c].astype(float) / h[a] for a, c in enumerate("xyz")]
    i = [np.floor(v).astype(int) for v in s]
    f = [v - k for v, k in zip(s, i)]
    for d in np.ndindex(2, 2, 2):
        w = P["rho"].astype(float)
        for a in range(3):
            w = w * (f[a] if d[a] else 1 - f[a])
        np.add.at(want, tuple(i[a] + 2 + d[a] for a in range(3)), w)
    want = want[own]
    # a sum of `count` terms, and positions to a few units in the last place of s < 12
    bar = (count + 200) * 2.0 ** -53 * np.abs(P["rho"]).sum()
    assert np.abs(want).max() > 0 and np.abs(got - want).max() <= bar
    r.close()
