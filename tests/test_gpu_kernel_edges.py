"""Kernels at the sizes where their tiling can go wrong: one workgroup's edge,
a remainder, the first size of another variant, the smallest and a large input.
"""
import numpy as np
import pytest
import torch

from rt_amd import scheme as S

pytestmark = pytest.mark.gpu


def spot_reference(x, y, f, G):
    """n, centroid, variance and RMS radius per group, two passes in numpy"""
    out = np.zeros((G, 6))
    for g in range(G):
        m = f[g::G] == 1
        xs, ys = x[g::G][m], y[g::G][m]
        if xs.size:
            vx, vy = xs.var(), ys.var()
            out[g] = [xs.size, xs.mean(), ys.mean(), vx, vy, np.sqrt(vx + vy)]
    return out


# a workgroup covers 256 // G strides of the groups 8 times (2048 rays in one
# group); 257 groups take a second block of groups; above 2^21 rays a workgroup
# walks its chunk in two passes
@pytest.mark.parametrize("n,G", [(1, 1), (2047, 1), (2048, 1), (2049, 1), (2040, 5), (2041, 5), (7, 255), (4097, 256),
                                 (257 * 8 + 1, 257), (3000, 1000), ((1 << 21) - 1, 3), ((1 << 21) + 4095, 1)])
def test_group_spots_at_chunk_edges(hip, n, G):
    print(f"[group spots] n={n} groups={G}", flush=True)
    g = torch.Generator().manual_seed(n + G)
    rays = torch.zeros((7, n), dtype=torch.float64)
    rays[0] = torch.randn(n, generator=g, dtype=torch.float64) * 0.01 + 12.5
    rays[1] = torch.randn(n, generator=g, dtype=torch.float64) * 0.3 - 2.0
    flag = (torch.rand(n, generator=g) < 0.9).to(torch.int8)
    dev, fd = rays.cuda(), flag.cuda()
    out = torch.full((G, hip.SPOT_STRIDE), float("nan"), dtype=torch.float64, device="cuda")
    got = hip.group_spots(dev, fd, G, out=out).cpu().numpy()
    want = spot_reference(rays[0].numpy(), rays[1].numpy(), flag.numpy(), G)
    assert np.array_equal(got[:, 0], want[:, 0])
    # centroids: a few roundings of values near 12.5; variances: squares of
    # differences that carry 12.5 * 2^-53 each, against a variance of 1e-4
    assert np.all(np.abs(got[:, 1:3] - want[:, 1:3]) <= 1e-13)
    assert np.all(np.abs(got[:, 3:6] - want[:, 3:6]) <= 1e-10 * np.abs(want[:, 3:6]) + 1e-28)


# one lane, one wave, the counting stages' workgroups of 256 lanes and of 1024
# (from 3 * 2^18 rays on), more rays than their largest grids hold at once
@pytest.mark.parametrize("n", [1, 64, 255, 257, 1023, 1024, 1025, 512 * 256 + 1, 512 * 1024 + 1, (3 << 18) - 1,
                               3 << 18, (3 << 18) + 1])
def test_mask_counts_and_flags(hip, n):
    print(f"[mask] n={n}", flush=True)

    g = torch.Generator().manual_seed(n)
    xy = torch.randn((2, n), generator=g, dtype=torch.float64)
    if n > 64:
        xy[0, 5], xy[1, 7] = float("nan"), float("inf")
    rec = S.Scheme([S.Surface(S.RT_PLANE, S.RT_MIRROR, S.RT_CIRCLE, size=(1.25, 0.0), center=(0.1, -0.2))],
                   S.Beam()).table
    dev, flag = xy.cuda(), torch.ones(n, dtype=torch.int8, device="cuda")
    bad = torch.full((2,), 3, dtype=torch.int64, device="cuda")
    hip.check(hip.lib().rt_hip_stage_mask(hip._dptr(np.ascontiguousarray(rec)), n, dev[0].data_ptr(), dev[1].data_ptr(),
                                          flag.data_ptr(), bad.data_ptr(), torch.cuda.current_stream().cuda_stream), "mask")
    # the aperture rejects what compares outside it: a NaN stays
    x, y = xy[0].numpy() - 0.1, xy[1].numpy() + 0.2
    lost = x * x + y * y > 1.25 * 1.25
    assert np.array_equal(flag.cpu().numpy() == 0, lost)
    assert bad.cpu().tolist() == [3 + int(lost.sum()), 3]


# every pattern of shifted coordinates and applied rotations: what moves moves
# as in plain arithmetic, what the frame change leaves alone keeps its bits
@pytest.mark.parametrize("dist", [(0.0, 0.0, 5.0), (1.5, 0.0, 0.0), (0.0, -2.0, 0.0), (0.3, 0.4, -7.0), (0.0, 0.0, 0.0)])
@pytest.mark.parametrize("ang", [(0.0, 0.0, 0.0), (0.2, 0.0, 0.0), (0.0, -0.3, 0.0), (0.0, 0.0, 1.1), (0.1, 0.2, 0.3)])
def test_transform_touches_what_it_moves(hip, dist, ang):
    print(f"[transform] dist={dist} ang={ang}", flush=True)
    n = 300
    g = torch.Generator().manual_seed(1)
    st = torch.randn((6, n), generator=g, dtype=torch.float64) * 50.0
    st[0, 3], st[4, 9] = -0.0, float("nan")
    dev = st.cuda()
    ptr = [dev[k].data_ptr() for k in range(6)]
    a, d = np.array(ang), np.array(dist)
    hip.check(hip.lib().rt_hip_stage_transform(hip._dptr(a), hip._dptr(d), n, *ptr,
                                               torch.cuda.current_stream().cuda_stream), "transform")
    want, moved = st.numpy().copy(), [False] * 6
    for k in range(3):
        want[k] -= dist[k]
        moved[k] = dist[k] != 0.0
    for k, (u, v) in enumerate(((0, 2), (1, 2), (0, 1))):
        if ang[k] == 0.0:
            continue
        s, c = np.sin(ang[k]), np.cos(ang[k])
        for w in (0, 3):
            want[u + w], want[v + w] = want[u + w] * c - want[v + w] * s, want[u + w] * s + want[v + w] * c
            moved[u + w] = moved[v + w] = True
    got = dev.cpu().numpy()
    for k in range(6):
        if not moved[k]:
            assert got[k].tobytes() == st[k].numpy().tobytes(), k
        else:
            # up to three rotations of values near 150: a few units of 150 * 2^-53
            assert np.allclose(got[k], want[k], rtol=0.0, atol=3e-13, equal_nan=True), k


def reference_order(codes):
    """Beam::Rearrange after every stage that lost rays, one swap at a time"""
    perm, G = list(range(len(codes))), len(codes)
    for c in range(1, 255):
        bad = [codes[r] == c for r in perm[:G]]
        if not any(bad):
            continue
        i, j = 0, G - 1
        while True:
            while i < G and not bad[i]:
                i += 1
            while j >= 0 and bad[j]:
                j -= 1
            if i >= j:
                break
            perm[i], perm[j] = perm[j], perm[i]
            bad[i], bad[j] = bad[j], bad[i]
        G -= sum(bad)
    return perm


# a tile is 4096 positions of 16 a lane; codes read four at a time from an
# aligned start, one at a time from any other
@pytest.mark.parametrize("n,offset", [(1, 0), (3, 0), (17, 1), (4095, 0), (4096, 0), (4097, 2), (3 * 4096 + 7, 3)])
@pytest.mark.parametrize("lost", [0.01, 0.6, 1.0])
def test_rearrange_order_and_counts(hip, n, offset, lost):
    print(f"[rearrange] n={n} offset={offset} lost={lost}", flush=True)
    rng = np.random.default_rng(n)
    codes = np.where(rng.random(n) < lost, rng.integers(1, 9, n), 0).astype(np.uint8)
    dev = torch.zeros(n + offset, dtype=torch.uint8, device="cuda")
    dev[offset:].copy_(torch.from_numpy(codes))
    perm, counts = hip.rearrange(dev[offset:])
    assert np.array_equal(perm.cpu().numpy(), reference_order(codes))
    assert np.array_equal(counts, np.bincount(codes, minlength=256))


# one ray, a partial workgroup, and more rays than the resident workgroups take
# in one round (so that each meets rays inside and outside its bounds)
@pytest.mark.parametrize("n", [1, 300, (1 << 18) - 1, 1 << 18, 700003])
def test_recorded_extents_equal_dumped_states(hip, n):
    print(f"[extents] n={n}", flush=True)
    from rt_amd import scheme as S, schemes
    sc = schemes.echelle_fixed_order(n, 1)
    ds = hip.DeviceScheme(sc)
    rays, flag = torch.empty((7, n), dtype=torch.float64, device="cuda"), torch.empty(n, dtype=torch.int8, device="cuda")
    loss = torch.empty(n, dtype=torch.uint8, device="cuda")
    ext = torch.zeros((sc.n_surf, hip.EXT_PER_SURF), dtype=torch.float64, device="cuda")
    ds.trace_record(rays, flag, loss, seed=4, extents=ext)
    dump = torch.empty((sc.n_surf, 7, n), dtype=torch.float64, device="cuda")
    dflag = torch.empty((sc.n_surf, n), dtype=torch.int8, device="cuda")
    ds.trace(None, None, seed=4, n=n, flags=S.RT_TRACE_GENERATE, dump=dump, dump_flag=dflag)
    e, codes = ext.cpu().numpy(), loss.cpu().numpy()
    for s in range(sc.n_surf):
        st, alive = dump[s].cpu().numpy(), dflag[s].cpu().numpy() != 0
        # X, Y at the intersection: the rays that met the surface, those lost at
        # its aperture or action too (they stay where they are); after the
        # aperture: the rays past it.  cZ on entry: where the frame change does
        # not rotate, the one that left the surface before
        passed = alive | (codes == 3 + 3 * s)
        met = passed | (codes == 2 + 3 * s)
        checks = [(1, st[0], met), (2, st[1], met), (3, st[0], passed), (4, st[1], passed), (5, st[5], alive)]
        if s > 0 and not any(sc.surfaces[s].angles):
            checks.append((0, dump[s - 1].cpu().numpy()[5], dflag[s - 1].cpu().numpy() != 0))
        for q, row, on in checks:
            v = row[on]
            want = (v.min(), v.max()) if v.size else (np.nan, np.nan)
            assert np.array_equal(e[s, 2 * q:2 * q + 2], want, equal_nan=True), (s, q)
    # all twelve of every surface in workgroups of another size
    ds.set_launch(256, 7, 16)
    other = torch.zeros_like(ext)
    ds.trace_record(rays, flag, loss, seed=4, extents=other)
    assert torch.equal(other.nan_to_num(12345.0), ext.nan_to_num(12345.0))
    ds.close()


# extents are optional: without them the generic kernel records the same codes
# and rays as with them, and as the generated kernel
@pytest.mark.parametrize("n", [1, 700])
def test_recording_without_extents(hip, n):
    from rt_amd import schemes
    sc = schemes.echelle_fixed_order(n, 1)
    out = []
    for jit, want in ((False, True), (False, False), (True, False)):
        print(f"[recording] n={n} generated={jit} extents={want}", flush=True)
        prev = hip.set_jit(jit)
        try:
            ds = hip.DeviceScheme(sc)
            rays = torch.empty((7, n), dtype=torch.float64, device="cuda")
            flag, loss = (torch.empty(n, dtype=d, device="cuda") for d in (torch.int8, torch.uint8))
            ext = torch.zeros((sc.n_surf, hip.EXT_PER_SURF), dtype=torch.float64, device="cuda") if want else None
            ds.trace_record(rays, flag, loss, seed=6, extents=ext)
            out.append((rays.cpu().numpy(), flag.cpu().numpy(), loss.cpu().numpy()))
            ds.close()
        finally:
            hip.set_jit(prev)
    for got in out[1:]:
        assert np.array_equal(got[1], out[0][1]) and np.array_equal(got[2], out[0][2])
    assert np.array_equal(out[1][0], out[0][0])
    # two kernels from the same stage code: 1e-12 of the scheme's length, of a
    # unit direction and of the wavelength
    L = max(1.0, max(abs(d) for q in sc.surfaces for d in q.distance))
    scale = np.array([L, L, L, 1.0, 1.0, 1.0, 1.0])[:, None]
    assert np.all(np.abs(out[2][0] - out[0][0]) <= 1e-12 * scale)


# recordings of another size than the one before them, captured in a graph:
# nothing is allocated then, whatever launch the size takes, nor for a launch
# of smaller workgroups set in between
@pytest.mark.parametrize("first,then,block", [(1 << 18, 5000, None), (5000, 1 << 18, None), (1 << 18, 1 << 18, 64)])
def test_recording_captured_after_another_size(hip, first, then, block):
    print(f"[captured recording] {first} then {then}, {block}", flush=True)
    from rt_amd import schemes
    sc = schemes.echelle_fixed_order(1 << 18, 1)
    m = max(first, then)
    rays = torch.empty((7, m), dtype=torch.float64, device="cuda")
    flag, loss = (torch.empty(m, dtype=d, device="cuda") for d in (torch.int8, torch.uint8))
    ext = torch.zeros((sc.n_surf, hip.EXT_PER_SURF), dtype=torch.float64, device="cuda")
    stream = torch.cuda.Stream()

    def record(ds, n):
        ds.trace_record(rays, flag, loss, seed=4, n=n, extents=ext, stream=stream.cuda_stream)
    ds = hip.DeviceScheme(sc)
    with torch.cuda.stream(stream):
        record(ds, then)                                   # the kernels of both sizes are compiled
        want = ext.clone()
        record(ds, first)
    stream.synchronize()
    ds.close()
    ds = hip.DeviceScheme(sc)                              # a scheme without working memory yet
    with torch.cuda.stream(stream):
        record(ds, first)
    stream.synchronize()
    if block:
        ds.set_launch(block, 8, 16)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=stream, capture_error_mode="thread_local"):
        record(ds, then)
    for k in range(3):
        ext.zero_()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(ext, want), k
        with torch.cuda.stream(stream):
            record(ds, first)
        torch.cuda.synchronize()
    ds.close()


def two_detectors(n):
    """a detector that the rays pass, one behind it, a frame too small for all
    of them on each and an aperture in between"""
    ccd = dict(xdim=64, ydim=64, xpix=0.25, ypix=0.25)
    b = S.Beam(type=S.RT_BEAM_CONIC, shape=S.RT_CIRCLE, params=(n, 0.0, 9.0, 1.0), range=(0.5, 0.6), nlambda=1)

    def detector(size, z):
        return S.Surface(S.RT_PLANE, S.RT_DETECTOR, S.RT_RECTANGLE, size=(size, size), distance=(0, 0, z), ccd=ccd)
    stop = S.Surface(S.RT_PLANE, S.RT_STOP, S.RT_CIRCLE, size=(8.5, 0.0), distance=(0, 0, 10.0))
    return S.Scheme([detector(17.0, 5.0), stop, detector(60.0, 400.0)], b, name="two detectors")


# counters derived from the losses: into the caller's own counters (at most 64
# workgroups) and through the copies; rays generated, and given with dead ones
@pytest.mark.parametrize("n", [1, 257, 64 * 256, 64 * 256 + 1, 100001])
@pytest.mark.parametrize("given", [False, True])
@pytest.mark.parametrize("jit", [True, False])
def test_counters_of_two_detectors(hip, n, given, jit):
    from oracle import oracle as O
    print(f"[two detectors] n={n} given={given} generated={jit}", flush=True)
    sc = two_detectors(n)
    kw = {}
    if given:
        kw["rays"] = O.trace(S.Scheme(sc.surfaces[:1], sc.beam), seed=9).rays
        kw["flag"] = (np.arange(n) % 5 != 0).astype(np.int8)
    ref = O.trace(sc, seed=9, hist=True, **kw)
    prev = hip.set_jit(jit)
    try:
        ds = hip.DeviceScheme(sc)
        rays = torch.from_numpy(kw.get("rays", np.zeros((7, n)))).cuda()
        flag = torch.from_numpy(kw.get("flag", np.zeros(n, dtype=np.int8))).cuda()
        hist = torch.zeros(64 * 64, dtype=torch.int32, device="cuda")
        stats = torch.full((S.STATS_LEN,), 7, dtype=torch.int64, device="cuda")
        flags = S.RT_TRACE_STORE | S.RT_TRACE_HIST | (0 if given else S.RT_TRACE_GENERATE)
        ds.trace(rays, flag, seed=9, n=n, flags=flags, hist=hist, stats=stats)
        assert np.array_equal(flag.cpu().numpy(), ref.flag)
        assert np.array_equal(hist.cpu().numpy().view(np.uint32), ref.hist)
        assert np.array_equal(stats.cpu().numpy().view(np.uint64) - np.uint64(7), ref.stats)
        ds.close()
    finally:
        hip.set_jit(prev)
    if n > 1000:
        assert ref.stats[S.ST_CCD_OFFCHIP] > 0 and ref.stats[S.ST_CCD_HITS] > ref.stats[S.ST_GOOD] > 0


def test_tuned_launch_holds_for_traces_like_the_timed_ones(hip, monkeypatch, capfd):
    """The launch of every trace as the library reports it: the tuner's for
    generated traces with the frames it timed, the defaults of their kind for
    the others, the caller's for all."""
    from rt_amd import schemes
    monkeypatch.setenv("RT_HIP_VERBOSE", "1")
    n = 1 << 18
    sc = schemes.czerny_turner(n, 1)
    px = sc.detector().ccd["xdim"] * sc.detector().ccd["ydim"]
    rays = torch.empty((7, n), dtype=torch.float64, device="cuda")
    flag, loss = (torch.empty(n, dtype=d, device="cuda") for d in (torch.int8, torch.uint8))
    ext = torch.zeros((sc.n_surf, hip.EXT_PER_SURF), dtype=torch.float64, device="cuda")
    hist, flux = (torch.zeros(px, dtype=d, device="cuda") for d in (torch.int32, torch.float64))
    gen, store, count = S.RT_TRACE_GENERATE, S.RT_TRACE_STORE, S.RT_TRACE_HIST
    both = count | S.RT_TRACE_FLUX

    def launches(ds):
        calls = dict(generated=lambda: ds.trace(rays, flag, n=n, flags=gen | store | count, hist=hist),
                     frames=lambda: ds.trace(rays, flag, n=n, flags=gen | store | both, hist=hist, flux=flux),
                     given=lambda: ds.trace(rays, flag, n=n, flags=count, hist=hist),
                     recorded=lambda: ds.trace_record(rays, flag, loss, extents=ext),
                     few=lambda: ds.trace_record(rays, flag, loss, n=1000, extents=ext),
                     spots=lambda: ds.trace_spots(1, n=n))
        out = {}
        for k, call in calls.items():
            capfd.readouterr()
            call()
            torch.cuda.synchronize()
            line = [v for v in capfd.readouterr().err.splitlines() if "generated kernel" in v][0]
            out[k] = tuple(int(line.split(w)[1].split(",")[0]) for w in ("block ", "waves "))
        return out
    ds = hip.DeviceScheme(sc)
    rules = dict(generated=(256, 7), frames=(256, 7), given=(256, 8), recorded=(1024, 8), few=(256, 7), spots=(256, 7))
    assert launches(ds) == rules
    ds.autotune(n_sample=20000, flags=store | count)
    if ds.get_unroll():
        assert launches(ds) == dict(rules, generated=ds.get_launch()[:2])
    ds.set_unroll(True)
    ds.set_launch(128, 5, 2)
    assert set(launches(ds).values()) == {(128, 5)}
    # a large sample into both frames: the launch that an untuned trace takes is
    # among those timed
    monkeypatch.setenv("RT_HIP_AUTOTUNE_LOG", "1")
    for sample, there in ((1 << 20, True), ((1 << 20) - 1, False)):
        capfd.readouterr()
        ds.autotune(n_sample=sample, flags=both)
        assert ("autotune: 512,7,16 " in capfd.readouterr().err) == there, sample
    ds.close()


def test_more_parameters_do_not_take_a_second_tape(hip):
    """A batched adjoint over more parameters than the one before needs more
    partials, not another tape: the tape (hundreds of MB here) stays."""
    from rt_amd import diff, schemes
    sch = schemes.echelle(8, 16)
    inst, _ = schemes.tolerance_instances(sch, 16, seed=1)
    db = hip.DeviceBatch(inst, np.full(16, 30000))
    pairs = [(p.surface, p.field) for p in diff.echelle_design_params(sch).params]
    ps, pf = zip(*pairs)
    seeds = torch.ones((16, 4, 3), dtype=torch.float64, device="cuda")
    used = []
    for m in (1, len(pairs)):
        print(f"[adjoint memory] {m} parameters", flush=True)
        grad = torch.zeros((16, m), dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        before = torch.cuda.mem_get_info()[0]
        db.adjoint(seeds, ps[:m], pf[:m], seed=3, grad=grad)
        torch.cuda.synchronize()
        used.append(before - torch.cuda.mem_get_info()[0])
    db.close()
    # 1,888 tiles of 256 lanes, tens of rows of 8 bytes each; the partials of 48
    # parameters are 1,888 * 4 * 48 * 8 bytes = 2.9 MB
    assert used[0] > 64 << 20 and used[1] < 32 << 20, used


def every_surface_kind():
    """a lens, a rotated auxiliary frame, a rotated stop, an aspheric lens, two
    unrotated stops in a row (the first loses rays), a toric lens, a plane lens
    face, both kinds of grating, a spherical and a toric mirror, a detector:
    every branch of the reverse step, and directions that pass one surface and
    two unchanged"""
    s = [S.Surface(S.RT_CONIC, S.RT_LENS, S.RT_CIRCLE, params=(1 / 400.0, -0.3, 0), size=(40.0, 0.0),
                   distance=(0.1, -0.2, 20.0), angles=(0.3, -0.2, 0.0), n1=1.0, n2=1.5),
         S.Surface(S.RT_PLANE, S.RT_AUXTYPE, distance=(0.0, 0.1, 3.0), angles=(0.0, 0.5, 1.0)),
         S.Surface(S.RT_PLANE, S.RT_STOP, S.RT_CIRCLE, size=(40.0, 0.0), distance=(0.0, 0.0, 2.0),
                   angles=(0.2, 0.0, 0.4)),
         S.Surface(S.RT_PLANE, S.RT_LENS, S.RT_CIRCLE, size=(40.0, 0.0), distance=(0.0, 0.0, 5.0),
                   angles=(0.0, 1.0, 0.0), n1=1.5, n2=1.0),
         S.Surface(S.RT_CONIC, S.RT_LENS, S.RT_CIRCLE, params=(-1 / 300.0, 0.2, 3, 1e-6, 1e-9, 1e-13),
                   size=(40.0, 0.0), distance=(0.0, 0.0, 10.0), n1=1.0, n2=1.6),
         S.Surface(S.RT_PLANE, S.RT_STOP, S.RT_CIRCLE, size=(6.0, 0.0), distance=(0.0, 0.0, 1.0)),
         S.Surface(S.RT_PLANE, S.RT_STOP, S.RT_CIRCLE, size=(40.0, 0.0), distance=(0.05, 0.0, 2.0)),
         S.Surface(S.RT_TORIC, S.RT_LENS, S.RT_CIRCLE, params=(1 / 500.0, 0.1, 1, 1e-7, 1 / 350.0),
                   size=(40.0, 0.0), distance=(0.2, 0.0, 6.0), n1=1.6, n2=1.0),
         S.Surface(S.RT_PLANE, S.RT_GRATING, S.RT_CIRCLE, size=(60.0, 0.0), distance=(0.0, 0.0, 30.0),
                   angles=(2.0, 0.0, 0.0), grating_type=S.RT_TRANSPARENT, order=1, gr_const=10.0),
         S.Surface(S.RT_CONIC, S.RT_MIRROR, S.RT_CIRCLE, params=(-1 / 900.0, 0.0, 0), size=(90.0, 0.0),
                   distance=(0.0, 0.0, 60.0), angles=(3.0, 0.0, 0.0)),
         S.Surface(S.RT_TORIC, S.RT_MIRROR, S.RT_CIRCLE, params=(1 / 1200.0, 0.0, 0, 1 / 1500.0),
                   size=(120.0, 0.0), distance=(0.0, 0.0, -70.0), angles=(0.0, 1.0, 0.0)),
         S.Surface(S.RT_PLANE, S.RT_GRATING, S.RT_CIRCLE, size=(150.0, 0.0), distance=(0.0, 0.0, 80.0),
                   grating_type=S.RT_REFLECTIVE, order=-1, gr_const=20.0),
         S.Surface(S.RT_PLANE, S.RT_DETECTOR, S.RT_RECTANGLE, size=(400.0, 400.0), distance=(0.0, 0.0, -90.0),
                   angles=(0.5, 0.2, 0.0), ccd=dict(xdim=64, ydim=64, xpix=5.0, ypix=5.0))]
    return s


@pytest.mark.parametrize("n", [1, 65, 600])
@pytest.mark.parametrize("beam", ["conic", "parallel"])
def test_generated_adjoint_equals_the_generic_one(hip, n, beam):
    # the generated reverse step reads the state after each surface from the
    # tape where the generic one replays it: the same derivatives, to the sums'
    # and the directions' rounding (1e-11 of the largest derivative by the same
    # field of a surface: those of one field are formed by like terms)
    from oracle import oracle as O
    kind = S.RT_BEAM_CONIC if beam == "conic" else S.RT_BEAM_PARALLEL
    b = S.Beam(type=kind, shape=S.RT_CIRCLE, params=(n, 0.0, 6.0, 1.0, 2.0), range=(0.5, 0.6), nlambda=1)
    surf = every_surface_kind()
    sch = S.Scheme(surf, b, name="kinds")
    good = int(O.trace(sch, seed=11).flag.sum())
    assert 0 < good and (n < 600 or good < n)
    ps, pf = [], []
    for i, q in enumerate(surf):
        fields = [S.S_DIST + k for k in range(3)] + [S.S_ANG + k for k in range(3)]
        if q.cls != S.RT_PLANE:
            fields += [S.S_C, S.S_K] + [S.S_A + k for k in range(int(q.params[2]))]
        if q.cls == S.RT_TORIC:
            fields.append(S.S_CR)
        if q.type == S.RT_GRATING:
            fields.append(S.S_GRCONST)
        ps += [i] * len(fields)
        pf += fields
    G = 3
    rng = np.random.default_rng(3)
    seeds = torch.from_numpy(rng.normal(size=(G, 3))).cuda()
    out = []
    for jit in (True, False):
        prev = hip.set_jit(jit)
        try:
            ds = hip.DeviceScheme(sch)
            st = torch.zeros(S.STATS_LEN, dtype=torch.int64, device="cuda")
            out.append(ds.adjoint(seeds, ps, pf, seed=11, n=n, stats=st).cpu().numpy())
            st = st.cpu().numpy()
            assert st[S.ST_RAYS] == n and st[S.ST_GOOD] == good and st[S.ST_ADJ_SKIP] == 0
            ds.close()
        finally:
            hip.set_jit(prev)
    assert np.all(np.isfinite(out[0])) and np.all(np.isfinite(out[1]))
    for f in set(pf):
        q = np.array(pf) == f
        scale = float(np.max(np.abs(out[1][q])))
        err = float(np.max(np.abs(out[0] - out[1])[q]))
        assert scale > 0 and err <= 1e-11 * scale, (f, err / scale)
