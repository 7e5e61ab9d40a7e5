"""The stage arithmetic over the whole exponent range.

The device forms quotients with shared reciprocals and unscaled square roots
where the face's or tile's values lie in a checked range of exponents, and
with the full sequences elsewhere: values on both sides of every limit, exact
zeros of both signs, infinities and NaN must give the oracle's bits."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

# around the limits 2^60 (faces), 2^-800 (numerators, tiles), 2^-860 (momenta), and the underflow threshold
EXPONENTS = [0, 30, 59, 60, 61, 100, 101, 300, 480, 799, 800, 801, 859, 861, 968, 1000, 1021, 1060]


def _same_bits(a, b):
    return (a.view(np.int64) == b.view(np.int64)) | (np.isnan(a) & np.isnan(b))


@pytest.mark.parametrize("method", ["RUSA", "HLLE", "HLLC", "HLLD"])
@pytest.mark.parametrize("direction", ["x", "y"])
def test_riemann_batch_exponents(method, direction):
    torch = pytest.importorskip("torch")
    import amr2d_mhd_amd as A

    rng = np.random.default_rng(77 + len(method) + (direction == "y"))
    n = 512
    L, R = [], []
    for e in EXPONENTS:
        w = np.zeros((2, n, 8))
        w[:, :, 0] = rng.uniform(0.1, 3.0, (2, n))
        w[:, :, 4] = rng.uniform(0.05, 3.0, (2, n))
        w[:, :, 1:4] = rng.normal(0, 1, (2, n, 3))
        w[:, :, 5:8] = rng.normal(0, 1, (2, n, 3))
        # each of the six vector components of each state: kept, scaled down by 2^-e, +0 or -0
        pick = rng.integers(0, 4, (2, n, 6))
        v = w[:, :, [1, 2, 3, 5, 6, 7]]
        v = np.where(pick == 1, v * 2.0 ** -e, np.where(pick == 2, 0.0, np.where(pick == 3, -0.0, v)))
        w[:, :, [1, 2, 3, 5, 6, 7]] = v
        w[1, : n // 4] = w[0, : n // 4]  # equal states: numerators cancel
        if e < 300:  # density or pressure on either side of the range
            k = slice(n // 2, n // 2 + 32)
            w[:, k, 0] *= 2.0 ** -e
            k = slice(n // 2 + 32, n // 2 + 64)
            w[:, k, 4] *= 2.0 ** -e
            k = slice(n // 2 + 64, n // 2 + 96)
            w[:, k, 0] *= 2.0 ** e
            w[:, k, 4] *= 2.0 ** e
            k = slice(n // 2 + 96, n // 2 + 128)
            w[0, k, 1:4] *= 2.0 ** e
        w[0, -1, 4] = -1.0
        w[0, -2, 2] = np.nan
        w[0, -3, 6] = np.inf
        L.append(w[0])
        R.append(w[1])
    wL, wR = np.concatenate(L), np.concatenate(R)
    with np.errstate(all="ignore"):
        fo, so = O.riemann(method, direction, 1.4, wL, wR)
    fg, sg = A.riemann_batch(method, direction, 1.4, torch.from_numpy(wL).cuda(), torch.from_numpy(wR).cuda())
    fg, sg = fg.cpu().numpy(), sg.cpu().numpy()
    assert np.array_equal(so != 0, sg != 0)
    ok = so == 0
    same = _same_bits(fg[ok], fo[ok])
    assert same.all(), f"{method} {direction}: {int((~same).sum())} flux components differ"


@pytest.mark.parametrize("lim,ng", [("1st", 2), ("noSL", 2), ("minmod", 2), ("VanLeer", 2), ("Superbee", 2),
                                    ("MC", 2), ("Koren", 2), ("Cada3rd", 2), ("WENO3", 2), ("WENO5", 4)])
@pytest.mark.parametrize("variant", [2, 3, 7])
@pytest.mark.parametrize("planar", [True, False])
def test_stage_exponents(lim, ng, variant, planar):
    """Stage 1 of four blocks whose velocities and fields span the range, each
    stage kernel, with and without z components, against the oracle's stage."""
    import amr2d_mhd_amd as A

    cfg = dict(ic="rotor", limiter=lim, flux="HLLD", cfl=0.4, nx=16, nghosts=ng, maxlevs=1)
    sim, dom = A.Simulation(cfg), O.Domain(**cfg)
    sim.init()
    assert dom.init() == 0
    sim.set_stage_variant(variant)
    rng = np.random.default_rng(5)
    NT = 16 + 2 * ng
    for lo in (60, 805, 1020):  # inside the tiles' range, across its end, into underflow
        U = np.zeros((4, 8, NT, NT))
        e = rng.integers(0, lo, (4, 6, NT, NT)).astype(np.float64)
        U[:, 0] = rng.uniform(0.5, 2, (4, NT, NT))
        U[:, 4] = rng.uniform(5, 9, (4, NT, NT))
        vec = rng.normal(0, 0.3, (4, 6, NT, NT)) * np.exp2(-e) * (rng.random((4, 6, NT, NT)) < 0.8)
        if planar:
            vec[:, [2, 5]] = 0.0
        U[:, [1, 2, 3, 5, 6, 7]] = vec
        U[3, 1:4], U[3, 5:8] = 0.0, 0.0  # a block at rest
        Bi = np.ascontiguousarray(U[:, 5:7])
        sim.upload("U", U)
        sim.upload("Bi", Bi)
        dom.set_field(O.U, U)
        dom.set_field(O.BI, Bi)
        sim.set_time(0.0, 1e-3, 1e-3, 1)
        dom.set_time(0.0, 1e-3, 1e-3, 1)
        sim.stage(1)
        assert dom.stage(1) == 0
        for f, of in (("Us", O.US), ("ff", O.FF), ("gg", O.GG)):
            a, b = sim.download(f, nslots=4), dom.get_field(of, 4)
            same = _same_bits(np.ascontiguousarray(a), np.ascontiguousarray(b))
            assert same.all(), f"{lim} below 2^-{lo}: {f} differs in {int((~same).sum())} values"
    sim.close()


@pytest.mark.parametrize("lim,ng", [("1st", 2), ("noSL", 2), ("minmod", 1), ("VanLeer", 2), ("Superbee", 2),
                                    ("MC", 2), ("Koren", 2), ("Cada3rd", 2), ("WENO3", 2), ("WENO5", 3), ("WENO5", 4)])
@pytest.mark.parametrize("NT", [12, 17, 20, 28, 30])
def test_recon_batch_exponents_and_sizes(lim, ng, NT):
    """Tiles in LDS (up to 28 cells a side) and beyond: values in and out of
    the range against the oracle; entries outside the computed range are zeros
    from the binding and untouched by the C entry point."""
    torch = pytest.importorskip("torch")
    import amr2d_mhd_amd as A
    from amr2d_mhd_amd._lib import lib

    if NT < 2 * ng + 4:
        pytest.skip("smaller than the ghost depth allows")
    rng = np.random.default_rng(3 + NT)
    nt = 4
    W = rng.uniform(0.2, 2.0, (nt, 8, NT, NT))
    for t, lo in ((1, 700), (2, 830), (3, 1070)):
        W[t] *= np.exp2(-rng.integers(0, lo, W[t].shape).astype(np.float64)) * (rng.random(W[t].shape) < 0.9)
    dW = torch.from_numpy(W).cuda()
    torch.full((nt, 4, 8, NT, NT), 7.0, dtype=torch.float64, device="cuda")  # what an allocation may hold
    out = A.recon_batch(dW, lim, ng, dx=1.0 / 30).cpu().numpy()
    raw = torch.full((nt, 4, 8, NT, NT), 7.0, dtype=torch.float64, device="cuda")
    rc = lib().amr_recon_batch(NT, ng, lim.encode(), 1.0 / 30, nt, dW.data_ptr(), raw.data_ptr(),
                               torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    raw = raw.cpu().numpy()
    weno = lim.startswith("WENO")
    lo, hi = (ng - 1, NT - ng) if weno else (0, NT - 2)
    inside = np.zeros(out.shape, bool)
    inside[:, :, :, lo:hi + 1, lo:hi + 1] = True
    inside[:, 0:2, 5] = inside[:, 2:4, 6] = False
    for t in range(nt):
        (xl, xr, yl, yr), _ = O.recon_tile(W[t], lim, ng, dx=1.0 / 30)
        same = _same_bits(out[t], np.stack([xl, xr, yl, yr]))[inside[t]]
        assert same.all(), f"{lim}: tile {t} differs in {int((~same).sum())} entries"
    assert _same_bits(raw, out)[inside].all()
    assert (out[~inside].view(np.int64) == 0).all() and (raw[~inside] == 7.0).all()


@pytest.mark.parametrize("lim,ng", [("1st", 2), ("noSL", 2), ("minmod", 2), ("VanLeer", 2), ("Superbee", 2),
                                    ("MC", 2), ("Koren", 2), ("Cada3rd", 2), ("WENO3", 2), ("WENO5", 4)])
def test_recon_batch_upper_exponents(lim, ng):
    """Tiles on either side of the upper limit 2^100 and far beyond (WENO's weights
    are fourth powers: 2^254 squares of squares below overflow, 2^300 beyond), whole and
    mixed with small values."""
    torch = pytest.importorskip("torch")
    import amr2d_mhd_amd as A

    rng = np.random.default_rng(13)
    NT, scales = 20 if ng == 2 else 24, [98, 99, 100, 101, 200, 253, 300, 1000]
    W = np.empty((2 * len(scales), 8, NT, NT))
    for t, e in enumerate(scales):
        w = rng.uniform(0.5, 2.0, (2, 8, NT, NT)) * rng.choice([-1.0, 1.0], (2, 8, NT, NT))
        W[2 * t] = np.ldexp(w[0], e)
        W[2 * t + 1] = np.ldexp(w[1], rng.integers(-e, e + 1, w[1].shape))
    out = A.recon_batch(torch.from_numpy(W).cuda(), lim, ng, dx=1.0 / 30).cpu().numpy()
    lo, hi = (ng - 1, NT - ng) if lim.startswith("WENO") else (0, NT - 2)
    inside = np.zeros(out.shape[1:], bool)
    inside[:, :, lo:hi + 1, lo:hi + 1] = True
    inside[0:2, 5] = inside[2:4, 6] = False
    compared = 0
    for t in range(len(W)):
        with np.errstate(all="ignore"):
            (xl, xr, yl, yr), status = O.recon_tile(W[t], lim, ng, dx=1.0 / 30)
        if status:  # the oracle stops at a NaN edge
            continue
        compared += 1
        same = _same_bits(out[t], np.stack([xl, xr, yl, yr]))[inside]
        assert same.all(), f"{lim}, 2^{scales[t // 2]}: tile {t} differs in {int((~same).sum())} entries"
    assert compared >= (12 if lim.startswith("WENO") else 15)


@pytest.mark.parametrize("lim,ng", [("minmod", 2), ("MC", 2), ("Cada3rd", 2), ("WENO3", 2), ("WENO5", 4)])
@pytest.mark.parametrize("variant", [2, 3, 7])
def test_stage_upper_exponents(lim, ng, variant):
    """Stage 1 with densities around 2^+-60 and 2^+-100, momenta around 2^400, flux
    differences around 2^480 and cells around 2^+-100, against the oracle's stage.  (Noise small enough that no edge
    state is negative.)"""
    import amr2d_mhd_amd as A

    NT = 16 + 2 * ng
    # exponents of density, pressure and the domain's length
    cases = [(60, 60, 0), (-61, 59, 0), (98, 0, 0), (101, 0, 0), (-98, 0, 0), (-102, 0, 0), (99, 99, 0), (250, 540, 0),
             (250, 560, 0), (0, 470, 0), (0, 490, 0), (0, 0, 98), (0, 0, 110), (0, 0, -92), (0, 0, -110),
             (101, 101, -110)]
    for er, ep, el in cases:
        if lim.startswith("WENO") and ep > 240:  # its weights' fourth powers overflow
            continue
        cfg = dict(ic="rotor", limiter=lim, flux="HLLD", cfl=0.4, nx=16, nghosts=ng, maxlevs=1, lenx=2.0 ** el)
        sim, dom = A.Simulation(cfg), O.Domain(**cfg)
        sim.init()
        assert dom.init() == 0
        sim.set_stage_variant(variant)
        rng = np.random.default_rng(abs(er) + 7)
        v, b = 2.0 ** ((ep - er) / 2), 2.0 ** (ep / 2)
        U = np.zeros((4, 8, NT, NT))
        U[:, 0] = np.ldexp(rng.uniform(0.9, 1.1, (4, NT, NT)), er)
        w = rng.normal(0, 0.1, (4, 6, NT, NT))
        U[:, 1:4] = U[:, :1] * (w[:, :3] * v)
        U[:, 5:8] = w[:, 3:] * b
        U[:, 4] = np.ldexp(rng.uniform(9.5, 10.5, (4, NT, NT)), ep)
        U[2:, [3, 7]] = 0.0  # blocks without z components
        Bi = np.ascontiguousarray(U[:, 5:7])
        dt = 1e-3 * 2.0 ** el / v
        sim.upload("U", U)
        sim.upload("Bi", Bi)
        dom.set_field(O.U, U)
        dom.set_field(O.BI, Bi)
        sim.set_time(0.0, dt, dt, 1)
        dom.set_time(0.0, dt, dt, 1)
        sim.stage(1)
        assert dom.stage(1) == 0
        for f, of in (("Us", O.US), ("ff", O.FF), ("gg", O.GG)):
            a, o = sim.download(f, nslots=4), dom.get_field(of, 4)
            same = _same_bits(np.ascontiguousarray(a), np.ascontiguousarray(o))
            assert same.all(), f"{lim}, rho 2^{er}, p 2^{ep}, length 2^{el}: {f} differs in {int((~same).sum())} values"
        sim.close()
