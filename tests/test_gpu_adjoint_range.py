"""The frozen-mesh reverse over the whole exponent range.

The device forms its quotients with shared reciprocals where the values that it
meets lie within a checked range, and with plain divisions elsewhere.  Either
way every quotient is the correctly rounded one, so the reverse must equal, bit
for bit, the same reverse on the host: the pointwise pieces built for the host
(amr_debug_*), put together in numpy in the kernels' order.  Cotangents up to
overflow and down to underflow, components that decay through 2^-1060, and
states too large for the shared reciprocals."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GAMMA = 5.0 / 3.0


def _faces_reverse(W, Bn, d, fb, flux):
    """Contributions S[s, k, j, i] to the four stencil cells of every face of
    direction d, and the normal field's adjoint."""
    from amr2d_mhd_amd._lib import lib

    L = lib()
    solver = L.amr_debug_hlld_vjp if flux == "HLLD" else L.amr_debug_hlle_vjp
    n = W.shape[-1]
    S, Bnb, nc = np.zeros((4, 8, n, n)), np.zeros((n, n)), 5 + d
    axis = 2 - d
    st = np.ascontiguousarray(np.moveaxis(np.stack([np.roll(W, 2 - s, axis) for s in range(4)]), (0, 1), (3, 2)))
    order = [0, 2, 1, 3, 4, 6, 5, 7] if d else list(range(8))  # the grid frame's components in the face's
    vb, wlr, f = np.zeros(4), np.zeros(2), np.zeros(8)
    for j in range(n):
        for i in range(n):
            w = np.zeros((2, 8))
            for k in range(8):
                L.amr_debug_recon_minmod_vjp(st[j, i, k].ctypes.data, 0.0, 0.0, vb.ctypes.data, wlr.ctypes.data)
                w[:, k] = wlr
            w[:, nc] = Bn[j, i]
            wl, wr = np.ascontiguousarray(w[0, order]), np.ascontiguousarray(w[1, order])
            g, lb, rb = np.ascontiguousarray(fb[order, j, i]), np.zeros(8), np.zeros(8)
            args = [wl.ctypes.data, wr.ctypes.data, GAMMA, g.ctypes.data, lb.ctypes.data, rb.ctypes.data]
            solver(*(args + [f.ctypes.data] if flux == "HLLD" else args))
            lb, rb = lb[order], rb[order]
            Bnb[j, i] = lb[nc] + rb[nc]
            for k in range(8):
                if k != nc:
                    L.amr_debug_recon_minmod_vjp(st[j, i, k].ctypes.data, lb[k], rb[k], vb.ctypes.data,
                                                 wlr.ctypes.data)
                    S[:, k, j, i] = vb
    return S, Bnb


def _stage_reverse(Q, pre, Bx, By, Binx, Biny, W, Bnx, Bny, s, dx, flux):
    """Reverse of a stage: the updated faces' adjoints (x, y), the pre-sync state's,
    what the fluxes add to the stage input's, and the normal fields' parts."""
    xm, xp = (lambda a: np.roll(a, 1, -1)), (lambda a: np.roll(a, -1, -1))
    ym, yp = (lambda a: np.roll(a, 1, -2)), (lambda a: np.roll(a, -1, -2))
    bbx, bby = Q[5] + Q[4] * (0.5 * (xp(Bx) + Bx)), Q[6] + Q[4] * (0.5 * (yp(By) + By))
    x, y = Binx + 0.5 * (bbx + xm(bbx)), Biny + 0.5 * (bby + ym(bby))
    rx, ry = s * x, s * y
    Eb = (1.0 / dx) * (ym(rx) - rx) - (1.0 / dx) * (xm(ry) - ry)
    q = Q.copy()
    q[5], q[6] = -Q[4] * pre[0], -Q[4] * pre[1]
    fx, fy = (s * xm(q) - s * q) / dx, (s * ym(q) - s * q) / dx
    fx[6] -= 0.25 * (Eb + yp(Eb))
    fy[5] += 0.25 * (Eb + xp(Eb))
    Sx, bx = _faces_reverse(W, Bnx, 0, fx, flux)
    Sy, by = _faces_reverse(W, Bny, 1, fy, flux)
    wb = np.zeros_like(Q)
    for t in range(4):  # position t of the face t - 2 cells below: this cell's is 2 - t above
        wb = wb + np.roll(Sx[t], t - 2, -1)
    for t in range(4):
        wb = wb + np.roll(Sy[t], t - 2, -2)
    g1, iw0, pb, ub = GAMMA - 1, 1.0 / W[0], wb[4], np.zeros_like(Q)
    w0b = wb[0] + pb * (-g1 * 0.5 * (W[1] * W[1] + W[2] * W[2] + W[3] * W[3]))
    ub[4] += pb * g1
    for k in (1, 2, 3):
        wkb = wb[k] - pb * g1 * W[0] * W[k]
        ub[k] += wkb * iw0
        w0b = w0b - wkb * W[k] * iw0
    ub[0] += w0b
    for k in (5, 6, 7):
        ub[k] += wb[k] - pb * g1 * W[k]
    return x, y, q, ub, bx, by


def _host_vjp(tape, Bx, By, dt, dx, cot, flux):
    n = Bx.shape[0]
    t = tape.reshape(24, n, n)
    W1, W2, Bxs, Bys, pre1, pre2, Bxo, Byo = t[:8], t[8:16], t[16], t[17], t[18:20], t[20:22], t[22], t[23]
    Uob, Bxob, Byob = cot
    x, y, q, ub, bx, by = _stage_reverse(Uob, pre2, Bxo, Byo, Bxob, Byob, W2, Bxs, Bys, -0.5 * dt, dx, flux)
    Ub, Usb = 0.5 * q, 0.5 * q + ub
    Bxb, Byb, Bsbx, Bsby = 0.5 * x, 0.5 * y, 0.5 * x + bx, 0.5 * y + by
    x, y, q, ub, bx, by = _stage_reverse(Usb, pre1, Bxs, Bys, Bsbx, Bsby, W1, Bx, By, -dt, dx, flux)
    return (Ub + q) + ub, (Bxb + x) + bx, (Byb + y) + by


def _state(kind, n, rng):
    """Controls (rho, v, p, Bx, By) and Bz of a noisy vortex; `decayed`: the vector
    components times 2^-e, e up to 1060, cell by cell; `large`, `small`: density and
    pressure times 2^+-180."""
    import torch

    from amr2d_mhd_amd import adjoint as AD

    rho, v, p, Bx, By = AD.orszag_tang_controls(n, modulation=0.05, noise=1e-2)
    r = lambda *s: torch.from_numpy(rng.standard_normal(s)).cuda()
    v[2] = 0.3 * r(n, n)
    Bz = 0.2 * r(n, n)
    if kind == "decayed":
        f = lambda *s: torch.from_numpy(np.exp2(-rng.integers(0, 1061, s).astype(float)) * (rng.random(s) < 0.8)).cuda()
        v, Bz, Bx, By = v * f(3, n, n), Bz * f(n, n), Bx * f(n, n), By * f(n, n)
    elif kind != "vortex":
        a = 2.0 ** (180 if kind == "large" else -180)
        rho, p, Bx, By, Bz = rho * a, p * a, Bx * a ** 0.5, By * a ** 0.5, Bz * a ** 0.5
    U = AD.cons_from_controls(rho, v, p, Bx, By, GAMMA)
    U[4] += 0.5 * Bz * Bz
    U[7] = Bz
    return U.contiguous(), Bx.contiguous(), By.contiguous()


@pytest.mark.parametrize("flux", ["HLLE", "HLLD"])
@pytest.mark.parametrize("kind,scales", [
    ("vortex", (0, -600, -960, -1040, 600, 960, 1010, 1016)),
    ("decayed", (0, -600, 900)),
    ("large", (0, -960, 700)),
    ("small", (0, -960, 960)),
])
def test_reverse_equals_host_bitwise(flux, kind, scales):
    import torch

    from amr2d_mhd_amd import adjoint as AD
    from amr2d_mhd_amd._lib import lib

    n = 18  # two tiles a side, the second of two columns (16 x 13 cells a tile)
    rng = np.random.default_rng(11)
    U, Bx, By = _state(kind, n, rng)
    mesh = AD.FrozenMesh(n, 1.0 / n, GAMMA, flux)
    dt = 0.2 / n
    tape = mesh.new_tapes(1, U.device)[0]
    mesh.step(U, Bx, By, dt, tape)
    base = [rng.standard_normal(s) for s in ((8, n, n), (n, n), (n, n))]
    bx, by, tp = Bx.cpu().numpy(), By.cpu().numpy(), tape.cpu().numpy()
    for e in scales:
        cot = [np.ldexp(c, e) for c in base]
        with np.errstate(all="ignore"):
            want = _host_vjp(tp, bx, by, dt, 1.0 / n, cot, flux)
        gc = [torch.from_numpy(c).cuda() for c in cot]
        for mode in (1, 2):
            assert lib().amr_debug_adj_set_fused(mesh.h, mode) == 0
            got = [t.cpu().numpy() for t in mesh.vjp(tape, Bx, By, dt, *gc)]
            for name, a, b in zip(("U", "Bx", "By"), got, want):
                same = (a.view(np.int64) == b.view(np.int64)) | (np.isnan(a) & np.isnan(b))
                assert same.all(), f"{kind}, cotangents 2^{e}, form {mode}: {int((~same).sum())} values of {name} differ"
    mesh.close()
