"""The frozen-mesh step and its reverse in place (outputs on the inputs they
replace) against the same calls with buffers of their own, bitwise: every entry
point of the C interface, whole buffers and x and y faces exchanged, grids of one
tile, of odd sizes and of several tiles."""
import ctypes as C

import pytest

pytestmark = pytest.mark.gpu

GAMMA = 5.0 / 3.0


def _setup(n, flux):
    import torch

    from amr2d_mhd_amd import adjoint as AD

    rho, v, p, Bx, By = AD.orszag_tang_controls(n, modulation=0.05, noise=1e-2)
    U = AD.cons_from_controls(rho, v, p, Bx, By, GAMMA).contiguous()
    gen = torch.Generator().manual_seed(n)
    cot = [torch.randn(t.shape, generator=gen, dtype=torch.float64).cuda() for t in (U, Bx, By)]
    return AD.FrozenMesh(n, 1.0 / n, GAMMA, flux), (U, Bx, By), cot, 0.2 / n


def _ptrs(*ts):
    return [C.c_void_p(t.data_ptr()) for t in ts]


@pytest.mark.parametrize("n", [4, 16, 61, 200])
@pytest.mark.parametrize("flux", ["HLLE", "HLLD"])
def test_step_in_place(n, flux):
    import torch

    from amr2d_mhd_amd._lib import lib

    mesh, state, _, dt = _setup(n, flux)
    tape = mesh.new_tapes(2, "cuda")
    want = mesh.step(*state, dt, tape[0])
    st = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    for call in ("step", "tape", "noalloc", "exchanged"):
        U, Bx, By = (t.clone() for t in state)
        a = _ptrs(U, Bx, By)
        out = [a[0], a[2], a[1]] if call == "exchanged" else a
        if call == "noalloc":
            rc = lib().amr_adj_step_noalloc(n, 1.0 / n, GAMMA, flux.encode(), *a, dt, *out, st)
        elif call == "tape":
            rc = lib().amr_adj_step_tape(mesh.h, *a, dt, *out, C.c_void_p(tape[1].data_ptr()), st)
        else:
            rc = lib().amr_adj_step(mesh.h, *a, dt, *out, st)
        assert rc == 0
        got = (U, By, Bx) if call == "exchanged" else (U, Bx, By)
        assert all(torch.equal(x, y) for x, y in zip(got, want)), call
    assert torch.equal(tape[0], tape[1])
    mesh.close()


@pytest.mark.parametrize("n", [4, 16, 61, 200, 300])
@pytest.mark.parametrize("flux", ["HLLE", "HLLD"])
def test_reverse_in_place(n, flux):
    import torch

    from amr2d_mhd_amd._lib import lib

    mesh, state, cot, dt = _setup(n, flux)
    tape = mesh.new_tapes(1, "cuda")[0]
    mesh.step(*state, dt, tape)
    want = mesh.vjp(tape, state[1], state[2], dt, *cot)
    st = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    for call in ("tape", "recomputing", "exchanged", "faces only"):
        g = [t.clone() for t in cot]
        a = _ptrs(*g)
        o = [torch.empty_like(t) for t in g]
        out = {"exchanged": [a[0], a[2], a[1]], "faces only": [_ptrs(o[0])[0], a[1], a[2]]}.get(call, a)
        if call == "recomputing":
            rc = lib().amr_adj_step_vjp(mesh.h, *_ptrs(*state), dt, *a, *out, st)
        else:
            rc = lib().amr_adj_vjp_tape(mesh.h, *_ptrs(tape, state[1], state[2]), dt, *a, *out, st)
        assert rc == 0
        got = {"exchanged": (g[0], g[2], g[1]), "faces only": (o[0], g[1], g[2])}.get(call, g)
        assert all(torch.equal(x, y) for x, y in zip(got, want)), call
    mesh.close()
