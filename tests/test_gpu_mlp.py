"""The flux-correction network's BF16 MFMA kernels against the FP64 oracle
(oracle/mlp_oracle.py), and the solver hooks of the learned correction.

Tolerances: the device rounds weights and activations to BF16 (8-bit
mantissa) and accumulates in FP32, the oracle uses the same BF16-rounded
weights and inputs with FP64 activations. Outputs agree to 2e-2 of their
scale, gradients to 3e-2 relative L2 per parameter block.
"""
import numpy as np
import pytest

from fall3d_amd import ads
from fall3d_amd.problem import random_problem
from oracle import mlp_oracle as mo

pytestmark = pytest.mark.gpu


def _params(seed):
    rng = np.random.default_rng(seed)
    p = mo.init_params(seed)
    p["b1"] = rng.standard_normal(mo.NH) * 0.2
    p["b2"] = rng.standard_normal(mo.NH) * 0.2
    p["b3"] = np.asarray(0.1)
    return p


def _bf16_params(p):
    return {k: mo.bf16_round(v) for k, v in p.items()}


def _inputs(n, seed):
    rng = np.random.default_rng(seed)
    x = rng.uniform(-1.0, 1.0, (n, 32))
    x[:, 31] = 0.0
    bits = ads.bf16_bits(x)
    return bits, ads.bf16_value(bits).astype(np.float64)


def test_forward_matches_oracle():
    p = _params(3)
    net = ads.Network(params=mo.flatten(p).astype(np.float32))
    bits, x = _inputs(1000, 4)  # not a multiple of the 16-row tile
    y = net.forward(bits)
    yr, _ = mo.forward(_bf16_params(p), x)
    err = np.abs(y - yr).max() / np.abs(yr).max()
    print(f"forward max err {err:.3e}", flush=True)
    assert err <= 2e-2
    net.release()


def test_gradient_matches_oracle():
    p = _params(5)
    net = ads.Network(params=mo.flatten(p).astype(np.float32))
    bits, x = _inputs(2050, 6)
    rng = np.random.default_rng(7)
    t = rng.standard_normal(x.shape[0]).astype(np.float32)
    g, sse = net.gradient(bits, t)
    loss_r, gr = mo.loss_and_grad(_bf16_params(p), x, t.astype(np.float64))
    assert abs(sse / x.shape[0] - loss_r) <= 2e-2 * loss_r
    gd = mo.unflatten(g.astype(np.float64))
    for k, _ in mo.PARAM_SHAPES:
        a, b = np.ravel(gd[k]), np.ravel(gr[k])
        e = np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30)
        print(f"grad {k}: rel L2 {e:.3e}", flush=True)
        assert e <= 3e-2, k
    net.release()


def test_training_fits_a_teacher_network():
    """Adam on random batches of rows generated by a fixed teacher network:
    the student's loss falls by more than 10x."""
    teacher = _params(11)
    teacher["w3"] = teacher["w3"] * 0.5
    bits, x = _inputs(200_000, 12)
    t, _ = mo.forward(_bf16_params(teacher), x)
    net = ads.Network(capacity=x.shape[0], params=mo.flatten(mo.init_params(13)).astype(np.float32))
    net.append(bits, t.astype(np.float32))
    assert net.count() == x.shape[0]
    loss = net.train(400, batch=8192, lr=2e-3, seed=1)
    print(f"loss {loss[0]:.4e} -> {loss[-1]:.4e}", flush=True)
    assert loss[-20:].mean() < 0.1 * loss[:5].mean()
    net.release()


@pytest.mark.parametrize("nx,cpt", [(21, 0), (150, 2)])
def test_face_flux_output_is_the_update_divergence(nx, cpt):
    """With face-flux output on, one drop-in x (y) sweep changes each interior
    cell by exactly -(Phi(f+1) - Phi(f)) / dxb (FP32 rounding), and the
    boundary faces carry the conservation ledger's fluxes; also with x lines
    over two waves (150 cells at 2 per lane: 76 lanes)."""
    p = random_problem(nx, 17, 6, 2, seed=3, stretched=False)
    g = ads.ADS(p.nx, p.ny, p.nz, p.nb, "minmod", "rk", 8, "fp32", grid=p.grid)
    if cpt:
        g.set_tiling(0, cells_per_thread=cpt)
    u, v, w = g.get_vcomps()
    u[...] = p.u1
    v[...] = p.v1
    g.set_flux_output(True)
    c0 = p.c0.copy(order="F")
    c1 = c0.copy(order="F")
    dt = 30.0
    g.solve_along_x(0.0, 0.0, dt, c1, p.k1)
    fx = g.face_flux(0)  # (nx+3, ny, nz, nb), face f between cells f-1 and f
    dxb = p.grid["dX1_b"][1:p.nx + 1]
    dc = c1[2:p.nx + 2, 2:p.ny + 2, 2:p.nz + 2, :] - c0[2:p.nx + 2, 2:p.ny + 2, 2:p.nz + 2, :]
    div = -(fx[2:p.nx + 2] - fx[1:p.nx + 1]) / dxb[:, None, None, None]
    scale = np.abs(c0).max()
    assert np.abs(dc - div).max() <= 2e-6 * scale
    g.set_flux_output(True)  # zero the accumulators
    c2 = c1.copy(order="F")
    g.solve_along_y(0.0, 0.0, dt, c2, p.k2)
    fy = g.face_flux(1)  # (nx, ny+3, nz, nb)
    dyb = p.grid["dX2_b"][1:p.ny + 1]
    dc = c2[2:p.nx + 2, 2:p.ny + 2, 2:p.nz + 2, :] - c1[2:p.nx + 2, 2:p.ny + 2, 2:p.nz + 2, :]
    div = -(fy[:, 2:p.ny + 2] - fy[:, 1:p.ny + 1]) / dyb[None, :, None, None]
    assert np.abs(dc - div).max() <= 2e-6 * scale
    g.release()


def test_zero_network_leaves_the_plain_step_unchanged():
    from fall3d_amd.problem import operational_problem
    p = operational_problem(40, 36, 12, 2, seed=2)
    out = []
    for learned in (False, True):
        g = ads.ADS(p.nx, p.ny, p.nz, p.nb, "minmod", "rk", 8, "fp32")
        g.set_problem(p)
        net = ads.Network(params=np.zeros(ads.Network().nparam, dtype=np.float32)) if learned else None
        g.set_learned(net)
        dt = g.time_step(0.0, 2, 0.9)
        g.run(dt, 6, 0)
        out.append(g.get_state()[0])
        g.release()
    assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize("rows", [1, 31, 33, 127, 129, 512, 16385, 17000])
def test_gradient_sums_at_the_sizes_of_the_reduction(rows):
    """Batches that end inside a 32-row chunk, inside a workgroup's four, and
    with fewer and more chunks per slot than the rows a slot reads ahead:
    the gradient against the oracle (BF16 tolerances as above)."""
    p = _params(21)
    net = ads.Network(params=mo.flatten(p).astype(np.float32))
    bits, x = _inputs(rows, rows)
    t = np.random.default_rng(rows).standard_normal(rows).astype(np.float32)
    g, sse = net.gradient(bits, t)
    loss_r, gr = mo.loss_and_grad(_bf16_params(p), x, t.astype(np.float64))
    assert abs(sse / rows - loss_r) <= 2e-2 * loss_r
    gd = mo.unflatten(g.astype(np.float64))
    for k, _ in mo.PARAM_SHAPES:
        a, b = np.ravel(gd[k]), np.ravel(gr[k])
        assert np.linalg.norm(a - b) <= 3e-2 * max(np.linalg.norm(b), 1e-30), k
    net.release()


def test_one_update_packs_what_it_learned():
    """After an update the next pass runs on the new parameters: the network's
    outputs equal those of a fresh network given the parameters read back
    (the operands packed by the update against the ones packed from scratch)."""
    bits, x = _inputs(5000, 31)
    net = ads.Network(capacity=5000, params=mo.flatten(_params(32)).astype(np.float32))
    net.append(bits, np.sin(x.sum(1)).astype(np.float32))
    net.train(3, batch=777, lr=1e-2, seed=5)
    fresh = ads.Network(params=net.params())
    assert np.array_equal(net.forward(bits[:1000]), fresh.forward(bits[:1000]))
    g0, _ = net.gradient(bits[:500], np.zeros(500, np.float32))
    g1, _ = fresh.gradient(bits[:500], np.zeros(500, np.float32))
    assert np.array_equal(g0, g1)
    net.release()
    fresh.release()
