"""Learned warm start on the GPU: FP16-MFMA inference and FP32 training
kernels against the FP64 CNN oracle (oracle/cnn_oracle.py), and the fallback
rule of the warm start."""
import ctypes

import cnn_oracle as C
import numpy as np
import pyoracle
import pytest
import torch

from cup3d_amd import workloads as W
from cup3d_amd.poisson import PoissonSolver, lib, solver_for
from helpers import grid_cases, nbr_table, random_field

pytestmark = pytest.mark.gpu


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a, np.float64).reshape(-1)).cuda()


def smooth_fields(blocks, h0, seed):
    from helpers import cell_centres
    X, h = cell_centres(blocks, h0)
    rng = np.random.default_rng(seed)
    k = rng.uniform(1, 3, (2, 3))
    prev = np.cos(2 * np.pi * (X @ k[0])) + 0.1 * rng.standard_normal(X.shape[:-1])
    rhs = (h ** 3)[:, None, None, None] * np.sin(2 * np.pi * (X @ k[1]))
    return rhs, prev, h


def residual(blocks, bpd, h0, bc, rhs, prev):
    """b - A p_prev with the oracle's operator (bMean = 0)."""
    O = pyoracle.Oracle(blocks, bpd, h0, bc, 0)
    return rhs.reshape(-1) - O.spmv(prev.reshape(-1))


@pytest.mark.parametrize("name", ["uniform_walls_3x2x2", "amr2_periodic_offcentre", "amr3_walls"])
def test_predict_matches_oracle(gpu, name):
    blocks, bpd, h0, bc = grid_cases()[name]
    S = PoissonSolver(bpd, h0, bc, bmean=0).set_topology(blocks)
    w = C.init_weights(5)
    w[C.NW - 1] = 0.05
    S.cnn_set_weights(w.astype(np.float32))
    rhs, prev, h = smooth_fields(blocks, h0, 1)
    out = torch.zeros(len(blocks) * 512, dtype=torch.float64, device=gpu)
    S.cnn_predict(dev(rhs), dev(prev), out)
    res = residual(blocks, bpd, h0, bc, rhs, prev)
    ref = C.predict(w, res, prev, h, nbr_table(blocks, bpd, bc))
    inc_g = out.cpu().numpy().reshape(ref.shape) - prev
    inc_o = ref - prev
    # FP16 weights and activations, FP32 accumulation: ~1e-3 of the increment
    rel = np.linalg.norm(inc_g - inc_o) / np.linalg.norm(inc_o)
    assert rel < 1e-2, rel


@pytest.mark.parametrize("lam", [0.0, 0.6])
def test_gradient_matches_oracle(gpu, lam):
    blocks, bpd, h0, bc = grid_cases()["amr2_periodic_offcentre"]
    S = PoissonSolver(bpd, h0, bc, bmean=0).set_topology(blocks)
    w = C.init_weights(7)
    w[C.NW - 1] = 0.02
    S.cnn_set_weights(w.astype(np.float32))
    rhs, prev, h = smooth_fields(blocks, h0, 2)
    p = prev + 0.3 * random_field(len(blocks), 3)
    S.cnn_add_sample(dev(rhs), dev(prev), dev(p))
    L = lib()
    f = L.cup3d_debug_cnn_gradient
    f.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_float, ctypes.c_void_p,
                  ctypes.POINTER(ctypes.c_double)]
    g = np.zeros(C.NW, np.float32)
    loss = ctypes.c_double()
    assert f(S.h, 0, lam, g.ctypes.data, ctypes.byref(loss)) == 0
    res = residual(blocks, bpd, h0, bc, rhs, prev)
    x, s_r, _ = C.inputs(res, prev, h, nbr_table(blocks, bpd, bc))
    h3 = (h ** 3)[:, None, None, None]
    target = (p - prev - np.sum(h3 * (p - prev)) / (512 * np.sum(h3))) / s_r
    th = C.halo(target, nbr_table(blocks, bpd, bc))
    lo, go = C.loss_and_grad(w.astype(np.float32).astype(np.float64), x, target, lam, th)
    assert abs(loss.value - lo) < 1e-4 * lo
    assert np.linalg.norm(g - go) < 1e-3 * np.linalg.norm(go)


def test_training_reduces_loss_and_fallback(gpu):
    """Train on a short sequence of solver triples at small size; the loss
    falls, and the warm start never uses a guess worse than p_prev."""
    w = W.c4_uniform_sequence((8, 4, 4))
    S = solver_for(w, tol_rel=0.0, tol_rhs=1e-9, bmean=1)
    prev = torch.zeros(w.ncells, dtype=torch.float64, device=gpu)
    rhs0 = dev(w.rhs(step=0))
    S.solve_device(rhs0, prev)
    sols = []
    for t in range(1, 11):
        b = dev(w.rhs(step=t))
        x = prev.clone()
        S.solve_device(b, x)
        sols.append((b, prev.clone(), x.clone()))
        prev = x
    for b, pp, x in sols[:8]:
        S.cnn_add_sample(b, pp, x)
    l0, _ = S.cnn_train(1, batch=64, lr=1e-3, seed=1)
    _, l1 = S.cnn_train(200, batch=64, lr=1e-3, seed=2)
    assert l1 < 0.5 * l0, (l0, l1)
    # held-out step: warm start with fallback
    Sg = solver_for(w, tol_rel=0.0, tol_rhs=1e-7, guess="cnn")
    Sg.cnn_set_weights(S.cnn_get_weights())
    b, pp, _ = sols[9]
    x = pp.clone()
    rep = Sg.solve_device(b, x)
    Sp = solver_for(w, tol_rel=0.0, tol_rhs=1e-7)
    x2 = pp.clone()
    rep2 = Sp.solve_device(b, x2)
    assert rep["status"] == 0 and rep2["status"] == 0
    assert rep["guess_resid"] <= rep2["err_init"] * (1 + 1e-12)
    # what the trained net gains: on this held-out step its guess (scaled by
    # the residual-minimising step) starts the solve from a residual at least
    # 10 % below the previous pressure's (0.58 of it in the runs so far)
    assert rep["guess_used"] == 2 and rep["guess_resid"] < 0.9 * rep2["err_init"]
    print("guess used", rep["guess_used"], "resid net/prev", rep["guess_resid"] / rep2["err_init"],
          "iters", rep["iterations"], "vs", rep2["iterations"])


@pytest.mark.parametrize("batch", [1, 17, 9000])
def test_training_is_the_same_for_every_batch_of_one_item(gpu, batch):
    """On a grid of one block with one sample every item of every minibatch is
    the same one, so the mean gradient and the Adam steps do not depend on the
    batch size: 1 (empty groups of the gradient sum), 17 (a ragged one) and
    9000 (one step per uploaded item list) against 16. Adding n equal terms in
    FP32 is off by at most n / 16 + 16 roundings, 3.5e-5 relative, and an Adam
    step by about twice that; the bar is 1e-3 of the length of three steps."""
    blocks = np.zeros((1, 4), np.int32)
    S = PoissonSolver((1, 1, 1), 0.125, (2, 2, 2), bmean=0).set_topology(blocks)
    rhs, prev, _ = smooth_fields(blocks, 0.125, 3)
    S.cnn_add_sample(dev(rhs), dev(prev), dev(1.1 * prev))
    w0 = C.init_weights(6).astype(np.float32)
    out = []
    for n in (16, batch):
        S.cnn_set_weights(w0)
        loss = S.cnn_train(3, batch=n, lr=1e-3, seed=4, res_weight=0.5)
        out.append((S.cnn_get_weights(), loss))
    moved = np.linalg.norm(out[0][0] - w0)
    assert moved > 0.5 * 1e-3 * np.sqrt(len(w0))
    assert np.linalg.norm(out[1][0] - out[0][0]) <= 1e-3 * 3e-3 * np.sqrt(len(w0))
    assert np.allclose(out[1][1], out[0][1], rtol=1e-4)


@pytest.mark.parametrize("name", ["uniform_walls_3x2x2", "amr3_walls"])
@pytest.mark.parametrize("bmean", [0, 1])
def test_predict_in_place_equals_out_of_place(gpu, name, bmean):
    """Where out overlaps prev (or the mean constraint zeroes a cell) the net
    reads a copy and its scales are summed in passes of their own, otherwise
    residual and scales are one pass over rhs and prev. The scales then differ
    by FP64 rounding at most, which moves an FP16 input by one rounding in
    2^42 cases: the predictions agree to 1e-6 of the increment."""
    blocks, bpd, h0, bc = grid_cases()[name]
    S = PoissonSolver(bpd, h0, bc, bmean=bmean).set_topology(blocks)
    S.cnn_set_weights(C.init_weights(5).astype(np.float32))
    rhs, prev, _ = smooth_fields(blocks, h0, 2)
    rhs, prev = dev(rhs), dev(prev)
    out, inplace = torch.zeros_like(prev), prev.clone()
    S.cnn_predict(rhs, prev, out)
    S.cnn_predict(rhs, inplace, inplace)
    assert torch.linalg.norm(out - inplace) <= 1e-6 * torch.linalg.norm(out - prev)


@pytest.mark.parametrize("bpd,bc", [((1, 1, 1), 2), ((1, 1, 1), 1), ((2, 1, 3), 1), ((3, 3, 3), 0)])
def test_predict_of_rough_fields_cell_by_cell(gpu, bpd, bc):
    """White-noise inputs on the smallest grids (a block that is its own
    neighbour, walls on all sides), the largest error of any cell: a halo cell
    or a zero of the padding taken from the wrong place moves cells next to it
    by one of 27 taps, about 0.2 of a typical increment. FP16 inputs, weights
    and two layers of activations each round by 2^-12 RMS of a term, so a cell
    of three layers is off by about 1e-3, and the worst of 14 000 by 5e-3."""
    blocks = W.uniform_blocks(*bpd)
    S = PoissonSolver(bpd, 0.125, (bc,) * 3, bmean=0).set_topology(blocks)
    w = C.init_weights(9)
    S.cnn_set_weights(w.astype(np.float32))
    rng = np.random.default_rng(11)
    shape = (len(blocks), 8, 8, 8)
    prev = rng.standard_normal(shape)
    rhs = 0.125 ** 3 * rng.standard_normal(shape)
    out = torch.zeros(prev.size, dtype=torch.float64, device=gpu)
    S.cnn_predict(dev(rhs), dev(prev), out)
    res = residual(blocks, bpd, 0.125, (bc,) * 3, rhs, prev)
    ref = C.predict(w, res, prev, np.full(len(blocks), 0.125), nbr_table(blocks, bpd, (bc,) * 3))
    err = np.abs(out.cpu().numpy().reshape(shape) - ref).max()
    inc = np.sqrt(np.mean((ref - prev) ** 2))
    assert err <= 0.02 * inc, (err, inc)
