"""The surrogate's HIP kernels against the FP64 FNO oracle: the bf16
matrix-core GEMM (operand and result lane layout), the forward pass, every
parameter gradient, and a few Adam steps.  Tolerances are those of bf16
operands with FP32 accumulation (8 significant bits per product operand)."""
import numpy as np
import pytest

from ehd_amd import fno as G
from oracle import fno_oracle as F

pytestmark = pytest.mark.gpu


def _bf16(x):
    """Round float32 to bf16 (nearest even) and back, as the kernel stages operands."""
    u = np.ascontiguousarray(x, dtype=np.float32).view(np.uint32).astype(np.uint64)
    u = (u + 0x7FFF + ((u >> 16) & 1)) >> 16
    return (u.astype(np.uint32) << 16).view(np.float32)


@pytest.mark.parametrize("mnk", [(16, 16, 16), (37, 45, 29), (130, 70, 200), (64, 1, 7), (1, 129, 33)])
def test_gemm_matches_bf16_reference(mnk):
    M, N, K = mnk
    rng = np.random.default_rng(M * 1000 + N)
    A = rng.standard_normal((M, K)).astype(np.float32)
    B = rng.standard_normal((K, N)).astype(np.float32)
    got = G.gemm(A, B)
    ref = _bf16(A).astype(np.float64) @ _bf16(B).astype(np.float64)   # bf16 products are exact in FP32
    scale = np.abs(_bf16(A)).astype(np.float64) @ np.abs(_bf16(B)).astype(np.float64)
    assert np.all(np.abs(got - ref) <= 1e-5 * scale + 1e-6), np.max(np.abs(got - ref) / (scale + 1e-30))


def _up4(v):
    return (v + 3) // 4 * 4


def _operand(layout, R, K, nb, rng):
    """Flat host array of nb (R x K) matrices (R = m for A, n for B) in the
    given layout; returns (flat, (r stride, k stride, batch stride), dense)."""
    if layout == "k":        # k unit-stride, rows 16-byte aligned
        sr, sk = _up4(K + 1), 1
    elif layout == "r":      # m / n unit-stride
        sr, sk = 1, _up4(R + 1)
    else:                    # odd strides: element staging
        sr, sk = 3, 3 * R + 1
    sb = _up4((R - 1) * sr + (K - 1) * sk + 5)
    flat = rng.standard_normal(nb * sb).astype(np.float32)
    r, k = np.meshgrid(np.arange(R), np.arange(K), indexing="ij")
    dense = np.stack([flat[b * sb + r * sr + k * sk] for b in range(nb)])
    return flat, (sr, sk, sb), dense


def _result_strides(layout, M, N, ns):
    """(cm, cn, c1, c2) of C: n unit-stride with every offset a multiple of 4
    floats ("n"), the same along m ("m"), or odd offsets ("x")."""
    if layout == "n":
        cm, cn = _up4(N + 1), 1
        c2 = M * cm + 4
        return cm, cn, ns * c2 + 8, c2
    if layout == "m":
        cm, cn = 1, _up4(M + 1)
        c2 = N * cn + 4
        return cm, cn, ns * c2 + 8, c2
    cm, cn = N + 3, 1
    c2 = M * cm + 1
    return cm, cn, ns * c2 + 7, c2


@pytest.mark.parametrize("la", ["k", "r", "x"])
@pytest.mark.parametrize("lb", ["k", "r", "x"])
@pytest.mark.parametrize("lc", ["n", "m", "x"])
@pytest.mark.parametrize("mnk", [(64, 128, 96), (36, 44, 28), (37, 45, 29), (8, 300, 4), (130, 24, 64)])
def test_gemm_strided_layouts(la, lb, lc, mnk):
    """Every staging layout of A (k, m or neither unit-stride) and B (k, n or
    neither), every result layout (16-byte stores along n or m, or element
    stores), full and ragged tiles, several k-steps, batches, alpha, beta and
    split-K slices, against FP64 products of the bf16-rounded operands."""
    M, N, K = mnk
    nb = 3
    rng = np.random.default_rng(M * 7 + N * 3 + K + ord(la) * 11 + ord(lb) + ord(lc) * 5)
    A, (am, ak, a1), Ad = _operand(la, M, K, nb, rng)
    Bt, (bn, bk, b1), Btd = _operand(lb, N, K, nb, rng)     # B stored as its transpose's layout: rows n
    for ksplit in (0, 32):
        ns = -(-K // ksplit) if ksplit else 1
        cm, cn, c1, c2 = _result_strides(lc, M, N, ns)
        C0 = rng.standard_normal(nb * c1).astype(np.float32)
        alpha, beta = (1.0, 0.0) if ksplit else (-0.75, 0.5)
        got = G.gemm_strided(M, N, K, A, (am, ak, a1), Bt, (bk, bn, b1), C0.copy(), (cm, cn, c1, c2), nb=nb,
                             ksplit=ksplit, alpha=alpha, beta=beta)
        for b in range(nb):
            Ab = _bf16(Ad[b]).astype(np.float64)
            Bb = _bf16(Btd[b]).astype(np.float64).T
            for sl in range(ns):
                k0, k1 = (sl * ksplit, min(K, (sl + 1) * ksplit)) if ksplit else (0, K)
                m, n = np.meshgrid(np.arange(M), np.arange(N), indexing="ij")
                idx = b * c1 + sl * c2 + m * cm + n * cn
                ref = alpha * (Ab[:, k0:k1] @ Bb[k0:k1]) + beta * C0[idx].astype(np.float64)
                scale = np.abs(Ab[:, k0:k1]) @ np.abs(Bb[k0:k1]) + abs(beta) * np.abs(C0[idx])
                err = np.abs(got[idx] - ref)
                assert np.all(err <= 1e-5 * scale + 1e-6), (b, sl, float(np.max(err / (scale + 1e-30))))
        # elements outside C's tiles are untouched
        mask = np.ones(C0.size, bool)
        for b in range(nb):
            for sl in range(ns):
                m, n = np.meshgrid(np.arange(M), np.arange(N), indexing="ij")
                mask[(b * c1 + sl * c2 + m * cm + n * cn).ravel()] = False
        assert np.array_equal(got[mask], C0[mask])


# (imaginary A, imaginary B, imaginary C written, sa, sb): the forms the
# spectral layers use (complex x complex, complex x real, real part only)
# and the rest
CMODES = [(True, True, True, 1, 1), (True, True, True, -1, 1), (True, True, True, 1, -1),
          (True, False, True, -1, 1), (True, True, False, -1, 1), (False, True, True, 1, -1),
          (False, False, True, 1, 1)]


@pytest.mark.parametrize("la", ["k", "r", "x"])
@pytest.mark.parametrize("lb", ["k", "r", "x"])
@pytest.mark.parametrize("lc", ["n", "m", "x"])
@pytest.mark.parametrize("mnk", [(36, 44, 40), (37, 45, 29)])
def test_cgemm_strided_forms(la, lb, lc, mnk):
    """The one-launch complex product in every staging and result layout,
    each form of it (an absent imaginary plane, the real part only,
    conjugates), alpha and beta, against FP64 complex products of the
    bf16-rounded planes; elements outside C are untouched."""
    M, N, K = mnk
    nb = 2
    rng = np.random.default_rng(M * 5 + N + K * 3 + ord(la) * 7 + ord(lb) * 13 + ord(lc) * 17)
    Ar, (am, ak, a1), Ard = _operand(la, M, K, nb, rng)
    Br, (bn, bk, b1), Brd = _operand(lb, N, K, nb, rng)
    Ai, Bi = rng.standard_normal(Ar.size).astype(np.float32), rng.standard_normal(Br.size).astype(np.float32)
    r, k = np.meshgrid(np.arange(M), np.arange(K), indexing="ij")
    Aid = np.stack([Ai[b * a1 + r * am + k * ak] for b in range(nb)])
    r, k = np.meshgrid(np.arange(N), np.arange(K), indexing="ij")
    Bid = np.stack([Bi[b * b1 + r * bn + k * bk] for b in range(nb)])
    cm, cn, c1, _ = _result_strides(lc, M, N, 1)
    m, n = np.meshgrid(np.arange(M), np.arange(N), indexing="ij")
    for hai, hbi, hci, sa, sb in CMODES:
        alpha, beta = (0.75, -0.5) if hci else (1.0, 0.0)
        C0r = rng.standard_normal(nb * c1).astype(np.float32)
        C0i = rng.standard_normal(nb * c1).astype(np.float32)
        gr, gi = G.cgemm_strided(M, N, K, Ar, Ai if hai else None, (am, ak, a1), Br, Bi if hbi else None,
                                 (bk, bn, b1), C0r.copy(), C0i.copy() if hci else None, (cm, cn, c1), nb=nb, sa=sa,
                                 sb=sb, alpha=alpha, beta=beta)
        mask = np.ones(C0r.size, bool)
        for b in range(nb):
            Ab = _bf16(Ard[b]) + 1j * sa * (_bf16(Aid[b]) if hai else 0)
            Bb = (_bf16(Brd[b]) + 1j * sb * (_bf16(Bid[b]) if hbi else 0)).T
            idx = b * c1 + m * cm + n * cn
            mask[idx.ravel()] = False
            prod = Ab.astype(np.complex128) @ Bb.astype(np.complex128)
            scale = np.abs(Ab) @ np.abs(Bb) + abs(beta) * (np.abs(C0r[idx]) + np.abs(C0i[idx]))
            ref_r = alpha * prod.real + beta * C0r[idx]
            err = np.abs(gr[idx] - ref_r)
            assert np.all(err <= 1e-5 * scale + 1e-6), ("re", b, hai, hbi, hci, sa, sb, float(np.max(err / scale)))
            if hci:
                ref_i = alpha * prod.imag + beta * C0i[idx]
                err = np.abs(gi[idx] - ref_i)
                assert np.all(err <= 1e-5 * scale + 1e-6), ("im", b, hai, hbi, sa, sb, float(np.max(err / scale)))
        assert np.array_equal(gr[mask], C0r[mask])
        if hci:
            assert np.array_equal(gi[mask], C0i[mask])


CFG = F.FNOConfig(X=16, Y=12, Z=8, width=8, modes=(4, 3, 3), layers=3, d_in=6, d_hidden=16, d_out=5)


def _setup(seed=0, B=3):
    rng = np.random.default_rng(seed)
    p = F.init_params(CFG, seed=seed)
    for k in p:
        if k in ("Pb", "Q1b", "Q2b") or k.startswith("b"):
            p[k] = 0.1 * rng.standard_normal(p[k].shape)
        if k.startswith("R"):
            p[k] = p[k] * 20.0           # spectral path comparable to the pointwise path
    a = rng.standard_normal((B, CFG.d_in, CFG.Z, CFG.Y, CFG.X))
    t = rng.standard_normal((B, CFG.d_out, CFG.Z, CFG.Y, CFG.X))
    net = G.FNO(CFG.X, CFG.Y, CFG.Z, width=CFG.width, modes=CFG.modes, layers=CFG.layers, d_in=CFG.d_in,
                d_hidden=CFG.d_hidden, d_out=CFG.d_out, max_batch=4)
    net.set_params(p)
    return p, a, t, net


def _rel(a, b):
    return float(np.linalg.norm(np.asarray(a, np.float64) - b) / max(np.linalg.norm(b), 1e-30))


def test_forward_matches_oracle():
    p, a, _, net = _setup()
    ref, _ = F.forward(CFG, p, a)
    got = net.forward(a)
    err = _rel(got, ref)
    print(f"FNO forward rel-L2 vs FP64 oracle: {err:.3e}")
    assert err < 2e-2
    assert np.array_equal(net.get_params(), G.flatten(net.cfg, p))


def test_gradients_match_oracle():
    p, a, t, net = _setup(seed=1)
    out, cache = F.forward(CFG, p, a)
    loss_ref, dout = F.mse(out, t)
    gref = F.backward(CFG, p, cache, dout)
    loss, g = net.gradients(a, t)
    assert abs(loss / loss_ref - 1) < 1e-2, (loss, loss_ref)
    gg = G.unflatten(net.cfg, g)
    errs = {k: _rel(gg[k], gref[k]) for k in gref}
    print("gradient rel-L2 per tensor:", {k: f"{v:.2e}" for k, v in errs.items()})
    assert max(errs.values()) < 5e-2, errs


def test_gradients_with_split_k_slices_match_oracle():
    """A grid of more points than one split-K chunk of the weight-gradient
    GEMMs (16x16x12 = 3072 > 2048), so those gradients are sums over several
    slices per sample."""
    cfg = F.FNOConfig(X=16, Y=16, Z=12, width=8, modes=(3, 4, 2), layers=2, d_in=6, d_hidden=16, d_out=5)
    rng = np.random.default_rng(5)
    p = F.init_params(cfg, seed=5)
    for k in p:
        if k in ("Pb", "Q1b", "Q2b") or k.startswith("b"):
            p[k] = 0.1 * rng.standard_normal(p[k].shape)
        if k.startswith("R"):
            p[k] = p[k] * 20.0
    a = rng.standard_normal((2, cfg.d_in, cfg.Z, cfg.Y, cfg.X))
    t = rng.standard_normal((2, cfg.d_out, cfg.Z, cfg.Y, cfg.X))
    net = G.FNO(cfg.X, cfg.Y, cfg.Z, width=cfg.width, modes=cfg.modes, layers=cfg.layers, d_in=cfg.d_in,
                d_hidden=cfg.d_hidden, d_out=cfg.d_out, max_batch=2)
    net.set_params(p)
    out, cache = F.forward(cfg, p, a)
    loss_ref, dout = F.mse(out, t)
    gref = F.backward(cfg, p, cache, dout)
    loss, g = net.gradients(a, t)
    assert abs(loss / loss_ref - 1) < 1e-2, (loss, loss_ref)
    gg = G.unflatten(net.cfg, g)
    errs = {k: _rel(gg[k], gref[k]) for k in gref}
    print("gradient rel-L2 per tensor (split-K):", {k: f"{v:.2e}" for k, v in errs.items()})
    assert max(errs.values()) < 5e-2, errs


def _small_net(width, modes, batch, seed, grid=(12, 8, 6), layers=2):
    cfg = F.FNOConfig(X=grid[0], Y=grid[1], Z=grid[2], width=width, modes=modes, layers=layers, d_in=6, d_hidden=24,
                      d_out=5)
    rng = np.random.default_rng(seed)
    p = F.init_params(cfg, seed=seed)
    for k in p:
        if k in ("Pb", "Q1b", "Q2b") or k.startswith("b"):
            p[k] = 0.1 * rng.standard_normal(p[k].shape)
        if k.startswith("R"):
            p[k] = p[k] * width * width * 0.3
    net = G.FNO(cfg.X, cfg.Y, cfg.Z, width=width, modes=modes, layers=layers, d_in=cfg.d_in, d_hidden=cfg.d_hidden,
                d_out=cfg.d_out, max_batch=batch)
    net.set_params(p)
    a = rng.standard_normal((batch, cfg.d_in, cfg.Z, cfg.Y, cfg.X)).astype(np.float32)
    t = rng.standard_normal((batch, cfg.d_out, cfg.Z, cfg.Y, cfg.X)).astype(np.float32)
    return cfg, p, net, a, t


# Widths 16 and 32 take kernels of their own up to 16 samples: 17 samples go through
# the batched GEMMs, and every sample alone or in a smaller batch has to come out
# the same bit for bit (mode counts that are and are not whole groups of 16).
@pytest.mark.parametrize("width", [16, 32])
@pytest.mark.parametrize("modes", [(3, 3, 1), (4, 2, 3)])
def test_small_batches_match_the_batched_gemms_bitwise(width, modes):
    _, _, net, a, _ = _small_net(width, modes, 17, seed=3)
    every = net.forward(a)
    assert np.all(np.isfinite(every))
    for i, n in ((0, 1), (1, 3), (4, 8), (1, 16)):
        assert np.array_equal(net.forward(a[i:i + n]), every[i:i + n]), (i, n)


@pytest.mark.parametrize("width,batch", [(16, 2), (32, 8), (32, 9), (16, 16), (32, 17)])
def test_gradients_of_every_width_and_batch_path_match_oracle(width, batch):
    cfg, p, net, a, t = _small_net(width, (3, 3, 2), batch, seed=11)
    out, cache = F.forward(cfg, p, a.astype(np.float64))
    loss_ref, dout = F.mse(out, t)
    gref = F.backward(cfg, p, cache, dout)
    loss, g = net.gradients(a, t)
    gg = G.unflatten(net.cfg, g)
    assert abs(loss / loss_ref - 1) < 1e-2, (loss, loss_ref)
    errs = {k: _rel(gg[k], gref[k]) for k in gref}
    assert max(errs.values()) < 5e-2, errs


# Widths 16 and 32 mix the modes in kernels of their own up to 16 samples, forward and
# backward; inside a width of 48 whose further channels have zero weights the batched
# GEMMs do it, and those channels stay zero: outputs, loss and the gradients of the shared
# channels are the same bit for bit.  One sample to two groups of 8; modes that are and
# are not whole groups of 16.  The backward kernel's two products are one launch, as
# GEMMs two.
@pytest.mark.parametrize("modes", [(3, 3, 1), (4, 2, 3), (5, 4, 3)])
@pytest.mark.parametrize("batch", [1, 2, 8, 9, 16])
@pytest.mark.parametrize("width", [16, 32])
def test_mixing_matches_the_gemms_bitwise(width, batch, modes):
    cfg, p, net, a, t = _small_net(width, modes, batch, seed=29)
    wide = G.FNO(cfg.X, cfg.Y, cfg.Z, width=48, modes=modes, layers=2, d_in=cfg.d_in, d_hidden=cfg.d_hidden,
                 d_out=cfg.d_out, max_batch=batch)

    def embed(small, large):
        out = np.zeros(large)
        out[tuple(slice(n) for n in small.shape)] = small
        return out

    wide.set_params({k: embed(np.asarray(p[k]), shape) for k, shape in G.param_shapes(wide.cfg)})
    res = []
    for n in (net, wide):
        n.gemm_work(reset=True)
        loss, g = n.gradients(a, t)
        res.append((n.gemm_work(reset=True).launches, loss, n.forward(a), G.unflatten(n.cfg, g)))
        n.close()
    (launches, loss, out, g), (launches_w, loss_w, out_w, g_w) = res
    # the transforms' kernel, from 256 channels of all samples on, is a launch less a layer and direction
    transforms = 4 * ((48 * batch >= 256) - (width * batch >= 256))
    assert launches + 2 == launches_w + transforms
    assert loss == loss_w and np.array_equal(out, out_w)
    for k in g:
        shared = g_w[k][tuple(slice(n) for n in g[k].shape)]
        assert np.all(np.isfinite(g[k])) and np.any(g[k]) and np.array_equal(g[k], shared), k


# A projection of 128 hidden channels takes kernels of its own; with 32 more channels
# whose weights are zero it goes through the pointwise GEMMs, and adds only zeros: outputs,
# loss and every gradient are the same bit for bit.  Points: 20 beyond the last
# whole tile of 32; two slices of 2048, the second part full; ragged in both; too few
# slices for the backward kernel.
@pytest.mark.parametrize("grid,batch", [((6, 6, 5), 128), ((16, 16, 10), 64), ((18, 14, 9), 64), ((18, 14, 9), 3)])
@pytest.mark.parametrize("width,d_out", [(16, 1), (32, 2), (16, 8), (32, 5)])
def test_projection_matches_the_pointwise_gemms_bitwise(grid, batch, width, d_out):
    cfg = F.FNOConfig(X=grid[0], Y=grid[1], Z=grid[2], width=width, modes=(2, 3, 2), layers=2, d_in=3, d_hidden=128,
                      d_out=d_out)
    rng = np.random.default_rng(17)
    p = F.init_params(cfg, seed=17)
    for k in ("Q1b", "Q2b"):
        p[k] = 0.3 * rng.standard_normal(p[k].shape)
    wide = dict(p)
    wide["Q1w"] = np.concatenate([p["Q1w"], np.zeros((width, 32))], axis=1)
    wide["Q1b"] = np.concatenate([p["Q1b"], np.zeros(32)])
    wide["Q2w"] = np.concatenate([p["Q2w"], np.zeros((32, d_out))], axis=0)
    a = rng.standard_normal((batch, 3, cfg.Z, cfg.Y, cfg.X)).astype(np.float32)
    t = rng.standard_normal((batch, d_out, cfg.Z, cfg.Y, cfg.X)).astype(np.float32)
    res = []
    for hidden, q in ((128, p), (160, wide)):
        net = G.FNO(cfg.X, cfg.Y, cfg.Z, width=width, modes=cfg.modes, layers=2, d_in=3, d_hidden=hidden, d_out=d_out,
                    max_batch=batch)
        net.set_params(q)
        loss, g = net.gradients(a, t)
        res.append((net.forward(a), loss, G.unflatten(net.cfg, g)))
        net.close()
    (out, loss, g), (out_w, loss_w, g_w) = res
    assert np.array_equal(out, out_w) and loss == loss_w
    g_w["Q1w"], g_w["Q1b"], g_w["Q2w"] = g_w["Q1w"][:, :128], g_w["Q1b"][:128], g_w["Q2w"][:128]
    for k in g:
        assert np.all(np.isfinite(g[k])) and np.array_equal(g[k], g_w[k]), k


# Widths 16 and 32 end their layers in a kernel of its own; inside a width of 48 whose
# further channels have zero weights the layers go through the GEMMs, and those channels
# stay zero: outputs, loss and the gradients of the shared channels are the same
# bit for bit.  Planes with a last tile of 8 points and of whole tiles; z of less
# than, of whole and of ragged groups of 16; 1 to all 16 modes; batches that fill
# rounds of 512 workgroups.
@pytest.mark.parametrize("grid,mz,batch", [((12, 6, 10), 1, 341), ((16, 16, 32), 16, 64), ((20, 10, 50), 12, 73)])
@pytest.mark.parametrize("width", [16, 32])
def test_layer_ends_match_the_gemms_bitwise(grid, mz, batch, width):
    cfg = F.FNOConfig(X=grid[0], Y=grid[1], Z=grid[2], width=width, modes=(3, 2, mz), layers=3, d_in=3, d_hidden=24,
                      d_out=2)
    rng = np.random.default_rng(23)
    p = F.init_params(cfg, seed=23)
    for k in p:
        if k in ("Pb", "Q1b", "Q2b") or k.startswith("b"):
            p[k] = 0.3 * rng.standard_normal(p[k].shape)
        if k.startswith("R"):
            p[k] = p[k] * width * width * 0.3
    a = rng.standard_normal((batch, 3, cfg.Z, cfg.Y, cfg.X)).astype(np.float32)
    t = rng.standard_normal((batch, 2, cfg.Z, cfg.Y, cfg.X)).astype(np.float32)

    def net(w):
        return G.FNO(cfg.X, cfg.Y, cfg.Z, width=w, modes=cfg.modes, layers=3, d_in=3, d_hidden=24, d_out=2, max_batch=batch)

    def embed(small, large):   # every axis of the width's length grows, zeros beyond
        out = np.zeros(large)
        out[tuple(slice(n) for n in small.shape)] = small
        return out

    res = []
    for w in (width, 48):
        n = net(w)
        n.set_params({k: embed(np.asarray(p[k]), shape) for k, shape in G.param_shapes(n.cfg)})
        loss, g = n.gradients(a, t)
        res.append((n.forward(a), loss, G.unflatten(n.cfg, g)))
        n.close()
    (out, loss, g), (out_w, loss_w, g_w) = res
    assert np.array_equal(out, out_w) and loss == loss_w
    for k in g:
        assert np.all(np.isfinite(g[k])) and np.array_equal(g[k], g_w[k][tuple(slice(n) for n in g[k].shape)]), k


def test_adam_steps_reduce_loss():
    p, a, t, net = _setup(seed=2)
    losses = [net.train_step(a, t, 3e-3) for _ in range(30)]
    print("losses:", [f"{x:.4f}" for x in losses[::5]])
    assert losses[-1] < 0.9 * losses[0]


def test_resident_batch_steps_match_host_batches():
    """Training steps on the batch left on the device (no host transfer) give
    bit for bit what the same steps with the host arrays give; a forward call
    in between invalidates the resident batch."""
    p, a, t, n1 = _setup(seed=3)
    _, _, _, n2 = _setup(seed=3)
    l1 = [n1.train_step(a, t, 2e-3) for _ in range(3)]
    l2 = [n2.train_step(a, t, 2e-3)] + [n2.train_step(None, None, 2e-3) for _ in range(2)]
    assert l1 == l2
    assert np.array_equal(n1.get_params(), n2.get_params())
    n2.forward(a)
    with pytest.raises(Exception):
        n2.train_step(None, None, 2e-3, batch=a.shape[0])


# Up to 16 modes along z the transforms along z and y share a kernel; with 17 modes, the
# further ones of zero weights, they go through the GEMMs: outputs, loss and the
# gradients of the shared modes are the same bit for bit.  Rows of less than, of
# whole and of ragged groups of 16; y and z of one and two steps of 32; 258
# channels of all samples make 256 workgroups.
@pytest.mark.parametrize("grid", [(12, 6, 34), (16, 32, 34), (36, 40, 70)])
@pytest.mark.parametrize("mz", [1, 16])
def test_transforms_match_the_gemms_bitwise(grid, mz):
    def net(m):
        return G.FNO(*grid, width=43, modes=(3, 3, m), layers=2, d_in=2, d_hidden=8, d_out=2, max_batch=6)

    rng = np.random.default_rng(31)
    a, t = (rng.standard_normal((6, 2) + grid[::-1]).astype(np.float32) for _ in range(2))
    small, large = net(mz), net(17)
    p = {k: 0.3 * rng.standard_normal(shape) for k, shape in G.param_shapes(small.cfg)}
    small.set_params(p)
    for k in p:
        if k.startswith("R"):
            p[k] = np.concatenate([p[k], np.zeros((17 - mz,) + p[k].shape[1:])])
    large.set_params(p)
    (loss, g), (loss_l, g_l) = small.gradients(a, t), large.gradients(a, t)
    assert loss == loss_l and np.array_equal(small.forward(a), large.forward(a))
    g, g_l = G.unflatten(small.cfg, g), G.unflatten(large.cfg, g_l)
    for k in g:
        assert np.all(np.isfinite(g[k])) and np.array_equal(g[k], g_l[k][:mz] if k.startswith("R") else g_l[k]), k


# The same over the sizes of the kernel: its three forms by the pieces of a wave (up
# to 3, 6 and 8), one to three tiles of 16 along ky, whole and ragged, the
# mode counts of the trained network and the most that fit.  The network with
# 17 modes runs one launch more a layer, so the smaller one does take the kernel; with
# 16 modes it does not (its LDS holds at most 15).
@pytest.mark.parametrize("grid,my,mz", [((12, 16, 34), 8, 8), ((36, 24, 34), 12, 12), ((64, 64, 64), 12, 12),
                                        ((20, 32, 34), 10, 14), ((34, 48, 40), 24, 10), ((12, 36, 70), 17, 9)])
def test_transform_kernels_forms_match_the_gemms_bitwise(grid, my, mz):
    def net(m):
        return G.FNO(*grid, width=43, modes=(3, my, m), layers=2, d_in=2, d_hidden=8, d_out=2, max_batch=6)

    rng = np.random.default_rng(37)
    a, t = (rng.standard_normal((6, 2) + grid[::-1]).astype(np.float32) for _ in range(2))
    nets = [net(m) for m in (mz, 16, 17)]
    p = {k: 0.3 * rng.standard_normal(shape) for k, shape in G.param_shapes(nets[0].cfg)}
    out, launches, grads = [], [], []
    for n, m in zip(nets, (mz, 16, 17)):
        n.set_params({k: np.concatenate([v, np.zeros((m - mz,) + v.shape[1:])]) if k.startswith("R") else v
                      for k, v in p.items()})
        n.gemm_work(reset=True)
        out.append(n.forward(a))
        launches.append(n.gemm_work(reset=True).launches)
        loss, g = n.gradients(a, t)
        grads.append(dict(G.unflatten(n.cfg, g), loss=np.float64(loss)))
        n.close()
    assert launches[0] + 2 == launches[1] == launches[2]
    assert np.all(np.isfinite(out[0])) and np.array_equal(out[0], out[2])
    for k, v in grads[0].items():
        assert np.all(np.isfinite(v)) and np.array_equal(v, grads[2][k][:mz] if k.startswith("R") else grads[2][k]), k


# The gather takes 64 samples a launch; the loss and its gradient, like the gather,
# work on quads (samples of 6 and 4 of them, fewer than the threads; of 300 and 200).
@pytest.mark.parametrize("grid", [(2, 2, 2), (10, 8, 5)])
@pytest.mark.parametrize("batch", [64, 65, 130])
def test_large_gathered_batches_match_host_batches(grid, batch):
    nets = [G.FNO(*grid, width=4, modes=(1, 1, 1), layers=2, d_in=3, d_hidden=8, d_out=2, max_batch=130)
            for _ in range(2)]
    rng = np.random.default_rng(4)
    p = (0.3 * rng.standard_normal(nets[0].n)).astype(np.float32)
    a = rng.standard_normal((9, 3) + grid[::-1]).astype(np.float32)
    t = rng.standard_normal((9, 2) + grid[::-1]).astype(np.float32)
    idx = rng.integers(0, 9, batch).tolist()
    for n in nets:
        n.set_params(G.unflatten(n.cfg, p))
    nets[1].set_dataset(a, t)
    loss = nets[0].train_step(a[idx], t[idx], 1e-3)
    assert nets[1].train_step_indices(idx, 1e-3) == loss
    assert np.array_equal(nets[0].get_params(), nets[1].get_params())
    out = nets[0].forward(a[idx])
    nets[1].set_params(G.unflatten(nets[1].cfg, p))
    first = nets[1].forward(a[idx]).astype(np.float64)
    ref = np.mean((first - t[idx].astype(np.float64)) ** 2)
    # float differences carry 2^-24 of the larger of the two each, their squares twice that: far within 1e-6
    assert abs(loss / ref - 1) < 1e-6 and out.shape == first.shape


@pytest.mark.parametrize("batch", [3, 65])
def test_prediction_after_a_gathered_batch_is_the_host_batchs(batch):
    """Predictions before and after one step on a gathered batch: the values of a network trained on the same batch
    from the host, and not those of before."""
    nets = [G.FNO(10, 8, 5, width=4, modes=(1, 1, 1), layers=2, d_in=3, d_hidden=8, d_out=2, max_batch=65)
            for _ in range(2)]
    rng = np.random.default_rng(6)
    p = (0.3 * rng.standard_normal(nets[0].n)).astype(np.float32)
    a = rng.standard_normal((9, 3, 5, 8, 10)).astype(np.float32)
    t = rng.standard_normal((9, 2, 5, 8, 10)).astype(np.float32)
    idx = rng.integers(0, 9, batch).tolist()
    for n in nets:
        n.set_params(G.unflatten(n.cfg, p))
    nets[1].set_dataset(a, t)
    before = nets[0].forward(a[idx])
    nets[0].train_step(a[idx], t[idx], 1e-3)
    nets[1].train_step_indices(idx, 1e-3)
    out, gathered = (n.forward(a[idx]) for n in nets)
    assert np.all(np.isfinite(out)) and np.array_equal(gathered, out) and not np.array_equal(out, before)


def test_resident_dataset_steps_match_host_batches():
    """Steps on mini-batches gathered on the device from a resident training
    set give bit for bit what the same steps on host copies of those samples
    give; out-of-range indices and a batch above max_batch are refused."""
    rng = np.random.default_rng(11)
    _, _, _, n1 = _setup(seed=5)
    _, _, _, n2 = _setup(seed=5)
    ds_a = rng.standard_normal((7, CFG.d_in, CFG.Z, CFG.Y, CFG.X)).astype(np.float32)
    ds_t = rng.standard_normal((7, CFG.d_out, CFG.Z, CFG.Y, CFG.X)).astype(np.float32)
    n2.set_dataset(ds_a, ds_t)
    for idx in ([6, 0, 3], [2, 2, 5, 1], [4]):
        l1 = n1.train_step(ds_a[idx], ds_t[idx], 2e-3)
        l2 = n2.train_step_indices(idx, 2e-3)
        assert l1 == l2
    assert np.array_equal(n1.get_params(), n2.get_params())
    with pytest.raises(Exception):
        n2.train_step_indices([0, 7], 2e-3)
    with pytest.raises(Exception):
        n2.train_step_indices([0, 1, 2, 3, 4], 2e-3)
    # a new set replaces the old one
    n2.set_dataset(ds_a[:2], ds_t[:2])
    with pytest.raises(Exception):
        n2.train_step_indices([2], 2e-3)
