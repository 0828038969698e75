"""Warm-start network kernels (csrc/cnn.hip) against the FP64 oracle
(oracle/cnn.py) with the same bfloat16 rounding points.  The grid shape is
not a multiple of the kernels' point tiles, and dilations > 1 wrap around
the periodic cell."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPE = (12, 10, 15)
DIL = (1, 2, 1, 3, 2, 1)
# middle layers, forward and backward-data: (12, 10, 15) on the point-tiled
# kernel; (6, 8, 32) with d = 1 and 2 on the row-tiled one; (4, 16, 64),
# (4, 8, 96) and (4, 8, 160) with d = 1 and 2 on the ring-staged one, with d = 3
# on the point-tiled one; (6, 12, 40) on the ring-staged one with a partial z
# block (40 = 32 + 8) and partial y groups (12 / d rows per residue class,
# d = 1, 2, 3).  test_middle_layer_kernels has every instance.
SHAPES = [(12, 10, 15), (6, 8, 32), (4, 16, 64), (4, 8, 96), (4, 8, 160), (6, 12, 40)]


def _setup(seed=0, scale=1.5, shape=SHAPE):
    from oracle import cnn
    rng = np.random.default_rng(seed)
    p = cnn.init_params(seed + 10, scale=scale)
    for k in p:
        if k.startswith("b"):
            p[k] = rng.normal(0, 0.2, p[k].shape)
    p = {k: v.astype(np.float32).astype(np.float64) for k, v in p.items()}
    x0 = rng.normal(0, 1, (2,) + shape).astype(np.float32).astype(np.float64)
    target = rng.normal(0, 0.3, shape).astype(np.float32).astype(np.float64)
    return p, x0, target


def _net(p, dil=DIL):
    from dftpy_amd.learned import WarmStartNet
    net = WarmStartNet(dil=dil)
    net.set_params(p)
    return net


def _rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("train", [False, True])
def test_forward_matches_oracle(train, shape):
    from oracle import cnn
    p, x0, _ = _setup(shape=shape)
    ref, _ = cnn.forward(p, x0, DIL, bf16=True)
    net = _net(p)
    x = torch.as_tensor(x0.reshape(2, -1), dtype=torch.float32, device="cuda")
    out = net.forward(x, shape, train=train).cpu().numpy().astype(np.float64).reshape(shape)
    print("forward rel L2 %.2e max %.2e (|ref| max %.2e)" % (_rel(out, ref), np.abs(out - ref).max(), np.abs(ref).max()))
    assert _rel(out, ref) < 2e-3
    assert np.abs(out - ref).max() < 2e-2 * np.abs(ref).max()


@pytest.mark.parametrize("dil", [(2, 1, 1, 1, 1, 1), (3, 1, 1, 1, 1, 2)])
def test_forward_first_layer_dilations(dil):
    """The row-staged first layer with d > 1 (its periodic z halo in LDS is d
    points each side) and the one-pass output layer with d = 2."""
    from oracle import cnn
    shape = (5, 24, 48)  # ny % 4d == 0 for d = 2, 3
    p, x0, _ = _setup(4, shape=shape)
    ref, _ = cnn.forward(p, x0, dil, bf16=True)
    net = _net(p, dil)
    x = torch.as_tensor(x0.reshape(2, -1), dtype=torch.float32, device="cuda")
    out = net.forward(x, shape).cpu().numpy().astype(np.float64).reshape(shape)
    print("forward rel L2 %.2e" % _rel(out, ref))
    assert _rel(out, ref) < 2e-3
    assert np.abs(out - ref).max() < 2e-2 * np.abs(ref).max()


@pytest.mark.parametrize("shape", SHAPES)
def test_backward_matches_oracle(shape):
    from oracle import cnn
    from dftpy_amd import DirectGrid
    p, x0, target = _setup(1, shape=shape)
    ref_out, cache = cnn.forward(p, x0, DIL, bf16=True)
    ref_loss, dout = cnn.loss(ref_out, target)
    gref = cnn.backward(p, cache, dout)
    net = _net(p)
    grid = DirectGrid(np.eye(3) * 5.0, shape, full=False, dtype=torch.float32)
    plan = grid.plan(torch.float32)
    x = torch.as_tensor(x0.reshape(2, -1), dtype=torch.float32, device="cuda")
    tgt = torch.as_tensor(target.reshape(-1), dtype=torch.float32, device="cuda")
    loss = net.train_step(plan, x, shape, tgt, lr=0.0)  # lr 0: gradients only
    assert abs(float(loss.item()) - ref_loss) < 1e-2 * ref_loss
    for k, g in gref.items():
        got = net.param(k, net.grad).cpu().numpy().astype(np.float64)
        print("%s rel %.2e" % (k, _rel(got, g)))
        assert _rel(got, g) < 1e-2, k


@pytest.mark.parametrize("shape", [(8, 16, 96), (8, 16, 160), (8, 20, 72)])
def test_shipped_dilations_match_oracle(shape):
    """The shipped network's dilations (1, 2, 4, 4, 2, 1) with nx and ny
    multiples of d for every layer: inference, training forward and backward
    run all four middle layers on the ring-staged kernel.  96 is the training
    grid's z size, 160 the 500-atom cell's; (8, 20, 72) is a batch-cell z size
    (72 = 2 x 32 + 8) with y groups that end short for d = 4 (20 / 4 = 5 rows
    per residue class)."""
    from oracle import cnn
    from dftpy_amd import DirectGrid
    from dftpy_amd.learned import WarmStartNet
    dil = WarmStartNet().dil
    assert dil == (1, 2, 4, 4, 2, 1)
    p, x0, target = _setup(3, shape=shape)
    ref, cache = cnn.forward(p, x0, dil, bf16=True)
    net = _net(p, dil)
    x = torch.as_tensor(x0.reshape(2, -1), dtype=torch.float32, device="cuda")
    for train in (False, True):
        out = net.forward(x, shape, train=train).cpu().numpy().astype(np.float64).reshape(shape)
        print("forward (train=%s) rel L2 %.2e" % (train, _rel(out, ref)))
        assert _rel(out, ref) < 2e-3
        assert np.abs(out - ref).max() < 2e-2 * np.abs(ref).max()
    ref_loss, dout = cnn.loss(ref, target)
    gref = cnn.backward(p, cache, dout)
    grid = DirectGrid(np.eye(3) * 5.0, shape, full=False, dtype=torch.float32)
    tgt = torch.as_tensor(target.reshape(-1), dtype=torch.float32, device="cuda")
    loss = net.train_step(grid.plan(torch.float32), x, shape, tgt, lr=0.0)
    assert abs(float(loss.item()) - ref_loss) < 1e-2 * ref_loss
    for k, g in gref.items():
        got = net.param(k, net.grad).cpu().numpy().astype(np.float64)
        print("%s rel %.2e" % (k, _rel(got, g)))
        assert _rel(got, g) < 1e-2, k


def _mid(shape, d, mode, x, w, bias, resid, mask, off):
    """One 32 -> 32 layer through its C entry.  off: elements by which the
    fields that only need their element's alignment are moved in their
    buffers, which keeps the layer off the ring-staged kernel's training modes.
    Mode 0: (x + relu, relu), mode 1: (FP32 sum, masked BF16 copy)."""
    from dftpy_amd import _lib
    n = int(np.prod(shape))
    nr = np.ascontiguousarray(shape, dtype=np.int32)

    def moved(t):
        v = torch.empty(n * 32 + 8, device="cuda", dtype=t.dtype)[off:off + n * 32]
        return v.copy_(t.reshape(-1))

    out1 = moved(torch.full((n, 32), float("nan"), device="cuda", dtype=torch.bfloat16))
    if mode == 0:
        out0 = torch.full((n * 32,), float("nan"), device="cuda", dtype=torch.bfloat16)
        args = (bias.data_ptr(), None, None)
    else:
        out0, mask = moved(resid), moved(mask)
        args = (None, out0.data_ptr(), mask.data_ptr())  # the residual in place, as the backward pass has it
    _lib.check(_lib.lib.ofdft_cnn_conv_mid(_lib.iptr(nr), d, mode, x.data_ptr(), w.data_ptr(), *args, out0.data_ptr(),
                                           out1.data_ptr(), _lib.stream()))
    return out0.view(n, 32), out1.view(n, 32)


def _mid_inputs(shape, seed=8):
    n = int(np.prod(shape))
    gen = torch.Generator(device="cuda").manual_seed(seed)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=gen)  # noqa: E731
    return rnd(n, 32).bfloat16(), (0.1 * rnd(27, 32, 32)).bfloat16(), rnd(32), rnd(n, 32), rnd(n, 32).bfloat16()


# Row-tiled kernel, every instance (nz / 32 = 1 to 5): nz below the ring's 36,
# nx no multiple of d, d above the ring's 4, or unaligned fields (off) on shapes
# the ring takes otherwise; the point-tiled kernel likewise; the ring with
# partial z blocks and row groups
ROWS_CASES = [((6, 8, 32), 2, 0), ((5, 8, 64), 2, 0), ((5, 8, 96), 2, 0), ((7, 8, 128), 2, 0), ((6, 16, 160), 4, 0),
              ((6, 20, 64), 5, 0), ((6, 20, 96), 5, 0), ((4, 16, 64), 1, 1), ((4, 8, 96), 2, 1), ((4, 8, 128), 1, 3),
              ((8, 16, 160), 4, 1)]
OTHER_CASES = [((6, 12, 40), 3, 1), ((5, 7, 48), 4, 1), ((6, 12, 40), 3, 0), ((4, 8, 96), 2, 0), ((8, 20, 72), 4, 0),
               ((8, 16, 160), 4, 0)]


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("shape,d,off", ROWS_CASES + OTHER_CASES)
def test_middle_layer_kernels(shape, d, off, mode):
    """Each kernel of a 32 -> 32 layer, forward with the ReLU kept and
    backward-data, against FP64: an FP32 sum of 864 products, the bias or
    residual is within 866 ulps / 2 of the sum of the magnitudes; its BF16
    copies are roundings (2^-9) of it, the masked one exactly that of out0."""
    x, w, bias, resid, mask = _mid_inputs(shape)
    out0, out1 = _mid(shape, d, mode, x, w, bias, resid, mask, off)
    add = bias if mode == 0 else resid
    ref, mag = add.double().expand(x.shape), add.double().abs().expand(x.shape)
    for t in range(27):
        sh = [-d * (i - 1) for i in (t // 9, t // 3 % 3, t % 3)]
        xs = torch.roll(x.double().view(*shape, 32), sh, (0, 1, 2)).view(-1, 32)
        wt = w[t].double().T.contiguous()
        ref, mag = ref + xs @ wt, mag + xs.abs() @ wt.abs()
    tol = 866 * 2.0 ** -24 * mag
    if mode == 0:
        ref = ref.clamp(min=0.0)
        assert ((out1.double() - ref).abs() <= tol + 2.0 ** -8 * ref).all()
        ref = ref + x.double()
        assert ((out0.double() - ref).abs() <= tol + 2.0 ** -8 * ref.abs()).all()
    else:
        assert ((out0.double() - ref).abs() <= tol).all()
        assert torch.equal(out1, torch.where(mask > 0, out0, torch.zeros_like(out0)).bfloat16())


@pytest.mark.parametrize("d", [2, 4])
def test_ring_forward_matches_row_kernel_at_160(d):
    """At the 500-atom cell's full 160^3 grid (where FP64 sums are too slow),
    one middle layer on the ring-staged kernel (aligned fields) against the
    row-tiled kernel (fields off by an element; its instances are compared with
    FP64 above): the same products, FP32 sums in a different order, forward
    (BF16 outputs: a sum near a rounding boundary moves by 2^-8) and
    backward-data.  The inference form of the ring, which keeps no ReLU, stores
    the same sums bit for bit."""
    from dftpy_amd import _lib
    shape = (160, 160, 160)
    x, w, bias, resid, mask = _mid_inputs(shape)
    ring, rows = (_mid(shape, d, 0, x, w, bias, resid, mask, off) for off in (0, 1))
    for a, b in zip(ring, rows):
        a, b = a.float(), b.float()
        assert float((a - b).norm() / b.norm()) < 1e-3
        assert bool(((a - b).abs() <= 2.0 ** -7 * b.abs() + 1e-3).all())
    plain = torch.full_like(ring[0], float("nan"))
    nr = np.ascontiguousarray(shape, dtype=np.int32)
    _lib.check(_lib.lib.ofdft_cnn_conv_mid(_lib.iptr(nr), d, 0, x.data_ptr(), w.data_ptr(), bias.data_ptr(), None, None,
                                           plain.data_ptr(), None, _lib.stream()))
    assert torch.equal(plain, ring[0])
    ring, rows = (_mid(shape, d, 1, x, w, bias, resid, mask, off) for off in (0, 1))
    assert float((ring[0] - rows[0]).norm() / rows[0].norm()) < 1e-5
    assert float((ring[0] - rows[0]).abs().max()) < 1e-3


@pytest.mark.parametrize("shape,dil", [((12, 10, 15), 1), ((4, 8, 160), 1), ((9, 6, 40), 2), ((8, 7, 300), 3),
                                       ((160, 160, 160), 1)])
def test_output_layer_one_pass_equals_tap_planes(shape, dil):
    """The output layer's one-pass form (work NULL: projections of a plane
    in LDS while the layer walks x) against the two-pass form through 27 FP16
    tap planes: the same FP16 projections summed in the same tap order, so the
    outputs are identical.  Shapes: walk cycles gcd(nx, d) > 1 (9, 6, 40; d 2
    is coprime to 9 and ny 6 = 3 y-blocks of 2 rows wrap), nz above one LDS
    block (300), and the 160^3 grid of the 500-atom cell."""
    from dftpy_amd import _lib
    n = int(np.prod(shape))
    g = torch.Generator(device="cuda").manual_seed(11)
    h = (torch.randn((n, 32), device="cuda", generator=g) * 2).to(torch.bfloat16)
    w = torch.randn((27, 32), device="cuda", generator=g) * 0.1
    b = torch.tensor([0.25], device="cuda")
    nr = np.ascontiguousarray(shape, dtype=np.int32)
    one = torch.full((n,), float("nan"), device="cuda")
    two = torch.full((n,), float("nan"), device="cuda")
    work = torch.empty(27 * n, device="cuda")
    s = _lib.stream()
    L = _lib.lib
    _lib.check(L.ofdft_cnn_conv_out(_lib.iptr(nr), dil, h.data_ptr(), w.data_ptr(), b.data_ptr(), one.data_ptr(),
                                    None, s))
    _lib.check(L.ofdft_cnn_conv_out(_lib.iptr(nr), dil, h.data_ptr(), w.data_ptr(), b.data_ptr(), two.data_ptr(),
                                    work.data_ptr(), s))
    assert bool(torch.isfinite(one).all())
    assert torch.equal(one, two)
    if n <= 20000:  # and both against the FP64 convolution of the FP16-rounded operands
        hh = h.float().cpu().numpy().astype(np.float64).reshape(shape + (32,))
        ww = w.half().double().cpu().numpy()
        ref = np.full(shape, 0.25)
        for t in range(27):
            dx, dy, dz = t // 9 - 1, (t // 3) % 3 - 1, t % 3 - 1
            ref += np.roll(hh @ ww[t], shift=(-dx * dil, -dy * dil, -dz * dil), axis=(0, 1, 2))
        err = np.abs(one.cpu().numpy().reshape(shape) - ref).max()
        print("one-pass vs FP64: max %.2e (|ref| max %.2e)" % (err, np.abs(ref).max()))
        assert err < 2e-3 * np.abs(ref).max()


def _oracle_adam(p, x0, tgt, lr, steps):
    from oracle import cnn
    q = {k: v.copy() for k, v in p.items()}
    m = {k: 0 * v for k, v in q.items()}
    v2 = {k: 0 * v for k, v in q.items()}
    losses = []
    for t in range(1, steps + 1):
        out, c = cnn.forward(q, x0, DIL, bf16=True)
        loss, d = cnn.loss(out, tgt)
        g = cnn.backward(q, c, d)
        losses.append(loss)
        for k in q:  # Adam, Kingma & Ba (2015), with bias correction
            m[k] = 0.9 * m[k] + 0.1 * g[k]
            v2[k] = 0.999 * v2[k] + 0.001 * g[k] ** 2
            q[k] -= lr * (m[k] / (1 - 0.9 ** t)) / (np.sqrt(v2[k] / (1 - 0.999 ** t)) + 1e-8)
    return losses


def test_training_trajectory_matches_oracle():
    """Sixty Adam steps on a learnable target (a linear map of the inputs)
    with the GPU forward, backward and Adam kernels follow the oracle's
    training trajectory and lower the loss."""
    from dftpy_amd import DirectGrid
    p, x0, _ = _setup(2, scale=1.0)
    tgt64 = 0.3 * x0[0] - 0.1 * x0[1]
    ref = _oracle_adam(p, x0, tgt64, 5e-4, 60)
    net = _net(p)
    grid = DirectGrid(np.eye(3) * 5.0, SHAPE, full=False, dtype=torch.float32)
    plan = grid.plan(torch.float32)
    x = torch.as_tensor(x0.reshape(2, -1), dtype=torch.float32, device="cuda")
    tgt = torch.as_tensor(tgt64.reshape(-1), dtype=torch.float32, device="cuda")
    losses = [float(net.train_step(plan, x, SHAPE, tgt, lr=5e-4).item()) for _ in range(60)]
    print(["%.4f" % v for v in losses[::6]])
    print(["%.4f" % v for v in ref[::6]])
    assert np.max(np.abs(np.array(losses) - ref) / np.array(ref)) < 0.02
    assert min(losses[-10:]) < 0.5 * losses[0]


def test_spectral_loss_matches_numpy():
    """Spectral (Hessian-metric) loss and its gradient against numpy's rfftn;
    w = 1 reduces to the mean squared error (Parseval)."""
    from dftpy_amd import DirectGrid
    from dftpy_amd import _lib
    rng = np.random.default_rng(4)
    grid = DirectGrid(np.eye(3) * 5.0, SHAPE, full=False, dtype=torch.float32)
    plan = grid.plan(torch.float32)
    pred = rng.normal(0, 1, SHAPE).astype(np.float32)
    tgt = rng.normal(0, 1, SHAPE).astype(np.float32)
    nzc = SHAPE[2] // 2 + 1
    for w in (np.ones(SHAPE[:2] + (nzc,), np.float32), rng.uniform(0, 3, SHAPE[:2] + (nzc,)).astype(np.float32)):
        d = pred.astype(np.float64) - tgt
        D = np.fft.rfftn(d)
        m = np.full(nzc, 2.0)
        m[0] = 1.0
        if SHAPE[2] % 2 == 0:
            m[-1] = 1.0
        n = d.size
        ref = float((m * w * np.abs(D) ** 2).sum() / n ** 2)
        gref = 2.0 / n * np.fft.irfftn(w * D, s=SHAPE)
        tp = torch.as_tensor(pred.reshape(-1), device="cuda")
        tt = torch.as_tensor(tgt.reshape(-1), device="cuda")
        tw = torch.as_tensor(w, device="cuda").contiguous()
        dp = torch.empty_like(tp)
        loss = torch.zeros(1, dtype=torch.float64, device="cuda")
        _lib.check(_lib.lib.ofdft_cnn_loss_spectral(plan.handle, tp.data_ptr(), tt.data_ptr(), tw.data_ptr(),
                                                    dp.data_ptr(), loss.data_ptr(), _lib.stream()))
        assert abs(float(loss.item()) - ref) < 1e-5 * ref
        g = dp.cpu().numpy().astype(np.float64).reshape(SHAPE)
        assert np.abs(g - gref).max() < 1e-5 * np.abs(gref).max()
        if np.all(w == 1):
            assert abs(ref - float((d * d).mean())) < 1e-9 * ref


@pytest.mark.parametrize("nr,d,nblk", [((12, 10, 14), 1, 512), ((9, 8, 33), 4, 7), ((40, 36, 40), 30, 64), ((5, 6, 96), 2, 1),
                                       ((40, 41, 70), 36, 512), ((70, 66, 128), 65, 512), ((12, 12, 48), 3, 512),
                                       ((34, 33, 48), 31, 100), ((20, 20, 64), 8, 512), ((2, 2, 2), 1, 512),
                                       # tiles of 32 whose stage has fewer vectors than the workgroup threads (d = 1
                                       # and 2), many steps a workgroup
                                       ((9, 40, 32), 1, 2), ((8, 37, 30), 2, 3), ((4, 66, 17), 2, 1),
                                       ((12, 96, 32), 2, 8), ((12, 96, 24), 1, 16), ((6, 50, 32), 3, 4)])
def test_weight_gradients_of_one_layer(nr, d, nblk):
    """Each layer's weight-gradient kernel against FP64 sums: FP32 sums of m
    products in a workgroup (m its share of the points, with the rounding of
    the product and the final addition) are within (m + 2) ulps / 2 of the sum
    of the magnitudes.  Tiles of 64, 48 and 32 points, dilations beyond a tile,
    closed chains of rows, more workgroups than work."""
    from dftpy_amd import _lib
    L, n = _lib.lib, int(np.prod(nr))
    gen = torch.Generator(device="cuda").manual_seed(1)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=gen)  # noqa: E731
    h, h2, f2, f1 = rnd(n, 32).bfloat16(), rnd(n, 32).bfloat16(), rnd(2, n), rnd(n)
    nrc = np.ascontiguousarray(nr, dtype=np.int32)
    for layer, g, x in ((0, h, f2), (1, h, h2), (2, f1, h)):
        K = int(L.ofdft_cnn_wgrad_partials(layer, 1))
        part = torch.full((K * nblk,), float("nan"), device="cuda")
        dw = torch.empty(K, device="cuda")
        _lib.check(L.ofdft_cnn_wgrad(_lib.iptr(nrc), d, layer, g.data_ptr(), x.data_ptr(), part.data_ptr(), nblk,
                                     dw.data_ptr(), _lib.stream()))
        rows = min(nblk, (n + 255) // 256) if layer != 1 else min(nblk, nr[0] * nr[1] * -(-nr[2] // 64))
        for mag in (False, True):
            G, X = (g.double().abs(), x.double().abs()) if mag else (g.double(), x.double())
            sh = lambda a, t: torch.roll(a, [-d * (i - 1) for i in (t // 9, t // 3 % 3, t % 3)], (0, 1, 2))  # noqa: E731
            out = []
            for t in range(27):
                if layer == 0:
                    out += [G.T @ sh(X[c].view(*nr), t).reshape(-1) for c in range(2)]
                elif layer == 1:
                    out.append((G.T @ sh(X.view(*nr, 32), t).reshape(-1, 32)).reshape(-1))
                else:
                    out.append(G @ sh(X.view(*nr, 32), t).reshape(-1, 32))
            out.append(G.sum(0).reshape(-1))
            out = torch.cat(out)
            if not mag:
                ref = out
        m = -(-n // rows) + 64
        assert ((dw.double() - ref).abs() <= (m + 2) * 2.0 ** -24 * out).all()


@pytest.mark.parametrize("nr,d", [((7, 6, 9), 2), ((32, 4, 5), 3), ((2, 2, 2), 1), ((16, 8, 33), 4)])
def test_output_layer_backward(nr, d):
    """dh against FP64 (27 products: 28 ulps / 2 of the magnitudes) and its
    masked BF16 copy exactly."""
    from dftpy_amd import _lib
    n = int(np.prod(nr))
    gen = torch.Generator(device="cuda").manual_seed(2)
    dout, w = torch.randn(n, device="cuda", generator=gen), torch.randn(27, 32, device="cuda", generator=gen)
    mask = torch.randn(n, 32, device="cuda", generator=gen).bfloat16()
    dh = torch.empty(n, 32, device="cuda")
    go = torch.empty(n, 32, device="cuda", dtype=torch.bfloat16)
    nrc = np.ascontiguousarray(nr, dtype=np.int32)
    _lib.check(_lib.lib.ofdft_cnn_out_backward(_lib.iptr(nrc), d, dout.data_ptr(), w.data_ptr(), mask.data_ptr(),
                                               dh.data_ptr(), go.data_ptr(), _lib.stream()))
    ref = mag = 0.0
    for t in range(27):
        s = torch.roll(dout.double().view(*nr), [d * (i - 1) for i in (t // 9, t // 3 % 3, t % 3)], (0, 1, 2)).reshape(-1, 1)
        ref, mag = ref + s * w[t].double(), mag + s.abs() * w[t].double().abs()
    assert ((dh.double() - ref).abs() <= 28 * 2.0 ** -24 * mag).all()
    assert torch.equal(go, torch.where(mask > 0, dh, torch.zeros_like(dh)).bfloat16())
