"""Batches of every tile count modulo 8 (the tiles that do not come in eights are cut into slices over the XCDs):
every row of every tile is computed exactly once."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from flyguy_amd._lib import call
from flyguy_amd.fly_hip import HopHip
from flyguy_amd.synth import scaled_3hop, synth_3hop
from gpu_helpers import NAMES, Core, rel

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def net():
    return scaled_3hop(16)


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("tiles", [1, 2, 3, 4, 5, 6, 7, 9, 13, 16, 23, 67])
def test_any_tile_count(gpu_lib, net, tiles, bf16):
    """Logits bit for bit those of single tiles (a sample's sums do not depend on its batch), the gradients the sum of
    the tiles' gradients (float32 sums in another order)."""
    s, params = net
    w = 64 if bf16 else 32
    rng = np.random.default_rng(tiles)
    obs = rng.standard_normal((tiles * w, s["obs_dim"])).astype(np.float32)
    dl = rng.standard_normal((tiles * w, s["n_act"])).astype(np.float32)
    core = Core(s, params, tiles * w, int(bf16))
    core.zero_grad()
    logits = core.forward(obs)
    core.backward(dl)
    got = core.get(4)
    core.zero_grad()
    for i in range(0, tiles * w, w):
        assert np.array_equal(core.forward(obs[i:i + w]), logits[i:i + w]), i // w
        core.backward(dl[i:i + w])
    for name, a, b in zip(NAMES, got, core.get(4)):
        # both add the same per-tile terms in float32: a few rounding errors of 6e-8 of the larger partial sums
        assert rel(a, b) <= 2e-6, (name, rel(a, b))


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("B", [32, 96, 160, 288, 352, 416, 736])
def test_hop_of_any_tile_count(gpu_lib, net, B, half):
    """HopHip: product and state gradient bit for bit those of single tiles (binary16 tiles hold 64 samples; the scale of
    the gradient is the batch's, so it is held to one shared largest value)."""
    s, params = net
    h = s["hop"][1]
    put = lambda a, t: torch.as_tensor(np.ascontiguousarray(a, dtype=t)).cuda()      # noqa: E731
    base = int(h["widx"].min())
    index = (put(h["crow"], np.int64), put(h["col"], np.int32), put(h["tcrow"], np.int64), put(h["tcol"], np.int32),
             put(h["twidx"] - base, np.int64))
    weights = put(params[0][h["widx"]], np.float32)
    g = torch.Generator(device="cuda").manual_seed(B)
    x = torch.randn(len(h["tcrow"]) - 1, B, device="cuda", generator=g)
    gz = torch.randn(len(h["crow"]) - 1, B, device="cuda", generator=g).clamp(-2, 2)
    gz[0] = 2.0

    def run(x, gz):
        x, w = x.contiguous().requires_grad_(), weights.clone().requires_grad_()
        out = HopHip.apply(w, x, *index, half)
        return (out.detach(),) + torch.autograd.grad(out, (w, x), gz.contiguous())
    out, gw, gh = run(x, gz)
    parts = [run(x[:, i:i + 64], gz[:, i:i + 64]) for i in range(0, B, 64)]
    assert torch.equal(out, torch.cat([p[0] for p in parts], 1))
    assert torch.equal(gh, torch.cat([p[2] for p in parts], 1))
    assert rel(gw.cpu(), sum(p[1] for p in parts).cpu()) <= 2e-6


@pytest.fixture(scope="module")
def uneven():
    """A network whose first hop's plan has waves of 1 to 10 steps, the longest four times the middle one."""
    return synth_3hop(sizes=(3000, 20000, 500, 40), edges=(300_000, 9_000, 900), redrive=(300, 20, 2), sigma=2.5)


@pytest.mark.parametrize("tiles", [1, 2, 3, 5, 7, 12])
def test_few_tiles(gpu_lib, uneven, monkeypatch, tiles):
    """Batches of few tiles (several steps' gathers in flight, one wave per workgroup, four steps on the uneven hop up
    to 2 tiles) against the kernel of larger batches, which firing bitmaps at every batch select: logits and every
    layer's states bit for bit."""
    s, params = uneven
    B = 32 * tiles
    obs = np.random.default_rng(tiles).standard_normal((B, s["obs_dim"])).astype(np.float32)
    got = []
    for mode in ("", "1"):
        if mode:
            monkeypatch.setenv("FLYGUY_SKIP_SILENT", mode)
        core = Core(s, params, B)
        got.append([core.forward(obs)] + [core.state(k, 0, n, B) for k, n in enumerate(s["sizes"])])
    for a, b in zip(*got):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("bias", [False, True])
def test_rows_of_many_segments(gpu_lib, bias):
    """Rows of 1 to 130 partial sums (64 of them are loaded at once for few tiles, 8 for many): bit for bit the same for
    one tile and for a batch of 1,000, and within float32 sums of the float64 product."""
    segments = [1, 2, 7, 8, 9, 63, 64, 65, 128, 130]
    rng = np.random.default_rng(3)
    n_src, B = 4000, 32000
    deg = [16 * k - 3 for k in segments]
    crow = np.concatenate([[0], np.cumsum(deg)])
    col = np.concatenate([np.sort(rng.choice(n_src, d, replace=False)) for d in deg])
    order = np.argsort(col, kind="stable")
    tcrow = np.concatenate([[0], np.cumsum(np.bincount(col, minlength=n_src))])
    row = np.repeat(np.arange(len(deg)), deg)
    put = lambda a, t: torch.as_tensor(np.ascontiguousarray(a, dtype=t)).cuda()      # noqa: E731
    index = (put(crow, np.int64), put(col, np.int32), put(tcrow, np.int64), put(row[order], np.int32),
             put(order, np.int64))
    g = torch.Generator(device="cuda").manual_seed(1)
    w = torch.randn(len(col), device="cuda", generator=g)
    h = torch.randn(B // 32, n_src, 32, device="cuda", generator=g)
    b = torch.randn(len(deg), device="cuda", generator=g) if bias else None
    layer = (False, b, None, None, None)
    many = HopHip.apply(w, h, *index, *layer)
    for tile in (0, 1, B // 32 - 1):
        assert torch.equal(HopHip.apply(w, h[tile:tile + 1].contiguous(), *index, *layer)[0], many[tile])
    dense = torch.zeros(len(deg), n_src, device="cuda", dtype=torch.float64)
    dense[put(row, np.int64), put(col, np.int64)] = w.double()
    want = dense @ h[0].double() + (b.double()[:, None] if bias else 0)
    # a sum of n terms in float32 is off by at most n 2^-24 of the sum of their magnitudes
    bound = (put(deg, np.float64)[:, None] + 2) * 2.0 ** -24 * (dense.abs() @ h[0].double().abs() + 4)
    assert ((many[0].double() - want).abs() <= bound).all()


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("n_dn", [500, 513, 1332, 1700])
def test_read_out_of_any_batch(gpu_lib, n_dn, bf16):
    """The read-out keeps more of a wave's 8-row groups in flight up to 1,024 samples (1, 2, 3 or 4 groups at these
    sizes): logits bit for bit those of a larger batch."""
    s, params = synth_3hop(sizes=(600, 900, 800, n_dn), edges=(9_000, 8_000, 12_000), redrive=(60, 20, 2))
    obs = np.random.default_rng(n_dn).standard_normal((1088, s["obs_dim"])).astype(np.float32)
    core = Core(s, params, 1088, int(bf16))
    want = core.forward(obs)
    for n in (64, 1024):
        assert np.array_equal(core.forward(obs[:n]), want[:n]), n


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("n", [1, 31, 32, 33, 64, 65, 96, 100])
def test_any_number_of_samples(gpu_lib, net, n, bf16):
    """fc_forward_n and fc_backward_n against whole tiles padded by the caller (the last row repeated, no gradient):
    logits and gradients bit for bit, and nothing written past the n-th sample's logits."""
    s, params = net
    B = 128
    rng = np.random.default_rng(n)
    obs = rng.standard_normal((n, s["obs_dim"])).astype(np.float32)
    dl = rng.standard_normal((n, s["n_act"])).astype(np.float32)
    core = Core(s, params, B, int(bf16))
    whole = -(-n // (64 if bf16 else 32)) * (64 if bf16 else 32)
    core.zero_grad()
    want = core.forward(np.concatenate([obs, np.repeat(obs[-1:], whole - n, 0)]))
    core.backward(np.concatenate([dl, np.zeros((whole - n, s["n_act"]), np.float32)]))
    grads = core.get(4)
    core.zero_grad()
    x, d = torch.as_tensor(obs).cuda(), torch.as_tensor(dl).cuda()
    logits = torch.full((n + 1, s["n_act"]), 7.0, device="cuda")
    call("fc_forward_n", core.h, x.data_ptr(), n, logits.data_ptr(), 0)
    call("fc_backward_n", core.h, d.data_ptr(), n)
    torch.cuda.synchronize()
    assert np.array_equal(logits[:n].cpu().numpy(), want[:n]) and bool((logits[n] == 7).all())
    for name, a, b in zip(NAMES, grads, core.get(4)):
        assert np.array_equal(a, b), name
    for bad in (0, -1, 129, 2**31 - 1):
        with pytest.raises(RuntimeError):
            call("fc_forward_n", core.h, x.data_ptr(), bad, logits.data_ptr(), 0)


@pytest.mark.parametrize("bf16", [False, True])
def test_a_gradient_of_another_batch_is_refused(gpu_lib, net, bf16):
    """fc_backward_n takes the last forward's number of samples and fc_backward a batch that was whole: the samples that
    filled the last tile have no gradient, and no real one is left out."""
    s, params = net
    core = Core(s, params, 128, int(bf16))
    x = torch.randn(128, s["obs_dim"], device="cuda", generator=torch.Generator(device="cuda").manual_seed(0))
    d = torch.ones(128, s["n_act"], device="cuda")
    logits = torch.empty(128, s["n_act"], device="cuda")
    core.zero_grad()
    call("fc_forward_n", core.h, x.data_ptr(), 100, logits.data_ptr(), 0)
    for name, n in (("fc_backward_n", 99), ("fc_backward_n", 101), ("fc_backward_n", 128), ("fc_backward", 128)):
        with pytest.raises(RuntimeError):
            call(name, core.h, d.data_ptr(), n)
    assert not any(g.any() for g in core.get(4))
    call("fc_backward_n", core.h, d.data_ptr(), 100)
    call("fc_forward", core.h, x.data_ptr(), 128, logits.data_ptr(), 0)
    with pytest.raises(RuntimeError):
        call("fc_backward_n", core.h, d.data_ptr(), 100)
    call("fc_backward", core.h, d.data_ptr(), 128)
    call("fc_backward_n", core.h, d.data_ptr(), 128)


@pytest.mark.parametrize("share", [0.0, 0.1, 0.3, 0.9])
@pytest.mark.parametrize("bf16", [False, True])
def test_order_of_waves_over_silent_rows(gpu_lib, uneven, monkeypatch, bf16, share):
    """A plan of unequal rows is walked in one order or another by the share of silent source rows: logits and every
    layer's states bit for bit those of a forward that skips none."""
    s, params = uneven
    params = list(params)
    params[2] = np.where(np.random.default_rng(1).random(params[2].size) < share, np.float32(30), params[2]).astype(np.float32)
    B = 64 * 11
    obs = np.random.default_rng(2).standard_normal((B, s["obs_dim"])).astype(np.float32)
    got = []
    for mode in ("0", "1"):
        monkeypatch.setenv("FLYGUY_SKIP_SILENT", mode)
        core = Core(s, params, B, int(bf16))
        got.append([core.forward(obs)] + [core.state(k, 0, n, B) for k, n in enumerate(s["sizes"])])
    for a, b in zip(*got):
        assert np.array_equal(a, b)
