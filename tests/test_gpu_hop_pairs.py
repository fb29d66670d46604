"""The tiled and binary16 products (fh_*, HopHip) on a graph whose plans have at least three steps a wave, so that they
take 6-byte pairs, and whose longest waves are at least four times the middle one, so that the forward's waves are dealt
out anew with empty places at the end; and their backwards with one and with two tiles per workgroup."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from flyguy_amd import fly_hip
from flyguy_amd._lib import call, plan_rows
from flyguy_amd.fly_hip import FireHip, HopHip, _args, _plan
from flyguy_amd.synth import scaled_3hop
from test_gpu_layer import rows, tiled

pytestmark = pytest.mark.gpu

HEAVY, LIGHT, N_SRC = 1000, 6013, 3000


def put(a, t):
    return torch.as_tensor(np.ascontiguousarray(a, dtype=t)).cuda()


def _index(crow, col, n_src):
    """(crow, col, tcrow, tcol, tperm) on the GPU, as HopHip takes them, and the row of every connection."""
    order = np.argsort(col, kind="stable")
    row = np.repeat(np.arange(len(crow) - 1), np.diff(crow))
    tcrow = np.concatenate([[0], np.cumsum(np.bincount(col, minlength=n_src))])
    return (put(crow, np.int64), put(col, np.int32), put(tcrow, np.int64), put(row[order], np.int32),
            put(order, np.int64)), row


@pytest.fixture(scope="module")
def graph():
    """1,000 rows of about 280 connections (split) among 6,013 of 0 to 9, in a drawn order; 3,000 sources."""
    rng = np.random.default_rng(11)
    deg = np.concatenate([rng.integers(240, 320, HEAVY), rng.integers(0, 10, LIGHT)])
    rng.shuffle(deg)
    crow = np.concatenate([[0], np.cumsum(deg)]).astype(np.int64)
    col = np.concatenate([np.sort(rng.choice(N_SRC, d, replace=False)) for d in deg]).astype(np.int32)
    index, row = _index(crow, col, N_SRC)
    w = torch.as_tensor(rng.standard_normal(len(col)).astype(np.float32)).cuda()
    return index, put(row, np.int64), w, plan_rows(crow)


def _narrow(p) -> bool:
    return len(p["pos"]) % 64 == 0 and len(p["pos"]) // 64 >= 3 * len(p["wave"])


def test_the_graphs_are_of_their_kinds(graph, light):
    index, _, _, p = graph
    dealt = fly_hip._striped(p)
    assert dealt is not p and _narrow(dealt) and p["nslot"] > 0
    assert len(p["wave"]) % 4 and len(dealt["wave"]) % 4 == 0          # (empty places)
    assert _narrow(plan_rows(index[2].cpu().numpy()))                  # the transposed plan
    assert not any(_narrow(plan_rows(light[0][k].cpu().numpy())) for k in (0, 2))


def _states(B, seed, n_rows=HEAVY + LIGHT, n_src=N_SRC):
    g = torch.Generator(device="cuda").manual_seed(seed)
    h = torch.relu(torch.randn(n_src, B, device="cuda", generator=g))
    gz = torch.randn(n_rows, B, device="cuda", generator=g).clamp(-2, 2)
    gz[0] = 2.0                                 # (one largest value, so that any piece of the batch has the same scale)
    return h, gz


@pytest.mark.parametrize("B", [32, 96, 160, 288])
def test_float32_products_against_eight_byte_pairs(gpu_lib, graph, B):
    """HopHip against fh_spmm / fh_spmm_bwd on row-major states, whose pairs take 8 bytes and whose plan is taken in a
    row: output, state gradient and strengths' gradient bit for bit."""
    index, _, w, _ = graph
    h, gz = _states(B, B)
    wd, hd = w.clone().requires_grad_(), h.clone().requires_grad_()
    got = HopHip.apply(wd, hd, *index, False)
    gw, gh = torch.autograd.grad(got, (wd, hd), gz)
    st = torch.cuda.current_stream().cuda_stream
    E, n_rows = w.numel(), gz.shape[0]

    def plan(*a):
        d = _plan(*a, E)
        return (d, torch.empty(d["npos"], 2, dtype=torch.int32, device="cuda"),
                torch.empty(max(d["nslot"] * B, 1), device="cuda"))
    d, cw, part = plan(index[0], index[1], None)
    out = torch.full_like(gz, float("nan"))
    call("fh_spmm", *_args(d), w.data_ptr(), h.data_ptr(), out.data_ptr(), n_rows, N_SRC, B, cw.data_ptr(),
         part.data_ptr(), st)
    assert torch.equal(got.detach(), out)
    d, cw, part = plan(index[2], index[3], index[4])
    want_h, want_w = torch.full_like(h, float("nan")), torch.zeros_like(w)
    gwpart = torch.empty(d["npos"] * (B // 32), device="cuda")
    call("fh_spmm_bwd", *_args(d), w.data_ptr(), gz.data_ptr(), h.data_ptr(), want_h.data_ptr(), want_w.data_ptr(),
         n_rows, N_SRC, B, cw.data_ptr(), gwpart.data_ptr(), part.data_ptr(), st)
    assert torch.equal(gh, want_h) and torch.equal(gw, want_w)


@pytest.fixture(scope="module")
def light():
    """Hop 2 of the benchmark network divided by 16: two steps a wave, 8-byte pairs."""
    s, params = scaled_3hop(16)
    h = s["hop"][1]
    base = int(h["widx"].min())
    index = (put(h["crow"], np.int64), put(h["col"], np.int32), put(h["tcrow"], np.int64), put(h["tcol"], np.int32),
             put(h["twidx"] - base, np.int64))
    return index, put(params[0][h["widx"]], np.float32)


def _take(monkeypatch, pair):
    """HopHip's backwards with two tiles per workgroup (pair) or one, whatever the graph."""
    monkeypatch.setattr(fly_hip, "bwd_pairs", lambda crow: pair)
    monkeypatch.setattr(fly_hip, "PAIR_FROM", 33)
    monkeypatch.setattr(fly_hip, "_plans", type(fly_hip._plans)())


@pytest.mark.parametrize("pair", [False, True])
@pytest.mark.parametrize("B", [32, 64, 96, 416])
@pytest.mark.parametrize("extra", ["bias", "drive"])
@pytest.mark.parametrize("kind", ["narrow", "wide"])
def test_layer_form(gpu_lib, graph, light, monkeypatch, kind, extra, B, pair):
    """The layer form, its bias or re-driven rows (in whole and in split rows, of a re-dealt plan where the pairs are
    narrow), against the row-major form with PyTorch's additions."""
    _take(monkeypatch, pair)
    index, w0 = (graph[0], graph[2]) if kind == "narrow" else light
    n_rows, n_s = len(index[0]) - 1, 500
    h0, gz = _states(B, 7 * B, n_rows, len(index[2]) - 1)
    g = torch.Generator(device="cuda").manual_seed(5)
    d0 = torch.randn(n_s, B, device="cuda", generator=g)
    b0 = torch.randn(n_rows, device="cuda", generator=g)
    gain = 1 + 0.1 * torch.randn(n_rows, device="cuda", generator=g)
    thr = 0.1 * torch.rand(n_rows, device="cuda", generator=g)
    redriven = torch.randperm(n_rows, device="cuda", generator=g)[:n_s - 20].sort().values
    drive_rows = torch.randperm(n_s, device="cuda", generator=g)[:n_s - 20]

    def run(form):
        w, h, d, b = (a.clone().requires_grad_() for a in (w0, h0, d0, b0))
        if form == "tiled":
            args = (b, None, None, None) if extra == "bias" else (None, tiled(d), redriven, drive_rows)
            z = HopHip.apply(w, tiled(h), *index, False, *args)
            out = rows(FireHip.apply(z, gain, thr))
            z = rows(z)
        else:
            z = HopHip.apply(w, h, *index, False)
            z = z + b[:, None] if extra == "bias" else z.index_add(0, redriven, d.index_select(0, drive_rows))
            out = FireHip.apply(z, gain, thr)
        grads = torch.autograd.grad(out, (w, h, b if extra == "bias" else d), gz)
        return z.detach(), grads
    (z1, g1), (z2, g2) = run("tiled"), run("rows")
    assert torch.equal(z1, z2) and torch.equal(g1[1], g2[1])
    if extra == "drive":
        assert torch.equal(g1[2], g2[2])
    if not pair:
        assert torch.equal(g1[0], g2[0])
    # a pair of tiles is added before the rest, and the bias in another order: sums of B terms in float32, off by at
    # most B 2^-24 of the sum of their magnitudes each way (a term: gain gz h, or gain gz)
    bound = 2 * float(gain.abs().max()) * B * 2.0 ** -24
    if pair and B > 32:
        row = torch.repeat_interleave(torch.arange(n_rows, device="cuda"), index[0].diff())
        size = torch.cat([(gz[r].abs() * h0[c.long()]).sum(1) for r, c in zip(row.split(50000), index[1].split(50000))])
        assert ((g1[0] - g2[0]).abs() <= bound * size + 1e-30).all()
    if extra == "bias":
        assert ((g1[2] - g2[2]).abs() <= bound * gz.abs().sum(1) + 1e-30).all()


@pytest.mark.parametrize("pair", [False, True])
@pytest.mark.parametrize("B", [32, 64, 96, 160, 416])
@pytest.mark.parametrize("kind", ["narrow", "wide"])
def test_binary16_product(gpu_lib, graph, light, monkeypatch, kind, B, pair):
    """The binary16 product and its backward, tiles alone and in pairs, with 6-byte (narrow) and 8-byte pairs: output and
    state gradient bit for bit those of single 64-sample tiles, and both and the strengths' gradient within float32 sums
    of the float64 product of the rounded operands."""
    _take(monkeypatch, pair)
    index, w0 = (graph[0], graph[2]) if kind == "narrow" else light
    crow, col, tcrow, tcol, tperm = index
    n_rows, n_src = len(crow) - 1, len(tcrow) - 1
    h, gz = _states(B, B, n_rows, n_src)

    def run(h, gz):
        w, h = w0.clone().requires_grad_(), h.contiguous().requires_grad_()
        out = HopHip.apply(w, h, *index, True)
        return (out.detach(),) + torch.autograd.grad(out, (w, h), gz.contiguous())
    out, gw, gh = run(h, gz)
    parts = [run(h[:, i:i + 64], gz[:, i:i + 64]) for i in range(0, B, 64)]
    assert torch.equal(out, torch.cat([p[0] for p in parts], 1))
    assert torch.equal(gh, torch.cat([p[2] for p in parts], 1))
    h16, g16, w = h.half().double(), (gz / 2).half().double() * 2, w0.double()
    row = torch.repeat_interleave(torch.arange(n_rows, device="cuda"), crow.diff())

    def dense(vals):
        return torch.zeros(n_rows, n_src, device="cuda", dtype=torch.float64).index_put_((row, col.long()), vals)
    a, aa = dense(w), dense(w.abs())
    u = 2.0 ** -24                              # n float32 additions are off by at most n u of the magnitudes' sum
    deg, tdeg = crow.diff()[:, None].double(), tcrow.diff()[:, None].double()
    assert ((out.double() - a @ h16).abs() <= (deg + 2) * u * (aa @ h16)).all()
    assert ((gh.double() - a.t() @ g16).abs() <= (tdeg + 4) * u * (aa.t() @ g16.abs()) + 1e-30).all()
    for i in range(0, len(row), 50000):
        r, c = row[i:i + 50000], col[i:i + 50000].long()
        terms = g16[r] * h16[c]
        assert ((gw[i:i + 50000].double() - terms.sum(1)).abs() <= (B + 4) * u * terms.abs().sum(1) + 1e-30).all()


def test_pairs_of_tiles_from_a_batch_up(gpu_lib, light, monkeypatch):
    """Below PAIR_FROM samples the backwards take one tile per workgroup whatever the graph: the gradients of both forms
    bit for bit those with pairs turned off; from there up a graph that pairs has them."""
    index, w0 = light
    n_rows, n_src = len(index[0]) - 1, len(index[2]) - 1
    assert fly_hip.bwd_pairs(index[0].cpu().numpy())

    def grads(B):
        g = torch.Generator(device="cuda").manual_seed(B)
        h = torch.relu(torch.randn(n_src, B, device="cuda", generator=g))
        gz = torch.randn(n_rows, B, device="cuda", generator=g)
        out = []
        for args, a, b in (((False, None, None, None, None), tiled(h), tiled(gz)), ((True,), h, gz)):
            w, a = w0.clone().requires_grad_(), a.clone().requires_grad_()
            out += torch.autograd.grad(HopHip.apply(w, a, *index, *args), (w, a), b)
        return out
    sizes = (32, 64, 96, fly_hip.PAIR_FROM - 32, fly_hip.PAIR_FROM)
    got = [grads(B) for B in sizes]
    monkeypatch.setattr(fly_hip, "bwd_pairs", lambda crow: False)
    monkeypatch.setattr(fly_hip, "_plans", type(fly_hip._plans)())
    for B, a in zip(sizes, got):
        same = [torch.equal(x, y) for x, y in zip(a, grads(B))]
        assert same == ([True] * 4 if B < fly_hip.PAIR_FROM else [False, True, False, True]), B


# ------------------------------------------------------------------------------------------------ plans of a caller's own
def _forward_c(d, w, h, half):
    """A product as a C caller makes it on the plan d, over tiled or binary16 states."""
    n_src, B = h.shape
    n_rows, st = HEAVY + LIGHT, torch.cuda.current_stream().cuda_stream
    cw = torch.empty(d["npos"], 2, dtype=torch.int32, device="cuda")
    part = torch.empty(max(d["nslot"] * (-(-B // 64) * 64), 1), device="cuda")
    out = torch.full((n_rows, B), 7.0, device="cuda")
    if half:
        src = torch.empty(-(-B // 64) * n_src * 64, dtype=torch.float16, device="cuda")
        call("fh_to_half", h.data_ptr(), n_src, B, None, src.data_ptr(), st)
        call("fh_spmm_h", *_args(d), w.data_ptr(), src.data_ptr(), out.data_ptr(), n_rows, n_src, B, cw.data_ptr(),
             part.data_ptr(), st)
    else:
        src = tiled(h)
        call("fh_spmm_tiled", *_args(d), w.data_ptr(), src.data_ptr(), out.data_ptr(), n_rows, n_src, B, cw.data_ptr(),
             part.data_ptr(), st)
    torch.cuda.synchronize()
    return out


@pytest.mark.parametrize("half", [False, True])
def test_a_source_past_the_states_reads_zeros(gpu_lib, graph, half):
    """A plan position whose source is no row of the states (65,536 + r among them, which 16 bits would turn into r) adds
    nothing: the product with those connections' strengths zero."""
    index, _, w, _ = graph
    d = dict(_plan(index[0], index[1], None, w.numel(), forward=True))
    h, _ = _states(64, 3)
    pcol, pidx = d["pcol"].clone(), d["pidx"].long()
    at = torch.nonzero(pidx >= 0).flatten()[::7]
    pcol[at[0::3]] += 65536
    pcol[at[1::3]] = N_SRC + (pcol[at[1::3]] % 60000)
    pcol[at[2::3]] = 0x01FFFFFF - pcol[at[2::3]]
    silent = w.clone()
    silent[pidx[at]] = 0
    want = _forward_c(d, silent, h, half)
    got = _forward_c(dict(d, pcol=pcol), w, h, half)
    assert torch.equal(got, want)


@pytest.mark.parametrize("half", [False, True])
def test_a_wave_off_the_steps_boundary_is_no_wave(gpu_lib, graph, half):
    """The positions of a wave start at a multiple of 64 (fc_plan_rows); with 6-byte pairs a record that says otherwise
    is refused like any other outside the plan: its rows are left alone, no other step's pairs are summed into them."""
    index, _, w, p = graph
    d = dict(_plan(index[0], index[1], None, w.numel()))               # (not dealt out anew: wave 0 has the longest rows)
    h, _ = _states(64, 4)
    last = len(p["wave"]) - 1
    while p["wave"][last, 1] == 0:
        last -= 1
    wave = d["wave"].clone()
    wave[last, 0] -= 32
    touched = p["seg"][8 * last:8 * last + 8]
    touched = put(touched[(touched[:, 0] >= 0) & (touched[:, 1] < 0), 0], np.int64)
    want = _forward_c(d, w, h, half)
    got = _forward_c(dict(d, wave=wave), w, h, half)
    assert len(touched) and (got[touched] == 7).all()
    want[touched] = 7
    assert torch.equal(got, want)


def test_a_re_drive_field_past_the_drive_is_none(gpu_lib, graph):
    """fh_layer on a plan whose re-drive fields name rows past the drive, in whole and in split rows: as with -1 there
    (the drive is the front of a larger buffer)."""
    index, _, w, _ = graph
    B, n_s, n_rows = 96, 50, HEAVY + LIGHT
    h, _ = _states(B, 5)
    drive = torch.randn(B // 32 + 1, n_s, 32, device="cuda", generator=torch.Generator(device="cuda").manual_seed(6))
    d = dict(_plan(index[0], index[1], None, w.numel()))
    seg, split = d["seg"].clone(), d["split"].clone()
    seg[:, 2] = torch.where(seg[:, 0] >= 0, seg[:, 0] % (2 * n_s), -1).to(torch.int32)
    split[:, 3] = split[:, 0] % (2 * n_s)

    def layer(seg, split):
        out = torch.full((B // 32, n_rows, 32), 7.0, device="cuda")
        cw = torch.empty(d["npos"], 2, dtype=torch.int32, device="cuda")
        part = torch.empty(max(d["nslot"] * B, 1), device="cuda")
        src = tiled(h)
        call("fh_layer", *_args(dict(d, seg=seg, split=split)), w.data_ptr(), src.data_ptr(), None, drive.data_ptr(), n_s,
             out.data_ptr(), n_rows, N_SRC, B, cw.data_ptr(), part.data_ptr(), torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        return out
    got = layer(seg, split)
    seg[:, 2][seg[:, 2] >= n_s] = -1
    split[:, 3][split[:, 3] >= n_s] = -1
    assert torch.equal(got, layer(seg, split))
    assert not torch.equal(got, layer(d["seg"], d["split"]))
