"""The tiled and binary16 products (fh_*, HopHip) on a graph whose plans have at least three steps a wave, so that they
take 6-byte pairs, and whose longest waves are at least four times the middle one, so that the forward's waves are dealt
out anew with empty places at the end."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from flyguy_amd import fly_hip
from flyguy_amd._lib import call, plan_rows
from flyguy_amd.fly_hip import _args, _plan
from test_gpu_layer import tiled

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


def test_the_graph_is_of_that_kind(graph):
    index, _, _, p = graph
    dealt = fly_hip._striped(p)
    assert dealt is not p and _narrow(dealt) and p["nslot"] > 0
    assert len(p["wave"]) % 4 and len(dealt["wave"]) % 4 == 0          # (empty places)
    assert _narrow(plan_rows(index[2].cpu().numpy()))                  # the transposed plan


def _states(B, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    h = torch.relu(torch.randn(N_SRC, B, device="cuda", generator=g))
    gz = torch.randn(HEAVY + LIGHT, B, device="cuda", generator=g).clamp(-2, 2)
    gz[0] = 2.0                                 # (one largest value, so that any piece of the batch has the same scale)
    return h, gz


# ------------------------------------------------------------------------------------------------ plans of a caller's own
def _forward_c(d, w, h, half):
    """A caller's product through the C entry points on a plan d: (with row-major states or none, tiled or binary16)."""
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
