"""The tiled layer form of HopHip and FireHip (fh_layer, fh_layer_bwd, fh_redrive_bwd, fh_fire_tiled, fh_fire_bwd_tiled)
against the row-major form with PyTorch's own additions."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from flyguy_amd.fly_hip import FireHip, HopHip
from gpu_helpers import rel
from test_gpu_hop_random import random_product

pytestmark = pytest.mark.gpu


def tiled(x):
    return x.view(x.shape[0], -1, 32).transpose(0, 1).contiguous()


def rows(x):
    return x.transpose(0, 1).reshape(x.shape[1], -1)


@pytest.mark.parametrize("seed", range(10))
@pytest.mark.parametrize("extra", ["bias", "drive", "shared drive", "none"])
def test_layer_against_the_row_major_form(gpu_lib, seed, extra):
    n_rows, n_src, B, crow, col, r, tcrow, tcol, tperm, w, rng = random_product(seed)
    n_s = 37
    put = lambda a: torch.as_tensor(np.ascontiguousarray(a)).cuda()      # noqa: E731
    index = tuple(put(a) for a in (crow, col, tcrow, tcol, tperm))
    leaf = lambda a: put(np.asarray(a, np.float32)).requires_grad_()     # noqa: E731
    h0, d0, b0 = rng.random((n_src, B)), rng.standard_normal((n_s, B)), rng.standard_normal(n_rows)
    g0, t0 = 1 + 0.1 * rng.standard_normal(n_rows), 0.1 * rng.random(n_rows)
    m = min(n_rows, n_s) // 2
    redriven = put(np.sort(rng.choice(n_rows, m, replace=False)).astype(np.int64))
    drive_rows = put(rng.integers(0, max(1, n_s // 4), m) if extra == "shared drive"
                     else rng.choice(n_s, m, replace=False).astype(np.int64)).long()
    gh = put(rng.standard_normal((n_rows, B)).astype(np.float32))

    def run(form):
        wd, h, d, b, g, t = leaf(w), leaf(h0), leaf(d0), leaf(b0), leaf(g0), leaf(t0)
        if form == "tiled":
            args = (b if extra == "bias" else None,) + ((tiled(d), redriven, drive_rows) if "drive" in extra
                                                        else (None, None, None))
            z = HopHip.apply(wd, tiled(h), *index, False, *args)
            out, z = rows(FireHip.apply(z, g, t)), rows(z)
        else:
            z = HopHip.apply(wd, h, *index, False)
            if extra == "bias":
                z = z + b[:, None]
            elif "drive" in extra:
                z = z.index_add(0, redriven, d.index_select(0, drive_rows))
            out = FireHip.apply(z, g, t)
        grads = torch.autograd.grad(out, (wd, h, d, b, g, t), gh, allow_unused=True)
        return z.detach(), out.detach(), grads
    (z1, o1, g1), (z2, o2, g2) = run("tiled"), run("rows")
    assert torch.equal(z1, z2) and torch.equal(o1, o2)
    for name, a, b in zip(("w", "h", "drive", "bias", "gain", "threshold"), g1, g2):
        assert (a is None) == (b is None), name
        if a is None:
            continue
        if name in ("h", "gain", "threshold") or (name == "drive" and extra == "drive"):
            assert torch.equal(a, b), name
        else:
            # w: two tiles' partials summed first; bias and a shared drive row: another order.  Sums of up to 256 float32
            # terms, a few rounding errors of 6e-8 of the larger partial sums
            assert a.numel() == 0 or rel(a.cpu(), b.cpu()) <= 2e-6, name
