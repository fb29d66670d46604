"""fc_copy's one-launch copies, and the gradient a teaching step leaves when one was copied in before it."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from flyguy_amd._lib import LibraryError, call, lib
from flyguy_amd.synth import scaled_3hop
from gpu_helpers import NAMES, Core

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("offset", [0, 1, 2, 3, 4])
def test_copies_at_any_alignment(gpu_lib, offset):
    """Arrays that start at any float of a 16-byte unit, and a null pointer in between: copied in and out unchanged,
    nothing written around them."""
    s, params = scaled_3hop(64)
    core = Core(s, params, 32)
    rng = np.random.default_rng(offset)
    want = [rng.standard_normal(n).astype(np.float32) for n in core.sizes]
    kept = core.get(2)[3]
    bufs = [torch.full((n + 16,), 7.0, device="cuda") for n in core.sizes]
    for b, w in zip(bufs, want):
        b[offset:offset + w.size] = torch.as_tensor(w).cuda()
    ptrs = (ctypes.c_void_p * 7)(*[b.data_ptr() + 4 * offset for b in bufs])
    ptrs[3] = None
    call("fc_copy", core.h, 2, 1, ptrs)
    for k, (name, got) in enumerate(zip(NAMES, core.get(2))):
        assert np.array_equal(got, kept if k == 3 else want[k]), name
    out = [torch.full((n + 16,), 7.0, device="cuda") for n in core.sizes]
    ptrs = (ctypes.c_void_p * 7)(*[b.data_ptr() + 4 * offset for b in out])
    ptrs[3] = None
    call("fc_copy", core.h, 2, 0, ptrs)
    for k, b in enumerate(out):
        b = b.cpu().numpy()
        n = core.sizes[k]
        assert (b[:offset] == 7).all() and (b[offset + n:] == 7).all()
        assert np.array_equal(b[offset:offset + n], np.full(n, 7, np.float32) if k == 3 else want[k])


def test_host_memory_still_goes_through_the_runtime(gpu_lib):
    """Pinned host memory, which the runtime's copy takes, is copied as before."""
    s, params = scaled_3hop(64)
    core = Core(s, params, 32)
    host = [torch.empty(n).pin_memory() for n in core.sizes]
    try:
        call("fc_copy", core.h, 0, 0, (ctypes.c_void_p * 7)(*[h.data_ptr() for h in host]))
    except LibraryError:
        pytest.skip("the runtime refuses host memory here")
    for h, p in zip(host, params):
        assert np.array_equal(h.numpy(), p.reshape(-1))


@pytest.mark.parametrize("bf16", [False, True])
def test_step_after_a_copied_gradient(gpu_lib, bf16):
    """A teaching step's gradient does not depend on what the gradient held: entries no backward writes (here the
    neurons of no layer) are zero after it."""
    s, params = scaled_3hop(64)
    s = dict(s, n_neurons=s["n_neurons"] + 5)                 # five neurons in no layer
    params = list(params)
    params[1] = np.concatenate([params[1], np.ones(5, np.float32)])
    params[2] = np.concatenate([params[2], np.zeros(5, np.float32)])
    rng = np.random.default_rng(0)
    obs = torch.as_tensor(rng.standard_normal((64, s["obs_dim"])).astype(np.float32)).cuda()
    tl = torch.as_tensor(rng.standard_normal((64, s["n_act"])).astype(np.float32)).cuda()
    got = []
    for dirty in (False, True):
        core = Core(s, params, 64, int(bf16))
        if dirty:
            core.set(4, [np.full(n, 3.0, np.float32) for n in core.sizes])
        call("fc_teach_step", core.h, obs.data_ptr(), tl.data_ptr(), 64, 1.0, 1e-3, 1e-3, 1e-3, 0.0, 0.9, None)
        got.append(core.get(4))
    for name, a, b in zip(NAMES, *got):
        assert np.array_equal(a, b), name
    assert not got[0][1][-5:].any() and not got[0][2][-5:].any()


def _lone_neurons():
    """A network with five neurons in no layer, whose gradient entries no backward writes, and a batch for it."""
    s, params = scaled_3hop(64)
    s = dict(s, n_neurons=s["n_neurons"] + 5)
    params = list(params)
    params[1] = np.concatenate([params[1], np.ones(5, np.float32)])
    params[2] = np.concatenate([params[2], np.zeros(5, np.float32)])
    rng = np.random.default_rng(0)
    return s, params, *(torch.as_tensor(rng.standard_normal((64, n)).astype(np.float32)).cuda()
                        for n in (s["obs_dim"], s["n_act"]))


def _step(core, obs, tl):
    call("fc_teach_step", core.h, obs.data_ptr(), tl.data_ptr(), 64, 1.0, 0.0, 0.0, 0.0, 0.0, 0.9, None)


def test_a_captured_step_clears_what_was_copied_in_since(gpu_lib):
    """A teaching step in a HIP graph (its rates zero, so that every replay sees the same weights), with a gradient
    copied in before each replay: the eager step's gradient every time."""
    s, params, obs, tl = _lone_neurons()
    core = Core(s, params, 64)
    _step(core, obs, tl)
    want = core.get(4)
    stream = torch.cuda.Stream()
    lib().fc_set_stream(core.h, stream.cuda_stream)
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        _step(core, obs, tl)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        _step(core, obs, tl)
    for i in range(3):
        core.set(4, [np.full(n, 3.0 + i, np.float32) for n in core.sizes])
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        for name, a, b in zip(NAMES, want, core.get(4)):
            assert np.array_equal(a, b), (i, name)


def test_a_captured_clearing_has_cleared_nothing_yet(gpu_lib):
    """fc_zero_grad recorded into a graph that has not run: the next step still clears the gradient copied in before."""
    s, params, obs, tl = _lone_neurons()
    core = Core(s, params, 64)
    _step(core, obs, tl)
    want = core.get(4)
    core.set(4, [np.full(n, 3.0, np.float32) for n in core.sizes])
    stream = torch.cuda.Stream()
    lib().fc_set_stream(core.h, stream.cuda_stream)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        core.zero_grad()
    lib().fc_set_stream(core.h, 0)
    _step(core, obs, tl)
    for name, a, b in zip(NAMES, want, core.get(4)):
        assert np.array_equal(a, b), name
