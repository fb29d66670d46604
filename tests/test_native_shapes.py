"""NativeFlyActor hands the library whole observations only: the library reads obs_dim values a sample, so a batch of
another width would be read across its samples (CPU; the library calls are recorded, not made)."""
from __future__ import annotations

import pytest
import torch

from flyguy_amd import fly_native


@pytest.fixture
def session(monkeypatch):
    s = fly_native._Session.__new__(fly_native._Session)
    s.handle, s.stream, s.obs_dim, s.evaluations, s.calls = None, None, 12, 0, []
    monkeypatch.setattr(fly_native._Session, "on_current_stream", lambda self, device: None)
    monkeypatch.setattr(fly_native, "call", lambda name, *args: s.calls.append((name, args[2])))
    return s


@pytest.mark.parametrize("n", [1, 5, 32, 64])
@pytest.mark.parametrize("shape", [(13,), (11,), (24,), (1,), (), (3, 5)])
def test_another_width_is_refused(session, n, shape):
    with pytest.raises(ValueError):
        session.evaluate(torch.zeros(n, *shape), 90)
    assert not session.calls and session.evaluations == 0


@pytest.mark.parametrize("n", [1, 5, 32, 64])
@pytest.mark.parametrize("shape", [(12,), (3, 4)])
def test_whole_observations_at_any_batch(session, n, shape):
    assert session.evaluate(torch.zeros(n, *shape), 90).shape == (n, 90)
    assert session.calls == [("fc_forward_n", n)]
