"""Whether a call keeps its prefix states: never more than the stated fraction of the memory that is free, however small they are."""
import types

import pytest
import torch

from fastmax_amd import attention


@pytest.mark.parametrize("need,free,fits", [(100, 400, True), (101, 400, False), (8 << 20, 1 << 20, False), (4096, 0, False), (0, 0, True)])
def test_kept_states_stay_within_the_fraction_of_free_memory(monkeypatch, need, free, fits):
    ext = types.SimpleNamespace(saved_state_bytes=lambda *a: need, saved_state_bytes_strided=lambda *a: need)
    monkeypatch.setattr(attention._ext, "load", lambda: ext)
    monkeypatch.setattr(torch.cuda, "mem_get_info", lambda device=None: (free, 1 << 38))
    monkeypatch.setattr(attention, "SAVE_STATES_MEMORY_FRACTION", 0.25)
    t = torch.empty(1, 4, 32)
    assert attention._states_fit(t, t, True, 2) is fits
    assert attention._states_fit_bytes(ext, t, t, True, 2) is fits
