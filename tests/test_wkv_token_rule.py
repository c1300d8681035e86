"""Which steps of single tokens take their decays, recurrence, norm and gate in one launch: sizes on both sides of each line as measured in whole decode steps, and a mixer that asks the rule."""
from types import SimpleNamespace

import pytest
import torch

from torchlet_amd.kernels import ops
from torchlet_amd.parts import wkv


@pytest.mark.parametrize("requests, heads, dim, vdim, rank, one", [
    (1, 32, 64, 64, 64, True), (32, 32, 64, 64, 64, True), (64, 32, 64, 64, 64, False), (8, 64, 64, 64, 64, True), (32, 64, 64, 64, 64, False), (32, 48, 64, 64, 64, False), (16, 32, 32, 32, 64, True),
    (64, 32, 32, 32, 64, False), (1, 16, 128, 128, 64, True), (32, 16, 128, 128, 64, True), (64, 16, 128, 128, 64, False), (32, 24, 96, 96, 64, False), (1, 32, 64, 64, 96, False), (16, 32, 64, 64, 128, False)])
def test_one_launch_where_it_was_faster(monkeypatch, requests, heads, dim, vdim, rank, one):
    monkeypatch.setattr(ops, "compute_units", lambda: 256)
    assert ops.wkv_token_pays(requests, heads, dim, vdim, rank) == one


@pytest.mark.parametrize("requests, one", [(16, True), (64, False)])
def test_the_mixer_asks_the_rule(monkeypatch, requests, one):
    """A mixer of 32 heads of 64 x 64 with every kernel replaced by a note that it was called."""
    heads, dim, hidden, rank = 32, 64, 16, 8
    called = []
    note = lambda name, result=None: monkeypatch.setattr(ops, name, lambda *a, **k: (called.append(name), result)[1])
    for name in ("linear_groups_beside", "channel_decay", "wkv_scan", "gated_head_norm"):
        note(name)
    note("wkv_token", True)
    monkeypatch.setattr(ops, "compute_units", lambda: 256)
    monkeypatch.setattr(ops, "settle_shift", lambda residual, *a: residual)
    monkeypatch.setattr(wkv, "project_out", lambda mixed, *a: mixed)
    mixer = SimpleNamespace(heads=heads, dim=dim, vdim=dim, hidden=hidden, k_width=heads * dim, v_width=heads * dim, dtype=torch.float32, state_floats=heads * dim * dim, mu=None, w_rkvg=None,
                            w_rk=None, w_vg=None, w1=torch.zeros(rank, hidden), w2t=None, w0=None, bonus=None, w_norm=None, w_o=None, spec=SimpleNamespace(norm_eps=1e-5))
    note("linear_groups")
    ctx = SimpleNamespace(max_new_tokens=1, req_indptr=torch.arange(requests + 1, dtype=torch.int32), slots=None, token_req=None)
    wkv.WKV.forward(mixer, torch.zeros(requests, hidden), ctx, SimpleNamespace(state=None))
    assert ("wkv_token" in called) == one and ("wkv_scan" in called) != one
