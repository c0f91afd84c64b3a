"""CPU tier: the host path of the module calls. The memo of resident forms (moe._memo): an entry is reused only
while every source it was built from is the same object at the same version, and a source that goes away is a
change like any other. The config struct of the reference-dtype block, and the stream query."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from quanta_amd import moe as M


def _calls(anchor, kind):
    """(run, built): run(sources) through the memo, and the values built so far."""
    built = []

    def run(sources):
        return M._memo(anchor, kind, sources, lambda: built.append(len(built)) or built[-1])
    return run, built


@pytest.mark.parametrize("leaf", [lambda: torch.ones(3), lambda: np.ones(3), lambda: M.TiledExperts(a=1),
                                  lambda: M.MixedExperts(n_experts=1)])
def test_a_source_that_goes_away_rebuilds(leaf):
    anchor = torch.zeros(1)
    run, built = _calls(anchor, "gone")
    v = leaf()
    assert run([anchor, v]) == run([anchor, v]) == 0
    del v   # nothing else holds it: the entry's weak reference is dead
    assert run([anchor, None]) == 1 and run([anchor, None]) == 1
    w = leaf()
    assert run([anchor, w]) == 2


def test_a_prepared_block_without_its_optional_sources(monkeypatch):
    """prepare() after the shared expert's gate and the correction bias were removed, their tensors freed."""
    monkeypatch.setattr(M, "_build_prepared", lambda p, cfg, **kw: sorted(k for k, v in p.items() if v is not None))
    p = {"gate": torch.zeros(4, 8), "experts_gate_up": torch.zeros(1), "experts_down": torch.zeros(1),
         "shared_expert_gate": torch.zeros(1, 8), "e_score_correction_bias": torch.zeros(4)}
    cfg = M.MoEConfig(8, 4, 2, 4)
    assert "shared_expert_gate" in M.prepare(p, cfg)
    del p["shared_expert_gate"]
    p["e_score_correction_bias"] = None
    assert M.prepare(p, cfg) == ["experts_down", "experts_gate_up", "gate"]


def test_changes_that_rebuild_and_calls_that_do_not():
    anchor, t = torch.zeros(1), torch.ones(3)
    run, built = _calls(anchor, "changes")
    d = {"packed": t, "bits": 4, "group_size": 64}
    assert run([d, None]) == run([dict(reversed(d.items())), None]) == 0   # the same leaves and values
    t.add_(1)
    assert run([d, None]) == 1                  # written in place
    assert run([dict(d, bits=3), None]) == 2    # another value
    assert run([{"packed": t, "bits": 3}, None]) == 3
    assert run([{"packed": t, "bits": 3}, (t, 1)]) == 4
    assert run([{"packed": t, "bits": 3}, [t, 1]]) == 4
    assert run([t, [t, 1]]) == 5


@pytest.mark.parametrize("value", [lambda v: v, np.array, torch.tensor, np.float32])
def test_general_config_values(value):
    """The reference-dtype block's config struct: kept for plain values, read again from a config that holds an
    array or a tensor, which may have no hash or be written in place."""
    from types import SimpleNamespace

    limit = value(7.0)
    cfg = SimpleNamespace(hidden_size=32, num_experts=4, num_experts_per_tok=2, moe_intermediate_size=64,
                          swiglu_limit=limit)
    get = lambda: M._general_config(cfg, 2, 0, 0, (True, 0, 4, 32), None, None, False, False)
    assert get().act_limit == 7.0 and get().top_k == 2
    if isinstance(limit, (np.ndarray, torch.Tensor)):
        limit -= 2.0
    else:
        cfg.swiglu_limit = value(5.0)
    assert get().act_limit == 5.0
    assert len(M._GENERAL_CFG) <= M._GENERAL_CFG_MAX


def test_raw_stream_without_the_private_query(monkeypatch):
    from types import SimpleNamespace

    from quanta_amd import ops

    monkeypatch.setattr(ops, "_current_raw_stream", None)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda dev: SimpleNamespace(cuda_stream=(dev.type, 7)))
    assert ops._raw_stream(torch.zeros(1)) == ("cpu", 7)
