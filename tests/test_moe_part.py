"""The mixture's part on the CPU: what it hands to the kernels."""
import torch

from zinfer_amd.config.specs import GatedExpertSpec, MoeSpec
from zinfer_amd.engine.batch import Scratch, StepContext
from zinfer_amd.parts import moe
from zinfer_amd.parts.base import BuildContext


def _part(prefix, W=64, ff=64, E=4, top=2, shared=False, dtype=torch.float32):
    spec = MoeSpec(hidden_size=W, n_experts=E, top_k=top, expert=GatedExpertSpec(ff),
                   shared=GatedExpertSpec(ff) if shared else None)
    part = moe.MoeFeedForward(spec, BuildContext(dtype, torch.device("cpu")), prefix)
    g = torch.Generator().manual_seed(1)
    part.bind({n: torch.randn(d.shape, generator=g) * 0.1 for n, d in part.declare().items()})
    return part


def _step(scratch):
    none = dict.fromkeys(("token_ids", "positions", "seq_index", "q_start", "ctx_len",
                          "state_slots", "want_rows"))
    return StepContext(n_tokens=3, n_seqs=3, n_want=3, kv=[], max_q_len=1, max_ctx_len=1,
                       q_lens=[1] * 3, ctx_lens=[1] * 3, slots=[0] * 3, _scratch=scratch, **none)


def test_engines_on_one_model_do_not_share_the_routers_counters(monkeypatch):
    """The router's sums and counters between workgroups are the engine's (its scratch memory's),
    not the model's: two engines on one model may run at the same time on two streams."""
    seen = []
    monkeypatch.setattr(moe.ops, "moe_route", lambda *a, work=None, **kw: seen.append(work))
    monkeypatch.setattr(moe.ops, "moe_experts", lambda *a, **kw: None)
    layers = [_part("a."), _part("b.")]
    engines = [Scratch(torch.device("cpu")) for _ in range(2)]
    h, residual = torch.zeros((3, 64)), torch.zeros((3, 64))
    for scratch in engines + engines:
        for part in layers:
            part.forward(h, residual, _step(scratch))
    first, second = seen[:2], seen[2:4]
    assert all(w is not None and not w.any() for w in seen)
    assert first[0] is first[1] and second[0] is second[1]      # (its launches follow each other)
    assert first[0].data_ptr() != second[0].data_ptr()
    assert seen[4] is first[0] and seen[6] is second[0]
