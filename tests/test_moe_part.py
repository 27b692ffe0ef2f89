"""The mixture's part on the CPU: what it hands to the kernels."""
import os
import re
import subprocess
from types import SimpleNamespace

import pytest
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


@pytest.mark.parametrize("W, ff, top, shared, tiled", [
    (256, 128, 8, False, False), (256, 128, 8, True, False), (1024, 512, 8, False, False),
    (1024, 1024, 4, True, False), (2048, 448, 4, True, False), (2048, 512, 2, True, True),
    (2048, 768, 4, False, False), (2048, 768, 4, True, True), (2048, 2048, 4, False, True),
    (2048, 2048, 2, False, False), (3072, 2048, 4, False, False), (3072, 2048, 2, True, True),
    (4096, 1024, 4, False, True)])
def test_experts_are_laid_out_anew_where_that_pays(monkeypatch, W, ff, top, shared, tiled):
    """Row by row where that is the faster form for a few tokens: narrow layers, few experts a token
    without a shared one."""
    asked, E = [], max(top, 2)
    monkeypatch.setattr(moe.ops, "moe_can_pretile", lambda gate_up, down: True)
    monkeypatch.setattr(moe.ops, "pretile_weight", lambda w: asked.append(w.shape) or w)
    monkeypatch.setattr(moe, "Linear", lambda w: SimpleNamespace(tiled=True, weight=w))
    spec = MoeSpec(hidden_size=W, n_experts=E, top_k=top, expert=GatedExpertSpec(ff),
                   shared=GatedExpertSpec(ff) if shared else None)
    part = moe.MoeFeedForward(spec, BuildContext(torch.bfloat16, torch.device("cpu")), "")
    part.bind({n: torch.zeros((1, 1), dtype=torch.bfloat16).expand(d.shape)
               for n, d in part.declare().items()})
    assert asked == ([(E * 2 * ff, W), (E * W, ff)] if tiled else [])


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


@pytest.mark.parametrize("W, ff, tiled", [(64, 64, False), (2048, 512, True)])
def test_bench_launches_a_mixture_as_the_engine_does(monkeypatch, W, ff, tiled):
    """Experts laid out by the same rule, work space for the router, the shared expert in the
    experts' kernels where it rides along there."""
    import bench
    T, E, top, calls = 4, 4, 2, []
    ops = moe.ops
    monkeypatch.setattr(ops, "moe_can_pretile", lambda gate_up, down: True)
    monkeypatch.setattr(ops, "moe_few_covers", lambda h, top: True)
    for name in ("moe_route", "moe_experts", "gemm", "gated_act"):
        monkeypatch.setattr(ops, name, lambda *a, name=name, **kw: calls.append((name, kw)))
    z = lambda *s, dt=torch.bfloat16: torch.zeros(s, dtype=dt)
    gate = z(T, 1, dt=torch.float32)
    run = bench._mixture_launcher(ops, z(T, W), z(E, W, dt=torch.float32),
                                  z(T, top, dt=torch.int32), z(T, top, dt=torch.float32),
                                  z(E, 2 * ff, W), z(E, W, ff), z(T, W, dt=torch.float32),
                                  shared=(z(128, W), z(W, 64), gate[:, 0]), scoring="sigmoid")
    run()
    (_, route), (_, experts) = calls[:2]
    assert route["work"] is not None and route["scoring"] == "sigmoid"
    assert experts["w_tiled"] == tiled and (experts["shared"] is not None) == tiled
    assert [name for name, _ in calls[2:]] == ([] if tiled else ["gemm", "gated_act", "gemm"])


def _compile_moe(arch, out):
    from zinfer_amd.ops import build
    if not os.path.exists("/opt/rocm/bin/hipcc"):
        pytest.skip("no compiler")
    flags = [f for f in build.FLAGS if f not in ("-shared", "-fPIC") and "offload-arch" not in f]
    return subprocess.run(["/opt/rocm/bin/hipcc", f"--offload-arch={arch}", *flags,
                           "--offload-device-only", "-S", "-I", build.CSRC,
                           os.path.join(build.CSRC, "moe.hip"), "-o", str(out)],
                          capture_output=True, text=True)


def test_the_routers_hand_over_between_workgroups(tmp_path):
    """In the code made for gfx950 the workgroups' sums leave past the caches before the count goes
    up (a wait for the stores), and the one that counts last reads them past the caches, behind
    the count's return.  For another target the file is refused: there the same source need not
    come out so."""
    out = tmp_path / "moe.s"
    assert _compile_moe("gfx950", out).returncode == 0
    bodies = re.findall(r"^(_Z18moe_route16_kernelI\wLb[01]ELb1EE\w+):[^\n]*\n(.*?)s_endpgm",
                        out.read_text(), re.S | re.M)
    assert len(bodies) == 4
    for name, body in bodies:
        code = [line.split(";")[0].strip() for line in body.splitlines()]

        def places(word, *more):
            return [i for i, c in enumerate(code) if c.startswith(word) and all(m in c for m in more)]
        count, = places("global_atomic_add")
        waits = places("s_waitcnt", "vmcnt(0)")
        stored = [i for i in places("global_store_dword", "sc1") if i < count]
        read = places("global_load_dwordx2", "sc1")
        assert len(stored) >= 4 and any(stored[-1] < i < count for i in waits), name
        assert read and all(any(count < i < r for i in waits) for r in read), name
    other = _compile_moe("gfx942", out)
    assert other.returncode != 0 and "written for gfx950's memory" in other.stderr
