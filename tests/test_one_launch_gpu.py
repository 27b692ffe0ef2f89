"""A decode step's layers in one launch: which sizes it takes (CPU), and on the GPU its logits against
the plain implementation and against a launch a product, where its work is dealt unevenly."""
import ctypes
import gc
import threading
import weakref

import numpy as np
import pytest
import torch

import plain
import tiny
from gpu_util import DEV
from test_engine_gpu import LOGITS_TOL_BF16
from zinfer_amd.config import Qwen3Config
from zinfer_amd.models import one_launch
from zinfer_amd.models.build import declare_tensors
from zinfer_amd.ops import build
from zinfer_amd.ops import decode_layers as kernel
from zinfer_amd.weights import draw_tensors


def test_the_sizes_python_accepts_are_accepted_by_the_entry():
    """No device here: the entry refuses sizes (-3) before it asks for one."""
    lib = build.load("decode_layers")
    accepted = 0
    for wgs in (32, 256, 304):
        for hidden in (448, 512, 576, 1000, 5120, 8192, 32768):
            for ff in (256, 512, 1088, 12288, 25600, 32768, 53248):
                for heads, kv in ((2, 1), (4, 4), (16, 1), (15, 1), (32, 8), (40, 8), (96, 96), (12, 5)):
                    for page, tokens in ((8, 1), (16, 1), (48, 2), (16, 3), (32, 4), (16, 5)):
                        p = kernel._Layers()
                        p.tokens, p.n_layers, p.hidden, p.ff = tokens, 1, hidden, ff
                        p.n_heads, p.n_kv_heads, p.page_size = heads, kv, page
                        p.max_splits = kernel.MAX_SPLITS
                        if kernel.sizes_covered(tokens, hidden, ff, heads, kv, 128, page, wgs):
                            accepted += 1
                            if not torch.cuda.is_available():      # (nothing is launched without one)
                                assert lib.zf_decode_layers(ctypes.byref(p), wgs, None) != -3, \
                                    (wgs, hidden, ff, heads, kv, page, tokens)
    assert accepted > 200


@pytest.mark.parametrize("shape,most_keys", [       # (per number of tokens)
    ((1024, 16, 8, 3072), (4096, 4096, 4096, 3072)), ((2048, 32, 8, 8192), (4096, 4096, 3072, 1024)),
    ((2560, 24, 8, 6912), (4096, 4096, 3072, 1024)), ((4096, 32, 8, 12288), (4096, 4096, 3072, 1024)),
    ((5120, 32, 8, 13824), (4096, 0, 0, 0)), ((4608, 36, 4, 14336), (0, 0, 0, 0)), ((5120, 40, 8, 17408), (0, 0, 0, 0)),
    ((5120, 64, 8, 25600), (0, 0, 0, 0))], ids=str)
def test_where_one_launch_pays(shape, most_keys):
    """As measured on 256 CUs: to which tables, if at all, a step of one to four tokens is the faster one so."""
    hidden, heads, kv, ff = shape
    for tokens, most in enumerate(most_keys, 1):
        for keys in (16, 256, 1024, 1040, 3072, 3088, 4096):
            assert kernel.pays(tokens, hidden, ff, heads, kv, keys, 256) == (keys <= most), (tokens, keys)


def _qwen3(hidden, heads, kv, ff, layers=2, vocab=1030):
    return dict(architectures=["Qwen3ForCausalLM"], model_type="qwen3", num_hidden_layers=layers,
                hidden_size=hidden, num_attention_heads=heads, num_key_value_heads=kv, head_dim=128,
                intermediate_size=ff, vocab_size=vocab, rope_theta=1000000.0, rms_norm_eps=1e-6,
                tie_word_embeddings=False, max_position_embeddings=4096, torch_dtype="bfloat16")


def _engine(cfg, weights, page=16, tokens=4096, graphs=True):
    from zinfer_amd.engine import Engine
    from zinfer_amd.models.build import build_model
    model = build_model(Qwen3Config.from_dict(cfg).model_spec(), weights, "bfloat16", DEV)
    return Engine(model, page_size=page, num_pages=(tokens + page - 1) // page + 2, max_requests=4,
                  use_graphs=graphs)


def _weights(cfg, seed):
    spec = Qwen3Config.from_dict(cfg).model_spec()
    drawn = draw_tensors(declare_tensors(spec), seed, torch.bfloat16, tied=False, device=DEV)
    return {k: t.cpu() for k, t in drawn.items()}


def _answer(eng, toks, singles):
    """The prompt's last row and every single token's, on the host."""
    from zinfer_amd.engine import StepEntry
    n = len(toks) - singles
    rows = [eng.step([StepEntry("r", toks[:n], [n - 1])]).float().cpu().numpy().copy()]
    for t in toks[n:]:
        rows.append(eng.step([StepEntry("r", [t], [0])]).float().cpu().numpy().copy())
    eng.release("r")
    return np.concatenate(rows)


# (width, heads, kv heads, feed-forward, page, tokens, of these alone): the narrowest; one head group of
# fifteen; a kv head a head; widths that leave waves without a tile and workgroups without a row group;
# pages of three times sixteen; contexts that begin and pass a wave's 32 keys and a split's 128; the
# served sizes with two to nine splits
SHAPES = [(512, 4, 2, 512, 16, 40, 36), (576, 15, 1, 1088, 48, 140, 16), (832, 4, 4, 832, 16, 262, 10),
          (1024, 16, 8, 3072, 16, 133, 8), (2560, 32, 8, 9728, 32, 70, 8), (4096, 32, 8, 12288, 16, 1030, 12)]


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_single_tokens_against_the_plain_implementation(shape, monkeypatch):
    """Logits of every single token; a launch a product stays within the same bound of them.  Workgroups
    that come and go (more than the CUs hold, fewer than there are) leave the bits as they are, and so does a
    graph."""
    hidden, heads, kv, ff, page, n, singles = shape
    cfg = _qwen3(hidden, heads, kv, ff)
    w = _weights(cfg, hidden + heads)
    toks = tiny.random_tokens(n, cfg["vocab_size"], n)
    ref = plain.model_forward_batched(cfg, w, toks).numpy()[-singles - 1:]
    monkeypatch.setattr(one_launch.OneLaunchLayers, "forward", _counted(calls := []))
    eng = _engine(cfg, w, page)
    assert eng.model.one_launch is not None
    got = _answer(eng, toks, singles)
    assert len(calls) >= 2, "the layers did not run in one launch"
    assert eng.graph_replays > 0
    scale = np.abs(ref).max()
    assert np.abs(got - ref).max() <= LOGITS_TOL_BF16 * scale
    assert np.array_equal(_answer(eng, toks, singles), got)
    assert np.array_equal(_answer(_engine(cfg, w, page, graphs=False), toks, singles), got)
    monkeypatch.setattr(kernel, "workgroups", lambda index: 2 * eng.model.one_launch.wgs)
    assert np.array_equal(_answer(_engine(cfg, w, page), toks, singles), got)
    fewer = 2 * max(ff // 256, hidden // 256, (heads + 2 * kv) // 2, kv * 8) + 3
    monkeypatch.setattr(kernel, "workgroups", lambda index: fewer)
    assert np.array_equal(_answer(_engine(cfg, w, page), toks, singles), got)
    apart = _engine(cfg, w, page)
    apart.model.one_launch = None
    assert np.abs(_answer(apart, toks, singles) - got).max() <= LOGITS_TOL_BF16 * scale


def _together(eng, requests, singles):
    """Prompts one after the other, then a token of every request a step: the rows of each."""
    from zinfer_amd.engine import StepEntry
    rows = {r: [] for r in requests}
    for r, t in requests.items():
        eng.step([StepEntry(r, t[:-singles], [])])
    for k in range(singles, 0, -1):
        logits = eng.step([StepEntry(r, [t[-k]], [0]) for r, t in requests.items()])
        for i, r in enumerate(requests):
            rows[r].append(logits[i].float().cpu().numpy().copy())
    for r in requests:
        eng.release(r)
    return {r: np.stack(v) for r, v in rows.items()}


@pytest.mark.gpu
@pytest.mark.parametrize("shape,lengths", [
    ((512, 4, 2, 512, 16), (9, 130)), ((576, 15, 1, 1088, 48), (140, 33, 12)), ((832, 4, 4, 832, 16), (8, 262, 40, 128)),
    ((1024, 16, 8, 3072, 16), (133, 10, 300, 31)), ((2560, 32, 8, 9728, 32), (70, 900)), ((4096, 32, 8, 12288, 16), (1030, 40, 129))],
    ids=str)
def test_several_requests_against_the_plain_implementation_and_alone(shape, lengths, monkeypatch):
    """Two to four tokens a step, with a graph and without: within the bound of the plain implementation, and of a
    request the bits it has alone."""
    hidden, heads, kv, ff, page = shape
    cfg = _qwen3(hidden, heads, kv, ff)
    w = _weights(cfg, hidden + heads)
    requests = {f"r{i}": tiny.random_tokens(n, cfg["vocab_size"], n) for i, n in enumerate(lengths)}
    monkeypatch.setattr(one_launch.OneLaunchLayers, "forward", _counted(calls := []))
    eng = _engine(cfg, w, page)
    got = _together(eng, requests, 6)
    assert len(calls) >= 2 and eng.graph_replays > 0
    plainly = _together(_engine(cfg, w, page, graphs=False), requests, 6)
    for r, toks in requests.items():
        ref = plain.model_forward_batched(cfg, w, toks).numpy()[-6:]
        assert np.abs(got[r] - ref).max() <= LOGITS_TOL_BF16 * np.abs(ref).max()
        assert np.array_equal(got[r], plainly[r])
        assert np.array_equal(got[r], _together(eng, {r: toks}, 6)[r])


def _counted(calls):
    forward = one_launch.OneLaunchLayers.forward

    def counted(self, *args):
        calls.append(1)
        return forward(self, *args)
    return counted


@pytest.mark.gpu
def test_two_engines_on_two_streams_at_once():
    """Launches that meet deal their work among the workgroups each has: the same bits as alone."""
    cfg = _qwen3(1024, 16, 8, 3072, layers=6)
    w = _weights(cfg, 5)
    toks = tiny.random_tokens(60, cfg["vocab_size"], 6)
    engines = [_engine(cfg, w, tokens=128) for _ in range(2)]
    alone = [_answer(e, toks, 40) for e in engines]
    assert np.array_equal(*alone)
    got = [[], []]

    def go(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(4):
                got[i].append(_answer(engines[i], toks, 40))
    threads = [threading.Thread(target=go, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for rows in got:
        assert len(rows) == 4 and all(np.array_equal(r, alone[0]) for r in rows)


@pytest.mark.gpu
def test_a_model_goes_with_its_last_reference():
    cfg = _qwen3(512, 4, 2, 512)
    eng = _engine(cfg, _weights(cfg, 7), tokens=128)
    assert eng.model.one_launch is not None
    model = weakref.ref(eng.model)
    gc.disable()
    try:
        del eng
        assert model() is None
    finally:
        gc.enable()


@pytest.mark.gpu
def test_a_failed_wait_is_an_error_of_the_next_step():
    """(the flag set by the host, as the kernel sets it when a wait comes to its end)"""
    from zinfer_amd.engine import StepEntry
    from zinfer_amd.errors import StepError
    cfg = _qwen3(512, 4, 2, 512)
    eng = _engine(cfg, _weights(cfg, 7), tokens=128)
    eng.step([StepEntry("r", [1, 2, 3], [2])])
    eng.step([StepEntry("r", [4], [0])])
    torch.cuda.synchronize()
    eng._scratch.kept(one_launch.STATUS)[0] = 1
    with pytest.raises(StepError, match="hear"):
        eng.step([StepEntry("r", [5], [0])])
    assert eng.length("r") == 4


def _flag(eng):
    eng._scratch.kept(one_launch.STATUS)[0] = 1


@pytest.mark.gpu
@pytest.mark.parametrize("reader", ["argmax", "to_host", "sample"])
def test_a_step_that_failed_is_taken_back_where_the_host_waits_for_it(reader):
    """(the flag set by the host, between the launch and the wait)  The step's request holds what it held
    before, and the same step then gives the same bits."""
    from zinfer_amd import ops
    from zinfer_amd.engine import StepEntry
    from zinfer_amd.errors import StepError
    cfg = _qwen3(512, 4, 2, 512)
    eng = _engine(cfg, _weights(cfg, 7), tokens=128)
    eng.argmax(eng.step([StepEntry("r", [1, 2, 3], [2])]))
    want = eng.to_host(eng.step([StepEntry("r", [4], [0])])).clone()
    logits = eng.step([StepEntry("r", [5], [0]), StepEntry("new", [9], [0])])
    records = np.zeros((2,), dtype=ops.SAMPLE_ROW_DTYPE)
    records[:] = (1.0, 1.0, 0.0, 1, 0.0)
    _flag(eng)
    with pytest.raises(StepError, match="hear"):
        eng.sample(logits, records) if reader == "sample" else getattr(eng, reader)(logits)
    assert eng.length("r") == 4 and not eng.has_request("new")
    eng.release("r")
    eng.argmax(eng.step([StepEntry("r", [1, 2, 3], [2])]))
    assert torch.equal(eng.to_host(eng.step([StepEntry("r", [4], [0])])), want)


@pytest.mark.gpu
def test_runs_of_steps_that_failed_return_no_tokens(monkeypatch):
    """The flag set while the steps run: as one graph and one by one."""
    from zinfer_amd import ops
    from zinfer_amd.engine import StepEntry
    from zinfer_amd.errors import StepError
    cfg = _qwen3(512, 4, 2, 512)
    eng = _engine(cfg, _weights(cfg, 7), tokens=128)
    eng.argmax(eng.step([StepEntry("r", [1, 2, 3], [2])]))
    pages = eng.cache.num_free_pages()
    go = lambda: eng.decode_steps([StepEntry("r", [4], [0])], 8)
    want = go()
    eng.release("r")
    for run in range(4):
        eng.argmax(eng.step([StepEntry("r", [1, 2, 3], [2])]))
        with monkeypatch.context() as m:
            upload = eng._upload
            m.setattr(eng, "_upload", lambda host: (upload(host), _flag(eng))[0])
            with pytest.raises(StepError, match="hear"):
                go()
        assert eng.length("r") == 3 and eng.cache.num_free_pages() == pages
        assert go() == want
        eng.release("r")
    assert eng.graph_replays > 8


@pytest.mark.gpu
def test_requests_of_a_failed_step_that_nobody_waited_for_can_only_be_released():
    from zinfer_amd.engine import StepEntry
    from zinfer_amd.errors import StepError
    cfg = _qwen3(512, 4, 2, 512)
    eng = _engine(cfg, _weights(cfg, 7), tokens=128)
    for r in ("r", "s"):
        eng.argmax(eng.step([StepEntry(r, [1, 2, 3], [2])]))
    eng.step([StepEntry("r", [4], [0])])
    torch.cuda.synchronize()
    _flag(eng)
    with pytest.raises(StepError, match="hear"):
        eng.step([StepEntry("s", [5], [0])])
    with pytest.raises(StepError, match="released"):
        eng.step([StepEntry("r", [5], [0])])
    assert np.isfinite(eng.to_host(eng.step([StepEntry("s", [5], [0])])).numpy()).all()
    eng.release("r")
    assert len(eng.argmax(eng.step([StepEntry("r", [5], [0])]))) == 1


@pytest.mark.gpu
def test_the_scheduler_accepts_no_token_of_a_failed_step(monkeypatch):
    from zinfer_amd.engine.scheduler import Scheduler
    from zinfer_amd.errors import StepError
    from zinfer_amd.sampling import SamplingParams
    cfg = _qwen3(512, 4, 2, 512)
    eng = _engine(cfg, _weights(cfg, 7), tokens=128)
    answers = []
    for spoiled in (False, True):
        for multi, top_k in ((1, 1), (4, 1), (1, 5000)):
            sched = Scheduler(eng, multi_step=multi)
            sched.add_request([1, 2, 3], SamplingParams(
                temperature=0.0 if top_k == 1 else 0.7, top_k=top_k, seed=3, max_new_tokens=9, ignore_eos=True))
            req = sched.waiting[-1]
            sched.step()
            if spoiled:
                sched.step()
                had = list(req.generated)
                upload = eng._upload
                monkeypatch.setattr(eng, "_upload", lambda host: (upload(host), _flag(eng))[0])
                with pytest.raises(StepError, match="hear"):
                    sched.step()
                monkeypatch.setattr(eng, "_upload", upload)
                assert list(req.generated) == had
            while not req.finished:
                sched.step()
            answers.append(list(req.generated))
    assert answers[:3] == answers[3:]


# (width, heads, kv heads, feed-forward, page), prompts' lengths, numbers of workgroups: one alone; a few; one less
# than hold a phase's sums, by its products or (the first) by its splits of contexts
FEW = [((512, 4, 4, 512, 16), (1500, 1410, 40, 1300), (1, 3, 31)), ((576, 15, 1, 1088, 48), (140, 33, 12), (2, 27)),
       ((832, 4, 4, 832, 16), (262, 40), (1, 11)), ((1024, 16, 8, 3072, 16), (133,), (1, 15)),
       ((4096, 32, 8, 12288, 16), (530,), (5, 23))]


@pytest.mark.gpu
@pytest.mark.parametrize("shape,lengths,numbers", FEW, ids=str)
def test_fewer_workgroups_than_hold_a_phase_give_the_same_bits(shape, lengths, numbers, monkeypatch):
    """Workgroups that are too few for a phase's sums take it a piece at a time."""
    hidden, heads, kv, ff, page = shape
    cfg = _qwen3(hidden, heads, kv, ff)
    w = _weights(cfg, hidden + heads)
    requests = {f"r{i}": tiny.random_tokens(n, cfg["vocab_size"], n) for i, n in enumerate(lengths)}
    want = _together(_engine(cfg, w, page, tokens=8192), requests, 5)
    monkeypatch.setattr(kernel, "sizes_covered", lambda *sizes: True)
    for n in numbers:
        monkeypatch.setattr(kernel, "workgroups", lambda index: n)
        monkeypatch.setattr(one_launch.OneLaunchLayers, "forward", _counted(calls := []))
        got = _together(_engine(cfg, w, page, tokens=8192), requests, 5)
        assert len(calls) >= 2
        for r in requests:
            assert np.array_equal(got[r], want[r]), (n, r)


@pytest.mark.gpu
@pytest.mark.parametrize("lengths", [(70,), (133, 10, 300, 31)], ids=str)
def test_workgroups_that_do_not_wait_for_the_others_give_the_same_bits(lengths, monkeypatch):
    """The meeting closes as soon as one has come: as many do the step as came by then."""
    cfg = _qwen3(1024, 16, 8, 3072)
    w = _weights(cfg, 3)
    requests = {f"r{i}": tiny.random_tokens(n, cfg["vocab_size"], n) for i, n in enumerate(lengths)}
    want = _together(_engine(cfg, w), requests, 6)
    monkeypatch.setattr(kernel, "MEET_TICKS", 0)
    monkeypatch.setattr(kernel, "MEET_MOST", 0)
    eng = _engine(cfg, w)
    for _ in range(4):
        got = _together(eng, requests, 6)
        assert all(np.array_equal(got[r], want[r]) for r in requests)


@pytest.mark.gpu
def test_three_engines_that_need_more_than_a_third_of_the_workgroups_each():
    """None of three launches that meet waits for what another holds: the same bits as alone."""
    from zinfer_amd.engine import StepEntry
    cfg = _qwen3(1024, 32, 8, 3072, layers=6)
    w = _weights(cfg, 5)
    requests = {f"r{i}": tiny.random_tokens(n, cfg["vocab_size"], n) for i, n in enumerate((40, 25, 61, 90))}
    engines = [_engine(cfg, w, tokens=512) for _ in range(3)]
    assert 3 * 96 > engines[0].model.one_launch.wgs >= 2 * 96       # (48 x 8 row groups of q, k and v, 4 a workgroup)
    want = [_together(e, requests, 20) for e in engines][0]
    for e in engines:
        for r, t in requests.items():
            e.step([StepEntry(r, t[:-20], [])])
    torch.cuda.synchronize()
    got = [{r: [] for r in requests} for _ in engines]

    def go(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            for k in range(20, 0, -1):
                logits = engines[i].step([StepEntry(r, [t[-k]], [0]) for r, t in requests.items()])
                rows = engines[i].to_host(logits).numpy()
                for j, r in enumerate(requests):
                    got[i][r].append(rows[j].copy())
    threads = [threading.Thread(target=go, args=(i,)) for i in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for rows in got:
        assert all(np.array_equal(np.stack(rows[r]), want[r]) for r in requests)


@pytest.mark.gpu
@pytest.mark.parametrize("shape,lengths,workgroups", [
    ((512, 4, 4, 512, 16), (1500, 1410, 40, 1300), None), ((1024, 16, 8, 3072, 16), (133,), None),
    ((576, 15, 1, 1088, 48), (140, 33, 12), 7)], ids=str)
def test_waits_that_give_up_hand_on_nothing_that_did_not_come(shape, lengths, workgroups, monkeypatch):
    """Every wait gives up at the first look that misses a word, in workgroups of every kind (some of the first
    shape's have attention alone) and in too few of them: rows of NaN, an error where the host waits, nothing in
    the pools that the whole step does not write, and the next step as if there had been none."""
    from zinfer_amd.engine import StepEntry
    from zinfer_amd.errors import StepError
    hidden, heads, kv, ff, page = shape
    cfg = _qwen3(hidden, heads, kv, ff)
    requests = {f"r{i}": tiny.random_tokens(n, cfg["vocab_size"], n) for i, n in enumerate(lengths)}
    if workgroups is not None:
        monkeypatch.setattr(kernel, "sizes_covered", lambda *sizes: True)
        monkeypatch.setattr(kernel, "workgroups", lambda index: workgroups)
    eng = _engine(cfg, _weights(cfg, hidden + heads), page, tokens=8192, graphs=False)
    for r, t in requests.items():
        eng.step([StepEntry(r, t[:-1], [])])
    pools = [p for view in eng.views for p in (view.k_pool, view.v_pool)]
    before = [p.clone() for p in pools]

    def step():
        return eng.step([StepEntry(r, t[-1:], [0]) for r, t in requests.items()])

    def back():
        for r, n in zip(requests, lengths):
            eng.cache.commit(r, n - 1)
            eng.cache.trim(r)
        for p, b in zip(pools, before):
            p.copy_(b)
    want = eng.to_host(step()).clone()
    written = [p.clone() for p in pools]
    for _ in range(3):
        back()
        with monkeypatch.context() as m:
            m.setattr(kernel, "SPIN_FROM", (1 << 21) | 15)
            rows = step()
        assert torch.isnan(rows).all().item()
        with pytest.raises(StepError, match="hear"):
            eng.to_host(rows)
        assert [eng.length(r) for r in requests] == [n - 1 for n in lengths]
        for p, b, w in zip(pools, before, written):
            assert ((p == b) | (p == w)).all().item()
        back()
        assert torch.equal(eng.to_host(step()), want)


@pytest.mark.gpu
def test_the_classes_and_the_step_they_add_up_to_are_of_one_program(monkeypatch):
    """A step measured by class, and all classes together, has a launch a product; the step itself has not."""
    from zinfer_amd import ops
    from zinfer_amd.engine import StepEntry
    cfg = _qwen3(512, 4, 2, 512)
    eng = _engine(cfg, _weights(cfg, 7), tokens=128)
    eng.step([StepEntry("r", [1, 2, 3], [2])])
    want = eng.to_host(eng.step([StepEntry("r", [4], [0])])).clone()
    measured, forward = [], one_launch.OneLaunchLayers.forward

    def counted(self, *args):
        measured.append(ops._class_filter is not None)
        return forward(self, *args)
    monkeypatch.setattr(one_launch.OneLaunchLayers, "forward", counted)
    times = eng.class_times([StepEntry("r", [5], [0])], repeats=5)
    assert set(times) == set(ops.KERNEL_CLASSES) | {"step"} and not any(measured)
    assert times["products"] > 0 and times["attention"] > 0 and times["step"] > 0
    eng.release("r")
    eng.step([StepEntry("r", [1, 2, 3], [2])])
    assert torch.equal(eng.to_host(eng.step([StepEntry("r", [4], [0])])), want)


@pytest.mark.gpu
def test_steps_where_it_does_not_pay_have_a_launch_a_product(monkeypatch):
    cfg = _qwen3(512, 4, 2, 512)
    w, toks = _weights(cfg, 7), tiny.random_tokens(40, cfg["vocab_size"], 2)
    apart = _engine(cfg, w)
    apart.model.one_launch = None
    monkeypatch.setattr(one_launch.OneLaunchLayers, "forward", _counted(calls := []))
    asked = []
    monkeypatch.setattr(kernel, "pays", lambda *sizes: asked.append(sizes))
    got = _answer(_engine(cfg, w), toks, 4)
    assert asked[0] == (1, 512, 512, 4, 2, 256, kernel.compute_units(0)) and not calls
    assert np.array_equal(got, _answer(apart, toks, 4))
