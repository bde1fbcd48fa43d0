"""The decode loop's runner on the CPU: what it hands the kernels of a step, on stand-ins for the engine and its kernels."""
import contextlib
from types import SimpleNamespace

import numpy as np
import pytest
import torch

from gesso_amd.engine.decode import DecodeRunner


def stand_in(pages=(40, 30), page_size=8, max_context=256, vocab=50):
    """As much of an engine as a runner asks of it; ``pages``: the page groups' sizes."""
    storage = SimpleNamespace(scratch_slot=9, num_pages=list(pages))
    return SimpleNamespace(device=torch.device("cpu"), max_context=max_context, page_size=page_size, storage=storage, dtype=torch.bfloat16,
                           DECODE_MAX_BATCH=64, spec=SimpleNamespace(vocab=vocab))


@pytest.fixture
def pinned(monkeypatch):
    """Pinned buffers asked for (there is no pinned memory without a GPU: the tensor itself)."""
    made = []
    monkeypatch.setattr(torch.Tensor, "pin_memory", lambda t: made.append(t.numel()) or t)
    return made


@pytest.mark.parametrize("groups", [0, 1, 2])
@pytest.mark.parametrize("B,cap", [(1, 1), (3, 4), (5, 8), (16, 16)])
def test_a_steps_facts_and_tables_come_by_one_copy(pinned, groups, B, cap):
    """What the rows' kernels read, against the same looked up row by row: pages that a window has given back and columns
    beyond a row's pages name the scratch page, rows beyond the batch the scratch page and slot."""
    eng = stand_in(pages=(40, 30)[:groups])
    runner = DecodeRunner(eng, cap)
    rng = np.random.default_rng(B)
    for turn in range(2):                          # (what the first filled in must not show in the second)
        lengths = [int(x) for x in rng.integers(1, 100 - 60 * turn, B)]
        tables = [[[-1 if rng.random() < 0.2 else int(rng.integers(0, 30)) for _ in range(-(-(n + 3) // 8) + int(rng.integers(0, 2)))]
                   for n in lengths] for _ in range(groups)]
        rcs = [SimpleNamespace(length=n, slot=None if i == 1 else i, tables=[t[i] for t in tables]) for i, n in enumerate(lengths)]
        tokens = rng.integers(0, 50, B)
        pinned.clear()
        runner._fill(rcs, tokens, 3)
        assert len(pinned) == 1
        assert runner.tok.tolist() == list(tokens) + [0] * (cap - B)
        assert runner.pos.tolist() == lengths + [0] * (cap - B)
        assert runner.kv_len.tolist() == [n + 1 for n in lengths] + [1] * (cap - B)
        assert runner.slots.tolist() == [9 if i == 1 else i for i in range(B)] + [9] * (cap - B)
        assert runner.live.tolist() == [1] * B + [0] * (cap - B)
        for g in range(groups):
            scratch = eng.storage.num_pages[g]
            for i in range(cap):
                reach = -(-(lengths[i] + 3) // 8) if i < B else max(-(-(n + 3) // 8) for n in lengths)
                want = [tables[g][i][c] if i < B and tables[g][i][c] >= 0 else scratch for c in range(reach)]
                assert runner.block_tables[g][i, :reach].tolist() == want


def test_the_runners_of_a_capacity_share_one_set_of_the_draws_scratch(monkeypatch):
    """A batch of drawing requests that grows from 129 to 512 passes runners of 160, 192, 256, 320, 384 and 512 rows; what
    their draws write to is one set a capacity, not one a runner."""
    from gesso_amd.engine.decode import _capacity
    from gesso_amd.engine.engine import Engine
    eng = stand_in(pages=())
    eng.rt = SimpleNamespace(ops=SimpleNamespace(choice_parts=lambda V: 3, choice_hist=lambda: 5, decode_choose=lambda *a, **kw: None),
                             stage=lambda name: contextlib.nullcontext())
    eng.choice_scratch = lambda rows: Engine.choice_scratch(eng, rows)
    monkeypatch.setattr(DecodeRunner, "_forward", lambda self: None)
    runners, sets = {}, {}
    for n in (129, 170, 200, 260, 330, 500, 150):
        cap = _capacity(n)
        runner = runners.setdefault(cap, DecodeRunner(eng, cap)).fit(n)
        runner.draws = True
        runner._body()
        assert runner.weights.numel() >= n * eng.spec.vocab
        sets.setdefault(cap, set()).add(runner.weights.data_ptr())
    assert {cap: len(s) for cap, s in sets.items()} == {256: 1, 512: 1}


def test_a_last_product_of_few_rows_asks_nothing_about_parts():
    """A prompt of some rows has thirty last products, each a host call of some microseconds: up to 64 rows, which never come in
    parts, cost no check of the operands for that."""
    from gesso_amd.parts.runtime import DeferredLinear, Runtime
    asked = []
    rt = object.__new__(Runtime)
    rt.ops = SimpleNamespace(mid_parts_pay=lambda x, w, wt: asked.append(x.shape[0]) or 3)
    rt.fused, rt.no_library, rt.many_rows, rt.streaming_rows_max, rt._tiles = False, False, "auto", 64, {}
    rt.linear = lambda x, w, bias=None: "computed"
    w = torch.zeros(16, 4096)
    for rows in (1, 13, 64):
        assert rt.project(torch.zeros(rows, 4096), w) == "computed"
    assert asked == []
    out = rt.project(torch.zeros(65, 4096), w)
    assert isinstance(out, DeferredLinear) and out.parts == 3 and asked == [65]


def hundred_rows_runtime(takes=lambda rows: True):
    """As much of a runtime as a last product of some hundred rows asks of it, and what was made."""
    from gesso_amd.parts.runtime import Runtime
    made = []
    rt = object.__new__(Runtime)
    rt.ops = SimpleNamespace(mid_parts_pay=lambda x, w, wt: 0, mid_residual_ok=lambda x, w, wt: takes(x.shape[0]),
                             gemm_mid_residual=lambda x, w, wt, res, nw, checked: made.append("stream") or ("rows", "sums"))
    rt.fused, rt.no_library, rt.many_rows, rt.streaming_rows_max, rt._tiles = False, False, "auto", 64, {}
    rt.linear = lambda x, w, bias=None: made.append("product") or "computed"
    rt.stage = lambda name: contextlib.nullcontext()
    return rt, made


def test_an_output_projection_of_some_hundred_rows_is_left_to_a_block_that_asks_for_it():
    """Called by itself, with a bias, for a block whose next reader does not take that many rows weighted, or where no one kernel
    adds it to the stream, it is computed at once."""
    from gesso_amd.parts.runtime import DeferredLinear
    w, x = torch.zeros(16, 32), torch.zeros(100, 32)
    rt, made = hundred_rows_runtime()
    out = rt.project(x, w, None, lambda rows: rows == 100)
    assert isinstance(out, DeferredLinear) and out.parts == 1 and made == []
    assert rt.project(x, w) == "computed" and rt.project(x, w, None, lambda rows: rows == 99) == "computed"
    assert rt.project(x, w, "bias", lambda rows: True) == "computed" and rt.project(x[:64], w, None, lambda rows: True) == "computed"
    rt, made = hundred_rows_runtime(takes=lambda rows: False)
    assert rt.project(x, w, None, lambda rows: True) == "computed" and made == ["product"]


@pytest.mark.parametrize("norm,weighted,into", [("fits", True, "stream"), ("fits", False, "product"), ("fits", None, "product"), ("no weight", True, "product"),
                                                ("other width", True, "product"), ("other type", True, "product"), (None, True, "product")])
def test_a_deferred_projection_meets_every_next_norm(norm, weighted, into):
    """Into the stream only where the next norm's weight fits its rows and their reader takes them weighted; else the ordinary
    product, pending for the norm's own pass."""
    from gesso_amd.parts.rmsnorm import ResidualStream
    from gesso_amd.parts.runtime import DeferredLinear
    rt, made = hundred_rows_runtime()
    weights = {"fits": torch.ones(16), "no weight": None, "other width": torch.ones(8), "other type": torch.ones(16).bfloat16()}
    after = None if norm is None else SimpleNamespace(row_weight=weights[norm])
    if norm == "no weight":
        after = object()
    stream = ResidualStream(torch.zeros(100, 16))
    stream.push(DeferredLinear(torch.zeros(100, 32), torch.zeros(16, 32), 1), rt, next_norm=after,
                weighted=None if weighted is None else lambda rows: weighted and rows == 100)
    assert made == [into]
    if into == "stream":
        assert (stream.xs, stream.ssq, stream.xs_for, stream.pending) == ("rows", "sums", after, None)
    else:
        assert (stream.xs, stream.ssq, stream.xs_for, stream.pending) == (None, None, None, "computed")


def test_a_block_says_what_reads_the_stream_next_while_its_mixer_runs_and_no_longer():
    from gesso_amd.parts.block import PreNormBlock
    rt, made = hundred_rows_runtime()
    said = []

    class Stream:
        following = None

        def push(self, out, rt, next_norm=None, weighted=None):
            said.append(("push", out, next_norm, weighted))

    class Mixer:
        def forward(self, x, ctx, cache):
            said.append(("mixer", ctx.takes_weighted))
            if x == "raises":
                raise RuntimeError("mixer")
            return "mixed"

    norm = lambda x: SimpleNamespace(add_norm=lambda stream: x)
    takes = lambda rows: True
    for ffn in (SimpleNamespace(takes_weighted=takes, forward=lambda x, ctx: said.append(("ffn", ctx.takes_weighted)) or "fed"),
                SimpleNamespace(forward=lambda x, ctx: said.append(("ffn", ctx.takes_weighted)) or "fed"), None):
        block = object.__new__(PreNormBlock)
        block.rt, block.mixer, block.mixer_norm, block.ffn, block.ffn_norm = rt, Mixer(), norm("rows"), ffn, norm("normed")
        ctx, asks = SimpleNamespace(), getattr(ffn, "takes_weighted", None)
        said.clear()
        block.forward(Stream(), ctx, None)
        assert said[0] == ("mixer", asks) and said[1][1] == "mixed" and said[1][3] is asks and ctx.takes_weighted is None
        assert said[2:] == ([("ffn", None), ("push", "fed", None, None)] if ffn is not None else [])
        block.mixer_norm = norm("raises")
        with pytest.raises(RuntimeError, match="mixer"):
            block.forward(Stream(), ctx, None)
        assert ctx.takes_weighted is None
