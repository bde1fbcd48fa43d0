"""An engine's calls from several threads and on several streams run one after another: steps share the decode loop's
buffers, the kernels' workspaces and the runtime's switches.  On stand-ins for streams and kernels, then on the GPU."""
import threading
import time
from types import SimpleNamespace

import pytest
import torch

from gesso_amd.engine import engine as engine_module
from gesso_amd.engine.batch import StepEntry
from gesso_amd.engine.engine import Engine


class Streams:
    """Stands for ``torch.cuda``'s streams and events: ``log`` has what was enqueued, in the order the host enqueued it."""

    def __init__(self):
        self.log, self.now = [], 1
        outer = self

        class Event:
            def record(self, stream=None):
                self.at = outer.now if stream is None else stream.cuda_stream
                outer.log.append(("record", self.at))

        self.Event = Event

    def current_stream(self, device=None):
        return SimpleNamespace(cuda_stream=self.now, wait_event=lambda e, s=self.now: self.log.append(("wait", s, e.at)))


def stand_in(monkeypatch, work, dtype="bfloat16", padding_free=True, page_size=16, context=512):
    """An engine whose steps call ``work()``, an ordinary one with ``["ordinary"]``, the loop's with the requests."""
    streams = Streams()
    for name in ("current_stream", "Event"):
        monkeypatch.setattr(torch.cuda, name, getattr(streams, name))
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.setattr(engine_module.ops, "_stream", lambda: streams.now)
    monkeypatch.setattr(engine_module, "Runtime", lambda *a: SimpleNamespace(
        streaming_rows_max=64, profile=None, ops=None, options=SimpleNamespace(record_portions=False)))
    monkeypatch.setattr(engine_module, "Model", lambda spec, rt: SimpleNamespace(
        graph_safe=True, padding_free=padding_free, bind=lambda t: None, cache_needs=lambda: [],
        forward=lambda ctx: work(streams, ["ordinary"])))
    monkeypatch.setattr(engine_module, "StepContext", lambda *a, **kw: None)
    monkeypatch.setattr(engine_module, "CacheStorage", lambda *a: SimpleNamespace(num_pages=[]))
    spec = SimpleNamespace(max_position=context, schedule=[], vocab=100)
    eng = Engine(spec, {}, dtype, device="cuda:0", page_size=page_size, num_pages=64, num_slots=65)
    eng._runner = lambda n: SimpleNamespace(step=lambda rids, ids: work(streams, rids), run=lambda rids, *a: work(streams, rids))
    for rid in "ab":
        eng.add_request(rid)
    return eng, streams


def test_a_call_on_another_stream_waits_for_the_one_before(monkeypatch):
    eng, streams = stand_in(monkeypatch, lambda st, rids: st.log.append(("work", st.now, rids[0])))
    for stream, rid in ((1, "a"), (1, "b"), (2, "a"), (1, "b")):
        streams.now = stream
        eng.step([StepEntry(rid, [3], [0])])
    streams.now = 2
    eng.decode(["a"], [3], 1)
    work = [(i, e[1]) for i, e in enumerate(streams.log) if e[0] == "work"]
    for (i, before), (k, at) in zip(work, work[1:]):
        between = streams.log[i + 1:k]
        assert before == at or between == [("record", before), ("wait", at, before)], streams.log
    assert [e for e in streams.log if e[0] == "wait"] == [("wait", 2, 1), ("wait", 1, 2), ("wait", 2, 1)]


def test_a_second_thread_waits_until_the_first_ones_call_has_returned(monkeypatch):
    inside, most = [], []

    def work(st, rids):
        inside.append(rids[0])
        most.append(len(inside))
        time.sleep(0.02)
        inside.remove(rids[0])

    eng, _ = stand_in(monkeypatch, work)

    def calls(rid, decode):
        for _ in range(5):
            eng.decode([rid], [3], 1) if decode else eng.step([StepEntry(rid, [3], [0])])

    threads = [threading.Thread(target=calls, args=(rid, rid == "b")) for rid in "ab"]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert len(most) == 10 and max(most) == 1


def test_a_call_that_fails_lets_the_next_one_in(monkeypatch):
    def work(st, rids):
        raise RuntimeError("no")

    eng, _ = stand_in(monkeypatch, work)
    for rid in "ab":
        with pytest.raises(Exception, match="no"):
            eng.step([StepEntry(rid, [3], [0])])
    assert eng._turn.depth == 0 and eng._turn.lock.acquire(blocking=False)
    eng._turn.lock.release()


@pytest.mark.parametrize("dtype,padding_free,loop", [
    ("bfloat16", True, range(1, 65)), ("bfloat16", False, (1, 2, 4, 8, 16, 24, 32, 48, 64)),
    ("float32", True, range(1, 17)), ("float32", False, (1, 2, 4, 8, 16))])
def test_which_steps_of_single_tokens_are_the_loops(monkeypatch, dtype, padding_free, loop):
    """By the number of requests alone: rows of padding that cost what live ones do are not added to a step that has none, nor
    any to a float32 step that keeps the device busy."""
    ran = []
    eng, _ = stand_in(monkeypatch, lambda st, rids: ran.append(rids[0] != "ordinary"), dtype, padding_free)
    for i in range(65):
        eng.add_request(i)
    for n in range(1, 66):
        eng.step([StepEntry(i, [3], [0]) for i in range(n)])
    assert [n for n, through in enumerate(ran, 1) if through] == list(loop)
    ran.clear()
    eng.step([StepEntry(0, [3], [0]), StepEntry(1, [3], [])])          # a request that wants no logits
    eng.step([StepEntry(0, [3, 4], [1])])                              # a portion of two tokens
    assert ran == [False, False]


@pytest.mark.parametrize("page_size,through", [(16, True), (20000, True), (32768, False), (40000, False)])
def test_pages_too_large_for_a_whole_contexts_table_leave_the_loop_out(monkeypatch, page_size, through):
    """A table of a whole context of 131,072 positions, and what the kernels divide positions by: 2^32 at most."""
    ran = []
    eng, _ = stand_in(monkeypatch, lambda st, rids: ran.append(rids[0] != "ordinary"), page_size=page_size, context=131072)
    eng.step([StepEntry("a", [3], [0])])
    assert ran == [through]


def tiny_engine(tmp_path, page_size=8, max_tokens=1024, **fields):
    import dataclasses
    from gesso_amd.weights import write_model_folder
    from tiny import STD, TINY_B
    d = write_model_folder(str(tmp_path / "b"), dataclasses.replace(TINY_B, **fields), 31, torch.bfloat16, std=STD)
    return Engine.from_folder(d, dtype="bfloat16", page_size=page_size, max_tokens=max_tokens, num_slots=8)


def tokens_of(eng, rid, n):
    return [(17 * i + 5 * len(str(rid)) + sum(map(ord, str(rid)))) % eng.spec.vocab for i in range(n)]


@pytest.mark.gpu
@pytest.mark.parametrize("recorded", [False, True])
def test_steps_of_two_streams_leave_each_others_requests_alone(tmp_path, recorded):
    """Two requests stepped in turn on two streams, nothing waited for in between: the logits of each alone."""
    def trace(rids, streams):
        eng = tiny_engine(tmp_path)
        if recorded:
            eng.add_request("other")
            eng.step([StepEntry("other", [1, 2, 3], [])])
            eng.decode(["other"], [4], 2)
        for r in rids:
            eng.add_request(r)
        torch.cuda.synchronize()
        rows = {r: [] for r in rids}
        for i in range(24):
            for r, s in zip(rids, streams):
                with torch.cuda.stream(s):
                    rows[r].append(eng.step([StepEntry(r, [tokens_of(eng, r, 24)[i]], [0])]))
        torch.cuda.synchronize()
        return {r: torch.cat(rows[r]).cpu() for r in rids}

    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    both = trace(["x", "y"], [a, b])
    for r in "xy":
        assert torch.equal(both[r], trace([r], [torch.cuda.current_stream()])[r])


@pytest.mark.gpu
def test_a_thread_that_decodes_beside_one_that_steps(tmp_path):
    """One thread runs the recorded loop, the other steps single tokens and prompts of the same engine; each gets what it gets
    alone."""
    def decoded(eng, out):
        eng.add_request("d")
        tok = int(eng.step([StepEntry("d", tokens_of(eng, "d", 9), [8])]).argmax())
        for _ in range(6):
            ids, bad = eng.decode(["d"], [tok], 8)
            assert not bad.any()
            out += ids[:, 0].tolist()
            tok = out[-1]

    def stepped(eng, out):
        for k in range(4):
            rid = ("s", k)
            eng.add_request(rid)
            out.append(eng.step([StepEntry(rid, tokens_of(eng, rid, 30), list(range(30)))]).cpu())
            for t in tokens_of(eng, rid, 12):
                out.append(eng.step([StepEntry(rid, [t], [0])]).cpu())
            eng.finish_request(rid)

    alone = []
    for f in (decoded, stepped):
        out = []
        f(tiny_engine(tmp_path), out)
        alone.append(out)
    eng, both, failed = tiny_engine(tmp_path), [[], []], []

    def guarded(f, out):
        try:
            f(eng, out)
        except BaseException as err:
            failed.append(err)

    threads = [threading.Thread(target=guarded, args=(f, o)) for f, o in zip((decoded, stepped), both)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed, failed
    assert both[0] == alone[0]
    assert len(both[1]) == len(alone[1]) and all(torch.equal(x, y) for x, y in zip(both[1], alone[1]))


@pytest.mark.gpu
def test_single_tokens_in_pages_that_hold_a_third_of_a_context(tmp_path):
    """Pages of 40,000 tokens with a context of 120,000: single tokens follow a prompt, as they do with small pages."""
    import plain_lfm2 as P
    from noise import NoiseBound
    eng = tiny_engine(tmp_path, 40000, 80000, max_position_embeddings=120000)
    d = str(tmp_path / "b")
    cfg, w = P.read_config(d), P.read_weights(d)
    eng.add_request("r")
    seq = tokens_of(eng, "r", 30)
    got = [eng.step([StepEntry("r", seq[:21], [20])])] + [eng.step([StepEntry("r", [t], [0])]) for t in seq[21:]]
    ref, rounded = P.forward(cfg, w, seq), P.forward(cfg, w, seq, store=P.to_bfloat16)
    bound = NoiseBound()
    for i, row in enumerate(got):
        bound.add(row[0].double().cpu(), ref[20 + i], rounded[20 + i], i)
    bound.check("single tokens in large pages,")
    assert eng.length("r") == 30


@pytest.mark.gpu
def test_two_engines_share_no_memory_that_their_kernels_write(tmp_path):
    """Two engines of one model, each on a stream of its own, nothing waited for in between: what the steps' kernels share keys'
    sums through is the engine's own, and the logits are those of each alone."""
    from tiny_makuzen import write_tiny
    d = write_tiny(str(tmp_path), "C", torch.bfloat16)

    def made():
        eng = Engine.from_folder(d, dtype="bfloat16", page_size=16, max_tokens=512, num_slots=2)
        eng.add_request("r")
        eng.step([StepEntry("r", tokens_of(eng, "r", 40), [])])
        torch.cuda.synchronize()
        return eng

    engines, streams = [made(), made()], [torch.cuda.Stream(), torch.cuda.Stream()]
    toks = [[(5 * i + 11 * k) % 97 for i in range(20)] for k in range(2)]
    rows = [[], []]
    for i in range(20):
        for k in range(2):
            with torch.cuda.stream(streams[k]):
                rows[k].append(engines[k].step([StepEntry("r", [toks[k][i]], [0])]))
    torch.cuda.synchronize()
    held = [{t.data_ptr() for v in e.rt.workspaces.values() for t in (v if isinstance(v, list) else [v])} for e in engines]
    assert held[0] and held[1] and not held[0] & held[1]
    for k in range(2):
        alone = made()
        want = [alone.step([StepEntry("r", [t], [0])]) for t in toks[k]]
        assert torch.equal(torch.cat(rows[k]), torch.cat(want))
