"""The split-K products' workspace: every engine's own, since its captured graphs hold the addresses; what it outgrows stays."""
import threading

import pytest
import torch

from mxserve.ops import decode_gemm
from mxserve.ops.decode_gemm import TABLE, Workspace, using, workspace

CPU = torch.device("cpu")


def test_growth_keeps_what_graphs_may_hold():
    ws = Workspace()
    a = ws.slabs(100, CPU)
    assert ws.slabs(60, CPU) is a and a.numel() == 100
    b = ws.slabs(101, CPU)
    assert b.numel() == 200 and ws.outgrown == [a]  # at least twice: those kept stay smaller than the last
    c = ws.slabs(1000, CPU)
    assert c.numel() == 1000 and len(ws.outgrown) == 2 and ws.outgrown[1] is b


def test_no_growth_while_a_graph_is_captured(monkeypatch):
    ws = Workspace()
    a = ws.slabs(100, CPU)
    monkeypatch.setattr(decode_gemm, "_capturing", lambda: True)
    assert ws.slabs(100, CPU) is a and ws.slabs(101, CPU) is None and ws.counters(CPU) is None and ws.part is a


def test_every_thread_and_engine_has_its_own():
    one, two = Workspace(), Workspace()
    outside = workspace()
    with using(one):
        t = TABLE.part = torch.zeros(4)
        seen = []
        th = threading.Thread(target=lambda: seen.append(workspace()))
        th.start()
        th.join()
        assert seen == [outside]
        with pytest.raises(KeyError), using(two):
            assert TABLE.part is None
            raise KeyError
        assert TABLE.part is t and one.part is t and two.part is None
    assert workspace() is outside and TABLE.part is outside.part


def test_another_engines_tuning_leaves_this_ones_alone(monkeypatch):
    """tune() of a second engine, larger or smaller: the first one's tensors stay where its graphs have them."""
    class Store:  # every choice is on file: the library
        hits = misses = 0
        tag = ""

        def __init__(self, *a):
            pass

        def get(self, key):
            return {"cfg": None}

        def save(self):
            pass

    from mxserve.ops import tuned
    monkeypatch.setattr(decode_gemm, "MODE", "auto")
    monkeypatch.setattr(tuned, "TunedStore", Store)
    monkeypatch.setattr(tuned, "device_tag", lambda d: "")
    for name in ("entries", "report", "store_stats"):
        monkeypatch.setattr(TABLE, name, type(getattr(TABLE, name))())
    w = torch.randn(16, 8)
    held = []
    for buckets in ([4], [2], [8]):
        ws = Workspace()
        with using(ws):
            decode_gemm.tune({"o": (w, 0)}, buckets, "cpu", torch.float32)
        assert ws.part is not None and all(ws.part is not p for _, p in held)
        held.append((ws, ws.part))
    assert all(ws.part is p for ws, p in held)
    ws, p = held[0]
    with using(ws):  # the same engine again
        decode_gemm.tune({"o": (w, 0)}, [2], "cpu", torch.float32)
        assert ws.part is p
        decode_gemm.tune({"o": (w, 0)}, [64], "cpu", torch.float32)
    assert ws.part is not p and ws.outgrown == [p]


@pytest.mark.gpu
def test_an_engines_graphs_after_another_engine(gpu, monkeypatch):
    """Split-K products everywhere: the first engine's graphs give the same tokens after a second, larger engine tuned, captured,
    ran and went."""
    from mxserve.config import EngineArgs
    from mxserve.engine.engine import LLMEngine
    from mxserve.engine.request import SamplingParams

    def split(lib, cands):
        cfg = next((c for c in cands if TABLE.splitk(c) > 1), None)
        return cfg, 1.0, 1.0

    monkeypatch.setenv("MXS_RETUNE", "1")
    monkeypatch.delenv("MXS_TUNED_SAVE", raising=False)
    monkeypatch.setattr(decode_gemm, "MODE", "auto")
    monkeypatch.setattr(decode_gemm, "pick", split)
    monkeypatch.setattr(TABLE, "entries", {})

    def engine(seqs):
        return LLMEngine(EngineArgs(model="small-llama", device="cuda", dtype="bfloat16", block_size=16, num_gpu_blocks=128,
                                    max_model_len=256, max_num_seqs=seqs, max_num_batched_tokens=256, load_format="random", seed=3))

    def tokens(eng):
        sp = SamplingParams(temperature=0.0, max_tokens=8, ignore_eos=True)
        return eng.generate([[5, 6, 7, 8], [9, 10, 11]], sp)

    a = engine(4)
    assert any(r["cfg"] is not None for r in a.runner.decode_gemm_report)
    first = tokens(a)
    b = engine(16)
    assert a.runner.gemm_ws.part is not None and a.runner.gemm_ws.part.data_ptr() != b.runner.gemm_ws.part.data_ptr()
    tokens(b)
    b.runner.close()
    torch.cuda.empty_cache()
    torch.cuda.synchronize()
    for _ in range(3):
        junk = torch.full((1 << 20,), float("nan"), device=gpu)
        assert tokens(a) == first
        del junk
