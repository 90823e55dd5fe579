"""States share one context's kept device blocks: a state made in a block that another one left behind
gives the same rollout as in fresh memory, also with other sizes, streams, models and threads."""
import threading

import numpy as np
import pytest
import torch

from burn_automata_amd import synthetic as syn
from burn_automata_amd.executor import HipAutomataExecutor
from burn_automata_amd.model import NpaModel
from burn_automata_amd.runtime import Context
from tests.helpers import to_np

pytestmark = pytest.mark.gpu


def _roll(ctx, w, steps=6):
    ex = HipAutomataExecutor(ctx=ctx)
    s = ex.create_state(NpaModel(w["model"], w["weights"]), w["positions"], w["states"], w["batch"], w["n"], w["grid"],
                        1.0, 0.5, 7)
    ex.step_state_many(s, steps)
    out = [to_np(x) for x in ex.read_state(s)]
    s.close()
    return out


def _fresh(w, steps=6):
    c = Context()
    out = _roll(c, w, steps)
    c.close()
    return out


def test_reused_blocks_give_the_same_rollout():
    # C4's build keeps counters between steps; sizes within and beyond a factor of two of each other
    loads = [syn.workload("c1", particles=2048), syn.workload("c4", particles=2048), syn.workload("c1", particles=1500),
             syn.workload("c2", particles=9000), syn.workload("c4", particles=16384), syn.workload("c1", particles=700)]
    want = [_fresh(w) for w in loads]
    ctx = Context()
    for _ in range(2):
        for w, ref in zip(loads, want):
            for a, b in zip(_roll(ctx, w), ref):
                np.testing.assert_array_equal(a, b)
    ctx.close()


def test_live_states_do_not_share_a_block():
    w = syn.workload("c1", particles=1024)
    ref = _fresh(w, 8)
    ctx = Context()
    ex = HipAutomataExecutor(ctx=ctx)
    m = NpaModel(w["model"], w["weights"])
    make = lambda: ex.create_state(m, w["positions"], w["states"], 1, w["n"], w["grid"], 1.0, 0.5, 7)  # noqa: E731
    make().close()  # leaves a block behind
    a, b = make(), make()
    for _ in range(8):
        ex.step_state(a)
        ex.step_state(b)
    for s in (a, b):
        for x, y in zip(ex.read_state(s), ref):
            np.testing.assert_array_equal(to_np(x), y)
        s.close()
    ctx.close()


def test_stream_change_and_threads():
    w = syn.workload("c4", particles=3000)
    ref = _fresh(w)
    ctx = Context()
    ex = HipAutomataExecutor(ctx=ctx)
    m = NpaModel(w["model"], w["weights"])
    side = torch.cuda.Stream()
    first = torch.cuda.current_stream().cuda_stream
    s = ex.create_state(m, w["positions"], w["states"], 1, w["n"], w["grid"], 1.0, 0.5, 7)
    ctx.set_stream(side.cuda_stream)
    ex.step_state_many(s, 50)
    ctx.set_stream(first)
    s.close()  # work may still be queued on the other stream
    for x, y in zip(_roll(ctx, w), ref):
        np.testing.assert_array_equal(x, y)
    states = [ex.create_state(m, w["positions"], w["states"], 1, w["n"], w["grid"], 1.0, 0.5, 7) for _ in range(6)]
    threads = [threading.Thread(target=st.close) for st in states]  # more than the pool keeps
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for x, y in zip(_roll(ctx, w), ref):
        np.testing.assert_array_equal(x, y)
    ctx.close()


def test_weights_staged_after_a_mode_change():
    """A state made on device pointers takes new weights from host arrays."""
    w = syn.workload("c1", particles=1024)
    ctx = Context()
    ex = HipAutomataExecutor(ctx=ctx)
    new = syn.seeded_weights(w["model"], 9)
    m = NpaModel(w["model"], w["weights"])
    a = ex.create_state(m, w["positions"], w["states"], 1, w["n"], w["grid"], 1.0, 0.5, 7)
    ex.update_state_model(a, new)
    ex.step_state_many(a, 4)
    ref = [to_np(x) for x in ex.read_state(a)]
    b = ex.create_state(m, w["positions"], w["states"], 1, w["n"], w["grid"], 1.0, 0.5, 7)
    from burn_automata_amd import _abi
    from burn_automata_amd._lib import lib
    import ctypes as C
    host = {k: np.ascontiguousarray(v, np.float32) for k, v in new.items()}
    wc = _abi.NpaWeightsC(*(C.c_void_p(host[k].ctypes.data) for k in ("w1", "b1", "w2", "b2")))
    ctx.host_io = True
    ctx.check(lib().npa_state_update_model(b.handle, C.byref(wc)))
    ctx.host_io = False
    ex.step_state_many(b, 4)
    for x, y in zip(ex.read_state(b), ref):
        np.testing.assert_array_equal(to_np(x), y)
    a.close()
    b.close()
    ctx.close()


def test_read_into_an_odd_address():
    """A destination off the word boundary goes through the runtime's copy, one on it through the library's kernel."""
    from burn_automata_amd._lib import lib

    w = syn.workload("c1", particles=700)
    ctx = Context()
    ex = HipAutomataExecutor(ctx=ctx)
    s = ex.create_state(NpaModel(w["model"], w["weights"]), w["positions"], w["states"], 1, w["n"], w["grid"], 1.0, 0.5, 7)
    ex.step_state_many(s, 2)
    want = to_np(ex.read_state(s)[2])
    for offset in (1, 2, 4):
        buf = torch.zeros(4 * w["n"] + 8, dtype=torch.uint8, device="cuda")
        torch.cuda.synchronize()
        ctx.check(lib().npa_state_read(s.handle, None, None, buf.data_ptr() + offset))
        torch.cuda.synchronize()
        np.testing.assert_array_equal(buf[offset: offset + 4 * w["n"]].cpu().numpy().view(np.float32), want)
        assert not buf[4 * w["n"] + offset:].any() and not buf[:offset].any()
    s.close()
    ctx.close()


def test_destroy_waits_for_work_on_other_streams():
    """A state's captured step, replayed on a stream that the context was never given, has finished when the state is
    destroyed: its block may be the next state's."""
    w = syn.workload("c1", particles=4096)
    ref = _fresh(w, 8)
    ctx = Context()
    ex = HipAutomataExecutor(ctx=ctx)
    m = NpaModel(w["model"], w["weights"])
    make = lambda: ex.create_state(m, w["positions"], w["states"], 1, w["n"], w["grid"], 1.0, 0.5, 7)  # noqa: E731
    capture, other = torch.cuda.Stream(), torch.cuda.Stream()
    ctx.set_stream(capture.cuda_stream)
    s = make()
    ex.step_state_many(s, 2)  # eager, outside the capture
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=capture):
        ex.step_state_many(s, 2)
    torch.cuda.synchronize()
    with torch.cuda.stream(other):
        for _ in range(500):  # about 40 ms of steps
            graph.replay()
    queued = not other.query()
    s.close()
    assert queued and other.query()
    t = make()
    ex.step_state_many(t, 8)
    for x, y in zip(ex.read_state(t), ref):
        np.testing.assert_array_equal(to_np(x), y)
    t.close()
    ctx.close()


def test_trim_gives_the_kept_memory_back():
    """The memory of destroyed states, and no live state's, is free again for other allocators after a trim."""
    w = syn.workload("c2", particles=200000)
    ctx = Context()
    ex = HipAutomataExecutor(ctx=ctx)
    m = NpaModel(w["model"], w["weights"])
    make = lambda: ex.create_state(m, w["positions"], w["states"], 1, w["n"], w["grid"], 1.0, 0.5, 7)  # noqa: E731
    live = make()
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    a, b = make(), make()
    two = before - torch.cuda.mem_get_info()[0]
    assert two > 100 << 20
    a.close()
    b.close()
    kept = before - torch.cuda.mem_get_info()[0]
    assert kept > two // 2
    ctx.trim()
    assert before - torch.cuda.mem_get_info()[0] <= two // 16
    ex.step_state_many(live, 6)
    for x, y in zip(ex.read_state(live), _fresh(w)):
        np.testing.assert_array_equal(to_np(x), y)
    live.close()
    ctx.close()
