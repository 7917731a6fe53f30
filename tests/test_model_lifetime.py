"""The life of a model's device memory.  What Model.logits_dev() returns keeps it
alive: a tensor over the logits was left with freed device memory once the last
reference to the Model was gone, or close() was called.  And a step that still
runs keeps its graph: it was destroyed before anything waited for the step."""
import gc
import types

import numpy as np
import pytest

import fake_hip


def test_logits_address_keeps_the_model(pe):
    freed = []
    lib = types.SimpleNamespace(prism_hip_model_logits_dev=lambda h: 4096, prism_hip_model_free=freed.append)
    m = pe.Model.__new__(pe.Model)
    m.ctx, m.h = types.SimpleNamespace(lib=lib), 7
    p = m.logits_dev()
    assert p == 4096 and isinstance(p, int)
    held = {"data": (p, False)}
    del m, p
    gc.collect()
    assert freed == []
    del held
    gc.collect()
    assert freed == [7]


@pytest.mark.gpu
def test_logits_tensor_outlives_the_model_reference(pe, gpu_ctx):
    import torch

    class View:
        def __init__(self, ptr, n):
            self.__cuda_array_interface__ = {"data": (ptr, False), "shape": (n,), "typestr": "<f2", "version": 3}

    cfg = pe.Qwen2Config(n_layers=1, hidden=128, n_heads=2, n_kv_heads=1, intermediate=64, vocab=300)
    embed, layers = pe.synth_weights(cfg, 5)
    m = pe.Model.from_tensors(gpu_ctx, cfg, embed, layers, max_seq=8)
    want = m.step(3, 0)
    logits = torch.as_tensor(View(m.logits_dev(), 300), device="cuda")
    del m
    gc.collect()
    assert np.array_equal(logits.cpu().numpy().view(np.uint16), want.view(np.uint16))


# ---- the order of waits and destructions, with the fake runtime

STREAM = 0x77000  # a stream of the caller's


def _model(hip, pe):
    cfg = pe.Qwen2Config(n_layers=1, hidden=128, n_heads=2, n_kv_heads=1, intermediate=64, vocab=304)
    ctx = pe.Context(0)
    m = pe.Model(ctx, cfg, max_seq=8)

    def upload(n, k):
        nbytes = n * 32 + n * k // 2
        return ctx.upload_dev(fake_hip.Tensor(hip, nbytes), n, k, 4)

    m.set_embedding(upload(cfg.vocab, cfg.hidden))
    layer = [upload(n, k) for n, k in cfg.shapes().values()]
    m.set_layer(0, layer)
    hip.clear()
    return ctx, m, layer


def release_in_flight(hip, pe, stream, how):
    ctx, m, layer = _model(hip, pe)
    m.step_dev(3, 0, stream)
    if how == "close":
        m.close()
    elif how == "new weights":
        m.set_layer(0, layer)
    elif how == "context first":
        ctx.close()
        m.close()
    return hip.log()


@pytest.mark.parametrize("stream", [None, STREAM])
@pytest.mark.parametrize("how", ["close", "new weights", "context first"])
def test_a_step_in_flight_is_waited_for(stream, how):
    """A model that is freed or gets new weights while a step runs, on the
    context's stream or the caller's: its executable, graph and capture stream
    are destroyed after a wait that covers the step."""
    log = fake_hip.call(__name__, "release_in_flight", stream, how)
    assert any(ln.startswith("graph launch") for ln in log) and any(ln.startswith("exec destroy") for ln in log)
    assert not [ln for ln in log if ln.endswith("IN FLIGHT")], log


def close_with_address(hip, pe):
    ctx, m, _ = _model(hip, pe)
    p = m.logits_dev()
    held = {"data": (p, False)}
    address = int(p)
    m.close()
    m.close()
    with pytest.raises(pe.PrismHipError):
        m.step_dev(3, 0)
    open_, lines = hip.room(address), hip.log()
    del p, m
    gc.collect()
    still = hip.room(address)
    del held
    gc.collect()
    return [open_, still, hip.room(address), [ln for ln in lines if ln.startswith("free")]]


def test_close_leaves_a_held_address_valid():
    """close() while an address of logits_dev() is held: the memory stays until
    the address is gone, and then it goes."""
    closed, dropped, gone, frees = fake_hip.call(__name__, "close_with_address")
    assert closed >= 608 and dropped >= 608 and frees == []
    assert gone == 0
