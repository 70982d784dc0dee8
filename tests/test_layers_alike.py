"""Which entries of a run order may run from one layer's launch list (no GPU): only layers that would launch
the same kernels with the same numbers. A layer that differs in one constant, or entries that do not each have a
cache plane of their own (or all read one), must run their own code."""

import dataclasses

import pytest

from conftest import TINY_B

import tie_amd  # noqa: F401  (registers the architecture and the parts)
from tie_amd.config.registry import resolve_architecture
from tie_amd.models.builder import Model
from tie_amd.models.spec import LayerCall, PartSpec


def qwen3_spec(layers):
    arch = resolve_architecture(TINY_B)
    return arch.build_spec(arch.read_config(dict(TINY_B, num_hidden_layers=layers)))


def alike(spec):
    model = Model(spec)
    model._find_layers_alike()
    return model._alike


def with_layer(spec, index, **changes):
    layers = list(spec.layers)
    layers[index] = dataclasses.replace(layers[index], **changes)
    return dataclasses.replace(spec, layers=tuple(layers))


def test_layers_of_one_shape_are_alike():
    assert alike(qwen3_spec(7)) == {0: 7}
    assert alike(qwen3_spec(3)) == {}          # fewer than four gain nothing


def test_a_layer_with_another_constant_is_not_alike():
    spec = qwen3_spec(9)
    norms = dict(spec.layers[4].norms)
    norms["pre_mixer"] = PartSpec("rms_norm", dict(norms["pre_mixer"].params, eps=1e-3))
    assert alike(with_layer(spec, 4, norms=norms)) == {0: 4, 5: 9}
    mixer = spec.layers[6].mixer
    other_scale = PartSpec(mixer.kind, dict(mixer.params, scale=0.5))
    assert alike(with_layer(spec, 6, mixer=other_scale)) == {0: 6}
    position = PartSpec("rope_neox", dict(mixer.params["position"].params, theta=10000.0))
    other_theta = PartSpec(mixer.kind, dict(mixer.params, position=position))
    assert alike(with_layer(spec, 2, mixer=other_theta)) == {3: 9}
    eps = PartSpec(mixer.kind, dict(mixer.params, qk_norm=dict(mixer.params["qk_norm"], eps=1e-2)))
    assert alike(with_layer(spec, 8, mixer=eps)) == {0: 8}


def test_entries_that_share_some_cache_planes_are_not_alike():
    spec = qwen3_spec(8)
    own = tuple(LayerCall(l) for l in range(8))
    assert alike(dataclasses.replace(spec, order=own)) == {0: 8}
    # entries 4 and 5 read entry 3's keys and values, 6 and 7 read entry 2's: the readers are of one shape and
    # write nothing, but they do not all read one plane, nor each its own
    shared = own[:4] + (LayerCall(4, 3), LayerCall(5, 3), LayerCall(6, 2), LayerCall(7, 2))
    assert alike(dataclasses.replace(spec, order=shared)) == {0: 4}
    one_plane = own[:4] + tuple(LayerCall(l, 3) for l in range(4, 8))
    assert alike(dataclasses.replace(spec, order=one_plane)) == {0: 4, 4: 8}


def launches_of_steps(monkeypatch, config, dtype, tensors, rows):
    """What steps of ``rows`` tokens launch with layers run from a launch list and with every layer running its own code,
    as ``(kernel, arguments)``: the model's host code with the launches themselves left out."""
    import torch

    from tie_amd import kernels
    from tie_amd.cache.manager import CacheManager
    from tie_amd.engine.batch import StepEntry
    from tie_amd.engine.runner import ModelRunner
    from tie_amd.models.builder import load_model_from_tensors

    log, got, replayed = [], [], 0

    def call(fn, what, *args):
        if kernels._recording is not None:
            kernels._recording.append((fn, args, what))
        log.append((what, args))

    monkeypatch.setattr(torch.Tensor, "is_cuda", property(lambda self: True), raising=False)
    monkeypatch.setattr(kernels, "_call", call)
    monkeypatch.setattr(kernels, "replay_call", lambda fn, what, args: log.append((what, tuple(args))))
    monkeypatch.setattr(kernels, "_stream", lambda: 0)
    model = load_model_from_tensors(config, tensors, dtype, "cpu")
    cache = CacheManager(model.cache_plan, block_size=16, num_blocks=32, dtype=dtype, device=torch.device("cpu"))
    runner = ModelRunner(model, cache)
    request = cache.new_request()
    assert cache.reserve(request, rows)
    for replay in (False, True, False):            # the first settles the scratch memory
        model.replay_layers, model.layers_replayed = replay, 0
        log.clear()
        runner.step([StepEntry(request, 0, list(range(rows)), [rows - 1])])
        got.append(list(log))
        replayed = max(replayed, model.layers_replayed)
    # A step's work lists are new tensors: only addresses of weights, of scratch memory and of the cache are compared.
    kept = [tensor for tensors in model._layer_tensors.values() for tensor in tensors]
    kept += [(t.data_ptr(), t.numel() * t.element_size()) for t in runner.workspace._buffers.values()]
    kept += [(t.data_ptr(), t.numel() * t.element_size()) for t in (*cache.kv.values(), *cache.state.values())]

    def comparable(args):
        return tuple(a if not isinstance(a, int) or a < 1 << 32 or any(0 <= a - at < size for at, size in kept)
                     else "the step's" for a in args)

    return [[(what, comparable(args)) for what, args in log] for log in got[1:]] + [model, replayed]


def norms_behind_two_mixers(layers):
    from vosurax_fixtures import _parallel

    return {"architecture": "Vosurax", "vocab": 64, "width": 48, "norm": {"eps": 1e-5},
            "layers": [{**_parallel((4, 2, 16, 32, 0.3, 40), (2, 40, 72, 5.0)), "mlp": None} for _ in range(layers)]}


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("rows", [5, 40])
@pytest.mark.parametrize("layers", [6, 7])
def test_a_pass_left_for_the_next_layer_keeps_its_own_layers_weights(monkeypatch, layers, rows, dtype):
    """A layer without a feed-forward leaves the norms behind its two mixers to the next layer's first pass: every pass
    reads the weights of the layer that left it, the last one's behind the last layer."""
    from vosurax_fixtures import make_tensors

    config = norms_behind_two_mixers(layers)
    listed, own, model, replayed = launches_of_steps(monkeypatch, config, dtype, make_tensors(config, 3, dtype), rows)
    assert model._alike == {0: layers}
    assert [args[4] for what, args in listed if what == "add_normed_results"] == \
        [layer.mixer.norm_weights[0].data_ptr() for layer in model.layers]
    assert listed == own


@pytest.mark.parametrize("rows", [3, 40])
@pytest.mark.parametrize("width", [64, 4096])
def test_a_launch_list_launches_what_every_layers_own_code_does(monkeypatch, width, rows):
    """In a step of a few rows every sub-layer leaves its last product to the next norm: over the weight of the layer it
    ends, which for a layer's first norm is the layer before."""
    import torch

    from tie_amd.models import expected_tensors_for_config
    from tie_amd.weights.random_init import random_tensors

    config = dict(TINY_B, num_hidden_layers=7, hidden_size=width, intermediate_size=128)
    specs = [s for s in expected_tensors_for_config(config) if not s.optional]
    tensors = dict(random_tensors(specs, 5, torch.bfloat16, device="cpu"))
    listed, own, model, replayed = launches_of_steps(monkeypatch, config, "bfloat16", tensors, rows)
    assert replayed == 4
    assert listed == own
    pending = sum(what == "skinny_gemm_bf16_norm" and args[15] is not None for what, args in own)   # a next norm's weight
    assert pending == (13 if rows == 3 else 0)


def test_a_launch_list_as_words(monkeypatch):
    """What one native call runs for several layers: pointers and whole numbers (negative ones too), a float's bits, None
    as a null pointer, and every layer's own addresses where they belong; a refused launch is reported by its name."""
    import ctypes
    import struct

    import numpy as np

    from tie_amd import kernels
    from tie_amd.errors import InvalidArgument

    norm = kernels._lib("elementwise").tie_rms_norm
    first = (norm, "rms_norm", (1000, 0, 2000, 1e-6, 3000, 1, None, 4, 256, 7), ((0, 1, 16), (4, 0, 0)))
    second = (norm, "second norm", (1000, 0, 2000, -0.5, 3000, 1, None, -4, 256, 7), ())
    assert kernels.LaunchList.takes([first, second])
    assert not kernels.LaunchList.takes([first, (kernels._order_streams, "order_streams", (None, None), ())])
    ran = {}

    class Recorder:
        @staticmethod
        def tie_run_launch_list(entries, first_word, count, words, words_a_layer, layers, failed):
            ran["words"] = np.ctypeslib.as_array(ctypes.cast(words, ctypes.POINTER(ctypes.c_uint64)), (layers, words_a_layer)).copy()
            return 0

    listed = kernels.LaunchList([first, second])
    real = kernels._lib
    monkeypatch.setattr(kernels, "_lib", lambda key, *a: Recorder if key == "launch_list" else real(key, *a))
    listed.run([[50, 60], [2 ** 40, 2 ** 41]])
    eps, half = (struct.unpack("<I", struct.pack("<f", v))[0] for v in (1e-6, -0.5))
    rest = [1000, 0, 2000, half, 3000, 1, 0, 2 ** 64 - 4, 256, 7]
    assert ran["words"].tolist() == [[76, 0, 2000, eps, 50, 1, 0, 4, 256, 7] + rest,
                                     [2 ** 41 + 16, 0, 2000, eps, 2 ** 40, 1, 0, 4, 256, 7] + rest]
    monkeypatch.setattr(kernels, "_lib", real)
    with pytest.raises(InvalidArgument, match="second norm"):       # refused before anything is launched
        kernels.LaunchList([second]).run([[0, 0]])


@pytest.mark.parametrize("layers,at_once", [(4, None), (6, None), (7, [2, 2]), (9, [2, 4]), (18, [2, 4, 8, 1])])
def test_a_launch_list_is_made_for_layers_enough_and_run_a_few_layers_first(monkeypatch, layers, at_once):
    """Three layers run their own code and show what the others launch. Making a list costs the host more than calls for a
    few layers do; and a long list is not written down whole before the GPU gets its first layers."""
    import torch

    from tie_amd import kernels

    model = Model(qwen3_spec(layers))
    made, ran, called = [], [], []

    class Listed:
        MIN_LAYERS = kernels.LaunchList.MIN_LAYERS

        @staticmethod
        def of(launches):
            made.append(launches)
            return Listed

        @staticmethod
        def run(addresses):
            ran.append([row[0] for row in addresses])

    class Step:
        device, pending_linear = "cuda", None
        cache_of = cache_places = staticmethod(lambda index: [])

    class Block:
        @staticmethod
        def forward(ctx, x, layer, cache):
            pass

    class Layer:
        block = Block

    monkeypatch.setattr(kernels, "LaunchList", Listed)
    monkeypatch.setattr(kernels, "replay_call", lambda fn, what, args: called.append(args[0]))
    monkeypatch.setattr(kernels, "start_recording", list)
    noted = kernels.rms_norm
    monkeypatch.setattr(Model, "_launch_list", staticmethod(lambda *a: [_launch(noted)]))
    model.layers = [Layer] * layers
    model._layer_tensors = {i: [(1000 + i, 1)] for i in range(layers)}
    model._layer_projections = {i: [] for i in range(layers)}
    model._run_alike(Step(), torch.zeros(1), 0, layers)
    rest = [1000 + i for i in range(3, layers)]
    if at_once is None:
        assert not made and not ran and called == rest
    else:
        assert len(made) == 1 and not called
        assert [len(part) for part in ran] == at_once and [a for part in ran for a in part] == rest


def _launch(fn):
    from tie_amd.models.builder import _Launch

    return _Launch(fn, "rms_norm", (0,), ((0, 0, 0),))


def test_arguments_that_fit_no_word_make_no_launch_list():
    from tie_amd import kernels

    norm = kernels._lib("elementwise").tie_rms_norm
    args = (1000, 0, 2000, 1e-6, 3000, 1, None, 4, 256, 7)
    assert kernels.LaunchList.of([(norm, "rms_norm", args, ())]) is not None
    for wrong in (args[:7] + (4.0,) + args[8:], args[:3] + ("eps",) + args[4:], args[:3] + (1e39,) + args[4:], args[:-1],
                  args[:7] + (2 ** 63,) + args[8:]):
        assert kernels.LaunchList.of([(norm, "rms_norm", wrong, ())]) is None


def test_lists_go_to_the_device_together():
    import torch

    from tie_amd import kernels

    a, none, b = kernels.upload_ints("cpu", [3, 1, 2], [], [7])
    assert none is None and a.dtype == b.dtype == torch.int32 and a.tolist() == [3, 1, 2] and b.tolist() == [7]
    assert kernels.upload_ints("cpu", [], []) == [None, None]
