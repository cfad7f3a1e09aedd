"""How much memory the packed copies of matrices may take, worked out without a GPU: the memory that is free is a number here, the copies are
made by ordinary tensors, and everything else is the engine's own."""
import importlib

import pytest
import torch

import tiny_configs as tc
import zogurax_configs as zc

K = importlib.import_module("daisi-llogos_amd.ops.kernels")
L = importlib.import_module("daisi-llogos_amd")
base = importlib.import_module("daisi-llogos_amd.parts.base")
moe = importlib.import_module("daisi-llogos_amd.parts.moe")
reg = importlib.import_module("daisi-llogos_amd.config.registry")
step = importlib.import_module("daisi-llogos_amd.engine.step")

EXPERTS = dict(zc.ZOG_C, layers=[dict(l, mlp={"kind": "moe", "router": {"experts": 4, "top": 2}, "expert": {"ff": 64}, "shared": {"ff": 32}})
                                 for l in zc.ZOG_C["layers"]])


@pytest.fixture(autouse=True)
def copies(monkeypatch):
    monkeypatch.setattr(K, "pack_weights", lambda w, gate_rows=0: K.PackedWeight(
        torch.zeros(K.packed_weight_bytes(*w.shape) // 2, dtype=torch.bfloat16), *w.shape, gate_rows))


def bound(monkeypatch, config, free, pack_weights=None):
    """The model of `config`, bound on the CPU with `free` bytes for copies beside its matrices and cache."""
    arch = reg.architecture_of(config)
    model = L.Model(arch.model_spec(arch.read_config(config)))
    rt = base.Runtime(torch.device("cpu"), torch.bfloat16)
    monkeypatch.setattr(step, "packed_weight_budget", lambda *a: free)
    step._packing(rt, model, 64, pack_weights)
    shapes = {s.name: s for s in model.tensor_specs()}

    def get(name):
        spec = shapes.get(name)
        if spec is None:
            return None
        return torch.zeros(spec.shape, dtype=torch.int32) if name.endswith("table") else torch.zeros(spec.shape)
    model.bind(get, rt)
    return model, rt


def experts_of(model):
    return [w for layer in model.layers for f in layer.feed_forwards() if f is not None for w in (f.packed_up, f.packed_down)]


@pytest.mark.parametrize("vocab", [331, 384])
def test_a_tied_heads_copy_is_not_given_away(monkeypatch, vocab):
    """The head is bound last and its copy, of a vocabulary that is no multiple of 64, is larger than the table: with memory to spare every
    matrix has its copy, and with just what they take too."""
    config = dict(tc.TINY_B, vocab_size=vocab, eos_token_id=1)
    model, rt = bound(monkeypatch, config, 1 << 40)
    assert model.head.packed is not None and rt.expert_budget == 0
    everything = model.packable_bytes()
    assert everything == model.packed_weight_bytes() and rt.pack_budget == (1 << 40) - everything
    model, rt = bound(monkeypatch, config, everything)
    assert model.head.packed is not None and rt.pack_budget == 0
    assert bound(monkeypatch, config, everything - 1)[0].head.packed is None


def test_experts_get_none_some_and_all(monkeypatch):
    """Experts' copies come after everybody else's and after the room for a second engine; none of the others loses its copy to them."""
    model, rt = bound(monkeypatch, EXPERTS, 1 << 40)
    copies = experts_of(model)
    own, others, each = step._own_bytes(model, torch.bfloat16, 64), model.packable_bytes(), [2 * 4 * 64 * 128] * len(copies)
    assert len(copies) == 8 and all(c is not None for c in copies) and sum(each) == 2 * model.expert_elements()
    assert model.packed_weight_bytes() == others + sum(each) and model.head.packed is not None
    for room, held in ((0, 0), (each[0] - 1, 0), (each[0], 1), (3 * each[0] + 5, 3), (sum(each), 8)):
        model, rt = bound(monkeypatch, EXPERTS, 2 * others + own + room)
        assert sum(c is not None for c in experts_of(model)) == held and model.head.packed is not None
        assert model.packed_weight_bytes() == others + sum(each[:held]) and rt.expert_budget == room - sum(each[:held])
        assert rt.pack_budget == others + own                 # what a second engine like this one needs is left
    model, _ = bound(monkeypatch, EXPERTS, others)            # just the others' copies
    assert model.packed_weight_bytes() == others and not any(experts_of(model))


def test_packing_all_and_none(monkeypatch):
    """True: every matrix but experts has its copy whatever is free, as before experts had any; experts as far as memory allows.  False: none."""
    model, rt = bound(monkeypatch, EXPERTS, 0, True)
    assert rt.pack_budget is None and model.packed_weight_bytes() == model.packable_bytes() and not any(experts_of(model))
    model, _ = bound(monkeypatch, EXPERTS, 1 << 40, True)
    assert all(c is not None for c in experts_of(model))
    model, _ = bound(monkeypatch, EXPERTS, 1 << 40, False)
    assert model.packed_weight_bytes() == 0 and not any(experts_of(model))


def test_no_memory_for_an_experts_copy_after_all(monkeypatch):
    """The allocation that fails leaves the row-major matrices to serve, there and in the layers behind it, and the other matrices their copies."""
    made = []

    def pack(w):
        made.append(w.shape)
        if len(made) == 3:
            raise torch.cuda.OutOfMemoryError("no room")
        return K.pack_weights(w.reshape(-1, w.shape[2]))
    monkeypatch.setattr(K, "pack_experts", pack)
    model, rt = bound(monkeypatch, EXPERTS, 1 << 40)
    assert [c is not None for c in experts_of(model)] == [True, True] + [False] * 6 and len(made) == 3
    assert rt.expert_budget == 0 and model.head.packed is not None
