"""Layer calls refuse host tensors before anything is enqueued, and a refused call leaves the layer as it was (CPU only)."""
import ctypes
import types

import pytest
import torch


def bare_layer(slots=None, topk=4):
    """A MoELayer as its argument checks see it: no device memory behind it (its table is on the meta device)."""
    import bmx
    m = bmx.MoELayer.__new__(bmx.MoELayer)
    m.num_experts_per_tok, m.num_local_experts, m.routing_first = topk, 8, 0
    m.hidden_size, m.intermediate_size = 256, 128
    m.table = types.SimpleNamespace(has_shared=False, device=torch.device("meta"))
    m.slots, m.li, m._ws, m._staged, m.router_weight, m.router = slots, 0, None, None, None, bmx._lib.RouterDesc()
    m.desc = m.slot_desc = bmx._lib.MoeDesc(256, 128, 8, topk, 0, 0, 1, 0.0, 16, None, 32)
    return m


def host_call(T):
    return torch.zeros((T, 256)).half(), torch.zeros((T, 4), dtype=torch.int64), torch.ones((T, 4)).half()


@pytest.mark.parametrize("T", [1, 3])
def test_refused_call_keeps_no_host_workspace(T):
    """The workspace a refused call leaves behind is the next call's: never host memory."""
    m = bare_layer()
    x, sel, w = host_call(T)
    for call in (lambda: m.run_bszN(x, sel, w), lambda: m.forward(x, torch.zeros((T, 8)).half())):
        with pytest.raises(ValueError, match="device tensor"):
            call()
        assert m._ws is None or m._ws.device.type != "cpu"


@pytest.mark.parametrize("T", [1, 3])
def test_slot_call_refuses_host_tensors(T):
    """A slot-table call with a host selection (host rows, host weights) raises: a kernel would read host addresses."""
    m = bare_layer(types.SimpleNamespace(agent=None, copied=[None], seq=[0], check=lambda: None))
    with pytest.raises(ValueError, match="device tensor"):
        m.run_bszN(*host_call(T))


class Dev:
    """Stands for a contiguous device tensor of a shape (the checks read nothing else)."""
    is_cuda, device = True, "cuda:0"

    def __init__(self, shape, dtype):
        self.shape, self.dtype = shape, dtype

    def is_contiguous(self):
        return True


@pytest.mark.parametrize("xs,ss,ws", [((2, 256), (2, 3), (2, 4)), ((2, 256), (2, 5), (2, 5)), ((2, 256), (1, 4), (2, 4)),
                                      ((2, 256), (2, 4), (2, 3)), ((2, 128), (2, 4), (2, 4)), ((2, 256), (8,), (2, 4))])
def test_slot_call_refuses_other_shapes(xs, ss, ws):
    """Picks or weights that are not the call's T rows of topk, or rows that are not H long, would be read out of range."""
    import bmx
    x, sel, w = Dev(xs, torch.float16), Dev(ss, torch.int64), Dev(ws, torch.float16)
    with pytest.raises(ValueError, match="of one T"):
        bmx.ops.moe_slots_forward(bare_layer().slot_desc, None, 0, x, sel, w)


def test_single_expert_is_a_layer_of_one(monkeypatch):
    """run_single_expert(e) calls the library for a layer of that expert alone (its record, one expert, no shared one), so
    the plans count on all rows being its."""
    import bmx
    m = bare_layer()
    got = {}
    m.act, m.gated, m.act_limit = 0, True, 0.0
    m.table.desc = lambda topk, first, *a: bmx._lib.MoeDesc(256, 128, 8, topk, first, 0, 1, 0.0, 4096, 8192, None)
    monkeypatch.setattr(bmx.ops, "dispatch", lambda sel, E, first, shared, rpg: got.update(sel=sel, E=E, first=first, shared=shared))
    monkeypatch.setattr(bmx.ops, "moe_experts", lambda desc, x, r, path: (got.update(desc=desc), (torch.full((3, 256), 7.0), None))[1])
    m.routing_first = 100
    y = m.run_single_expert(torch.zeros((3, 256)), 5, torch.zeros((3, 256)).half())
    d = got["desc"]
    assert (d.E, d.topk, d.first, d.shared, d.experts) == (1, 1, 0, None, 4096 + 5 * ctypes.sizeof(bmx._lib.Expert))
    assert got["E"] == 1 and got["first"] == 0 and not got["shared"] and got["sel"].tolist() == [[0]] * 3
    assert bool((y == 7.0).all())
