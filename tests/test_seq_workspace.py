"""A program may ask for a sequential model's workspace before it has the model's buffers: the size depends on the layers' shapes alone (no GPU needed)."""
import ctypes as C

import pytest

import helpers

capi = helpers.package().capi


def _layers(inputs, hidden, outputs, filled):
    layers = (capi.SeqLayer * 4)()
    for layer, (kind, i, o) in zip(layers, ((0, inputs, hidden), (1, hidden, hidden), (1, hidden, hidden), (0, hidden, outputs))):
        layer.kind = kind
        part = layer.gru if kind else layer.dense
        if kind:
            part.input_dim, part.hidden_dim, part.fast_tanh = i, o, 1
        else:
            part.in_dim, part.out_dim = i, o
        if filled:      # addresses that nothing here reads
            for name, ctype in part._fields_:
                if ctype is C.c_void_p:
                    setattr(part, name, 4096)
    return layers


@pytest.mark.parametrize("hidden", [8, 16, 32, 64])
@pytest.mark.parametrize("steps,batch", [(1, 1), (2, 3), (100, 100), (4000, 2)])
def test_workspace_size_depends_on_shapes_alone(hidden, steps, batch):
    size = helpers.package().load_library().rlt_rocm_seq_workspace_bytes
    size.restype, size.argtypes = C.c_size_t, [C.POINTER(capi.SeqLayer), C.c_int, C.c_int, C.c_int]
    empty, filled = (size(_layers(4, hidden, 2, f), 4, steps, batch) for f in (False, True))
    assert empty == filled > 0
