"""Arguments of the stack calls are checked for every layer before the first one runs (host code only: nothing is launched)."""
import ctypes as C

import pytest

from subspec_amd import _lib as L

ADDRESS = 1 << 20                                    # stands for device memory; never dereferenced


def _dims(rows):
    return L.DecoderLayerDims(L.BF16, 0, rows, 256, 256, 2, 1, 128, 1024, 100, rows, 1e-6, 1e4, None, None, None, 0, 0, 0)


def _call(kind, layers, dims):
    lib, n = L.lib(), len(layers)
    table = (type(layers[0]) * n)(*layers)
    caches = (C.c_void_p * n)(*[ADDRESS] * n)
    if kind == "prefill":
        return lib.subspec_prefill_stack(C.byref(dims), table, n, ADDRESS, ADDRESS, ADDRESS, caches, caches, None, None, ADDRESS,
                                         1 << 40, None)
    fn = lib.subspec_dense_decoder_stack if kind == "dense" else lib.subspec_int4_decoder_stack
    return fn(C.byref(dims), table, n, ADDRESS, ADDRESS, ADDRESS, ADDRESS, caches, caches, None, None, ADDRESS, 1 << 40, None)


@pytest.mark.parametrize("kind", ["int4", "dense", "prefill"])
def test_a_misaligned_projection_of_the_last_layer_is_refused(kind):
    cls = L.DecoderLayerWeights if kind == "int4" else L.DenseLayerWeights
    names = [name for name, _ in cls._fields_ if name not in ("input_norm", "post_norm", "qkv_bias")]
    assert len(names) == (8 if kind == "int4" else 4)
    for name in names:
        layers = [cls(**{f: ADDRESS for f, _ in cls._fields_}) for _ in range(3)]
        setattr(layers[-1], name, ADDRESS + 2)
        assert _call(kind, layers, _dims(100 if kind == "prefill" else 8)) == -1, name
        assert b"projection weights must be 16-byte aligned" in L.lib().subspec_last_error(), name
