"""The engine's context outlives every object made on it, in whatever order
Python finalises them: objects and engine dropped together in a reference cycle
(a traceback's frames after a failed call) are finalised in no particular order,
and an object destroyed on a freed context waits on a freed stream.  The native
library is replaced by a recorder."""
import gc
import types

import numpy as np
import pytest
import torch

import hala_amd as H


class recorder:
    def __init__(self):
        self.order = []

    def __getattr__(self, name):
        if not name.startswith("hala_"):
            raise AttributeError(name)
        return lambda *a: self.order.append(name) or 0


def build(eng):
    p = torch.tensor([0, 1, 2], dtype=torch.int32)
    i = torch.tensor([0, 1], dtype=torch.int32)
    v = torch.ones(2, dtype=torch.float64)
    return [H.gpu_sparse_matrix(eng, 2, 2, p, i, v), H.gpu_ilu(eng, p, i, None),
            H.gpu_triangular_matrix(eng, "L", "N", p, i, v), H.batch_solver(eng, p, p, i)]


@pytest.mark.parametrize("engine_first", [True, False])
@pytest.mark.parametrize("how", ["cycle", "engine dropped", "objects dropped", "failed creation"])
def test_context_destroyed_last(monkeypatch, how, engine_first):
    rec = recorder()
    monkeypatch.setattr(H, "lib", lambda: rec)

    def call(name, *a):
        if how == "failed creation" and name == "hala_ilu_create":
            raise H.HalaError(-2, "no")

    monkeypatch.setattr(H, "call", call)
    gc.collect()
    gc.disable()
    try:
        eng = H.gpu_engine(0, stream=types.SimpleNamespace(cuda_stream=0))
        if how == "failed creation":
            with pytest.raises(H.HalaError):
                build(eng)
            del eng
        else:
            objs = build(eng)
            if how == "engine dropped":
                for o in objs:
                    del o.engine  # a program may hold the objects alone
                del eng, o
                assert "hala_ctx_destroy" not in rec.order
                del objs
            elif how == "objects dropped":
                del objs, eng
            else:
                box = [eng] + objs if engine_first else objs[::-1] + [eng]
                for o in box:
                    o.box = box
                del box, eng, objs, o
    finally:
        gc.enable()
    gc.collect()
    assert rec.order.count("hala_ctx_destroy") == 1 and rec.order[-1] == "hala_ctx_destroy", rec.order
    assert how == "failed creation" or len(rec.order) == 5, rec.order
