"""Destruction of library objects from Python, over a stand-in for the library:
everything created on a context goes before it and once, also where the garbage
collector takes context and objects together (an exception's traceback holds
both, or the interpreter ends), when weak references are cleared before any
__del__ and the older object, the context, is finalised first."""
import ctypes as C
import gc

import pytest

import mag_amd as M
from mag_amd import _lib
from mag_amd import multi_md as MD
from mag_amd import serving as SV


class FakeLib:
    def __init__(self):
        self.log, self.next = [], 1

    def __getattr__(self, name):
        def call(*args):
            if name.endswith("_create"):
                h = C.cast(args[-1], C.POINTER(C.c_void_p))
                h[0] = self.next
                self.next += 1
            elif name.endswith("_destroy"):
                self.log.append((name, C.cast(args[0], C.c_void_p).value))
            return 0
        return call


@pytest.fixture
def lib(monkeypatch):
    fake = FakeLib()
    monkeypatch.setattr(_lib, "_lib", fake)
    yield fake
    gc.collect()


ALL = ["mag_ctx_destroy", "mag_chain_destroy", "mag_field_destroy", "mag_multi_destroy", "mag_server_destroy"]


def make():
    ctx = M.Context(0)
    arg = M.Arg_chmc()
    return [ctx, M.Field(ctx, (4, 4, 4, 4)), M.Chain(ctx, (4, 4, 4, 4), arg), SV.Server(ctx),
            MD.MultiChain(ctx, (8, 8, 8, 8), arg, MD.params(0.1, 1.0))]


def check(lib):
    names, handles = zip(*lib.log)
    assert sorted(names) == sorted(ALL) and len(set(handles)) == len(ALL) and None not in handles, lib.log
    assert names[-1] == "mag_ctx_destroy", lib.log


def test_collected_together(lib):
    cycle = make()
    cycle.append(cycle)
    del cycle
    gc.collect()
    check(lib)


def test_close_with_live_objects(lib):
    objs = make()
    objs[0].close()
    check(lib)
    with_handles = [o.handle for o in objs if hasattr(o, "handle")]
    assert not any(with_handles)
    del objs
    gc.collect()
    check(lib)


def test_objects_first(lib):
    objs = make()
    objs[3].close()
    while len(objs) > 1:
        objs.pop()
    assert len(lib.log) == len(ALL) - 1
    objs[0].close()
    check(lib)
