"""Device memory as the host code handles it, without a GPU: fs_host.c over a
HIP runtime of host memory (hip_stub.c) that counts allocations and frees."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from futspace_amd import View
from futspace_amd._native import FUTSPACE_SIGNATURES

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SIDE = 32
VIEW = View(x=3.0, y=4.0, height=300.0, angle=0.4, horizon=8.0, h=12, w=16, d=0.01, z0=0.5)


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("stub") / "libstub.so")
    subprocess.run(["gcc", "-std=gnu11", "-O1", "-fPIC", "-shared", "-ffp-contract=off", "-w",
                    "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-o", out,
                    os.path.join(ROOT, "futspace_amd", "csrc", "fs_host.c"),
                    os.path.join(ROOT, "tests", "hip_stub.c"), "-lm"], check=True)
    so = ctypes.CDLL(out)
    for name, (res, args) in FUTSPACE_SIGNATURES.items():
        if hasattr(so, name):
            getattr(so, name).restype, getattr(so, name).argtypes = res, args
    return so


class Ctx:
    """A context of the stub, freed at the end of the test."""

    def __init__(self, lib):
        self.lib, self.ptr = lib, lib.futhark_context_new(None)
        assert self.ptr

    def map(self, side=SIDE, want=0):
        p = ctypes.c_void_p()
        a = np.zeros((side, side), np.uint32)
        rc = self.lib.fsx_map_new(self.ptr, ctypes.byref(p), a.ctypes.data,
                                  a.ctypes.data, side, side, 8, side, 0.1, 0.1)
        assert rc == want
        return p.value

    def free(self, m):
        assert self.lib.fsx_map_free(self.ptr, m) == 0

    def output(self, nbytes=12 * 16 * 4):
        return ctypes.create_string_buffer(nbytes)


def _get(lib, name, kind=ctypes.c_int64):
    return kind.in_dll(lib, name).value


def _set(lib, name, value, kind=ctypes.c_int64):
    kind.in_dll(lib, name).value = value


@pytest.fixture
def contexts(lib):
    made = [Ctx(lib), Ctx(lib)]
    yield made
    _set(lib, "stub_capturing", 0, ctypes.c_int)
    _set(lib, "stub_limit", 2 ** 63 - 1)
    for c in made:
        lib.futhark_context_free(c.ptr)
    lib.hipGetLastError()


def _readers(lib, c, m):
    """The calls that queue work over a map's buffers."""
    view, f32 = VIEW.to_c(), ctypes.create_string_buffer(64 * SIDE * SIDE)
    ref = ctypes.byref(view)
    return {
        "render": lambda: lib.fsx_render(c.ptr, m, ref, f32, 0),
        "render2": lambda: lib.fsx_render2(c.ptr, m, ref, f32, 0),
        "shade_factor": lambda: lib.fsx_map_shade_factor(c.ptr, m, f32),
        "forward": lambda: lib.fsx_render_f32(c.ptr, m, ref, f32, f32, SIDE, SIDE, 0.1, f32, f32),
        "step": lambda: lib.fsx_render_f32_l2_step_noalloc(
            c.ptr, m, ref, f32, f32, SIDE, SIDE, 0.1, f32, 0, f32, f32, f32, f32, f32, f32),
    }


MAP_BUFFERS = 5      # heights twice, colours, shaded colours and their quads


@pytest.mark.parametrize("call", ["render", "render2", "shade_factor", "forward", "step"])
@pytest.mark.parametrize("where", ["own", "other", "graph"])
def test_buffers_read_elsewhere_are_freed_and_not_reused(lib, contexts, call, where):
    """A map that another context or a captured graph reads goes back to the
    driver, whose free waits for the device; only a map that the owner's own
    stream alone reads is kept for the next load."""
    a, b = contexts
    m = a.map()
    if where == "graph":
        assert lib.fsx_context_stream(a.ptr)      # as who captures it has to
    _set(lib, "stub_capturing", int(where == "graph"), ctypes.c_int)
    assert _readers(lib, b if where == "other" else a, m)[call]() == 0
    _set(lib, "stub_capturing", 0, ctypes.c_int)
    frees = _get(lib, "stub_frees")
    a.free(m)
    freed = _get(lib, "stub_frees") - frees
    # only render reads the shade's two buffers as well
    assert freed == (0 if where == "own" else MAP_BUFFERS if call == "render" else 3)


def test_buffers_read_on_a_callers_stream_under_capture_are_freed(lib, contexts):
    """A context moved onto a caller's stream, which the caller captures."""
    a = contexts[0]
    m = a.map()
    own = ctypes.create_string_buffer(8)
    assert lib.fsx_context_set_stream(a.ptr, ctypes.addressof(own)) == 0
    _set(lib, "stub_capturing", 1, ctypes.c_int)
    assert _readers(lib, a, m)["render"]() == 0
    _set(lib, "stub_capturing", 0, ctypes.c_int)
    assert lib.fsx_context_set_stream(a.ptr, None) == 0
    frees = _get(lib, "stub_frees")
    a.free(m)
    assert _get(lib, "stub_frees") - frees == MAP_BUFFERS


def test_a_map_freed_through_another_context_leaves_no_pool(lib, contexts):
    a, b = contexts
    m = a.map()
    frees = _get(lib, "stub_frees")
    b.free(m)
    assert _get(lib, "stub_frees") - frees == MAP_BUFFERS


def test_a_state_rendered_elsewhere_keeps_its_buffers_out_of_the_pool(lib, contexts):
    a, b = contexts
    maps = np.zeros((SIDE, SIDE), np.uint32)
    col = lib.futhark_new_u32_2d(a.ptr, maps.ctypes.data, SIDE, SIDE)
    hts = lib.futhark_new_i32_2d(a.ptr, maps.ctypes.data, SIDE, SIDE)
    s0, s1, out = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_void_p()
    assert lib.futhark_entry_init(a.ptr, ctypes.byref(s0), 0) == 0
    assert lib.futhark_entry_update_map(a.ptr, ctypes.byref(s1), ctypes.c_void_p(col),
                                        ctypes.c_void_p(hts), s0) == 0
    assert lib.futhark_entry_render(b.ptr, ctypes.byref(out), s1) == 0
    frees = _get(lib, "stub_frees")
    lib.futhark_free_opaque_state(a.ptr, s1)
    assert _get(lib, "stub_frees") - frees == MAP_BUFFERS
    lib.futhark_free_opaque_state(a.ptr, s0)
    lib.futhark_free_u32_2d(a.ptr, col)
    lib.futhark_free_i32_2d(a.ptr, hts)
    lib.futhark_free_u32_2d(b.ptr, out)


def test_a_shade_that_a_captured_graph_writes_is_freed_and_not_reused(lib, contexts):
    """A step under capture shades into a buffer that every replay of the graph
    writes again."""
    a = contexts[0]
    maps = np.zeros((SIDE, SIDE), np.uint32)
    col = lib.futhark_new_u32_2d(a.ptr, maps.ctypes.data, SIDE, SIDE)
    hts = lib.futhark_new_i32_2d(a.ptr, maps.ctypes.data, SIDE, SIDE)
    states = [ctypes.c_void_p() for _ in range(4)]
    init, loaded, keyed, stepped = states
    assert lib.futhark_entry_init(a.ptr, ctypes.byref(init), 0) == 0
    assert lib.futhark_entry_update_map(a.ptr, ctypes.byref(loaded), ctypes.c_void_p(col),
                                        ctypes.c_void_p(hts), init) == 0
    assert lib.futhark_entry_key(a.ptr, ctypes.byref(keyed), 0, ord("u"), loaded) == 0
    assert lib.fsx_context_stream(a.ptr)
    _set(lib, "stub_capturing", 1, ctypes.c_int)
    assert lib.futhark_entry_step(a.ptr, ctypes.byref(stepped), 0.016, keyed) == 0
    _set(lib, "stub_capturing", 0, ctypes.c_int)
    frees = _get(lib, "stub_frees")
    for s in states:
        lib.futhark_free_opaque_state(a.ptr, s)
    # the heights and colours that the graph reads, and the shade it writes;
    # the shade of the loaded state is read by nothing and kept
    assert _get(lib, "stub_frees") - frees == MAP_BUFFERS
    lib.futhark_free_u32_2d(a.ptr, col)
    lib.futhark_free_i32_2d(a.ptr, hts)


def _calls_that_allocate(lib, c, m):
    """Calls whose first use, or every use, takes device memory of its own."""
    view, buf = VIEW.to_c(), ctypes.create_string_buffer(4096)
    wide = View(**{**VIEW.__dict__, "w": 4096, "h": 1}).to_c()
    maps, off, out = (ctypes.c_void_p * 1)(m), ctypes.c_int64(0), ctypes.c_void_p()
    aligned = ctypes.c_void_p((ctypes.addressof(buf) + 63) & ~63)

    def batch():
        rc = lib.fsx_batch_new(c.ptr, maps, 1, ctypes.byref(view), 1, aligned,
                               ctypes.addressof(off), ctypes.byref(out))
        if rc == 0:
            lib.fsx_batch_free(c.ptr, out)
        return rc

    def load():
        p, a = ctypes.c_void_p(), np.zeros((40, 40), np.uint32)
        rc = lib.fsx_map_new(c.ptr, ctypes.byref(p), a.ctypes.data, a.ctypes.data, 40, 40, 8, 40,
                             0.1, 0.1)
        if rc == 0:
            c.free(p.value)
        return rc

    def array():
        a = lib.futhark_new_u32_2d(c.ptr, buf, 8, 8)
        if a:
            lib.futhark_free_u32_2d(c.ptr, a)
        return int(not a)

    return {"batch": batch, "load": load, "array": array,
            "loss": lambda: lib.fsx_l2_loss(c.ptr, aligned, aligned, 16, 0, aligned, aligned),
            "render2": lambda: lib.fsx_render2(c.ptr, m, ctypes.byref(wide), aligned, 0)}


@pytest.mark.parametrize("call", ["batch", "load", "array", "loss", "render2"])
def test_pooled_buffers_are_given_back_where_memory_runs_out(lib, contexts, call):
    """A call that fits once the pool is given back succeeds, whichever way it
    allocates, and so does the next launch; one that does not fit fails alone."""
    c = contexts[0]
    m = c.map()
    call = _calls_that_allocate(lib, c, m)[call]
    c.free(c.map(side=256))                      # 1.9 MB into the pool
    _set(lib, "stub_limit", _get(lib, "stub_live") + 16)
    assert call() == 0
    assert _readers(lib, c, m)["render"]() == 0
    assert lib.futhark_context_clear_caches(c.ptr) == 0


@pytest.mark.parametrize("call", ["batch", "load", "array", "loss", "render2"])
def test_a_refused_allocation_leaves_no_error_behind(lib, contexts, call):
    c = contexts[0]
    m = c.map()
    call = _calls_that_allocate(lib, c, m)[call]
    lib.futhark_context_clear_caches(c.ptr)
    _set(lib, "stub_limit", _get(lib, "stub_live") + 16)
    assert call() == 1
    assert _readers(lib, c, m)["render"]() == 0
    assert lib.futhark_context_sync(c.ptr) == 0


def _array(lib, c, rows):
    a = lib.futhark_new_u32_2d(c.ptr, None, rows, 4)
    assert a
    lib.futhark_free_u32_2d(c.ptr, a)


def test_map_loads_leave_a_render_loop_its_buffer(lib, contexts):
    """More freed map buffers than the pool has slots, and one of the frame's
    own size, take nothing from the output arrays."""
    c = contexts[0]
    lib.futhark_context_clear_caches(c.ptr)
    _array(lib, c, 16 * 16)
    for side in (64, 65, 66, 67, 16):
        c.free(c.map(side=side))
    kept = c.map(side=16)
    mallocs = _get(lib, "stub_mallocs")
    _array(lib, c, 16 * 16)
    assert _get(lib, "stub_mallocs") == mallocs
    c.free(kept)


def test_output_arrays_of_many_sizes_keep_their_slots(lib, contexts):
    """Frames of one size more than the pool has slots, one after the other:
    all but one find their buffer again."""
    c = contexts[0]
    lib.futhark_context_clear_caches(c.ptr)
    for _ in range(2):
        mallocs = _get(lib, "stub_mallocs")
        for rows in range(1, 18):
            _array(lib, c, rows)
    assert _get(lib, "stub_mallocs") - mallocs == 1


def test_map_buffers_are_reused_up_to_the_bound(lib, contexts):
    """A load after a load of its size allocates nothing; what is kept stays
    within 256 MiB, the newest first, and goes with the caches."""
    c = contexts[0]
    lib.futhark_context_clear_caches(c.ptr)
    before = _get(lib, "stub_live")
    for side in (2048, 1024, 1024):
        mallocs = _get(lib, "stub_mallocs")
        c.free(c.map(side=side))
    assert _get(lib, "stub_mallocs") == mallocs
    for side in range(1400, 1410):
        c.free(c.map(side=side))
        assert _get(lib, "stub_live") - before <= 256 << 20
    mallocs = _get(lib, "stub_mallocs")
    c.free(c.map(side=1409))
    assert _get(lib, "stub_mallocs") == mallocs
    lib.futhark_context_clear_caches(c.ptr)
    assert _get(lib, "stub_live") == before
