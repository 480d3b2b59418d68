"""The blocks a context keeps between particle steps, on a device allocator that the test bounds from the host."""
import ctypes as C
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
MIB = 1 << 20

# the host layer with an allocator of `room` bytes instead of the device's
SOURCE = r"""
#include "%s/earthbyte_underworld_amd/host/ust_context.c"
size_t room;
static struct { void *p; size_t n; } held[256];
int ust_dev_malloc(void **p, size_t bytes) {
    *p = NULL;
    if (bytes > room) return UST_ENOMEM;
    for (int i = 0; i < 256; i++)
        if (!held[i].p) {
            *p = held[i].p = malloc(1);
            held[i].n = bytes;
            room -= bytes;
            return UST_OK;
        }
    return UST_ENOMEM;
}
int ust_dev_free(void *p) {
    for (int i = 0; p && i < 256; i++)
        if (held[i].p == p) {
            room += held[i].n;
            held[i].p = NULL;
            free(p);
        }
    return UST_OK;
}
int ust_k_fill_f64(double *x, double v, size_t n, void *stream) { return UST_OK; }
ust_context *make(int np) {
    ust_context *ctx = (ust_context *)calloc(1, sizeof(*ctx));
    ctx->np = np;
    return ctx;
}
size_t idle(ust_context *ctx) { return ctx->pool_idle; }
int take(ust_context *ctx, void **p, size_t bytes) { return swarm_malloc(ctx, p, bytes); }
void give(ust_context *ctx, void **p) { swarm_free(ctx, p); }
int other(ust_context *ctx, void **p, size_t bytes) { return ust_dev_alloc_zero(ctx, p, bytes); }
"""


@pytest.fixture(scope="module")
def pool(tmp_path_factory):
    from earthbyte_underworld_amd import _lib
    d = tmp_path_factory.mktemp("pool")
    src, so = str(d / "pool.c"), str(d / "pool.so")
    with open(src, "w") as f:
        f.write(SOURCE % ROOT)
    here = os.path.dirname(_lib.LIB_PATH)
    subprocess.run(["gcc", "-std=gnu11", "-O1", "-shared", "-fPIC", "-Wl,-Bsymbolic", "-w", f"-I{ROOT}/include",
                    f"-I{ROOT}/earthbyte_underworld_amd/host", src, "-o", so, f"-L{here}", "-l:libust.so",
                    f"-Wl,-rpath,{here}"], check=True)
    _lib.load()
    lib = C.CDLL(so)
    lib.make.restype = C.c_void_p
    lib.idle.restype = C.c_size_t
    lib.idle.argtypes = [C.c_void_p]
    for f in (lib.take, lib.other):
        f.argtypes = [C.c_void_p, C.POINTER(C.c_void_p), C.c_size_t]
    lib.give.argtypes = [C.c_void_p, C.POINTER(C.c_void_p)]
    return lib


@pytest.mark.parametrize("kind,size", [("other", 60 * MIB), ("other", 8), ("take", MIB // 2), ("take", 60 * MIB)])
def test_idle_blocks_make_room_for_any_allocation(pool, kind, size):
    """64 MiB of a swarm step's blocks are idle in 100 MiB when the context asks for memory that only they leave room for: a
    solver's or an operator's array (60 MiB; 8 bytes, where nothing is left), a small or a large one of the next step."""
    room = C.c_size_t.in_dll(pool, "room")
    room.value = 100 * MIB
    ctx, p, q, rest = pool.make(1000000), C.c_void_p(), C.c_void_p(), C.c_void_p()
    assert pool.take(ctx, C.byref(p), 60 * MIB) == 0  # and a sixteenth more
    pool.give(ctx, C.byref(p))
    kept = pool.idle(ctx)
    assert kept == 60 * MIB // 16 * 17 and room.value == 100 * MIB - kept
    if size < MIB:
        assert pool.other(ctx, C.byref(rest), room.value) == 0 and room.value == 0
    elif kind == "take":  # larger than the idle block by more than the pool hands out
        size = 70 * MIB
    rc = getattr(pool, kind)(ctx, C.byref(q), size)
    assert rc == 0 and q.value and pool.idle(ctx) == 0


def test_refused_when_no_room_is_left_with_the_pool_empty(pool):
    room = C.c_size_t.in_dll(pool, "room")
    room.value = 10 * MIB
    ctx, q = pool.make(1000000), C.c_void_p()
    for f in (pool.take, pool.other):
        assert f(ctx, C.byref(q), 11 * MIB) == -3 and not q.value
    assert room.value == 10 * MIB
    assert pool.take(ctx, C.byref(q), 10 * MIB) == 0  # the exact size where a sixteenth more does not fit
    pool.give(ctx, C.byref(q))
    assert room.value == 10 * MIB
