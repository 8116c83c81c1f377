"""The host side of a short pass through a MoE layer on a library that notes its calls (no GPU): what happens to its buffers when
a call fails, and how the pool lets its workspaces go."""
import ctypes as C
import threading

import pytest


class Library:
    """Every entry point returns 0 (or what FAILS says); memory is numbers."""

    def __init__(self, fails=()):
        self.fails, self.log, self.held, self.next = dict(fails), [], set(), 0x1000

    def __getattr__(self, name):
        def f(*args):
            self.log.append(name)
            if name.endswith("_workspace"):
                return 4096
            if self.fails.get(name):
                return self.fails[name]
            if name == "ilt_malloc":
                args[0]._obj.value = self.next
                self.held.add(self.next)
                self.next += 0x1000
            if name == "ilt_free":
                self.held.remove(args[0].value)
            if name == "ilt_error_string":
                return b"made to fail"
            return 0
        return f


@pytest.fixture
def setting(monkeypatch):
    from illatio_amd import ds4f, hip

    def make(**fails):
        lib = Library(fails)
        monkeypatch.setattr(hip, "_lib", lib)
        dev = hip.Device(0, hip.DeviceInfo(), 0)
        pool = object.__new__(ds4f.ExpertPool)
        pool.dev, pool.d, pool.ff, pool._spare, pool._lock = dev, 256, 256, [], threading.Lock()
        pool.pool = pool.ptrs = None
        pool.host_buf = 0
        monkeypatch.setattr(ds4f, "step_weights", lambda pool, sh: C.c_int(0))
        b = hip.DBuf(0x100, 4096, dev)
        return lib, pool, lambda: ds4f.ffn_small(dev, pool, None, b, b, 3, 8, 2, 1.5, 0.0)
    return make


def test_the_workspace_is_kept_and_the_result_handed_over(setting):
    lib, pool, call = setting()
    first = call()
    second = call()
    assert len(pool._spare) == 1 and lib.held == {first.ptr, second.ptr, pool._spare[0].ptr}
    pool.free()
    assert lib.held == {first.ptr, second.ptr} and not pool._spare


@pytest.mark.parametrize("where", ["ilt_d4_ffn_small", "ilt_stream_sync"])
def test_a_failed_call_leaves_no_buffer_and_waits_before_it_frees(setting, where):
    from illatio_amd import hip
    lib, pool, call = setting(**{where: 1})
    with pytest.raises(hip.HipError):
        call()
    assert not lib.held and not pool._spare
    last = lib.log[lib.log.index("ilt_d4_ffn_small") + 1:]
    assert last.index("ilt_stream_sync") < last.index("ilt_free")


def test_a_failed_allocation_leaves_no_buffer(setting):
    from illatio_amd import hip
    lib, pool, call = setting()
    real, count = lib.__getattr__, []

    def second_fails(name):
        f = real(name)
        if name != "ilt_malloc":
            return f
        count.append(1)
        return f if len(count) == 1 else lambda *a: 2
    lib.__class__ = type("Failing", (Library,), {"__getattr__": lambda self, name: second_fails(name)})
    with pytest.raises(hip.HipError):
        call()
    assert lib.held == {b.ptr for b in pool._spare}


def test_free_takes_the_pools_lock(setting):
    lib, pool, call = setting()
    call()
    taken = []

    class Lock:
        def __enter__(self): taken.append(len(pool._spare))
        def __exit__(self, *a): pass
    pool._lock = Lock()
    pool.free()
    assert taken == [1] and not pool._spare
