"""libql_dns.so's host code without a GPU: what it does when a runtime call fails,
what it allocates and waits for, and which launch shapes it takes.  The library
runs on tests/cpp/hip_on_host.cpp, which serves its HIP calls from host memory
(kernels do nothing) and makes chosen ones fail.  Every scenario runs in a
process of its own."""
import ctypes
import os
import subprocess
import sys

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def runtime(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("hip_on_host") / "hip_on_host.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-Wall", "-Werror", "-o", so,
                    os.path.join(HERE, "cpp", "hip_on_host.cpp")], check=True)
    return so


def scenario(runtime, name, *args):
    r = subprocess.run([sys.executable, os.path.abspath(__file__), runtime, name] + [str(a) for a in args],
                       stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
    assert r.returncode == 0 and "scenario done" in r.stdout, r.stdout


# ---------------------------------------------------------------------------
# in the scenario's process
# ---------------------------------------------------------------------------
class Host:
    """The stand-in runtime's controls."""

    def __init__(self, so):
        # ahead of the library's own dependencies in symbol lookup
        self.L = ctypes.CDLL(so, mode=ctypes.RTLD_GLOBAL)
        for f in ("hoh_live", "hoh_limit"):
            getattr(self.L, f).restype = ctypes.c_size_t
        for f in ("hoh_races", "hoh_bad", "hoh_null_waits", "hoh_mallocs", "hoh_host_live", "hoh_sizes"):
            getattr(self.L, f).restype = ctypes.c_long
        for f in ("hoh_fail_malloc", "hoh_fail_host", "hoh_fail_new"):
            getattr(self.L, f).argtypes = [ctypes.c_long]
        self.L.hoh_limit.argtypes = [ctypes.c_size_t]
        self.L.hoh_sizes.argtypes = [ctypes.POINTER(ctypes.c_size_t), ctypes.c_long]

    def __getattr__(self, name):
        f = getattr(self.L, "hoh_" + name)
        setattr(self, name, f)
        return f

    def sizes(self):
        n = self.L.hoh_sizes(None, 0)
        a = (ctypes.c_size_t * n)()
        self.L.hoh_sizes(a, n)
        return list(a)

    def clean(self):
        """No copy outside its buffer and none that a late clearing could undo."""
        assert self.bad() == 0 and self.races() == 0, (self.bad(), self.races())


def _state(c, seed=3):
    rng = np.random.default_rng(seed)
    lin = rng.standard_normal((c.nxy, c.nLin, c.nz)) + 1j * rng.standard_normal((c.nxy, c.nLin, c.nz))
    lin[::c.params.NY // 2, 0::2, 0] = 0
    return lin, rng.standard_normal((c.nMF, c.nz)) + 0j


def _context(**kw):
    from ql_dns_amd.capi import QLContext
    from ql_dns_amd.params import QLParams
    kw.setdefault("NX", 8)
    kw.setdefault("NY", 6)
    kw.setdefault("NZ", 32)
    c = QLContext(QLParams(**kw))
    c.set_state(*_state(c))
    c.linear_ops_init(0.0)
    return c


def _fails(f, *args):
    from ql_dns_amd.capi import QLError
    try:
        f(*args)
    except QLError as e:
        assert e.code == -2 and "out of memory" in str(e), e
        return True
    return False


def _fails_state(f, *args):
    from ql_dns_amd.capi import QL_ERR_STATE, QLError
    try:
        f(*args)
    except QLError as e:
        return e.code == QL_ERR_STATE
    return False


def s_error_is_reported_once(host):
    c = _context()
    c.adjoint_forward(4, 2, 0.0)
    host.fail_malloc(1)
    assert _fails(c.adjoint_backward)
    # the calls after it launch kernels and check for their errors, not for an old one
    c.steps(3)
    c.get_state()


def _gradient(c, n=7, every=3):
    c.adjoint_forward(n, every, 0.0)
    c.adjoint_backward()


def _noisy_context(model):
    c = _context(model=model, NZ=64)
    c.set_noise(2.0)  # the driven step's buffer among the segment's
    return c


def s_backward_buffers(host, model):
    # the allocations of a backward, and what is allocated after one
    c = _noisy_context(model)
    c.adjoint_forward(7, 3, 0.0)
    n0 = host.mallocs()
    c.adjoint_backward()
    nalloc, sizes = host.mallocs() - n0, host.sizes()
    c.close()
    assert nalloc > 10 and host.live() == 0
    for k in range(1, nalloc + 1):
        c = _noisy_context(model)
        c.adjoint_forward(7, 3, 0.0)
        host.fail_malloc(k)
        assert _fails(c.adjoint_backward), k
        c.adjoint_backward()  # the same backward again, with memory to be had
        assert host.sizes() == sizes, k
        _gradient(c)
        assert host.sizes() == sizes, k
        c.close()
        assert host.live() == 0 and host.host_live() == 0, k
    host.clean()


def s_checkpoints(host):
    c = _context()
    n0 = host.mallocs()
    c.adjoint_forward(7, 2, 0.0)
    nalloc, sizes = host.mallocs() - n0, host.sizes()
    c.close()
    assert nalloc > 15 and host.live() == 0
    for k in range(1, nalloc + 1):
        c = _context()
        host.fail_malloc(k)
        assert _fails(c.adjoint_forward, 7, 2, 0.0), k
        assert _fails_state(c.adjoint_backward), k  # no forward has completed
        c.adjoint_forward(7, 2, 0.0)
        assert host.sizes() == sizes, k
        c.adjoint_backward()
        c.close()
        assert host.live() == 0, k
    host.clean()


def s_room_for_checkpoints(host):
    c = _context()
    c.adjoint_forward(40, 2, 0.0)
    need = host.live()
    c.close()
    c = _context()
    _gradient(c, 4, 2)
    host.limit(need)  # just what the forward takes on a new context
    c.adjoint_forward(40, 2, 0.0)
    assert host.live() <= need
    host.limit(1 << 40)
    c.adjoint_backward()
    c.close()
    assert host.live() == 0
    host.clean()


def _refused(f, *args):
    from ql_dns_amd.capi import QLError
    try:
        f(*args)
    except QLError as e:
        return e.code == -1
    return False


def s_transform_on_default_shape(host):
    from ql_dns_amd.capi import QLBatch
    from ql_dns_amd.params import QLParams
    for model in (0, 1, 2):
        for NZ in (32, 64):
            c = _context(model=model, NZ=NZ)
            before = c.config()[0]
            assert before["line"] == 64 and before["transform"] == 0
            c.set_transform(NZ, 1)
            assert c.config()[0]["transform"] == 1 and c.config()[0]["line"] == 256
            c.steps(2)
            c.set_transform(NZ, 0)
            assert c.config()[0] == before
            # a shape that was asked for stays
            c.set_config(NZ, 64, 128)
            assert _refused(c.set_transform, NZ, 1)
            assert c.config()[0]["line"] == 64 and c.config()[0]["transform"] == 0
            c.set_config(NZ, 128, 512)
            c.set_transform(NZ, 1)
            c.set_transform(NZ, 0)
            assert c.config()[0]["line"] == 128 and c.config()[0]["transform"] == 0
            c.close()
    b = QLBatch([QLParams(NX=8, NY=8, NZ=NZ) for NZ in (32, 64, 64)])
    b.set_transform(64, 1)
    assert [g["transform"] for g in b.config()] == [0, 1] and [g["line"] for g in b.config()] == [64, 256]
    b.close()
    for kw in (dict(NZ=128), dict(NZ=32, precision=1)):
        assert _refused(_context(**kw).set_transform, kw["NZ"], 1)


def s_large_boxes(host):
    from ql_dns_amd.capi import QLContext
    from ql_dns_amd.params import QLParams
    for model, NX, line in ((2, 160, 64), (2, 176, 256), (1, 176, 64), (1, 350, 256), (0, 176, 64), (0, 350, 64)):
        c = QLContext(QLParams(model=model, NX=NX, NY=NX, NZ=64))
        assert c.config()[0]["line"] == line, (model, NX)
        assert c.config()[0]["tail"] == (1 if line == 64 else 0)  # 256 workgroups, or 512
        c.close()


def s_tail_follows_the_shape(host):
    from ql_dns_amd.params import QLParams
    c = _context(NX=36, NY=60, NZ=64)

    def tail(line, target):
        c.set_config(64, line, target)
        g = c.config()[0]
        return g["tail"], g["workgroups"] * 64

    start = c.config()[0]
    assert start["tail"] == 1
    # one launch up to 16384 / NZ rows, two above, whatever the shape before
    for line, target in ((64, 256), (256, 512), (128, 4096), (64, 256), (64, 1 << 30), (128, 256), (64, 512)):
        t, rows = tail(line, target)
        assert t == (1 if rows <= 16384 else 0), (line, target, rows)
    # a tail that was asked for stays as far as it fits (65536 / NZ rows)
    c.set_tail(64, 1)
    assert tail(64, 512)[0] == 1 and tail(64, 1 << 30)[0] == 0 and tail(64, 512)[0] == 1
    c.set_tail(64, 0)
    assert tail(64, 256)[0] == 0
    c.close()
    # never by rule: variable steps, larger sets, mixed precision, NZ above 64
    for kw in (dict(NZ=64, dt=-0.01), dict(NZ=64, precision=1), dict(NZ=128)):
        c = _context(**kw)
        c.set_config(kw["NZ"], 64, 64)
        assert c.config()[0]["tail"] == 0
        c.close()
    from ql_dns_amd.capi import QLBatch
    b = QLBatch([QLParams(NX=8, NY=8, NZ=32)] * 5)
    b.set_config(32, 64, 64)
    assert b.config()[0]["tail"] == 0
    b.close()


def s_creation(host):
    from ql_dns_amd.capi import QLBatch, QLContext
    from ql_dns_amd.params import QLParams
    for kw in (dict(NX=16, NY=16, NZ=32), dict(NX=64, NY=64, NZ=256), dict(NX=16, NY=16, NZ=64, precision=1)):
        n = host.null_waits()
        c = QLContext(QLParams(**kw))
        assert host.null_waits() - n <= 2, host.null_waits() - n  # clearings in one wait, and the launch table's
        assert host.host_live() == 0  # pinned memory with the first result that takes it
        c.set_state(*_state(c))
        c.steps(1)
        assert host.host_live() == 0
        c.get_state()
        assert host.host_live() == 1
        c.get_state()
        assert host.host_live() == 1
        d = QLContext(QLParams(**kw))
        d.get_state()
        assert host.host_live() == 1  # the next handle's results take what is there
        c.close()
        c = d
        c.diagnostics(0.0)
        assert host.host_live() <= 2
        host.clean()
        c.close()
        assert host.live() == 0 and host.host_live() == 0  # and it goes with the last
    n = host.null_waits()
    b = QLBatch([QLParams(NX=8, NY=8, NZ=(32, 64, 128)[k % 3]) for k in range(12)])
    assert host.null_waits() - n <= 4
    b.steps(1)
    host.clean()
    # a shape with more workgroups than the set was created with: its buffers are cleared before they are used
    n = host.null_waits()
    b.set_config(64, 64, 1 << 30)
    b.steps(1)
    assert host.null_waits() - n <= 1
    host.clean()
    b.close()


def _downloads(c, lin, mf, kx0, before=lambda: None, after=lambda: None):
    """get_state with nothing but the call itself between before() and after()."""
    from ql_dns_amd.capi import _dp
    got = np.zeros_like(lin), np.zeros_like(mf), np.zeros_like(kx0)
    args = [c._h] + [_dp(a) for a in got]
    before()
    rc = c._L.ql_get_state(*args)
    after()
    c._check(rc)
    for a, b in zip(got, (lin, mf, kx0)):
        assert np.array_equal(a, b)


def s_downloads(host, NX, NZ, model):
    from ql_dns_amd.ic import mode_tables
    from ql_dns_amd.params import QLParams
    kw = dict(NX=NX, NY=NX, NZ=NZ, model=model)
    kx0 = mode_tables(QLParams(**kw))[0]
    c = _context(**kw)
    lin, mf = _state(c)
    for _ in range(3):
        _downloads(c, lin, mf, kx0)
    # no memory for what the copying takes on the host, a thread's start included
    for k in range(1, 13):
        _downloads(c, lin, mf, kx0, lambda: host.fail_new(k), lambda: host.fail_new(0))
    c.close()
    # no pinned memory, at the first result and after
    c = _context(**kw)
    held = host.host_live()
    for k in range(3):
        host.fail_host(1)
        _downloads(c, lin, mf, kx0)
    assert host.host_live() == held
    host.fail_host(0)
    c.steps(1)  # and the failure is not reported by a later call
    c.close()
    assert host.host_live() == 0
    host.clean()


def s_shape_without_memory(host, precision):
    c = _context(NX=36, NY=60, NZ=64, precision=precision)
    before, sizes = c.config(), host.sizes()
    n0 = host.mallocs()
    c.set_config(64, 128, 1 << 30)
    nalloc = host.mallocs() - n0
    after = c.config()
    c.close()
    assert nalloc == 3 and after != before
    for k in range(1, nalloc + 1):
        c = _context(NX=36, NY=60, NZ=64, precision=precision)
        host.fail_malloc(k)
        assert _fails(c.set_config, 64, 128, 1 << 30), k
        assert c.config() == before and host.sizes() == sizes, k  # the shape it had, buffers and all
        c.steps(1)
        c.set_config(64, 128, 1 << 30)
        assert c.config() == after
        c.close()
    host.clean()
    assert host.live() == 0


def s_tune_without_memory(host):
    from ql_dns_amd.capi import QLBatch
    from ql_dns_amd.params import QLParams
    ps = [QLParams(NX=8, NY=6, NZ=32), QLParams(NX=20, NY=20, NZ=64)]
    states = []
    for r, p in enumerate(ps):
        c = _context(NX=p.NX, NY=p.NY, NZ=p.NZ)
        states.append(_state(c, r))
        c.close()
    b = QLBatch(ps)
    shape = b.config()[1]
    n = host.mallocs()
    b.tune(1)
    n = host.mallocs() - n  # five buffers per group, and those of larger shapes
    assert n > 10
    b.close()
    for k in range(0, n + 1):
        b = QLBatch(ps)
        for r, st in enumerate(states):
            b.set_state(r, *st)
        live = host.live()
        if k:
            host.fail_malloc(k)
            assert _fails(b.tune, 1), k
            assert host.live() >= live and (host.live() == live or k > 10), k
            assert b.config()[1] == shape, k
            b.set_transform(64, 1)  # the shape is still nobody's
            b.set_transform(64, 0)
            assert b.config()[1] == shape, k
        else:
            b.tune(1)
        for r, (lin, mf) in enumerate(states):
            l, m, _ = b.get_state(r)
            assert np.array_equal(l, lin) and np.array_equal(m, mf), (k, r)
        b.close()
    host.clean()


def s_gradient_waits(host):
    c = _noisy_context(0)
    c.adjoint_forward(4, 2, 0.0)
    n = host.null_waits()
    c.adjoint_backward()
    assert host.null_waits() - n <= 2
    n = host.null_waits()
    c.adjoint_forward(6, 1, 0.0)  # four checkpoints more
    assert host.null_waits() - n <= 4
    c.adjoint_backward()
    host.clean()
    c.close()


def s_threads(host):
    from threading import Thread
    cs = [_context(NX=NX, NY=NX, NZ=NZ) for NX, NZ in ((6, 32), (34, 256), (34, 256), (70, 256), (24, 256), (8, 64))]
    want = [c.get_state() for c in cs]
    bad = []

    def work(k):
        for _ in range(12):
            if not all(np.array_equal(a, b) for a, b in zip(cs[k].get_state(), want[k])):
                bad.append(k)

    ts = [Thread(target=work, args=(k % len(cs),)) for k in range(2 * len(cs))]  # two threads per context
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
    for n, c in enumerate(cs):
        assert 1 <= host.host_live() <= 4
        c.close()
    assert host.host_live() == 0
    host.clean()


# ---------------------------------------------------------------------------
def test_gradients_wait_once_per_group_of_buffers(runtime):
    scenario(runtime, "gradient_waits")


def test_downloads_of_several_threads(runtime):
    """Threads on one context take turns, threads on several have memory of their own."""
    scenario(runtime, "threads")


def test_tuning_there_is_no_memory_for_keeps_the_state(runtime):
    """And the launch shapes."""
    scenario(runtime, "tune_without_memory")


@pytest.mark.parametrize("precision", [0, 1])
def test_a_shape_there_is_no_memory_for_changes_nothing(runtime, precision):
    scenario(runtime, "shape_without_memory", precision)


@pytest.mark.parametrize("NX,NZ,model", [(6, 32, 0), (34, 256, 0), (34, 256, 2), (70, 256, 0), (70, 256, 2)])
def test_results_arrive_whole_or_without_an_exception(runtime, NX, NZ, model):
    """States of one piece, of a few and of more than there are slots, in both
    layouts: the same values whatever the host has no memory for."""
    scenario(runtime, "downloads", NX, NZ, model)


def test_creation_waits_once_and_pins_nothing(runtime):
    """A new context waits for the clearing of its buffers as a whole, not for each
    (30 waits took 0.24 ms of a small context's 0.6), and has no pinned memory."""
    scenario(runtime, "creation")


def test_default_shapes_of_large_boxes(runtime):
    """At NZ = 64 large boxes of HD_fullU and MHD_BQlin are faster on the workgroup kernel."""
    scenario(runtime, "large_boxes")


def test_default_tail_follows_the_shape(runtime):
    """The one-launch tail a set has by default is a matter of the shape it has now,
    not of the one it was created with."""
    scenario(runtime, "tail_follows_the_shape")


def test_matrix_core_transform_on_a_default_shape(runtime):
    """ql_batch_set_transform takes a set no shape was asked for: it moves to the
    workgroup kernel, which has the variant, and back."""
    scenario(runtime, "transform_on_default_shape")


def test_longer_forward_after_a_gradient_takes_no_more_memory(runtime):
    """The buffers an earlier backward left make way for checkpoints."""
    scenario(runtime, "room_for_checkpoints")


def test_forward_after_a_failed_allocation(runtime):
    """Whichever buffer of a checkpoint could not be had, the next forward on the
    context finds all of them."""
    scenario(runtime, "checkpoints")


@pytest.mark.parametrize("model", [0, 1, 2])
def test_backward_after_a_failed_allocation(runtime, model):
    """Whichever of a gradient's buffers could not be had, the same backward and
    the next gradient find all of them, and none is lost."""
    scenario(runtime, "backward_buffers", model)


def test_a_failed_allocation_is_reported_once(runtime):
    scenario(runtime, "error_is_reported_once")


if __name__ == "__main__":
    sys.path.insert(0, os.path.dirname(HERE))
    host_ = Host(sys.argv[1])
    globals()["s_" + sys.argv[2]](host_, *[int(a) for a in sys.argv[3:]])
    print("scenario done")
