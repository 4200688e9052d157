"""Calls on a device with little memory left: scratch that only makes a call faster (the build's
packed particles and the levels taken together, the density solve's copy in slot order, the
search's rows and packed nodes) is done without when there is no room for it, with the same
results. A first context measures what a call takes when there is room; a second one gets less."""
import contextlib
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

N = 3000000
MB = 1 << 20


@pytest.fixture(scope="module")
def gz():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from gizmo_shared_memory_amd import tree
    return tree


@pytest.fixture(scope="module")
def P(gz):
    g = torch.Generator(device="cuda").manual_seed(5)
    x, y, z = (torch.rand(N, generator=g, device="cuda", dtype=torch.float64) for _ in range(3))
    return gz.Particles(x, y, z, torch.full_like(x, 1.0 / N), torch.full_like(x, 0.01))


def _free():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


@contextlib.contextmanager
def _context(gz):
    from gizmo_shared_memory_amd import _lib as L
    ctx = gz.Context(0)
    yield ctx
    L.load().gz_ctx_destroy(ctx.handle)


@contextlib.contextmanager
def _room(bytes_left):
    """Only so much device memory free."""
    from gizmo_shared_memory_amd import _lib as L
    hip = L.load()  # (its own hipMalloc: torch would serve a piece from buffers that it holds)
    held = []
    while (more := _free() - int(bytes_left)) >= 2 * MB:  # (in pieces: all of it is not one range)
        held.append(C.c_void_p())
        assert hip.hipMalloc(C.byref(held[-1]), C.c_size_t(min(more, 1 << 35))) == 0
    try:
        yield
    finally:
        for p in held:
            assert hip.hipFree(p) == 0


@pytest.fixture(scope="module", autouse=True)
def most_of_the_device(P):
    """The tests take the rest in turn: 280 GB take seconds to allocate."""
    with _room(8000 * MB):
        yield


def _limited(gz, prepare, less):
    """call = prepare(context): its result with room, and with `less` bytes less room than it took.
    (The first of three contexts leaves torch with the buffers that the call asks it for.)"""
    out, full = [], 0
    for i, lack in enumerate([None, None, *less]):
        with _context(gz) as c:
            call = prepare(c)
            before = _free()
            with _room(full - lack) if lack else contextlib.nullcontext():
                print(f"[memory] {_free() / MB:.0f} MB free", flush=True)
                assert not lack or abs(_free() - (full - lack)) < 16 * MB
                got = call()
                if i == 1:
                    full = before - _free()
                    print(f"[memory] the call takes {full / MB:.0f} MB", flush=True)
                    assert full > max(less)
            if i:
                out.append(got)
            del call
    for got in out[1:]:
        assert all(np.array_equal(a, b) for a, b in zip(out[0], got))


def test_build_without_room_for_its_packed_particles(gz, P):
    """192 MB of packed particles, some 40 MB for the levels together."""
    def prepare(c):
        def call():
            T = gz.build(P, ctx=c)
            d = T.download()
            return [d[k] for k in sorted(d) if isinstance(d[k], np.ndarray)]
        return call
    _limited(gz, prepare, (100 * MB, 150 * MB))


def test_density_without_room_for_its_copy(gz, P):
    """96 MB of the particles in slot order."""
    def prepare(c):
        T = gz.build(P, ctx=c)
        tg = T.device_orderbuf()
        h = torch.full((N,), 0.013, dtype=torch.float64, device="cuda")
        return lambda: [v.cpu().numpy() for v in gz.density(T, P, tg, 32.0, 1.0, h_start=h)]
    _limited(gz, prepare, (64 * MB,))


def test_search_without_room_for_rows_or_nodes(gz, P):
    """732 MB of rows, some 22 MB of nodes."""
    def prepare(c):
        T = gz.build(P, ctx=c)
        at = T.device_orderbuf().view(torch.int32).long()
        q = torch.stack([P.x[at], P.y[at], P.z[at]], 1).contiguous()
        r = torch.full((N,), 0.01, dtype=torch.float64, device="cuda")
        return lambda: [v.view(torch.int32 if v.dtype == torch.uint32 else v.dtype).cpu().numpy()
                        for v in gz.ngb_search(T, q, r)]
    _limited(gz, prepare, (400 * MB, 742 * MB))
