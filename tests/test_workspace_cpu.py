"""The skinny GEMM's workspaces under graph capture, with the captures played
on the host: which buffer a call gets and what was filled for it."""
import pytest
import torch

from lightserve_amd import _lib
from lightserve_amd.kernels import tiled_matmul as tm

STREAM, CPU = 7, torch.device("cpu")


@pytest.fixture
def capture(monkeypatch):
    """capture(id): the stream captures from now on (0: it does not)."""
    now = [0]
    monkeypatch.setattr(_lib, "capture_id", lambda stream: now[0], raising=False)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: now[0] != 0)
    tm.release_workspaces()
    yield lambda n: now.__setitem__(0, n)
    tm.release_workspaces()


def _use(nbytes=1 << 20):
    """One product: the counters it finds, and what it leaves beside them."""
    ws = tm._workspace(CPU, STREAM, nbytes)
    assert ws.numel() >= nbytes
    return ws


def _clean(ws):
    return bool((ws[:_lib.GEMV_COUNTER_BYTES] == 0).all())


@pytest.mark.parametrize("eager_first", [True, False])
def test_a_capture_shares_with_nothing(capture, eager_first):
    if eager_first:
        assert _use() is _use()
    capture(1)
    first = _use()
    assert first is _use() and _clean(first)
    first[:_lib.GEMV_COUNTER_BYTES] = 5  # nothing that a capture records has run
    capture(2)
    second = _use()
    assert second is not first and second is _use() and _clean(second)
    second[:_lib.GEMV_COUNTER_BYTES] = 5
    capture(0)
    eager = _use()
    assert eager is not first and eager is not second and eager is _use() and _clean(eager)


def test_growth_inside_a_capture_is_filled(capture):
    capture(3)
    small = _use()
    big = _use(small.numel() + 1)
    assert big is not small and _clean(big) and big is _use()


def test_the_cache_keeps_one_workspace_per_capture_stream(capture):
    import weakref
    seen = []
    for n in range(1, 6):
        capture(n)
        seen.append(weakref.ref(_use()))
    assert [r() is not None for r in seen] == [False] * 4 + [True]
