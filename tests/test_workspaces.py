"""The workspace tables of bitnet_tt._native, on the CPU (the device calls are
replaced): growth and release against other threads, finalizers and
check_errors, and the error words of workspaces that are gone."""

import gc
import threading
import types

import pytest
import torch

from bitnet_tt import _native as N

DEV = torch.device("cuda", 0)


class Owner:
    pass


@pytest.fixture(autouse=True)
def tables(monkeypatch):
    """Empty tables, one stream, host memory for device memory."""
    for name in ("_workspaces", "_fast", "_error_words", "_prepared_for", "_reset_hooks"):
        monkeypatch.setattr(N, name, {})
    for name in ("_retired", "_late_errors"):
        monkeypatch.setattr(N, name, [], raising=False)
    zeros = torch.zeros
    monkeypatch.setattr(torch, "zeros", lambda *a, device=None, **k: zeros(*a, **k))
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: types.SimpleNamespace(cuda_stream=7))
    monkeypatch.setattr(torch.cuda, "synchronize", lambda device=None: None)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)


def set_word(buf, off):
    buf[off] = 1


def test_error_word_of_a_released_owner_is_still_raised():
    o = Owner()
    n = N.owner_id(o)
    set_word(N.workspace(DEV, 64, "step", 16, n), 16)
    del o
    gc.collect()
    assert not N._workspaces
    with pytest.raises(RuntimeError, match="step workspace .* word at byte 16 = 1"):
        N.check_errors(DEV)
    N.check_errors(DEV)
    assert not N._retired


def test_error_word_of_a_replaced_workspace_is_still_raised():
    set_word(N.workspace(DEV, 64, "bitlinear", 16), 16)
    buf = N.workspace(DEV, 4 << 20, "bitlinear", 16)
    with pytest.raises(RuntimeError, match="bitlinear workspace"):
        N.check_errors(DEV)
    assert N.workspace(DEV, 64, "bitlinear", 16) is buf
    N.check_errors(DEV)


def test_retired_workspaces_are_bounded():
    for i in range(3 * N._RETIRED_MAX):
        o = Owner()
        buf = N.workspace(DEV, 64, "step", 16, N.owner_id(o))
        if i == 1:
            set_word(buf, 16)
        del o, buf
        gc.collect()
        assert len(N._retired) <= N._RETIRED_MAX + 1
    with pytest.raises(RuntimeError, match="step workspace"):
        N.check_errors(DEV)
    N.check_errors(DEV)


def test_owner_released_during_check_errors(monkeypatch):
    owners = [Owner() for _ in range(8)]
    bufs = [N.workspace(DEV, 64, "step", 16, N.owner_id(o)) for o in owners]
    set_word(bufs[3], 16)
    monkeypatch.setattr(torch.cuda, "synchronize", lambda device=None: (owners.clear(), gc.collect()))
    with pytest.raises(RuntimeError, match="step workspace"):
        N.check_errors(DEV)
    assert not N._workspaces


def test_owner_released_while_the_tables_are_held():
    o, other = Owner(), Owner()
    n = N.owner_id(o)
    N.workspace(DEV, 64, "step", 16, n)
    with N._ws_lock:
        before = dict(N._workspaces)
        del o
        gc.collect()
        assert N._workspaces == before  # not under the reader's feet
    N.workspace(DEV, 64, "step", 16, N.owner_id(other))
    assert not [k for k in N._workspaces if k[3] == n]


def test_growth_against_a_lookup(monkeypatch):
    """A lookup that another thread's growth overtakes does not bring the old
    buffer back."""
    old = N.workspace(DEV, 64, "bitlinear", 16)
    grown = threading.Event()
    started = []

    def grow():
        N.workspace(DEV, 4 << 20, "bitlinear", 16)
        grown.set()

    class Words(dict):
        def setdefault(self, *a):
            if not started:
                started.append(threading.Thread(target=grow))
                started[0].start()
                grown.wait(0.3)
            return super().setdefault(*a)

    monkeypatch.setattr(N, "_error_words", Words(N._error_words))
    N.workspace_ptr(0, 64, "bitlinear", 16, 7)
    started[0].join()
    hit = N.workspace_ptr(0, 64, "bitlinear", 16, 7)
    assert hit[1] == 4 << 20 and hit[0] != old.data_ptr()
    assert hit[2] is N._workspaces[("bitlinear", "cuda:0", 7)]


def test_stream_of_takes_what_current_stream_takes(monkeypatch):
    """None and indexless devices mean the current device, as for
    torch.cuda.current_stream; what that refuses is refused."""
    seen = []

    def current_stream(device=None):
        if device is not None and torch.device(device).type != "cuda":
            raise ValueError("not a GPU")
        seen.append(device)
        return types.SimpleNamespace(cuda_stream=9)

    monkeypatch.setattr(torch.cuda, "current_stream", current_stream)
    monkeypatch.setattr(N, "_raw_stream", lambda index: 100 + index)
    for device in (None, "cuda", torch.device("cuda"), 0):
        assert N.stream_of(device).value == 9
    assert seen == [None, "cuda", torch.device("cuda"), 0]
    assert N.stream_of(torch.device("cuda", 1)).value == 101
    with pytest.raises(ValueError):
        N.stream_of(torch.device("cpu"))
