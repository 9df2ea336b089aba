"""The binding's layout check accepts and refuses what looking at the slices
does, and the spans of a prompt pass are every row's window (no GPU)."""
import random

import numpy as np
import pytest
import torch

import needle_amd as nd


class OnDevice:
    """A CPU tensor that says it is on the device."""
    is_cuda = True

    def __init__(self, t):
        self.t = t

    def __getattr__(self, name):
        return getattr(self.t, name)

    def __getitem__(self, i):
        return self.t[i]


def _by_slices(t, numel, rows):
    if rows:
        ok = t.dim() == 0 or all(t[i].is_contiguous() for i in range(min(t.shape[0], 1)))
        if t.dim() > 1:
            ok = ok and t.stride(0) >= t[0].numel()
    else:
        ok = t.is_contiguous()
    return t.data_ptr() if ok and t.numel() >= numel else ValueError


def _outcome(f):
    try:
        return f()
    except (ValueError, IndexError) as e:
        return type(e)


def test_layout_check_over_shapes_and_strides():
    r = random.Random(1)
    for _ in range(20000):
        dims = r.randint(0, 4)
        shape = [r.choice([0, 1, 1, 2, 3, 4]) for _ in range(dims)]
        strides = [r.choice([0, 1, 2, 3, 4, 6, 8, 12, 24]) for _ in range(dims)]
        if r.random() < 0.6:  # contiguous, or but for its first stride
            strides, step = [0] * dims, 1
            for i in reversed(range(dims)):
                strides[i], step = step, step * max(shape[i], 1)
            if dims and r.random() < 0.5:
                strides[0] = max(0, strides[0] + r.choice([-1, 1, 5]))
        t = torch.empty(1000).as_strided(shape, strides)
        rows, numel = r.random() < 0.5, r.choice([0, 3, 24])
        want = _outcome(lambda: _by_slices(t, numel, rows))
        got = _outcome(lambda: nd._arg(OnDevice(t), torch.float32, "t", numel, rows))
        assert got == want, (shape, strides, rows, numel)


@pytest.fixture
def seen(monkeypatch):
    """What a prompt pass would hand to the cache and the attention."""
    seen = {}
    monkeypatch.setattr(nd, "_torch", lambda: torch)
    monkeypatch.setattr(nd, "kv_alloc", lambda g, n, device: (torch.zeros(1, dtype=torch.uint8), 1))
    monkeypatch.setattr(nd, "kv_write", lambda ctx, g, kv, stride, pos, k, v: seen.update(pos=pos))
    monkeypatch.setattr(nd, "attend_step_i8",
                        lambda ctx, g, kv, stride, lo, hi, *rest: seen.update(lo=lo, hi=hi))
    return seen


def test_prompt_spans(seen):
    for seq in range(20):
        for window in (0, 1, 2, 5, 19, 20, 21, 64):
            x = torch.zeros(seq, 16)
            nd.attend_i8_prefill(None, 1, 1, 16, 16, x, x, x, window=window)
            t = torch.arange(seq, dtype=torch.int32)
            assert torch.equal(seen["pos"], t) and torch.equal(seen["hi"], t)
            lo = torch.clamp(t + 1 - window, min=0) if window else torch.zeros_like(t)
            assert torch.equal(seen["lo"], lo) and seen["lo"].dtype == torch.int32
            assert seen["lo"].is_contiguous() and seen["hi"].is_contiguous()


@pytest.mark.parametrize("window", [None, False, -1, -7, 5.0, 2.5, 64.0, -2.0, np.int64(5), np.float32(3.0),
                                    torch.tensor(5), torch.tensor([3])])
def test_prompt_spans_of_any_number(seen, window):
    """A window is any number, or None for the whole prompt: spans as from
    row + 1 - window, a fraction cut off."""
    for seq in (1, 7, 20):
        x = torch.zeros(seq, 16)
        nd.attend_i8_prefill(None, 1, 1, 16, 16, x, x, x, window=window)
        t = torch.arange(seq, dtype=torch.int32)
        lo = torch.clamp(t + 1 - window, min=0).to(torch.int32) if window else torch.zeros_like(t)
        assert torch.equal(seen["lo"], lo) and torch.equal(seen["hi"], t)
        assert seen["lo"].dtype == seen["hi"].dtype == torch.int32
