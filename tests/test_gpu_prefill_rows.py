"""Prefill passes of many rows (several rows a workgroup in the MLP, gates of
four rows a wave, shared attention tiles) against stepping, bit for bit: row
counts on both sides of each change of kernel, ragged in every tile.

The 4-layer geometry has a 32-position window, so the local rings wrap, and
one global layer."""
import numpy as np
import pytest
import torch

import needle_amd as nd
import v3_synth as S

pytestmark = pytest.mark.gpu


def _bits(a):
    return a.cpu().numpy().view(np.uint32)


@pytest.fixture(scope="module")
def small(ctx):
    g, recs = S.build_records({**S.small_geometry(4), "max_seq_len": 4096}, seed=33)
    return nd.V3Model(ctx, g, recs, S.CODEBOOK)


@pytest.mark.parametrize("kv_int8", [True, False])
@pytest.mark.parametrize("sessions,passes", [
    (1, [1, 5]), (16, [16]), (1, [256, 3]), (3, [86, 2]), (2, [255, 1, 40]), (4, [129]), (7, [101, 7]),
    (5, [205, 30]), (13, [79, 33]), (8, [64] * 35)])
def test_pass_equals_stepping(small, sessions, passes, kv_int8):
    n = sum(passes)
    prompts = np.stack([S.prompt_tokens(n, 90 + i) for i in range(sessions)]).astype(np.int32)
    ref = nd.V3Batch(small, sessions, max_len=n + 3, kv_int8=kv_int8)
    got = nd.V3Batch(small, sessions, max_len=n + 3, max_chunk=max(passes), kv_int8=kv_int8)
    lr = torch.empty(sessions, small.rows, device="cuda")
    lg = torch.empty(sessions, small.rows, device="cuda")
    t = 0
    for c in passes:
        for k in range(t, t + c):
            ref.step(prompts[:, k], logits=lr, want_next=k == t + c - 1)
        got.prefill(prompts[:, t:t + c], logits=lg)
        t += c
        assert np.array_equal(_bits(lr), _bits(lg)), t
    tok = prompts[:, 0]
    for s in range(2):  # the caches and tails left behind
        ref.step(tok, logits=lr)
        got.step(tok, logits=lg)
        assert np.array_equal(_bits(lr), _bits(lg)), s
    ref.close()
    got.close()
