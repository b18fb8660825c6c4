"""The operators called from several Python threads: the interpreter's lock is free while they allocate and launch, and the launches of
one call stay together on their stream."""
import sys
import threading
import time

import numpy as np
import pytest
import torch

from tests.util import *  # noqa: F401,F403

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def qt():
    import qwen_tailor_amd as q
    q._lib.lib()
    return q


def test_another_thread_runs_while_launches_wait(qt, dev):
    """with a switch interval longer than the test nobody is made to give the lock up: another thread gets on only where the calls
    release it.  The launches take the GPU longer than the host, and there are more of them than a hardware queue holds.  (The results
    are kept: torch gives the lock back where a tensor ends.)"""
    q, k, Kp = (torch.ones(s, dtype=BF16, device=dev) for s in ((1, 8, 256), (1, 2, 256), (1, 2, 16384, 256)))
    slot, pos = torch.zeros(1, dtype=torch.int32, device=dev), torch.full((1,), 16000, dtype=torch.int32, device=dev)
    attn_b, args = qt._lib.host.attn_b, (q, k, k, Kp, Kp.clone(), slot, pos, 1, 128, None)
    attn_b(*args)
    turns, stop = [0], [False]

    def other():
        while not stop[0]:
            turns[0] += 1
            time.sleep(0)                                 # (gives the lock back)
    t = threading.Thread(target=other, daemon=True)
    before = sys.getswitchinterval()
    sys.setswitchinterval(1000.0)
    try:
        t.start()
        time.sleep(0.1)                                   # (from here on it waits for the lock with the long interval)
        at = turns[0]
        kept = [attn_b(*args) for _ in range(12000)]
        got = turns[0] - at
    finally:
        sys.setswitchinterval(before)
        stop[0] = True
        t.join()
    torch.cuda.synchronize()
    assert len(kept) == 12000 and got > 0, "the lock was held through every launch"


def test_threads_that_share_a_stream(qt, dev):
    """calls of two launches that meet in the stream's scratch memory, from two threads on one stream: every result has the bits of the
    call by itself"""
    def work(seed):
        rng = np.random.default_rng(seed)
        rb = lambda *s: to_dev(bf(rng.standard_normal(s)), dev, BF16)
        B, Lmax, S, L, T = 4, 600, 320, 1500, 130
        q, k, v, Kp, Vp = rb(B, 8, 256), rb(B, 2, 256), rb(B, 2, 256), rb(B, 2, Lmax, 256), rb(B, 2, Lmax, 256)
        slots, pos = to_dev(rng.permutation(B).astype(np.int32), dev), to_dev(rng.integers(300, Lmax - 1, B).astype(np.int32), dev)
        qs, K, V = rb(1, 8, S, 256), rb(1, 2, L, 256), rb(1, 2, L, 256)
        cw, A_log, dtb, gw = layer_params(seed)
        S0 = to_dev((rng.standard_normal((1, 16, 128, 128)) * 0.02).astype(np.float32), dev)
        ins = [rb(T, PW), rb(1, 3, CD), S0, to_dev(cw, dev, BF16), to_dev(A_log, dev), to_dev(dtb, dev), to_dev(gw, dev)]
        return lambda: [qt.batch.attn_b(q, k, v, Kp, Vp, slots, pos), qt.prefill.gdn_core(*ins)[0],
                        qt.attention.scaled_dot_product_attention(qs, K, V, scale=256 ** -0.5)]
    runs = [work(1), work(2)]
    want = [f() for f in runs]
    torch.cuda.synchronize()
    bad, errors = [0, 0], []

    def loop(i):
        try:
            for _ in range(150):
                for a, b in zip(runs[i](), want[i]):
                    bad[i] += int(not torch.equal(a, b))
        except Exception as e:                            # noqa: BLE001 (reported below)
            errors.append(e)
    threads = [threading.Thread(target=loop, args=(i,)) for i in range(2)]
    before = sys.getswitchinterval()
    sys.setswitchinterval(1e-6)
    try:
        for t in threads:
            t.start()
        for t in threads:
            t.join()
    finally:
        sys.setswitchinterval(before)
    assert not errors, errors
    assert bad == [0, 0]
