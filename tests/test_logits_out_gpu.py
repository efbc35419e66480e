"""Logits on their way to the caller: up to 1 MiB in one copy, more in pieces of 256 KiB through pinned memory of 32, which longer ones pass several times.  The same rows eight at a
time, bit for bit; several sessions at once, each from a thread of its own."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
VOCAB = 32000


@pytest.fixture(scope="module")
def model(gpu):
    return gpu.LlmModel(gpu.LlmHParams(1, 256, 8, 2, 64, 512, VOCAB, 1e-5, 10000.0, 0, 0, 0, 0, 1)).fill_synthetic(4)


def passes(gpu, model, rows, width, seed, session=None):
    s = session or gpu.LlmSession(model, 256, 8)
    toks = np.random.default_rng(seed).integers(3, VOCAB, rows).astype(np.int32)
    out = [s.forward(np.arange(r, min(r + width, rows)), np.zeros(min(width, rows - r)), toks[r:r + width]) for r in range(0, rows, width)]
    return np.concatenate([o[0] for o in out]), np.concatenate([o[1] for o in out])


@pytest.mark.parametrize("rows", [1, 8, 9, 33, 65, 66, 131, 256])
def test_logits_of_many_rows(gpu, model, rows):
    got, ids = passes(gpu, model, rows, 256, rows)
    want, want_ids = passes(gpu, model, rows, 8, rows)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32)) and np.array_equal(ids, want_ids)


def test_sessions_in_threads(gpu, model):
    rows = [70, 130, 33]
    got = [None] * len(rows)
    sessions = [gpu.LlmSession(model, 256, 8) for _ in rows]

    def work(i):
        got[i] = [passes(gpu, model, rows[i], 256, 7 + k, sessions[i])[0] for k in range(3)]
    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(rows))]
    [t.start() for t in threads]
    [t.join() for t in threads]
    for i, n in enumerate(rows):
        for k in range(3):
            assert np.array_equal(got[i][k].view(np.uint32), passes(gpu, model, n, 8, 7 + k)[0].view(np.uint32))


def test_halves_sent_in_any_order(gpu, model):
    """eight halves of the pinned memory, freed and sent again by whichever thread takes a half's last piece: one behind a later one is still waited for"""
    rows = 256
    s = gpu.LlmSession(model, 256, 8)
    want = passes(gpu, model, rows, 8, 3)[0]
    stop = threading.Event()

    def busy():  # threads that hold the others up in the middle of a piece
        a = np.zeros(1 << 22, np.uint8)
        while not stop.is_set():
            a[:] = a + 1
    others = [threading.Thread(target=busy) for _ in range(12)]
    [t.start() for t in others]
    try:
        for _ in range(60):
            got = passes(gpu, model, rows, 256, 3, s)[0]
            assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    finally:
        stop.set()
        [t.join() for t in others]
    s.close()


REFUSAL = r"""
#include <dlfcn.h>
#include <stddef.h>
int hipHostMalloc(void** p, size_t n, unsigned flags) {
    static int (*real)(void**, size_t, unsigned);
    if (n >= ((size_t)8 << 20)) { *p = 0; return 2; /* hipErrorOutOfMemory */ }
    if (!real) real = (int (*)(void**, size_t, unsigned))dlsym(dlopen("libamdhip64.so.7", RTLD_NOW | RTLD_NOLOAD), "hipHostMalloc");
    return real(p, n, flags);
}
"""
WITHOUT = r"""
import ctypes, sys
ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
sys.path[:0] = [sys.argv[2]]
import numpy as np
import trackiellm_amd as tk
m = tk.LlmModel(tk.LlmHParams(1, 256, 8, 2, 64, 512, 32000, 1e-5, 10000.0, 0, 0, 0, 0, 1)).fill_synthetic(4)
s = tk.LlmSession(m, 256, 8)
print("open", flush=True)
x = np.arange(3, 43, dtype=np.int32)
np.save(sys.argv[3], s.forward(np.arange(40), np.zeros(40), x)[0])
"""


def test_a_session_without_pinned_memory(gpu, model, tmp_path):
    """where the runtime refuses it (here: a definition in front of its own), a session opens all the same and its logits go by the plain copy"""
    import os
    import subprocess
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    shim, out = tmp_path / "refuse.so", tmp_path / "logits.npy"
    (tmp_path / "refuse.c").write_text(REFUSAL)
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(shim), str(tmp_path / "refuse.c"), "-ldl"], check=True)
    r = subprocess.run([sys.executable, "-c", WITHOUT, str(shim), root, str(out)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and "open" in r.stdout, r.stderr[-1000:]
    x = np.arange(3, 43, dtype=np.int32)
    want = gpu.LlmSession(model, 256, 8).forward(np.arange(40), np.zeros(40), x)[0]
    assert np.array_equal(np.load(out).view(np.uint32), want.view(np.uint32))
