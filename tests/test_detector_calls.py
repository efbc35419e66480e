"""Results of a detector call as they reach Python, and calls through an engine that several handles share."""
import ctypes as C
import threading
import time

import numpy as np
import pytest

import trackiellm_amd as tk
import trackiellm_amd.vision as V


@pytest.mark.parametrize("n", [0, 1, 3])
def test_results_are_read_as_the_fields_are(n):
    r = (V.DetectionResult * max(n, 1))()
    for i in range(n):
        r[i].class_id, r[i].confidence, r[i].label = 4000000000 + i, 0.1 * i, (None, b"a", b"some label")[i]
        r[i].bbox.x, r[i].bbox.y, r[i].bbox.w, r[i].bbox.h = -i, 2 - i, 1 << 30, i
    want = [(r[i].class_id, r[i].label, r[i].confidence, (r[i].bbox.x, r[i].bbox.y, r[i].bbox.w, r[i].bbox.h)) for i in range(n)]
    assert V._detections(C.cast(r, C.POINTER(V.DetectionResult)) if n else C.POINTER(V.DetectionResult)(), n) == want


@pytest.mark.gpu
def test_a_lone_caller_among_idle_handles_runs_its_frames_one_by_one(gpu):
    model = "synthetic://yolov8n?seed=5&cls_bias=-0.45"
    dets = [gpu.ObjectDetector(model=model, width=96, height=96, conf=0.4) for _ in range(3)]
    rng = np.random.default_rng(1)
    frames = [rng.integers(0, 256, (50 + 7 * i, 60, 3), np.uint8) for i in range(4)]
    first = [dets[0].detect(f) for f in frames]
    assert any(first)
    assert [dets[i % 3].detect(f) for i, f in enumerate(frames)] == first
    handles, batches, nframes, widest = dets[0].share_stats()
    assert (handles, batches, nframes, widest) == (3, 8, 8, 1)


def jobs_of(callers, requests, wait=400, job=450, frame=100, most=32):
    """[(caller, not before)] -> [(size, begin)]"""
    n = len(requests)
    who, at = (C.c_int * n)(*[r[0] for r in requests]), (C.c_int64 * n)(*[r[1] for r in requests])
    sizes, begins = (C.c_int * n)(), (C.c_int64 * n)()
    jobs = tk.lib().tk_mi355x_arrivals_simulate(callers, wait, job, frame, most, n, who, at, sizes, begins)
    assert sum(sizes[:jobs]) == n
    return list(zip(sizes[:jobs], begins[:jobs]))


@pytest.mark.parametrize("period", [2000, 33000])
@pytest.mark.parametrize("callers", [2, 8, 32])
def test_bursts_are_one_job_each(callers, period):
    rng = np.random.default_rng(callers)
    late = rng.integers(0, 300, (20, callers)) + period * np.arange(1, 21)[:, None]
    got = jobs_of(callers, [(c, int(late[b, c])) for b in range(20) for c in range(callers)], frame=10)
    assert got == [(callers, int(late[b].max())) for b in range(20)]


def test_callers_that_come_back_at_once_are_one_job():
    got = jobs_of(8, [(c, 0) for c in range(8) for _ in range(10)])
    assert [g[0] for g in got] == [8] * 10


def test_a_lone_caller_waits_once_for_idle_ones():
    at = [10000 * (i + 1) for i in range(6)]
    assert jobs_of(32, [(3, t) for t in at]) == [(1, at[0] + 400)] + [(1, t) for t in at[1:]]


@pytest.mark.parametrize("callers", [2, 3, 8])
@pytest.mark.parametrize("gap", [0, 100, 3000])
def test_handles_that_one_thread_uses_in_turn_do_not_wait_for_each_other(callers, gap):
    """a call, `gap`, the next handle's call: each of them is waited for twice at most"""
    step = 550 + gap
    at, requests = 1000, []
    for i in range(10 * callers):
        got = jobs_of(callers, requests + [(i % callers, at)])
        requests.append((i % callers, at))
        begin = got[-1][1]
        assert got[-1][0] == 1 and begin - at in (0, 400)
        assert begin == at or i < 2 * callers
        at = begin + step


@pytest.mark.parametrize("gap", [900, 2500])
def test_a_caller_that_has_been_served_is_not_waited_for(gap):
    """bursts of one, then the seven others `gap` later: the seven are one job, which begins when the last of them is in (or the first one's job ends)"""
    got = jobs_of(8, [(c, 33000 * b + (gap + 10 * c if c else 0)) for b in range(1, 9) for c in range(8)])
    assert [g[0] for g in got] == [1, 7] * 8
    for b in range(1, 8):  # (from the second burst on; in the first nobody has a history)
        one, seven = got[2 * b][1], got[2 * b + 1][1]
        assert one <= 33000 * (b + 1) + 400 and seven == max(33000 * (b + 1) + gap + 70, one + 550)


def test_a_burst_after_a_lone_call_is_one_job():
    """one caller between the bursts of all: neither is the burst cut to jobs of one and the rest, nor does the lone call wait (from the third burst on: the
    second is the first whose callers have a history)"""
    lone, bursts = [(0, 30000 * b + 15000) for b in range(1, 9)], [(c, 30000 * b + 20 * c) for b in range(1, 9) for c in range(6)]
    got = jobs_of(6, sorted(lone + bursts, key=lambda r: r[1]))
    got = [g for g in got if g[1] >= 90000]
    assert got == [(6, 30000 * b + 100) if k == 0 else (1, 30000 * b + 15000) for b in range(3, 9) for k in range(2)]


@pytest.mark.gpu
def test_bursts_of_threads_after_a_lone_call(gpu):
    model = "synthetic://yolov8n?seed=5&cls_bias=-0.45"
    dets = [gpu.ObjectDetector(model=model, width=128, height=128, conf=0.4) for _ in range(6)]
    frame = np.random.default_rng(1).integers(0, 256, (60, 60, 3), np.uint8)
    want = dets[0].detect(frame)
    gate, results = threading.Barrier(6), []

    def call(i):
        for _ in range(11):
            gate.wait()
            if i == 0:
                time.sleep(0.015)
                results.append(dets[0].detect(frame))
                time.sleep(0.015)
            gate.wait()
            results.append(dets[i].detect(frame))
    threads = [threading.Thread(target=call, args=(i,)) for i in range(6)]
    before = dets[0].share_stats()
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    after = dets[0].share_stats()
    assert all(r == want for r in results) and after[2] - before[2] == 77 and after[3] == 6
    assert after[1] - before[1] <= 28  # 22 and a few for threads that the host held up; cut bursts make 33
