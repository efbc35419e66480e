"""Results of a detector call as they reach Python, and calls through an engine that several handles share."""
import ctypes as C

import numpy as np
import pytest

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
