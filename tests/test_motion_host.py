"""Host side of the motion producer mirror (kvpersist.motion) on the CPU:
the trace post-processing against the oracle, and the CSV round trip the
CLI and the variance harness read (reference:
traces/gen_motion_from_video.py:121-149, src/run_policy_experiment.cu:45-69)."""

import csv
import threading

import numpy as np
import pytest
import torch

from kvpersist import motion
from oracle import farneback as fb


def test_trace_post_processing_matches_oracle():
    pairs = np.random.default_rng(2).random((7, 98)) * 9
    got = motion.trace_from_change(pairs, 40.0)
    want = fb.trace_from_change(pairs, 40.0)
    assert np.array_equal(got[0], want[0]) and got[1] == want[1]
    assert np.array_equal(got[2], want[2])


def test_csv_round_trip(tmp_path):
    pairs = np.random.default_rng(3).random((4, 98)) * 9
    change, tau, reuse = motion.trace_from_change(pairs)
    tr = motion.MotionTrace(change, tau, reuse, np.zeros((5, 30, 52)), 1560, 16, 50.0)
    p = tmp_path / "t.csv"
    with open(p, "w", newline="") as fh:
        w = csv.writer(fh)
        w.writerow(["frame_id", "tile_id", "motion_score", "is_static", "token_start",
                    "token_count", "reuse"])
        w.writerows(motion.trace_rows(tr))
    assert [r[:6] for r in motion.trace_rows(tr)] == [r[:6] for r in fb.trace_rows(
        change, tau, reuse, 1560, 16)]
    s = motion.read_trace_csv(p)
    assert s.shape == (5, 98) and s.dtype == np.float32
    want = np.array([[np.float32(f"{v:.6f}") for v in row] for row in change])
    assert np.array_equal(s, want)


@pytest.fixture
def on_host(monkeypatch):
    """motion._workspace with host tensors in place of device memory."""
    class Host:
        stream = idle_device = None
        made = []

        def __init__(self, device, stream, nbytes):
            self.buf = torch.empty(nbytes, dtype=torch.uint8)
            self.made.append((device, stream, nbytes))

    monkeypatch.setattr(motion, "_Workspace", Host)
    monkeypatch.setattr(motion, "_local", threading.local())
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    return torch.device("cuda", 0)


def test_workspaces_are_kept_by_device_stream_and_thread(on_host):
    def ws(stream, nbytes=64, device=on_host):
        return motion._workspace(device, stream, nbytes)

    a = ws(None)
    assert ws(0) is a and ws(None, 10) is a      # the null stream, smaller calls
    b = ws(0x1000)
    assert b is not a and ws(0x1000) is b
    assert ws(None, device=torch.device("cuda", 1)) is not a
    grown = ws(0x1000, 128)
    assert grown.numel() == 128 and ws(0x1000) is grown
    other = []
    t = threading.Thread(target=lambda: other.append(ws(0x1000)))
    t.start()
    t.join()
    assert other[0] is not grown and ws(0x1000) is grown


def test_a_thread_keeps_a_bounded_number_of_workspaces(on_host):
    first = motion._workspace(on_host, 0x100, 1)
    for i in range(2, 2 + motion._MAX_WORKSPACES - 1):
        motion._workspace(on_host, 0x100 * i, 1)
    assert motion._workspace(on_host, 0x100, 1) is first          # now the last used
    kept = motion._local.workspaces
    second = kept[0, 0x200].buf
    motion._workspace(on_host, 0x10000, 1)
    assert len(kept) == motion._MAX_WORKSPACES and (0, 0x200) not in kept
    assert motion._workspace(on_host, 0x200, 1) is not second


def test_copied_frames_belong_to_the_stream_that_reads_them(on_host, monkeypatch):
    """Host frames and strided ones are copied into memory of the call's stream."""
    made = motion._Workspace.made
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    frames = np.random.default_rng(4).integers(0, 256, (2, 12, 10), dtype=np.uint8)
    got = motion._frames_u8(frames[:, :, ::2], stream=0x1000)
    assert made == [(on_host, 0x1000, 120)] and np.array_equal(got.numpy(), frames[:, :, ::2])
    flows = torch.arange(48, dtype=torch.float32).view(4, 3, 4)[:, :, :2]
    got = motion._dense(flows, None, on_host)
    assert made[1] == (on_host, 0, 4 * 24) and torch.equal(got, flows) and got.is_contiguous()
