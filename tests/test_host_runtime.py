"""The host runtime (fastface.c) over a stand-in for the device
(host_runtime_check.c): which streams, events, graphs and copies a call uses,
and what it leaves behind when one of them fails.  CPU only."""
import os
import subprocess

import pytest

from fastface_amd import synth

ROOT = synth.REPO_ROOT
HOST = os.path.join(ROOT, "fastface_amd", "csrc", "host")
LIB = os.path.join(ROOT, "fastface_amd", "lib")


@pytest.fixture(scope="module")
def checker(tmp_path_factory):
    if not os.path.exists(os.path.join(LIB, "libfastface_amd.so")):
        pytest.skip("library not built")
    exe = str(tmp_path_factory.mktemp("host_runtime") / "host_runtime_check")
    srcs = [os.path.join(HOST, f) for f in ("fastface.c", "ff_model.c", "ff_plan.c")]
    subprocess.run(["gcc", "-O1", "-g", "-std=c99", "-pthread", "-ffp-contract=off", "-D_POSIX_C_SOURCE=200809L",
                    "-I" + HOST, "-I" + os.path.join(ROOT, "include"),
                    os.path.join(ROOT, "tests", "host_runtime_check.c"), *srcs, "-o", exe, "-L" + LIB, "-lfastface_amd",
                    "-Wl,-rpath," + LIB, "-lm"], check=True, capture_output=True)
    return exe


@pytest.fixture(scope="module")
def trace(checker, synth_ffw4):
    """scenario -> (stream numbers, [(call, its lines)])"""
    def run(scenario):
        r = subprocess.run([checker, synth_ffw4, synth.OPSC_PATH, synth.OPSC2_PATH, scenario], capture_output=True,
                           text=True, timeout=120)
        assert r.returncode == 0, r.stderr[-2000:]
        calls, streams = [], None
        for line in r.stdout.splitlines():
            if line.startswith("context "):
                t = line.split()
                streams = {"context": t[1], "mine": t[3]}
            elif line.startswith("call "):
                calls.append((line[5:], []))
            elif calls:
                calls[-1][1].append(line)
        return streams, calls
    return run


def rc(lines):
    return int([x for x in lines if x.startswith("rc ")][0].split()[1])


# the calls of a split batch in order: 2 launches; records of the fork, the
# join and the end; waits of the second stream and of the caller's
@pytest.mark.parametrize("what", ["launch-2", "record-2", "wait-2", "record-3"])
def test_half_of_a_split_batch_fails(trace, what):
    """A call that fails after its first half's launch leaves work in flight
    on the caller's stream: what frees the buffers afterwards waits for it."""
    streams, calls = trace("half-fails-" + what)
    assert [c for c, _ in calls] == ["device 30", "device 30", "reserve", "destroy"]
    ok, failed, reserve = (lines for _, lines in calls[:3])
    assert rc(ok) == 0 and sum(x.startswith("launch ") for x in ok) == 2
    assert rc(failed) != 0 and rc(reserve) == 0
    bad = next(i for i, x in enumerate(failed) if x.endswith("FAILED"))
    started = [x for x in failed[:bad] if x.startswith("launch ")]
    assert started and started[0].endswith("stream " + streams["mine"])
    # before the first buffer goes: a host wait for each stream that got work,
    # on an event recorded on it after its launch or on the stream itself
    lines = failed + reserve
    freed = next(i for i, x in enumerate(lines) if x in ("free", "graph_destroy " + started[0].split()[1]))
    for s in sorted({x.split()[3] for x in started}):
        at = max(i for i, x in enumerate(lines[:freed]) if x.startswith("launch ") and x.endswith("stream " + s))
        events = {s2: i for i, x in enumerate(lines[at:freed], at)
                  if x.startswith("record ") and x.endswith("stream " + s) for s2 in [x.split()[1]]}
        waited = [i for i, x in enumerate(lines[at:freed], at)
                  if x == "stream_sync " + s or (x.startswith("event_sync ") and x.split()[1] in events)]
        # (the second stream's work may also be joined into the caller's)
        joined = [x for x in lines[at:freed] if x.startswith("wait ") and x.split()[1] in events and not x.endswith("FAILED")
                  and x.split()[3] != s]
        assert waited or (s != streams["mine"] and joined), (s, lines)


def test_chains_of_different_sizes_do_not_queue(trace):
    """A device call whose batch differs from the unfinished one's waits for
    it on the host before it launches (or captures) anything, also where the
    buffers are the same and the I/O descriptor stays; an equal one queues."""
    streams, calls = trace("sizes")
    calls = [(c, lines) for c, lines in calls if c.startswith("device")]
    assert [c for c, _ in calls] == ["device %d" % n for n in (8, 8, 5, 36, 37, 37, 8)]
    end = None                                          # the event at the last call's end
    for k, (c, lines) in enumerate(calls):
        assert rc(lines) == 0
        first = next(i for i, x in enumerate(lines) if x.startswith(("launch ", "capture ")))
        waited = [x.split()[1] for x in lines[:first] if x.startswith("event_sync ")]
        if k:
            assert (end in waited) == (calls[k - 1][0] != c), (c, lines)
        records = [x.split()[1] for x in lines if x.startswith("record ") and x.endswith("stream " + streams["mine"])]
        end = records[-1]


def test_small_host_outputs_go_through_pinned_memory(trace):
    """Up to eight faces' embeddings reach the caller through the pinned
    buffer: one fp32 face (and six uint8) in place, more by a copy into it."""
    _, calls = trace("host")
    for c, lines in calls:
        if not c.startswith("host"):
            continue
        assert rc(lines) == 0
        out = [x.split()[3] for x in lines if x.startswith("d2h ")]
        n = int(c.split()[1])
        assert out == ([] if n == 1 else ["1"] if n <= 8 else ["0"]), (c, lines)


def test_mixed_host_batches_keep_the_descriptor(trace):
    """Calls that run in place and calls that go through the device buffers
    alternate without rewriting an I/O descriptor (32 bytes, a host wait
    before and after): each kind has its own."""
    _, calls = trace("host")
    calls = [(c, lines) for c, lines in calls if c.startswith("host")]
    copies = [sum(x.startswith(("h2d 16 ", "h2d 32 ")) for x in lines) for _, lines in calls]
    # (the first call in place, the first over the device buffers, the first
    # over the uint8 buffer)
    assert copies == [1, 1, 0, 0, 0, 0, 0, 0, 1], list(zip([c for c, _ in calls], copies))
