"""kernel_ms is read off the device's clock: a block's end is that of its last
wave, not of the wave that notes it (tests/cpp/clock_span.hip)."""
import os
import subprocess

import pytest

EXE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "bin", "clock_span")


@pytest.mark.gpu
@pytest.mark.parametrize("blocks,threads", [(1, 64), (1, 256), (3, 1024), (256, 512)])
def test_the_clock_covers_every_wave(gpu, blocks, threads):
    if not os.path.exists(EXE):
        pytest.fail("tests/cpp/bin/clock_span is not built: run __graft_entry__.build()")
    ticks = 20000  # 200 us
    r = subprocess.run([EXE, str(blocks), str(threads), str(ticks)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr
    # the waiting wave may start before block 0 notes its start, by no more than a launch
    assert int(r.stdout) >= 0.9 * ticks
