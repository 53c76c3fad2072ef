"""Reads of one engine's scenes by several threads at once against reads by one thread."""
import threading

import numpy as np
import pytest

from diploma_thesis_amd import Engine, scenes

pytestmark = pytest.mark.gpu


def test_reads_from_several_threads_equal_serial_reads():
    """Threads that read different scenes of one engine at the same time get what one thread reads."""
    print("reads: eight threads", flush=True)
    mix = [scenes.mix_scene(n, 50 + k) for k, n in enumerate((300, 2000, 7000, 9000, 12000, 4000, 1, 15000))]
    with Engine(mix) as e:
        e.step(3)
        e.sync()
        want = [(e.download(s), e.checksum(s), e.render_state(s), e.snapshot(s).to_arrays()) for s in range(len(mix))]
    with Engine(mix) as e:          # (its first read is one of the threads')
        e.step(3)
        wrong, start = [], threading.Barrier(len(mix))

        def reader(s):
            try:
                start.wait(60)
                for r in range(40):
                    down, check, render, snap = want[s]
                    got = e.download(s)
                    ok = all(np.array_equal(got[k], down[k]) for k in down) and e.checksum(s) == check
                    ok = ok and all(np.array_equal(a, b) for a, b in zip(e.render_state(s), render))
                    now = e.snapshot(s).to_arrays()
                    if not (ok and all(np.array_equal(now[k], snap[k]) for k in snap)):
                        wrong.append((s, r))
                        return
            except Exception as x:   # noqa: BLE001  (an assertion in a thread would be lost)
                wrong.append((s, repr(x)))

        threads = [threading.Thread(target=reader, args=(s,)) for s in range(len(mix))]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
    assert not wrong
