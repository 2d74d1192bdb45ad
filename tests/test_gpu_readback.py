"""GPU read-backs against the oracle: the state of networks either side of the
size up to which one kernel writes it to pinned memory (131,072 neurons), a
part of it only, the counters, and a step's spikes when they fit the pinned
buffer (256 KiB) and when they don't."""
import ctypes
import os

import numpy as np
import pytest

from helpers import OracleNet

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _restore_env(pkg):
    yield
    pkg.apply_env(pkg.config_dir("c0"))


@pytest.mark.parametrize("counts,side", [((1, 1, 1), 1), ((22, 21, 22), 1), ((60, 61, 30), 2), ((21, 21, 21), 45),
                                         ((21, 21, 21), 46)])
def test_readback_vs_oracle(pkg, oracle, tmp_path, counts, side):
    e, e2, i = counts
    # 30 Hz x 800 inputs of 0.5 mV: every neuron fires within a few ms
    (tmp_path / "column.txt").write_text(
        f"0 {e} 0.5 0.0 30 20 20 15 2 1 500 0.05\n"
        f"1 {e2} 0.5 0.0 30 7 20 15 2 1 500 0.05\n"
        f"2 {i} 0.5 0.0 30 10.3 20 15 2 0.25 333.3 0.01\n")
    for f in ("connectivity.txt", "bathEfficacy.txt"):
        (tmp_path / f).write_text(open(os.path.join(pkg.config_dir("c0"), f)).read())
    pkg.apply_env(pkg.config_dir("c0"), env_CFX=side, env_CFY=side, env_totalSimTime_ms=7)
    print(f"read-backs: {side}x{side} columns of {counts} vs oracle", flush=True)
    ora = OracleNet(oracle, str(tmp_path))
    try:
        with pkg.Network(str(tmp_path), keep_spikes=True) as net:
            spikes = 0
            for step in range(6):
                ora.fire()
                net.step(1)
                ids, te = net.last_spikes()
                oids, ote = ora.last_spikes()
                assert np.array_equal(ids, oids) and np.array_equal(te, ote), step
                a, b = net.state(), ora.state()
                for k in ("v", "c", "Tr", "Te"):
                    assert np.array_equal(a[k].view(np.uint64), b[k].view(np.uint64)), (step, k)
                spikes += int(a["fired"].astype(bool).sum())
                assert net.stats()["spikes"] == net.stats()["spikes"] == spikes
            assert spikes > 0
            st = net.state()
            part = np.zeros(len(st["c"]))
            rc = net._lib.dpsnn_get_state(net._h, None, part.ctypes.data_as(ctypes.POINTER(ctypes.c_double)), None, None,
                                          None)
            assert rc == 0 and np.array_equal(part, st["c"])
            last = net.state()["fired"].astype(bool)
            net.step(1)
            assert np.array_equal(np.flatnonzero(last), np.sort(net.last_spikes()[0]))
    finally:
        ora.close()
