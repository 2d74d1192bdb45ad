"""GPU parity of phase 2 (the merge of internal and bath events and the
dynamics) at the sizes where its staging can go wrong: tiles of 64 neurons
with a remainder, neurons with no event, chunks of 8 events and their
remainders, and baths with more events per ms than the LDS queue holds.
State and spikes are the oracle's, bit for bit."""
import os

import numpy as np
import pytest

from helpers import OracleNet

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _restore_env(pkg):
    yield
    pkg.apply_env(pkg.config_dir("c0"))


# (neurons per sub-population, grid side, bath Hz per input): 800 inputs, so
# 30 Hz is 24 bath events per ms and 0.05 Hz one in 25 ms; the bath is drawn
# ahead of phase 1 up to 128 events per neuron and ms at most (8 Hz: the most
# is 20 times the mean)
NETWORKS = [((1, 1, 1), 1, 3.0), ((21, 21, 21), 1, 30.0), ((22, 21, 21), 1, 0.05), ((22, 22, 21), 1, 5.5),
            ((60, 61, 30), 2, 8.0), ((97, 96, 47), 2, 3.0), ((150, 150, 75), 2, 12.0)]
FORMS = {"bath merged": dict(DPSNN_BATH="0"), "records": dict(DPSNN_PIPE="0"), "pipe": dict(DPSNN_PIPE="1"),
         "records window": dict(DPSNN_PIPE="0", DPSNN_WINDOW="1"),
         "pipe big sort": dict(DPSNN_PIPE="1", DPSNN_WINDOW="1", DPSNN_SORT_CAP="20"),
         "pipe general path": dict(DPSNN_PIPE="1", DPSNN_PHASE1_DENSE_MAX="30")}


@pytest.mark.parametrize("form", list(FORMS))
@pytest.mark.parametrize("counts,side,nu_ext", NETWORKS)
def test_phase2_bit_exact_vs_oracle(pkg, oracle, tmp_path, monkeypatch, counts, side, nu_ext, form):
    """form, from step 32 on: the bath merged in phase 2 or sorted in with
    the internal events by each of phase 1's sorts; one wave or three waves
    per tile in phase 2."""
    for k, v in FORMS[form].items():
        monkeypatch.setenv(k, v)
    e, e2, i = counts
    (tmp_path / "column.txt").write_text(
        f"0 {e} 0.5 0.0 {nu_ext} 20 20 15 2 1 500 0.05\n"
        f"1 {e2} 0.5 0.0 {nu_ext} 7 20 15 2 1 500 0.05\n"
        f"2 {i} 0.5 0.0 {nu_ext} 10.3 20 15 2 0.25 333.3 0.01\n")
    for f in ("connectivity.txt", "bathEfficacy.txt"):
        (tmp_path / f).write_text(open(os.path.join(pkg.config_dir("c0"), f)).read())
    pkg.apply_env(pkg.config_dir("c0"), env_CFX=side, env_CFY=side, env_totalSimTime_ms=70)
    print(f"phase 2, {form}: {side}x{side} columns of {counts}, bath {nu_ext} Hz, 70 ms vs oracle", flush=True)
    ora = OracleNet(oracle, str(tmp_path))
    try:
        with pkg.Network(str(tmp_path), keep_spikes=True) as net:
            for step in range(70):
                ora.fire()
                net.step(1)
                ids, te = net.last_spikes()
                oids, ote = ora.last_spikes()
                assert np.array_equal(ids, oids) and np.array_equal(te, ote), step
                a, b = net.state(), ora.state()
                for k in ("v", "c", "Tr", "Te"):
                    assert np.array_equal(a[k].view(np.uint64), b[k].view(np.uint64)), (step, k)
    finally:
        ora.close()
