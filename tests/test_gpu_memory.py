"""Device memory of a handle follows the state it holds."""
import ctypes

import numpy as np
import pytest

from icarion_amd import _abi
from icarion_amd import workloads as W

pytestmark = pytest.mark.gpu


def free_bytes():
    hip = ctypes.CDLL("libamdhip64.so")
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


BIG, SMALL = 4_000_000, 1000   # 24 bytes of positions alone per ion


def test_upload_gives_back_what_a_larger_cloud_took():
    from icarion_amd import gpu
    w = W.quadrupole_workload(n=BIG, seed=1, precision=_abi.PRECISION_FP32_KAHAN)
    small = w["ensemble"].subset(np.arange(SMALL))
    with gpu.Handle() as h:
        h.set_domain(w["domain"], w["physics"])
        h.set_species(w["species"])
        h.upload_state(small)
        before = free_bytes()
        h.upload_state(w["ensemble"])
        assert before - free_bytes() > 100 * BIG
        h.upload_state(small)
        assert before - free_bytes() < 24 * BIG
        st = h.step(0.0, w["dt"], 10)
        out = small.copy()
        h.download_state(out)
    assert st.ion_steps == 10 * SMALL and not np.array_equal(out.x, small.x)


def test_batch_gives_back_what_a_larger_batch_took_and_counts_large_clouds():
    from icarion_amd import gpu

    def clouds(n):
        w = W.quadrupole_workload(n=n, seed=1, precision=_abi.PRECISION_FP32_KAHAN)
        w["domain"].detector_z_m = 1e-4
        e = w["ensemble"]
        e.active[::7] = 0
        return [dict(kind="q", domain=w["domain"], physics=w["physics"], species=w["species"], ensemble=e, t0=0.0,
                     dt=w["dt"], n_steps=20, step_offset=0)]

    big, small = clouds(BIG + 77), clouds(SMALL)
    with gpu.Handle() as h:
        h.batch_upload(small)
        before = free_bytes()
        h.batch_upload(big)
        assert before - free_bytes() > 90 * BIG
        for _ in range(2):   # a second run starts its counts anew
            st, _ = h.batch_run(None, None)
        h.batch_download(big)
        e = big[0]["ensemble"]
        assert st[0].alive == int(((e.active != 0) & (e.born != 0)).sum()) > 0
        assert st[0].arrived == int((~np.isnan(e.arrival_time_s)).sum())
        h.batch_upload(small)
        assert before - free_bytes() < 24 * BIG
