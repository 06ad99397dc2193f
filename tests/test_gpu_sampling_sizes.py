"""GPU: top-p selection at the vocabulary sizes where its kernel changes (samp_select_radix_kernel's candidates a thread, then the streamed one,
nanollama_amd/csrc/nl_sample.h), against the integer restatement.  Reference: go/main.go:346-398."""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
import sampling_mirror as sm  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("V", [1, 3, 4097, 32767, 32768, 32769, 49152, 49153, 65535, 65536, 65537])
def test_sizes(V):
    from nanollama_amd import model as hip
    rng = np.random.default_rng(V)
    plain = (rng.standard_normal(V) * 2.0).astype(np.float32)
    last = plain.copy()
    last[V - 1] = plain.max() + np.float32(3.0)                    # the last candidate of the last thread
    ties = plain.copy()
    ties[rng.permutation(V)[:V // 2]] = np.float32(1.5)            # ranks among equal candidates, buckets beyond the list
    for lg in (plain, last, ties):
        for u in (0.0, 0.4, 0.999):
            recent = [int(t) for t in rng.integers(0, V, 5)]
            pick, _, rec = hip.op_sample(lg.copy(), 0.8, 0.9, 50, 1.0, 6, u, recent)
            assert pick == sm.device_top_p(lg, 0.8, 0.9, u)[0], u
            assert rec == sm.push_recent(recent, pick, 6)
