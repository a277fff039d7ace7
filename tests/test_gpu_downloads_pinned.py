"""Large results into pinned buffers, into pageable ones and into both at once
(each takes its own way to the host), whole and at odd addresses."""
import numpy as np
import pytest
import torch

from tests.test_gpu_downloads import _formula

pytestmark = pytest.mark.gpu
N = 400_001  # 4.8 MB of literals, 3.2 of offsets, 1.6 of LBDs, 0.4 of flags


@pytest.mark.parametrize("pinned", ["", "offsets", "lits", "offsets lits", "lbd flags", "offsets lits flags lbd"])
@pytest.mark.parametrize("shift", [0, 1])
def test_destinations(pinned, shift):
    from parafrost_amd.simplifier import Simplifier
    cnf = _formula(N, 3)

    def buf(name, n, dtype):
        return torch.zeros(n + shift + 1, dtype=dtype, pin_memory=name in pinned.split())

    b = [buf("offsets", N + 1, torch.int64), buf("lits", 3 * N, torch.int32), buf("flags", N, torch.uint8),
         buf("lbd", N, torch.int32)]
    assert b[1].is_pinned() == ("lits" in pinned)
    s = Simplifier(0)
    try:
        s.upload(cnf.maxvar, cnf.offsets, cnf.lits, flags=np.arange(N) % 4 * 16 + 1)
        for _ in range(2):
            for x in b:
                x.fill_(7)
            s._check(s._L.pfs_download_cnf(s._h, *[x[shift:].data_ptr() for x in b]), "pfs_download_cnf")
            got = [x.numpy() for x in b]
            assert np.array_equal(got[0][shift:-1], np.arange(N + 1) * 3)
            assert np.array_equal(got[1][shift:-1].view(np.uint32), cnf.lits)
            assert np.array_equal(got[2][shift:-1], np.arange(N) % 4 * 16 + 1) and not got[3][shift:-1].any()
            assert all(x[-1] == 7 and (x[:shift] == 7).all() for x in got)  # nothing around them
    finally:
        s.close()
