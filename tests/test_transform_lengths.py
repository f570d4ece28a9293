"""sddc_transform over lengths on both sides of every column count and of the row
counts between its kernels, against the oracle (Transforms.py:73-129)."""
import ctypes

import numpy as np
import pytest

from oracle import sddc_oracle as O
from spectraldoublediffusiveconvection_amd import _lib

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def run(kind, a, n_out):
    src = torch.as_tensor(a, device="cuda")
    dst = torch.empty((a.shape[0], n_out), dtype=torch.float64, device="cuda")
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    _lib.check(_lib.lib().sddc_transform(kind, ctypes.c_void_p(src.data_ptr()),
                                         ctypes.c_void_p(dst.data_ptr()), a.shape[0], a.shape[1],
                                         n_out, stream))
    return dst.cpu().numpy()


# 14 and 1001 have factors above 5
@pytest.mark.parametrize("L", [6, 14, 64, 72, 135, 192, 200, 256, 270, 384, 400, 500, 512, 540, 768,
                               800, 1001, 1024, 1080, 1536, 1600, 2048])
@pytest.mark.parametrize("rows", [1, 5, 2049, 4100])
def test_transforms_at_length(L, rows):
    """1e-14 of each row's norm: the tolerance of the drop-in's transforms."""
    K = max(2, 2 * L // 3)
    rng = np.random.default_rng(L + rows)
    a, x = rng.standard_normal((rows, K)), rng.standard_normal((rows, L))
    got = [run(_lib.SDDC_IDCT, a, L), run(_lib.SDDC_IDST, a, L), run(_lib.SDDC_DCT, x, K),
           run(_lib.SDDC_DST, x, K)]
    for b in sorted({0, rows // 2, rows - 1}):
        ref = [O.idct(a[b], L), O.idst(a[b], L), O.dct(x[b])[:K], O.dst(x[b])[:K]]
        for g, r in zip(got, ref):
            assert np.linalg.norm(g[b] - r) < 1e-14 * np.linalg.norm(r), b


# on both sides of the row counts at which the kernel changes: 4-8, 9-12, 13-16 and
# more columns, with three, four and two workgroups of k_transform on a CU
@pytest.mark.parametrize("L", [300, 384, 600, 810, 1080, 1280, 1728])
@pytest.mark.parametrize("rows", [1024, 1025, 1535, 1537, 2048])
def test_transforms_around_the_row_lines(L, rows):
    """1e-14 of each row's norm, as above, for the first and last rows."""
    K = 2 * L // 3
    rng = np.random.default_rng(L + rows)
    a, x = rng.standard_normal((rows, K)), rng.standard_normal((rows, L))
    got = [run(_lib.SDDC_IDCT, a, L), run(_lib.SDDC_IDST, a, L), run(_lib.SDDC_DCT, x, K),
           run(_lib.SDDC_DST, x, K)]
    for b in (0, 1, rows - 2, rows - 1):
        ref = [O.idct(a[b], L), O.idst(a[b], L), O.dct(x[b])[:K], O.dst(x[b])[:K]]
        for g, r in zip(got, ref):
            assert np.linalg.norm(g[b] - r) < 1e-14 * np.linalg.norm(r), b
