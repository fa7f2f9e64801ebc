"""The CSR product with 128, 64 and 16 rows a workgroup (rows of up to 9, up to 40 and more
entries on average): remainders, both sides of the lines between them, empty rows and rows
of several chunks of 1024 entries, against sums in extended precision."""
import numpy as np
import pytest

from fvmpor_amd.lib import CsrMatrix
from test_gemv_shapes_gpu import _matrix

pytestmark = pytest.mark.gpu

CASES = {"9 on average": (257, lambda n: np.full(n, 9)),
         "one more": (257, lambda n: np.r_[np.full(n - 1, 9), 10]),
         "one of 256": (4100, lambda n: np.r_[256, np.full(n - 1, 3)]),
         "one of 257": (4100, lambda n: np.r_[np.full(n - 1, 3), 257]),
         "half empty": (385, lambda n: np.arange(n) % 2 * 11),
         "127": (127, lambda n: np.full(n, 2)), "128": (128, lambda n: np.full(n, 2)), "129": (129, lambda n: np.full(n, 2)),
         "40 on average": (200, lambda n: np.full(n, 40)),
         "40 and one": (200, lambda n: np.r_[np.full(n - 1, 40), 41]),
         "15": (15, lambda n: np.full(n, n)), "17 of 61": (61 + 20, lambda n: np.full(n, 61)),
         "full": (1100, lambda n: np.full(n, n)),
         "long and empty": (1600, lambda n: np.where(np.arange(n) < 64, 1300, 0))}


@pytest.mark.parametrize("which", list(CASES))
@pytest.mark.parametrize("beta", [0.0, -0.5])
def test_rows_a_workgroup(which, beta):
    torch = pytest.importorskip("torch")
    n, rows_of = CASES[which]
    rng = np.random.default_rng(n)
    lengths = rows_of(n)
    ia, ja, a = _matrix(rng, n, lengths)
    x, y0 = rng.standard_normal(n), rng.standard_normal(n)
    A = CsrMatrix(ia, ja)
    da, dx, y = (torch.tensor(v, device="cuda") for v in (a, x, y0))
    torch.cuda.synchronize()
    A.set_values(da)
    A.gemv(2.0, dx, beta, y)
    torch.cuda.synchronize()
    rows = np.repeat(np.arange(n), lengths)
    ref, size = np.zeros(n, dtype=np.longdouble), np.zeros(n)
    np.add.at(ref, rows, a.astype(np.longdouble) * x[ja])
    np.add.at(size, rows, np.abs(a * x[ja]))
    ref = 2.0 * ref + beta * y0
    # one rounding per term of the sum, and of alpha, beta y and the last sum
    bound = (lengths + 3) * 2.0 ** -53 * 1.01 * (2.0 * size + np.abs(beta * y0))
    assert (np.abs(y.cpu().numpy() - ref) <= bound).all()
