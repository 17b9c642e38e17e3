"""BitLinear::forward on f32 activations where the choice between its kernels' forms changes (row-broadcast, 4 x 4 x 1
and 16 x 16 matrix cores): bit-exact against the oracle's sequential fold, non-finite activations among them."""
import numpy as np
import pytest

import oracle
from inputs import assert_bitexact, normal, raw_packed

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
from kore_amd import rocm  # noqa: E402
from kore_amd.rocm import HipBuffer  # noqa: E402

DEV = 0


def up(a):
    return HipBuffer.from_host(DEV, np.ascontiguousarray(a))


# out, tokens, in.  The last narrow tile and the first 64-column one; K one column short of where the expected
# times decide; the 4 x 4 form with one chunk of K, a column more, one less and more than two, below K = 2560 and past
# 192 tokens; the 16 x 16 form below 768 waves, and from 768 waves up to 32 tokens or little K (a row less takes the
# row-broadcast form); 4, 5 and 7 rows a lane of the row-broadcast form; K that is no multiple of 4.
FORMS = [(4096, 32, 40), (4096, 33, 37), (2048, 40, 79), (582, 839, 79), (582, 839, 80), (582, 839, 81), (582, 400, 159),
         (582, 400, 160), (582, 400, 161), (4100, 64, 161), (5376, 64, 897), (1021, 400, 1000), (1024, 257, 323),
         (2560, 96, 1283), (700, 1000, 163), (2375, 200, 1001), (6912, 96, 320), (6909, 130, 163), (24512, 17, 40),
         (24513, 32, 37), (49150, 5, 41), (49089, 16, 80), (3185, 65, 40), (4392, 66, 41), (6332, 70, 37), (64, 3000, 241),
         (33, 700, 84), (3, 900, 330)]


@pytest.mark.parametrize("m,n,k", FORMS)
def test_bit_linear_f32_forms(m, n, k):
    print(f"bit_linear f32 out={m} tokens={n} in={k}", flush=True)
    p, sa, bias = raw_packed(m, k, m + k), normal((m,), 3, 1.0, 0.1), normal((m,), 4)
    x = normal((n, k), n + k)
    x[n // 3, k // 2] = np.inf
    x[n - 1, 0] = np.nan
    x[n // 2] *= np.float32(2.0 ** 118)  # sums that overflow on the way
    x[0] = 0.0
    got = rocm.rocm_bit_linear_f32(DEV, up(p), up(sa), up(x), up(bias), m, n, k).to_host(np.float32).reshape(n, m)
    assert_bitexact(got, oracle.bit_linear_forward(p, sa, x, bias, m, n, k), "bit_linear_f32")
