"""Every form of the int8 ternary matmul around the sizes where the choice between them changes, on code rows and packed
rows of every alignment: bit-exact against the oracle (an exact integer sum, one epilogue)."""
import numpy as np
import pytest

import oracle
from inputs import assert_bitexact, normal, raw_packed, rng

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
from kore_amd import rocm  # noqa: E402
from kore_amd.rocm import HipBuffer  # noqa: E402

DEV = 0


def at(arr: np.ndarray, offset: int) -> HipBuffer:
    """arr's bytes on the device, `offset` bytes past a 16-byte boundary, with nothing of the allocation after them."""
    raw = torch.from_numpy(np.ascontiguousarray(arr).reshape(-1).view(np.uint8).copy())
    t = torch.empty(offset + raw.numel(), dtype=torch.uint8, device="cuda:0")
    t[offset:].copy_(raw)
    return HipBuffer.from_tensor(t[offset:])


# m, n, k, byte offset of the codes, of the packed rows.  Two to eight codes either side of the small-n path's rows and K; one block
# of 32 codes and the next; the number of workgroups around each form's limit (32 x 32 of 8 waves to 512, of 4 to 1024
# with two code tiles and little K, to 2047 with one; 64 x 32 beyond; 64 x 64 of 8 waves to 256, of 4 beyond; long K); 256
# tiles of 128 x 128 then the tile kernel; the rows from which aligned codes leave the skinny kernel and others stay; K of
# one partial piece, one block, and one column more or less.
FORMS = [(5, 1, 15, 0, 0), (5, 1, 16, 0, 0), (33, 1, 17, 1, 1), (7, 2, 8, 0, 0), (64, 2, 2048, 0, 0), (64, 2, 2056, 0, 0),
         (5120, 2, 2064, 0, 0), (5121, 2, 2064, 0, 0), (5121, 2, 2568, 0, 0), (8192, 2, 4104, 0, 1), (8193, 2, 4104, 0, 0),
         (5121, 2, 7680, 0, 0), (5121, 2, 7688, 0, 3), (1024, 4, 4616, 0, 0), (1025, 4, 4616, 0, 0), (1023, 3, 4616, 0, 1),
         (9, 4, 9000, 0, 2), (2048, 4, 7688, 0, 0), (2049, 3, 7688, 0, 0), (64, 3, 4608, 0, 0), (8192, 7, 8, 0, 0), (8193, 8, 8, 0, 0), (31, 3, 8, 0, 1),
         (7, 2, 2563, 3, 2), (300, 3, 2560, 0, 0), (129, 8, 2568, 0, 0), (31, 32, 31, 5, 3),
         (32, 33, 159, 0, 0), (65, 33, 160, 0, 0), (64, 31, 161, 9, 1), (97, 40, 1001, 7, 0), (6657, 45, 175, 15, 3),
         (8192, 64, 320, 0, 0), (8193, 64, 320, 0, 0), (4128, 45, 2576, 0, 1), (8192, 64, 2561, 3, 0), (8224, 64, 2576, 0, 0), (49152, 2, 2056, 0, 0),
         (49153, 2, 2056, 0, 1), (16384, 40, 163, 3, 1), (16385, 64, 176, 0, 0), (8200, 45, 1040, 0, 1),
         (16385, 9, 161, 0, 0), (65504, 5, 33, 1, 0), (65505, 32, 48, 0, 2), (40960, 33, 48, 0, 0), (40961, 33, 48, 0, 0),
         (57344, 33, 528, 0, 0), (57345, 33, 528, 0, 0), (57345, 40, 33, 2, 1), (8224, 33, 5136, 0, 0), (28672, 65, 32, 0, 0), (28673, 65, 32, 0, 3), (28673, 70, 37, 1, 0),
         (4096, 65, 163, 0, 0), (8200, 65, 336, 0, 0), (8192, 100, 164, 2, 1), (1024, 1000, 177, 0, 0),
         (2100, 1000, 1283, 1, 0), (4096, 1024, 165, 0, 2), (4100, 1024, 176, 0, 0), (4100, 1020, 171, 3, 1),
         (70, 3000, 335, 0, 0), (1, 4000, 480, 0, 0)]


@pytest.mark.parametrize("m,n,k,oq,oa", FORMS)
def test_ternary_i8_forms(m, n, k, oq, oa):
    print(f"ternary i8 m={m} n={n} k={k} codes+{oq} packed+{oa}", flush=True)
    p = raw_packed(m, k, m + k)
    q = rng(n + k).integers(-128, 128, size=(n, k), dtype=np.int64).astype(np.int8)
    sa, sq = normal((m,), 8, 1.0, 0.1), np.abs(normal((n,), 9, 0.02, 0.005))
    bias = normal((m,), 10)
    want = oracle.ternary_matmul_i8(p, sa, q, sq, m, n, k)
    ab, qb, sab, sqb = at(p, oa), at(q, oq), at(sa, 0), at(sq, 0)
    got = rocm.rocm_ternary_matmul_i8(DEV, ab, sab, qb, sqb, m, n, k).to_host(np.float32).reshape(m, n)
    assert_bitexact(got, want, "c[m, n]")
    got = rocm.rocm_bit_linear_i8(DEV, ab, sab, qb, sqb, at(bias, 0), m, n, k).to_host(np.float32).reshape(n, m)
    assert_bitexact(got, want.T + bias, "layer")


# 256 x 128 tiles from just past the skinny kernel's range: one and several K steps, more of them than the
# two-workgroup form takes on larger outputs, ragged in every dimension, packed rows at each byte offset; one tile column
# where there are 144 tiles of 256 x 256 too.
@pytest.mark.parametrize("m,n,k,oa", [(4100, 1025, 16, 0), (2048, 1025, 960, 0), (2048, 1024, 960, 1), (2049, 1023, 960, 0), (2049, 1024, 976, 0), (4097, 1030, 176, 1), (2600, 1700, 2736, 0), (2570, 1665, 4112, 3),
                                      (4101, 1026, 176, 0), (4102, 1027, 336, 2), (4103, 1028, 16, 0),
                                      (6912, 601, 2560, 0), (129, 33000, 336, 2), (128, 33000, 176, 0), (36900, 65, 1296, 1),
                                      (36900, 128, 16, 0)])
def test_ternary_i8_mid_sizes(m, n, k, oa):
    print(f"ternary i8 mid m={m} n={n} k={k} packed+{oa}", flush=True)
    p = raw_packed(m, k, m + k)
    q = rng(n + k).integers(-128, 128, size=(n, k), dtype=np.int64).astype(np.int8)
    sa, sq, bias = normal((m,), 8, 1.0, 0.1), np.abs(normal((n,), 9, 0.02, 0.005)), normal((m,), 10)
    b = p.astype(np.int32)
    trits = np.stack([np.where(b < 243, b // 3 ** i % 3 - 1, 0) for i in range(5)], -1).reshape(m, -1)[:, :k]
    # every partial sum is a whole number below 2^24: exact in f32 in any order
    acc = (torch.from_numpy(trits.astype(np.float32)) @ torch.from_numpy(q.astype(np.float32)).t()).numpy()
    want = (acc * sa[:, None]) * sq[None, :]
    ab, qb, sab, sqb = at(p, oa), at(q, 0), at(sa, 0), at(sq, 0)
    got = rocm.rocm_ternary_matmul_i8(DEV, ab, sab, qb, sqb, m, n, k).to_host(np.float32).reshape(m, n)
    assert_bitexact(got, want, "c[m, n]")
    got = rocm.rocm_bit_linear_i8(DEV, ab, sab, qb, sqb, at(bias, 0), m, n, k).to_host(np.float32).reshape(n, m)
    assert_bitexact(got, want.T + bias, "layer")
