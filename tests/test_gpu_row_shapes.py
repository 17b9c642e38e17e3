"""Row kernels on long and ragged rows: lengths around each change of plan,
views at every 4-byte offset, against the oracle (bit-exact where the entry
point is) with the tolerances of test_gpu_parity.py."""
import numpy as np
import pytest

import oracle
from inputs import assert_bitexact, assert_close, assert_close_scaled, normal, rmsnorm_inputs

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
from kore_amd import rocm  # noqa: E402
from kore_amd.rocm import HipBuffer  # noqa: E402

DEV = 0
U32 = 2.0 ** -24


def at(arr: np.ndarray, offset: int) -> HipBuffer:
    """arr on the device, starting `offset` floats past a 16-byte boundary."""
    flat = np.ascontiguousarray(arr).reshape(-1)
    t = torch.empty(flat.size + 8, dtype=torch.from_numpy(flat).dtype, device="cuda:0")
    v = t[offset:offset + flat.size]
    v.copy_(torch.from_numpy(flat))
    return HipBuffer.from_tensor(v)


def room(n: int, offset: int):
    """A NaN-filled buffer of n floats at `offset`, and the whole allocation, whose guards must stay NaN."""
    t = torch.full((n + 16,), float("nan"), device="cuda:0")
    return HipBuffer.from_tensor(t[8 + offset - 4:8 + offset - 4 + n]), t, 8 + offset - 4


def inside(t, start: int, n: int) -> np.ndarray:
    h = t.cpu().numpy()
    assert np.isnan(h[:start]).all() and np.isnan(h[start + n:]).all(), "written outside the output"
    return h[start:start + n]


# One float4 per lane and wave more or less around 256, 512, 1024, 4096, 6144, 8192, 12288 and 16384 columns, each with a
# row more than the generic path takes and odd numbers of rows; 16385 is the generic path's, as are the first rows of each
# range (a few of any length, more odd than even ones).  Rows: fewer than, and not a multiple of, a workgroup's.
@pytest.mark.parametrize("rows,cols,offset", [
    (1, 1, 0), (3, 5, 1), (45, 5, 1), (9, 255, 2), (44, 255, 2), (45, 255, 2), (601, 258, 3), (7, 513, 0), (44, 513, 0), (45, 513, 0), (73, 513, 0),
    (44, 1024, 1), (45, 1024, 1), (45, 769, 3), (46, 767, 2), (72, 1021, 1), (75, 1021, 1), (513, 1030, 2), (36, 2049, 0), (37, 2049, 0), (6, 3071, 3), (39, 3071, 3),
    (1100, 4095, 1), (4, 4096, 1), (37, 4096, 1), (3, 4097, 0), (9, 4097, 0), (8, 4100, 0), (9, 4100, 0), (8, 5120, 1),
    (2, 5121, 0), (18, 4100, 1), (19, 4100, 1), (10, 5120, 0), (11, 5120, 0), (9, 6144, 0), (11, 6144, 0), (18, 8189, 2),
    (19, 8189, 2), (20, 8192, 1), (4, 8196, 0), (9, 12285, 3), (11, 12285, 3), (515, 6143, 2), (2, 6144, 0), (3, 6145, 1), (520, 8192, 0), (2, 8191, 0), (3, 8193, 3), (2, 12288, 0),
    (2, 12291, 1), (259, 16384, 0), (2, 16383, 2), (2, 16385, 0)])
def test_rms_norm_backward_long_and_ragged(rows, cols, offset):
    print(f"rms_norm_backward rows={rows} cols={cols} offset={offset}", flush=True)
    x, g = rmsnorm_inputs(rows, cols, seed=rows + cols)
    dy = normal((rows, cols), rows * 3 + cols)
    dx, dx_all, dx_at = room(rows * cols, offset)
    dg, dg_all, dg_at = room(cols, offset)
    ws, ws_all, ws_at = room(rocm.rocm_rms_norm_backward_workspace_bytes(rows, cols) // 4, offset)
    rocm.rocm_rms_norm_backward_f32(DEV, at(dy, offset), at(x, offset), at(g, offset), rows, cols, 1e-5, ws, dx, dg)
    torch.cuda.synchronize()
    inside(ws_all, ws_at, ws.nbytes // 4)
    dx_w, dg_w = oracle.rms_norm_backward(dy, x, g, 1e-5)
    x64, dy64, g64 = (a.astype(np.float64) for a in (x, dy, g))
    inv = 1.0 / np.sqrt((x64 * x64).mean(1, keepdims=True) + 1e-5)
    terms = np.abs(x64 * dy64 * g64).sum(1, keepdims=True) * inv ** 3 / cols
    # dx is a difference of two terms, each with a sum of cols (rows for dgamma) roundings on either side
    assert_close_scaled(inside(dx_all, dx_at, rows * cols).reshape(rows, cols), dx_w,
                        np.abs(g64 * inv * dy64) + terms * np.abs(x64), rtol=1e-5 + cols * U32, what="dx")
    assert_close_scaled(inside(dg_all, dg_at, cols), dg_w, np.abs(dy64 * x64 * inv).sum(0), rtol=1e-5 + rows * U32,
                        what="dgamma")


@pytest.mark.parametrize("rows,cols", [(700, 8192), (85, 1001), (65, 1001)])
def test_rms_norm_backward_dgamma_over_gamma(rows, cols):
    """grad_gamma may be gamma's buffer; every row of dx uses the old gamma."""
    x, g = rmsnorm_inputs(rows, cols, seed=3)
    dy = normal((rows, cols), 4)
    want = rocm.rocm_rms_norm_backward_f32(DEV, at(dy, 0), at(x, 0), at(g, 0), rows, cols, 1e-5)
    gb = at(g, 0)
    dx, dg = rocm.rocm_rms_norm_backward_f32(DEV, at(dy, 0), at(x, 0), gb, rows, cols, 1e-5, grad_gamma=gb)
    torch.cuda.synchronize()
    assert dx.to_host().tobytes() == want[0].to_host().tobytes()
    assert dg.to_host()[:cols * 4].tobytes() == want[1].to_host()[:cols * 4].tobytes()


# ----------------------------------------------------------- softmax family
# Tolerances as in test_gpu_parity.py: 1e-5 against 64 bits; 1e-5 plus one rounding per term that the oracle's
# left-to-right sums take.  Lengths: each plan's first and last (wave, workgroup, the long kernel's 8, 16 and 24 float4 a
# thread and its LDS chunks, the loop), whole and ragged, at every 4-byte offset.
SM_LENGTHS = [(9, 3, 1), (5, 250, 2), (6, 257, 3), (7, 511, 0), (5, 1023, 1), (3, 1024, 2), (3, 2047, 0), (3, 2048, 1),
              (2, 4093, 3), (2, 8189, 0), (2, 16383, 2), (2, 16385, 0), (2, 16388, 0), (2, 32768, 0), (2, 32769, 1),
              (2, 65536, 0), (2, 65539, 0), (2, 98304, 3), (2, 98308, 0), (2, 131071, 0), (2, 135168, 0),
              (2, 135169, 0)]
# The same around the lengths and row counts where a row's kernel changes: a thread a float or a wave for a ragged
# backward of up to 512 columns, one or two waves a row to 1024, one wave, 256 or 512 threads from 2049 to 4096 (whole
# and ragged, forward and backward each have their own counts), 256 or 512 from 8193.
SM_LENGTHS += [(5, 513, 2), (5, 768, 1), (5, 769, 1), (3, 771, 0), (6, 960, 0), (6, 961, 0), (7, 964, 0), (5, 1021, 3),
               (1792, 101, 1), (1793, 102, 3), (1793, 301, 2), (1537, 1001, 1), (1537, 1024, 0), (2561, 1024, 0),
               (2049, 964, 0), (5120, 801, 2), (768, 2052, 0), (769, 2052, 0), (1537, 2052, 0), (2305, 2049, 3),
               (3073, 2564, 0), (3073, 3073, 1), (3073, 3076, 0), (512, 8196, 0), (513, 8196, 0), (513, 8193, 1)]


def _rows_with_specials(rows, cols, seed):
    x = normal((rows, cols), seed) * 3
    x[0, cols // 2:] -= 40.0          # a max early in the row, and late
    x[-1, :cols // 2] -= 40.0
    x[0, 0::7] = -np.inf              # threads that meet nothing but -inf
    return x


def _soft64(x):
    e = np.exp(x.astype(np.float64) - x.max(-1, keepdims=True).astype(np.float64))
    return e / e.sum(-1, keepdims=True)


@pytest.mark.parametrize("rows,cols,offset", SM_LENGTHS)
def test_softmax_family_long_and_ragged(rows, cols, offset):
    print(f"softmax family rows={rows} cols={cols} offset={offset}", flush=True)
    x = _rows_with_specials(rows, cols, cols)
    n = rows * cols

    def out_of(call):
        b, t, start = room(n, offset)
        call(b)
        torch.cuda.synchronize()
        return inside(t, start, n).reshape(rows, cols)

    want = _soft64(x)
    got = out_of(lambda b: rocm.rocm_softmax_f32(DEV, at(x, offset), rows, cols, b))
    assert_close(got, want, what="softmax vs f64")
    assert_close(got, oracle.softmax(x), rtol=1e-5 + cols * U32, what="softmax vs oracle")

    back = cols // 3  # row r keeps back + r + 1 columns
    got = out_of(lambda b: rocm.rocm_softmax_causal_f32(DEV, at(x, offset), rows, cols, back, b))
    want_c = np.zeros((rows, cols))
    for r in range(rows):
        keep = min(back + r + 1, cols)
        if np.isfinite(x[r, :keep]).any():
            want_c[r, :keep] = _soft64(x[r:r + 1, :keep])[0]
        else:
            want_c[r, :keep] = np.nan
        assert (got[r, keep:] == 0.0).all()
    assert_close(got, want_c, what="causal vs f64")

    y, dy = oracle.softmax(x), normal((rows, cols), cols + 1)
    got = out_of(lambda b: rocm.rocm_softmax_backward_f32(DEV, at(dy, offset), at(y, offset), rows, cols, b))
    y64, dy64 = y.astype(np.float64), dy.astype(np.float64)
    scale = np.abs(y64) * (np.abs(dy64) + np.abs(y64 * dy64).sum(-1, keepdims=True))
    assert_close_scaled(got, oracle.softmax_backward(dy, y), scale, rtol=1e-5 + cols * U32, what="backward")

    t = np.array([(cols - 1 - 5 * r) % cols for r in range(rows)], np.float32)  # the last columns, a ragged tail's too
    ref = want.copy()
    ref[np.arange(rows), t.astype(np.int64)] -= 1.0
    got = out_of(lambda b: rocm.rocm_cross_entropy_backward_f32(DEV, at(x, offset), at(t, 0), rows, cols, b))
    assert_close(got, ref / rows, what="cross entropy vs f64")
    b = at(x, offset)  # in place
    rocm.rocm_cross_entropy_backward_f32(DEV, b, at(t, 0), rows, cols, b)
    assert b.to_host(np.float32).tobytes() == got.tobytes()


@pytest.mark.parametrize("cols", [1001, 20000, 70001])
def test_softmax_long_and_ragged_nonfinite_rows(cols):
    x = normal((6, cols), cols) * 2
    x[0, 5] = np.nan
    x[1, :] = -np.inf
    x[2, cols - 1] = np.inf
    x[3, :-1] = -np.inf
    x[4] = -3e38
    x[5, 0] = 3e38
    for got, want in ((rocm.rocm_softmax_f32(DEV, at(x, 1), 6, cols), oracle.softmax(x)),
                      (rocm.rocm_softmax_causal_f32(DEV, at(x, 1), 6, cols, cols), oracle.softmax_causal(x, cols)),
                      (rocm.rocm_softmax_causal_f32(DEV, at(x, 0), 6, cols, 3), oracle.softmax_causal(x, 3))):
        got = got.to_host(np.float32).reshape(6, cols)
        assert_close(got, want, rtol=1e-5 + cols * U32, what="nonfinite rows")


# ------------------------------------------------- RMSNorm, pre-quant, gate
# Bit-exact for every plan: one wave a row to 3072 columns, two to 4096, four to 16384, each at its first and last
# length, whole, partly filled (a wave without any column) and ragged; 16385 is the scalar kernel's, as are the shortest rows and
# many of up to 48 columns.
NORM_LENGTHS = [(3, 1, 1), (5, 6, 3), (65, 3, 1), (70, 4, 0), (66, 7, 2), (511, 4, 0), (512, 4, 0), (4400, 8, 0),
                (4399, 8, 0), (3200, 8, 1), (3199, 9, 1), (12400, 16, 0), (12399, 16, 0), (8600, 17, 3), (17600, 32, 1),
                (17600, 32, 0), (18200, 33, 2), (18199, 33, 2), (26000, 46, 1), (28000, 49, 3), (65536, 25, 1),
                (65537, 25, 1), (98304, 25, 2), (98305, 25, 2), (140000, 24, 3), (300, 255, 2), (7, 1021, 1), (9, 1537, 0), (260, 2561, 3), (300, 3071, 0),
                (5, 3072, 0), (300, 3073, 0), (3, 3076, 0), (2, 4095, 2), (3, 4096, 1), (300, 4097, 0), (2, 4100, 0), (5, 5119, 1), (270, 5120, 0), (3, 6144, 0),
                (300, 6912, 0), (3, 6915, 2), (2, 7168, 0), (4, 7172, 0), (300, 8192, 0), (3, 8191, 3), (2, 8193, 0),
                (2, 9000, 0), (3, 10240, 0), (2, 12285, 1), (3, 12288, 0), (259, 14336, 0), (2, 16383, 2),
                (3, 16384, 0), (2, 16385, 0)]


def _norm_rows(rows, cols, seed):
    """Ordinary rows with outliers, and rows whose running sum creeps, overflows, vanishes or holds NaN."""
    x = normal((rows, cols), seed)
    x[normal((rows, cols), seed + 1) > 2.3] *= np.float32(20.0)
    if rows > 2:
        x[1] *= np.float32(2.0 ** -70)
        x[2] = np.float32(1e19)
    if rows > 6:
        x[3] = 0.0
        x[4, cols // 2] = np.nan
        x[5, -1] = np.inf
        x[6, cols // 2:] = 0.0
    return x


@pytest.mark.parametrize("rows,cols,offset", NORM_LENGTHS)
def test_norm_family_long_and_ragged_bit_exact(rows, cols, offset):
    print(f"norm family rows={rows} cols={cols} offset={offset}", flush=True)
    x, w = _norm_rows(rows, cols, cols), normal((cols,), cols + 2, 1.0, 0.02)
    n = rows * cols
    b, t, start = room(n, offset)
    rocm.rocm_rms_norm_f32(DEV, at(x, offset), at(w, offset), rows, cols, 1e-6, b)
    torch.cuda.synchronize()
    got = inside(t, start, n).reshape(rows, cols)
    assert_bitexact(got, oracle.rms_norm(x, w, 1e-6), "rms_norm")
    q = torch.full((n + 16,), 99, dtype=torch.int8, device="cuda:0")
    s, s_all, s_at = room(rows, offset)
    rocm.rocm_rms_norm_quant_i8(DEV, at(x, offset), at(w, offset), rows, cols, 1e-6,
                                HipBuffer.from_tensor(q[4 + offset:4 + offset + n]), s)
    torch.cuda.synchronize()
    q = q.cpu().numpy()
    assert (q[:4 + offset] == 99).all() and (q[4 + offset + n:] == 99).all()
    want_q, want_s = oracle.rms_norm_quant_i8(x, w, 1e-6)
    assert_bitexact(q[4 + offset:4 + offset + n].reshape(rows, cols), want_q, "codes")
    assert_bitexact(inside(s_all, s_at, rows), want_s, "scales")
    z = normal((rows, cols), cols + 3) * 3
    b, t, start = room(n, offset)
    rocm.rocm_fused_rms_norm_silu_gate_f32(DEV, at(x, offset), at(w, offset), at(z, offset), rows, cols, 1e-6, b)
    torch.cuda.synchronize()
    with np.errstate(all="ignore"):
        assert_close(inside(t, start, n).reshape(rows, cols), oracle.rms_norm_silu_gate(x, w, z, 1e-6),
                     what="silu gate")


@pytest.mark.parametrize("cols", [3584, 4097, 6912, 8192, 14336])
def test_norm_in_place_rows_of_several_waves(cols):
    x, w = normal((70, cols), 5), normal((cols,), 6, 1.0, 0.02)
    b = at(x, 0)
    rocm.rocm_rms_norm_f32(DEV, b, at(w, 0), 70, cols, 1e-6, out=b)
    assert_bitexact(b.to_host(np.float32).reshape(70, cols), oracle.rms_norm(x, w, 1e-6), "in place")
