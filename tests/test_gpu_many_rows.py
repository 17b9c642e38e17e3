"""Row counts at which a workgroup or a wave a row comes to 2^32 threads, more than one launch holds: the calls go in
bands of rows.  Rows around the buffer's ends, the bands' and the point where one launch would wrap, against the oracle."""
import numpy as np
import pytest

import oracle
from inputs import assert_bitexact, assert_close, int8_codes, normal, raw_packed

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
from kore_amd import rocm  # noqa: E402
from kore_amd.rocm import HipBuffer  # noqa: E402

DEV = 0
U32 = 2.0 ** -24


def big(rows, cols):
    """An unset device matrix, or a skip where the card has no room for it."""
    need = rows * cols * 4
    torch.cuda.empty_cache()
    if torch.cuda.mem_get_info()[0] < need + (4 << 30):
        pytest.skip(f"needs {need >> 30} GiB of device memory")
    return torch.empty((rows, cols), dtype=torch.float32, device="cuda:0")


def sample(rows):
    return sorted({r for r in (0, 1, 777, (1 << 21) - 1, 1 << 21, rows // 2, (1 << 23) + 1, rows - 5, rows - 1) if r < rows})


def fill(t, at, seed):
    x = normal((len(at), t.shape[1]), seed) * 3
    put(t, at, x)
    return x


def put(t, at, x):
    for r, row in zip(at, x):
        t[r].copy_(torch.from_numpy(row))


def rows_of(t, at):
    return np.stack([t[r].cpu().numpy() for r in at])


# Just past 2^32 threads at 512 and (1024 columns) at 128 threads a row.
@pytest.mark.parametrize("rows,cols", [((1 << 23) + 3, 2052), ((1 << 25) + 3, 1024)])
def test_softmax_many_rows(rows, cols):
    print(f"softmax rows={rows} cols={cols}", flush=True)
    t, at = big(rows, cols), sample(rows)
    b = HipBuffer.from_tensor(t.view(-1))
    x = fill(t, at, 1)
    rocm.rocm_softmax_f32(DEV, b, rows, cols, b)
    assert_close(rows_of(t, at), oracle.softmax(x), rtol=1e-5 + cols * U32, what="softmax")
    x = fill(t, at, 2)
    rocm.rocm_softmax_causal_f32(DEV, b, rows, cols, 5, b)
    want = np.concatenate([oracle.softmax_causal(x[i:i + 1], 5 + r) for i, r in enumerate(at)])
    assert_close(rows_of(t, at), want, rtol=1e-5 + cols * U32, what="causal")
    x = fill(t, at, 3)
    targets = torch.full((rows,), 7.0, device="cuda:0")
    rocm.rocm_cross_entropy_backward_f32(DEV, b, HipBuffer.from_tensor(targets), rows, cols, b)
    want = oracle.softmax(x).astype(np.float64)
    want[:, 7] -= 1.0
    assert_close(rows_of(t, at), want / rows, rtol=1e-5 + cols * U32, atol=1e-6 / rows, what="cross entropy")


@pytest.mark.parametrize("rows,cols", [((1 << 23) + 3, 1025), ((1 << 23) + 3, 2052)])
def test_softmax_backward_many_rows(rows, cols):
    print(f"softmax backward rows={rows} cols={cols}", flush=True)
    t, at = big(rows, cols), sample(rows)
    b = HipBuffer.from_tensor(t.view(-1))
    y = oracle.softmax(fill(t, at, 1))
    put(t, at, y)
    rocm.rocm_softmax_backward_f32(DEV, b, b, rows, cols, b)
    assert_close(rows_of(t, at), oracle.softmax_backward(y, y), rtol=1e-5 + cols * U32, atol=1e-6, what="backward")

# Just past 2^32 threads at a wave a row, and at a thread a row; odd bands start a ragged row anywhere.
@pytest.mark.parametrize("rows,cols", [((1 << 26) + 3, 17), ((1 << 26) + 3, 3), ((1 << 32) + 3, 1)])
def test_norm_family_many_rows(rows, cols):
    print(f"norm family rows={rows} cols={cols}", flush=True)
    t, at = big(rows, cols), sample(rows)
    w = normal((cols,), 4, 1.0, 0.02)
    xb, wb = HipBuffer.from_tensor(t.view(-1)), HipBuffer.from_host(DEV, w)
    x = fill(t, at, 1)
    q, scale = rocm.rocm_rms_norm_quant_i8(DEV, xb, wb, rows, cols, 1e-6)
    want_q, want_s = oracle.rms_norm_quant_i8(x, w, 1e-6)
    assert_bitexact(rows_of(q.tensor(torch.int8)[:rows * cols].view(rows, cols), at), want_q, "codes")
    assert_bitexact(rows_of(scale.tensor(torch.float32)[:rows].view(rows, 1), at)[:, 0], want_s, "scales")
    y = rocm.rocm_fused_rms_norm_silu_gate_f32(DEV, xb, wb, xb, rows, cols, 1e-6)
    assert_close(rows_of(y.tensor(torch.float32)[:rows * cols].view(rows, cols), at),
                 oracle.rms_norm_silu_gate(x, w, x, 1e-6), what="silu gate")
    rocm.rocm_rms_norm_f32(DEV, xb, wb, rows, cols, 1e-6, out=xb)
    assert_bitexact(rows_of(t, at), oracle.rms_norm(x, w, 1e-6), "rms_norm")


def test_elementwise_many_threads():
    n = (1 << 34) + 5
    print(f"silu and mul in place n={n}", flush=True)
    t = big(n, 1).view(-1)
    b = HipBuffer.from_tensor(t)
    spots = [0, 4096, (1 << 33) - 8, (1 << 33) + 100, n // 2 + 64, n - 8]
    x = normal((len(spots), 8), 5)
    put(t, [slice(i, i + 8) for i in spots], x)
    rocm.rocm_silu_f32(DEV, b, n, b)
    y = rows_of(t, [slice(i, i + 8) for i in spots])
    assert_close(y, oracle.silu(x), what="silu")
    rocm.rocm_mul_f32(DEV, b, b, n, b)
    assert_bitexact(rows_of(t, [slice(i, i + 8) for i in spots]), y * y, "mul")


def test_embedding_many_ids():
    n, dim, vocab = (1 << 26) + 3, 4, 1000
    print(f"embedding n={n}", flush=True)
    table = normal((vocab, dim), 6)
    ids = (torch.arange(n, device="cuda:0", dtype=torch.int32) * 7) % vocab
    out = rocm.rocm_embedding_f32(DEV, HipBuffer.from_host(DEV, table), HipBuffer.from_tensor(ids), n, vocab, dim)
    got = out.tensor(torch.float32).view(n, dim)
    at = sample(n)
    assert_bitexact(rows_of(got, at), oracle.embedding(table, np.array([int(ids[r]) for r in at], np.int32)), "rows")


# One long sequence and many short ones, at 128 threads a token of 32 floats.
@pytest.mark.parametrize("batch,seq", [(1, (1 << 25) + 3), ((1 << 22) + 1, 9)])
def test_rope_many_tokens(batch, seq):
    print(f"rope batch={batch} seq={seq}", flush=True)
    t = big(batch * seq, 32)
    at = sample(batch * seq)
    x = fill(t, at, 7)
    inv = rocm.rocm_rope_inv_freq_f32(DEV, 32, 10000.0)
    rocm.rocm_rope_f32(DEV, HipBuffer.from_tensor(t.view(-1)), inv, batch, seq, 1, 32, 3, False)
    want = np.concatenate([oracle.rope(x[i].reshape(1, 1, 1, 32), 3 + r % seq, 10000.0).reshape(1, 32)
                           for i, r in enumerate(at)])
    assert_close(rows_of(t, at), want, what="rope")


def test_rms_norm_backward_many_rows():
    rows, cols = (1 << 30) + 3, 4
    print(f"rms_norm_backward rows={rows}", flush=True)
    x, dy, dx = (big(rows, cols) for _ in range(3))
    x.fill_(1.0)
    dy.zero_()
    at, g = sample(rows), normal((cols,), 8, 1.0, 0.02)
    xs, ds = fill(x, at, 9), fill(dy, at, 10)
    dxb, dgb = rocm.rocm_rms_norm_backward_f32(
        DEV, HipBuffer.from_tensor(dy.view(-1)), HipBuffer.from_tensor(x.view(-1)), HipBuffer.from_host(DEV, g), rows,
        cols, 1e-5, grad_input=HipBuffer.from_tensor(dx.view(-1)))
    want_dx, want_dg = oracle.rms_norm_backward(ds, xs, g, 1e-5)  # the other rows' dy is 0
    assert_close(rows_of(dx, at), want_dx, rtol=1e-4, atol=1e-5, what="dx")
    assert_close(dgb.to_host(np.float32)[:cols], want_dg, rtol=1e-5, atol=1e-5, what="dgamma")


def ternary_rows(m, n, k):
    """Sampled weight rows with bytes, scales and bias of their own among rows of zero trits, scale 1 and bias 0."""
    torch.cuda.empty_cache()
    need = m * ((k + 4) // 5 + 8 + 4 * n)
    if torch.cuda.mem_get_info()[0] < need + (4 << 30):
        pytest.skip(f"needs {need >> 30} GiB of device memory")
    at = sample(m)
    a = torch.full((m, (k + 4) // 5), 121, dtype=torch.uint8, device="cuda:0")
    sa, bias = torch.ones(m, device="cuda:0"), torch.zeros(m, device="cuda:0")
    packed, scales, add = raw_packed(len(at), k, k), normal((len(at),), 11, 1.0, 0.1), normal((len(at),), 12)
    put(a, at, packed), put(sa.view(m, 1), at, scales[:, None]), put(bias.view(m, 1), at, add[:, None])
    c = torch.full((m * n,), 7.0, device="cuda:0")
    bufs = [HipBuffer.from_tensor(t.view(-1)) for t in (a, sa, bias, c)]
    return at, packed, scales, add, c, bufs


def check_ternary(c, m, n, at, want, add, matmul, layer):
    matmul()
    assert_bitexact(rows_of(c.view(m, n), at), want, "c[m, n]")
    if not want.any():
        assert torch.count_nonzero(c) == 0, "c[m, n] of no columns"
    c.fill_(7.0)
    layer()
    assert_bitexact(rows_of(c.view(n, m).T, at), want + add[:, None], "layer")


# Just past 2^32 threads: 16 a weight row for one code, 4 for two with K not a multiple of 8, one an output for K = 0.
# Then bands of 256 x 128 and 128 x 128 tiles, the last one short, and 256 x 192 and 256 x 256 tiles, which have none.
@pytest.mark.parametrize("m,n,k", [((1 << 28) + 5, 1, 8), ((1 << 30) + 5, 2, 17), ((1 << 26) + 3, 64, 0),
                                   ((1 << 24) + 5, 70, 16), ((1 << 24) + 261, 130, 1296), ((1 << 24) + 5, 200, 4176),
                                   ((1 << 24) + 133, 70, 17)])
def test_ternary_i8_many_rows(m, n, k):
    print(f"ternary i8 m={m} n={n} k={k}", flush=True)
    at, packed, scales, add, c, (ab, sab, bb, cb) = ternary_rows(m, n, k)
    q, sq = int8_codes(n, k, 13), np.abs(normal((n,), 14, 0.02, 0.005))
    qb, sqb = HipBuffer.from_host(DEV, q), HipBuffer.from_host(DEV, sq)
    want = oracle.ternary_matmul_i8(packed, scales, q, sq, len(at), n, k)
    check_ternary(c, m, n, at, want, add, lambda: rocm.rocm_ternary_matmul_i8(DEV, ab, sab, qb, sqb, m, n, k, out=cb),
                  lambda: rocm.rocm_bit_linear_i8(DEV, ab, sab, qb, sqb, bb, m, n, k, out=cb))


# Just past 2^32 threads: 7 a weight row for one column, 8 for five with K = 0; then bands of the 16 x 16 kernel.
@pytest.mark.parametrize("m,n,k", [((1 << 30) + 5, 1, 7), ((1 << 29) + 5, 5, 0), ((1 << 24) + 67, 20, 6)])
def test_ternary_f32_many_rows(m, n, k):
    print(f"ternary f32 m={m} n={n} k={k}", flush=True)
    at, packed, scales, add, c, (ab, sab, bb, cb) = ternary_rows(m, n, k)
    b = normal((k, n), 15)
    b0, b1 = HipBuffer.from_host(DEV, b), HipBuffer.from_host(DEV, np.ascontiguousarray(b.T))
    want = oracle.ternary_matmul(packed, scales, b, len(at), n, k)
    check_ternary(c, m, n, at, want, add, lambda: rocm.rocm_ternary_matmul_f32(DEV, ab, sab, b0, m, n, k, out=cb),
                  lambda: rocm.rocm_bit_linear_f32(DEV, ab, sab, b1, bb, m, n, k, out=cb))


# 64 threads a row of up to 1280 columns, whole float4 or not, and 256 of more than 2560.
@pytest.mark.parametrize("m,k", [((1 << 26) + 5, 4), ((1 << 26) + 5, 3), ((1 << 24) + 5, 2564)])
def test_pack_weights_many_rows(m, k):
    print(f"pack m={m} k={k}", flush=True)
    kp = (k + 4) // 5
    t, at = big(m, k + (kp + 7) // 4), sample(m)
    w = t.view(-1)[:m * k].view(m, k).zero_()
    x = fill(w, at, 16)
    p, sc = rocm.rocm_pack_weights_ternary(DEV, HipBuffer.from_tensor(w), m, k, 0.5)
    want_p, want_s = oracle.pack_weights_ternary(x, 0.5)
    assert_bitexact(rows_of(p.tensor(torch.uint8)[:m * kp].view(m, kp), at), want_p, "packed")
    assert_bitexact(rows_of(sc.tensor(torch.float32)[:m].view(m, 1), at)[:, 0], want_s, "scales")
