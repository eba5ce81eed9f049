"""End-to-end sparse decode layer on the GPU against the oracle.

BASELINE.json configs[0] against the golden fixture written by the compiled
reference; configs[2] (score N=32768 over the hot pool, select at the cap,
sparse attention) against the oracle: scores and ids bit-exact, attention
within 2e-3."""
from pathlib import Path

import numpy as np
import pytest
import torch

from hs_data import config1_inputs, f16_bits, from_dev, pool_rows, rng, rope_keys, to_dev
from test_gpu_attention import rel_err

pytestmark = pytest.mark.gpu
FIXTURE = Path(__file__).resolve().parent / "golden" / "config1.npz"


def test_config1_golden(hs):
    g = np.load(FIXTURE, allow_pickle=False)
    n = int(g["n"])
    q, k, _ = config1_inputs(0, n)
    partial = torch.zeros((n + 63) // 64, dtype=torch.int32, device="cuda")
    raw = hs.ops.score(to_dev(q), to_dev(k.reshape(-1)), n, head0_partial=partial)
    assert np.array_equal(from_dev(raw), g["raw"])
    ids, counts, _, status = hs.ops.select(raw, 32, n, n, float(g["alpha"]), float(g["ratio"]),
                                           scale_raw=True, head0_partial=partial)
    st = hs.ops.read_status(status)
    assert st["code"] == 0 and st["k"] == int(g["k"])
    assert st["boundary_tied_heads"] == int(g["boundary_tied_heads"])
    assert np.array_equal(from_dev(ids)[:, : st["k"]], g["ids"])
    assert np.array_equal(from_dev(counts), g["counts"])


@pytest.mark.parametrize("n,alpha", [(4096, 5.0), (32768, 5.0), (32768, 1.5)])
def test_config3_layer(hs, port, n, alpha):
    g = rng(3000 + n)
    k = rope_keys(n, 31 + n)
    v = f16_bits(g.standard_normal((n, 8, 128)))
    pool = pool_rows(k, v)
    q16 = f16_bits(g.standard_normal((32, 128)))
    q32 = g.standard_normal((32, 128)).astype(np.float32)
    scores, ids, counts, out, status = hs.ops.decode_layer(
        to_dev(q16), torch.from_numpy(q32).cuda(), to_dev(pool.reshape(-1)), n, alpha, 0.2)
    st = hs.ops.read_status(status)
    raw = port.score(q16, pool.reshape(-1), n, 2048)
    assert np.array_equal(from_dev(scores), raw)
    rc, kk, pids, pcounts, tied = port.select(port.scale(raw), 32, n, n, alpha, 0.2)
    assert st["code"] == 0 and st["k"] == kk and st["boundary_tied_heads"] == tied
    gids = from_dev(ids)[:, :kk]  # the layer lists each head's selection by ascending id
    assert np.array_equal(gids, np.sort(pids, axis=1)) and np.array_equal(from_dev(counts), pcounts)
    ref = port.attention(q32, pool.view(np.uint8).reshape(-1), [list(r) for r in pids])
    assert rel_err(out.cpu().numpy().astype(np.float64), ref) <= 2e-3
    if alpha == 5.0:
        assert kk == int(np.floor(n * np.float64(np.float32(0.2))))  # k reaches the cap


def test_layer_zero_selection_is_an_error(hs):
    n = 256
    g = rng(1)
    k = f16_bits(g.standard_normal((n, 8, 128)) * 0.01)
    k[7, 0, :] = f16_bits(np.full(128, 8.0))  # one token dominates head 0
    v = f16_bits(g.standard_normal((n, 8, 128)))
    pool = pool_rows(k, v)
    q16 = f16_bits(np.ones((32, 128)))
    q32 = np.ones((32, 128), dtype=np.float32)
    *_, status = hs.ops.decode_layer(to_dev(q16), torch.from_numpy(q32).cuda(),
                                     to_dev(pool.reshape(-1)), n, 0.5, 0.2)
    assert hs.ops.read_status(status)["code"] == hs.HS_ERR_ZERO_SELECTION


def test_layer_split_kv_arrays_equal_records(hs):
    # score over the K array's 2048 B rows and attention over the K and V
    # arrays: scores, ids, counts and output equal the 4096 B record layout's
    n = 32768
    g = rng(4242)
    k = rope_keys(n, 4243)
    v = f16_bits(g.standard_normal((n, 8, 128)))
    records = pool_rows(k, v)
    q16 = f16_bits(g.standard_normal((32, 128)))
    q32 = torch.from_numpy(g.standard_normal((32, 128)).astype(np.float32)).cuda()
    a = hs.ops.decode_layer(to_dev(q16), q32, to_dev(records.reshape(-1)), n, 5.0, 0.2)
    b = hs.ops.decode_layer(to_dev(q16), q32, to_dev(np.ascontiguousarray(records[:, :1024])), n,
                            5.0, 0.2, v_pool=to_dev(np.ascontiguousarray(records[:, 1024:])),
                            row_bytes=2048)
    sa, sb = hs.ops.read_status(a[4]), hs.ops.read_status(b[4])
    assert sa == sb and sa["code"] == 0
    kk = sa["k"]
    assert torch.equal(a[0], b[0])
    assert torch.equal(a[1][:, :kk], b[1][:, :kk])
    assert torch.equal(a[2], b[2]) and torch.equal(a[3], b[3])


@pytest.mark.parametrize("n", [1, 7, 64, 65, 1023, 1024, 2047, 2048, 2049, 4095, 8191, 8192, 8193])
def test_short_layer_edges(hs, port, n):
    # up to 8192 tokens one launch counts and selects, with 256 threads up
    # to 2048: runs of 8 ids, bitmap words and rows that end anywhere, ties
    # at the cut, signed zeros, all scores equal; 8193 takes the two launches
    for kind in ("gaussian", "coarse", "zero", "equal"):
        g = rng(n + len(kind))
        k = rope_keys(n, 5 + n)
        if kind == "coarse":  # few distinct scores: ties at the cut
            k = f16_bits(np.round(g.standard_normal((n, 8, 128))))
        elif kind == "zero":  # scores of both zeros at the cut
            k = f16_bits(np.where(g.random((n, 8, 1)) < 0.1, g.standard_normal((n, 8, 128)), 0.0))
        elif kind == "equal":
            k = np.broadcast_to(f16_bits(g.standard_normal((1, 8, 128))), (n, 8, 128)).copy()
        v = f16_bits(g.standard_normal((n, 8, 128)))
        pool = pool_rows(k, v)
        q16 = f16_bits(np.round(g.standard_normal((32, 128)) * 2) if kind == "coarse" else g.standard_normal((32, 128)))
        q32 = g.standard_normal((32, 128)).astype(np.float32)
        # (a few tokens: a margin that keeps every head's k above 0)
        alpha, ratio, fp32 = (4.0, 0.2, False) if n >= 64 else (100.0, 1.0, True)
        raw = port.score(q16, pool.reshape(-1), n, 2048)
        rc, kk, pids, pcounts, tied = port.select(port.scale(raw), 32, n, n, alpha, ratio, fp32)
        scores, ids, counts, out, status = hs.ops.decode_layer(
            to_dev(q16), torch.from_numpy(q32).cuda(), to_dev(pool.reshape(-1)), n, alpha, ratio, fp32_counts=fp32)
        st = hs.ops.read_status(status)
        assert np.array_equal(from_dev(scores), raw)
        assert st["code"] == rc == 0 and st["k"] == kk > 0 and st["boundary_tied_heads"] == tied, (kind, st, kk, tied)
        assert np.array_equal(from_dev(counts), pcounts)
        assert np.array_equal(from_dev(ids)[:, :kk], np.sort(pids, axis=1)), kind
        ref = port.attention(q32, pool.view(np.uint8).reshape(-1), [list(r) for r in pids])
        assert rel_err(out.cpu().numpy().astype(np.float64), ref) <= 2e-3


def test_short_layer_errors(hs, port):
    # the single launch's error paths: a nonfinite score in head 0 and in
    # another head, a threshold beyond F16; a call after each is clean
    n = 3000
    g = rng(77)
    v = f16_bits(g.standard_normal((n, 8, 128)))
    q32 = torch.from_numpy(g.standard_normal((32, 128)).astype(np.float32)).cuda()
    q16 = f16_bits(g.standard_normal((32, 128)))
    for bad_head, alpha, code in ((None, 5.0, 0), (0, 5.0, hs.HS_ERR_NONFINITE), (None, 5.0, 0),
                                  (7, 5.0, hs.HS_ERR_NONFINITE), (None, 70000.0, hs.HS_ERR_THRESHOLD), (None, 5.0, 0)):
        k = rope_keys(n, 5)
        if bad_head is not None:
            k[1234, bad_head] = 0x7C00  # inf: its products are inf or NaN
        *_, status = hs.ops.decode_layer(to_dev(q16), q32, to_dev(pool_rows(k, v).reshape(-1)), n, alpha, 0.2)
        st = hs.ops.read_status(status)
        assert st["code"] == code and (st["k"] == 600) == (code == 0)


@pytest.mark.parametrize("wait", [0, 1, 5000])
@pytest.mark.parametrize("n", [1500, 3001, 8192])
def test_short_layer_counts_missing_heads(hs, port, n, wait):
    # a workgroup that reads no other head's count (wait 0), or only those
    # published by its first look, counts the rest itself: the same layer,
    # errors included, on a workspace whose words all look published
    import ctypes
    g = rng(n)
    k, v = rope_keys(n, n), f16_bits(g.standard_normal((n, 8, 128)))
    q16 = f16_bits(g.standard_normal((32, 128)))
    q32 = g.standard_normal((32, 128)).astype(np.float32)
    kmax = int(np.floor(n * np.float64(np.float32(0.2))))
    dev = lambda shape, dt=torch.int32: torch.full(shape, -1, dtype=dt, device="cuda")
    P = lambda t: ctypes.c_void_p(t.data_ptr())
    ws = torch.full((hs.ops.decode_layer_workspace_bytes(n),), 0xFF, dtype=torch.uint8, device="cuda")
    for bad in (None, 0, 5):  # KV heads with a nonfinite key
        kk = k.copy()
        if bad is not None:
            kk[n // 2, bad] = 0x7C00  # inf: its products are inf or NaN
        pool = pool_rows(kk, v)
        pd, q16d, q32d = to_dev(pool.reshape(-1)), to_dev(q16), torch.from_numpy(q32).cuda()
        scores, ids, counts = dev((32, n), torch.float16), dev((32, kmax)), dev((32,))
        out, status = dev((32, 128), torch.float32), dev((4,))
        ws.fill_(0xFF)
        hs.check(hs.lib().hs_selftest_decode_layer(
            P(q16d), P(q32d), P(pd), ctypes.c_void_p(pd.data_ptr() + 2048), 4096, None, n, n, 4.0, 0.2, 0,
            P(scores), P(ids), kmax, P(counts), P(out), P(status), P(ws), wait,
            ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
        st = hs.ops.read_status(status)
        if bad is not None:  # no stale membership words: every head attends to nothing
            assert st["code"] == hs.HS_ERR_NONFINITE and torch.isnan(out).all()
            continue
        raw = port.score(q16, pool.reshape(-1), n, 2048)
        rc, k_want, pids, pcounts, tied = port.select(port.scale(raw), 32, n, n, 4.0, 0.2)
        assert np.array_equal(from_dev(scores), raw)
        assert rc == st["code"] == 0 and st["k"] == k_want > 0 and st["boundary_tied_heads"] == tied
        assert np.array_equal(from_dev(counts), pcounts)
        assert np.array_equal(from_dev(ids)[:, :k_want], np.sort(pids, axis=1))
        ref = port.attention(q32, pool.view(np.uint8).reshape(-1), [list(r) for r in pids])
        assert rel_err(out.cpu().numpy().astype(np.float64), ref) <= 2e-3


def test_selftest_layer_refuses_long_waits(hs):
    import ctypes
    assert hs.lib().hs_selftest_decode_layer(*[None] * 4, 4096, None, 1, 1, 1.0, 0.2, 0, None, None, 1, None, None,
                                             None, ctypes.c_void_p(256), 5001, None) == hs.HS_ERR_ARGUMENT
    assert "wait limit" in hs.last_error()


@pytest.mark.parametrize("n", [3001, 8192, 12001, 16384, 40001, 65536])
@pytest.mark.parametrize("row_bytes", [2048, 4096])
def test_row_mapped_layer_equals_plain(hs, n, row_bytes):
    # hs_decode_layer over a shuffled pool behind a row map, in every regime
    # of its launches (one launch of count and selection, chunks of 32, 64 and
    # 128 ids, streamed keys, two words per thread), as K and V arrays and as
    # KV records: every output equals the plain layer's bit for bit
    keys = torch.empty(n * 1024, dtype=torch.float16, device="cuda")
    values, q16 = torch.empty_like(keys), torch.empty(4096, dtype=torch.float16, device="cuda")
    hs.ops.fill_rope_keys(keys, n, 1024, 8, seed=n)
    hs.ops.fill_gaussian(values, seed=n + 1)
    hs.ops.fill_gaussian(q16, seed=n + 2)
    q32 = torch.randn((32, 128), generator=torch.Generator(device="cuda").manual_seed(n), device="cuda")
    k, v = keys.view(n, 1024), values.view(n, 1024)
    want = hs.ops.decode_layer(q16, q32, k, n, 5.0, 0.2, v_pool=v, row_bytes=2048)
    rows = n + 37  # rows of no token among them
    g = rng(n)
    place = torch.from_numpy(g.permutation(rows)[:n].astype(np.int64)).cuda()
    mk, mv = (torch.full((rows, 1024), float("nan"), dtype=torch.float16, device="cuda") for _ in range(2))
    mk[place], mv[place] = k, v
    pool = dict(pool=mk, v_pool=mv) if row_bytes == 2048 else dict(pool=torch.cat([mk, mv], dim=1).contiguous())
    got = hs.ops.decode_layer(q16, q32, pool.pop("pool"), n, 5.0, 0.2, rows=place.int(), row_bytes=row_bytes, **pool)
    st = hs.ops.read_status(want[4])
    assert hs.ops.read_status(got[4]) == st and st["code"] == 0 and st["k"] > 0
    kk = st["k"]
    assert torch.equal(got[0], want[0]) and torch.equal(got[1][:, :kk], want[1][:, :kk])
    assert torch.equal(got[2], want[2]) and torch.equal(got[3], want[3])
