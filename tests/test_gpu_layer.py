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


@pytest.mark.parametrize("n", [1500, 3001, 8192])
def test_short_layer_counts_missing_heads(hs, port, n):
    # a workgroup that stops waiting for the other heads' counts at once
    # counts them itself: the same selection, errors included
    import ctypes
    import subprocess
    names = subprocess.run(["nm", "-D", "--defined-only", str(hs.LIB_PATH)], capture_output=True, text=True,
                           check=True).stdout.split()
    fn = getattr(hs.lib(), next(x for x in names if "launch_layer_select" in x))
    P, U = ctypes.c_void_p, ctypes.c_uint32
    fn.restype = ctypes.c_int
    fn.argtypes = [P, U, ctypes.c_float, ctypes.c_float, U, P, P, ctypes.c_size_t, P, P, P, P, P, U]
    flags = hs.HS_SELECT_SCALE_RAW | hs.HS_SELECT_REQUIRE_K | hs.HS_SELECT_ID_ORDER
    g = rng(n)
    for bad in (None, 0, 9):
        raw = f16_bits(g.standard_normal((32, n)) * 20.0)
        if bad is not None:
            raw[bad, n // 2] = 0x7E00
        key = lambda b: np.where(b > 0x8000, b ^ 0xFFFF, (b & 0x7FFF) | 0x8000).astype(np.uint32)
        keys = np.where((raw[0] & 0x7FFF) > 0x7C00, 0, key(raw[0]))
        part = np.maximum.reduceat(keys, np.arange(0, n, 64)).astype(np.uint32)
        kmax = int(np.floor(n * np.float64(np.float32(0.2))))
        ids = torch.zeros((32, kmax), dtype=torch.int32, device="cuda")
        counts = torch.zeros(32, dtype=torch.int32, device="cuda")
        member = torch.zeros((32, (n + 31) // 32), dtype=torch.int32, device="cuda")
        status = hs.ops.new_status()
        ws = torch.zeros(hs.ops.select_workspace_bytes(32, n), dtype=torch.uint8, device="cuda")
        raw_d, part_d = to_dev(raw), to_dev(part)
        p = lambda t: t.data_ptr()
        assert fn(p(raw_d), n, 3.0, 0.2, flags, p(part_d), p(ids), kmax, p(counts), p(member), p(status), p(ws),
                  torch.cuda.current_stream().cuda_stream, 0) == 0
        st = hs.ops.read_status(status)
        if bad is not None:
            assert st["code"] == hs.HS_ERR_NONFINITE and not from_dev(member).any()
            continue
        rc, k, pids, pcounts, tied = port.select(port.scale(raw), 32, n, n, 3.0, 0.2)
        assert rc == st["code"] == 0 and st["k"] == k and st["boundary_tied_heads"] == tied
        assert np.array_equal(from_dev(counts), pcounts)
        assert np.array_equal(from_dev(ids)[:, :k], np.sort(pids, axis=1))
