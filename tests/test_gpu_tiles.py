"""Attention at every query shape the reference takes (sj_kvarn_cuda.cuh:102-135: any n_q x n_head): the query
rows of a KV head (n_q positions x the GQA group) are cut into 16-row tiles, up to 8 per launch, on the matrix-core
kernels (every scalar and trellis body at D = 128 and 256).

Bar: |gpu - oracle| <= 1e-3 + 1e-3 |oracle| per value against the oracle's position-ordered loop
(sj_kvarn.h:1535-1564), the BASELINE tolerance; the reference's own device test (tests/test_cuda.cu:84-135)
also reports the relative L2 error of each row, which is bounded here by 1e-3.
"""
import ctypes as C
import os
import sys
import threading

import numpy as np
import pytest

import cabi
import inputs

sys.path.insert(0, cabi.PKG)
import sjk  # noqa: E402

from test_gpu_layer import device_context, make_pair  # noqa: E402

pytestmark = pytest.mark.gpu
ATOL = RTOL = 1e-3
N_THREADS = min(16, os.cpu_count() or 1)


def say(*a):
    print(*a, flush=True)


@pytest.fixture(scope="module")
def lib():
    return sjk.load()


@pytest.fixture(scope="module")
def dev():
    d = sjk.Device()
    yield d
    d.free_all()


def oracle_rows(oracle, OL, B, N, q, qpos0, scale, rows):
    """the oracle's layer_attend_row for (iq, hq) pairs, on host threads"""
    n_q, n_head, D = q.shape
    gq = n_head // OL.cfg.n_head_kv
    out = {}

    def work(k):
        for iq, hq in rows[k::N_THREADS]:
            o = np.zeros(D, np.float32)
            qq = np.ascontiguousarray(q[iq, hq])
            oracle.layer_attend_row(C.byref(OL), B, N, cabi.ptr(qq, cabi.f32p), hq // gq, qpos0 + iq, scale,
                                    cabi.ptr(o, cabi.f32p))
            out[(iq, hq)] = o

    ths = [threading.Thread(target=work, args=(k,)) for k in range(N_THREADS)]
    for t in ths:
        t.start()
    for t in ths:
        t.join()
    return out


def check_rows(got, want):
    worst, worst_l2 = 0.0, 0.0
    for (iq, hq), w in want.items():
        g = got[iq, hq]
        err = np.abs(g - w)
        assert np.all(err <= ATOL + RTOL * np.abs(w)), "row (%d,%d) max abs err %g" % (iq, hq, err.max())
        worst = max(worst, float((err / (ATOL + RTOL * np.abs(w))).max()))
        n2 = float(np.sum(w.astype(np.float64) ** 2))
        worst_l2 = max(worst_l2, float(np.sqrt(np.sum((g - w).astype(np.float64) ** 2) / (n2 if n2 > 0 else 1.0))))
    return worst, worst_l2


def attend(lib, dev, view, B, N, qpos0, q, scale):
    dq, do = dev.put(q), dev.alloc(q.nbytes)
    sjk.check(lib.sjk_hip_attend(C.byref(view), B, N, qpos0, q.shape[0], q.shape[1], dq, scale, do, None), "attend")
    got = dev.get(do, q.nbytes, np.float32).reshape(q.shape)
    dev.free(dq)
    dev.free(do)
    return got


def test_reference_device_test_shape(oracle, lib):
    """The reference's own device attention test (tests/test_cuda.cu:84-135): D = 256, 2 KV heads, 3/3 trellis
    body, tail 256 / tail_max 512, 1200 positions stored in ubatches of 16 through the host API, then the last
    16 positions with 4 query heads each (32 query rows per KV head: two tiles). The cache is built through
    libsjk's sj_kvarn_* calls exactly as the reference test builds its own, and must equal the oracle's
    byte for byte."""
    D, H, NPOS, NQ, HQ = 256, 2, 1200, 16, 4
    rng = np.random.default_rng(99)
    x = (rng.standard_normal((NPOS, H * D)) / 1024.0).astype(np.float32)
    q = (rng.standard_normal((NPOS, HQ, D)) / 1024.0).astype(np.float32)
    layers = []
    for api in (oracle, lib):
        cfg = (cabi.Config if api is oracle else sjk.Config).from_buffer_copy(bytes(oracle.config_default(D, H, 2048, 64)))
        cfg.bits_k, cfg.bits_v, cfg.tail, cfg.tail_max = 3, 3, 256, 512
        L = cabi.Layer() if api is oracle else sjk.Layer()
        if api is oracle:
            assert oracle.layer_init(C.byref(L), C.byref(cfg)) == 0
            pol = cabi.Policy()
            oracle.policy_init(C.byref(pol), cfg.sink, cfg.tail, cfg.tail_max, 128, 0)
            begin, commit, seal, store = (oracle.policy_begin_ubatch, oracle.policy_commit, oracle.layer_seal,
                                          oracle.layer_store)
        else:
            sjk.check(lib.sj_kvarn_layer_init(C.byref(L), C.byref(cfg)), "layer_init")
            pol = sjk.Policy()
            lib.sj_kvarn_policy_init(C.byref(pol), cfg.sink, cfg.tail, cfg.tail_max, 128, 0)
            begin, commit, seal, store = (lib.sj_kvarn_policy_begin_ubatch, lib.sj_kvarn_policy_commit,
                                          lib.sj_kvarn_layer_seal, lib.sj_kvarn_layer_store)
        for p in range(0, NPOS, 16):
            if begin(C.byref(pol), p, 16) > pol.B:
                seal(C.byref(L), pol.B, pol.B_pending)
            commit(C.byref(pol))
            for i in range(p, p + 16):
                store(C.byref(L), i, x[i].ctypes.data_as(cabi.f32p), x[(i * 7) % NPOS].ctypes.data_as(cabi.f32p))
        layers.append((L, pol))
    (OL, opol), (PL, ppol) = layers
    d = sjk.Device()
    try:
        assert opol.B == ppol.B and opol.B > 128
        for name, nb in (("sink", 128 * H * D * 4), ("ring", OL.cap * H * 2 * OL.stage_bytes),
                         ("body", (opol.B - 128) // 128 * H * OL.lay.bytes)):
            got = d.get(C.c_void_p(getattr(PL, name)), nb, np.uint8)
            want = np.ctypeslib.as_array(C.cast(getattr(OL, name), cabi.u8p), shape=(nb,))
            assert np.array_equal(got, want), name
        qpos0 = NPOS - NQ
        qq = np.ascontiguousarray(q[qpos0:])
        view = lib.sjk_layer_view(C.byref(PL))
        got = attend(lib, d, view, ppol.B, NPOS, qpos0, qq, 1.0 / 16.0)
        want = oracle_rows(oracle, OL, opol.B, NPOS, qq, qpos0, 1.0 / 16.0,
                           [(iq, hq) for iq in range(NQ) for hq in range(HQ)])
        worst, l2 = check_rows(got, want)
        say("[tiles] reference shape: worst %.4f of the tolerance, max rel L2 %.2e" % (worst, l2))
        assert l2 <= 1e-3
    finally:
        d.free_all()
        oracle.layer_free(C.byref(OL))
        lib.sj_kvarn_layer_free(C.byref(PL))


@pytest.mark.parametrize("bk,bv,body,n_q,D", [(4, 4, 0, 512, 256), (3, 3, 1, 96, 256), (4, 4, 0, 512, 128)],
                         ids=["4/4s-ubatch512", "3/3t-ubatch96", "d128-4/4s-ubatch512"])
def test_prefill_ubatch(oracle, lib, dev, bk, bv, body, n_q, D):
    """A prefill ubatch of n_q positions x 16 query heads (GQA 4:1: 4 n_q rows per KV head) at the end of a context with a
    sealed body and a tq6_0 tail; the positions of the ubatch are both in the tail and (causally masked) in the body.
    The 4/4 bodies run on the 32-row kernel and, with the output over the queries, in many launches of 8 16-row tiles,
    as the trellis body does. Sampled rows from every part of the ubatch."""
    H, S, G = 4, 128, 128
    B = S + 12 * G
    n_pos = B + 700
    OL, PL = make_pair(oracle, lib, D, H, bk, bv, body, 256, 1024, n_ctx=n_pos + 64, n_ubatch=512)
    view = lib.sjk_layer_view(C.byref(PL))
    try:
        device_context(oracle, lib, dev, OL, PL, view, n_pos, B, seed=4000 + bk)
        n_head = 16
        q = np.random.default_rng(21).standard_normal((n_q, n_head, D)).astype(np.float32)
        qpos0 = n_pos - n_q
        got = attend(lib, dev, view, B, n_pos, qpos0, q, 0.0625)
        assert np.all(np.isfinite(got))
        rng = np.random.default_rng(n_q)
        rows = sorted({(0, 0), (0, 15), (n_q - 1, 0), (n_q - 1, 15), (n_q // 2, 5)} |
                      {(int(a), int(b)) for a, b in zip(rng.integers(0, n_q, 40), rng.integers(0, n_head, 40))})
        worst, l2 = check_rows(got, oracle_rows(oracle, OL, B, n_pos, q, qpos0, 0.0625, rows))
        say("[tiles] ubatch %d: %d rows, worst %.4f of the tolerance, rel L2 %.2e" % (n_q, len(rows), worst, l2))
        dq = dev.put(q)
        sjk.check(lib.sjk_hip_attend(C.byref(view), B, n_pos, qpos0, n_q, n_head, dq, 0.0625, dq, None), "attend over q")
        over = dev.get(dq, q.nbytes, np.float32).reshape(q.shape)
        worst, l2 = check_rows(over, oracle_rows(oracle, OL, B, n_pos, q, qpos0, 0.0625, rows))
        say("[tiles] ubatch %d over its queries: worst %.4f of the tolerance, rel L2 %.2e" % (n_q, worst, l2))
    finally:
        oracle.layer_free(C.byref(OL))
        lib.sj_kvarn_layer_free(C.byref(PL))


SHAPES = [
    # D, H, bk, bv, body, n_q, n_head
    (128, 1, 4, 4, 0, 4, 4),        # configs[0]'s shape (1 KV head, D = 128, 4/4), decode width 4: the 4/4
    (128, 1, 4, 4, 0, 40, 4),       # the same, 160 query rows: 10 tiles, two launches     matrix-core kernel
    (128, 8, 4, 4, 0, 4, 32),       # 8 KV heads, GQA 4:1, width 4 (the common D = 128 decode shape)
    (128, 2, 3, 3, 1, 4, 8),        # trellis at D = 128
    (128, 2, 4, 2, 0, 9, 8),        # 4/2 scalar at D = 128, 36 rows per KV head: the other scalar bodies' kernel
    (256, 4, 3, 3, 0, 4, 16),       # a scalar body other than 4/4 at D = 256
    (256, 4, 4, 2, 0, 9, 16),       # 4/2 scalar, 36 rows per KV head
]


@pytest.mark.parametrize("D,H,bk,bv,body,n_q,n_head", SHAPES,
                         ids=["c1-d128-w4", "c1-d128-160rows", "d128-h8-w4", "d128-3/3t", "d128-4/2s",
                              "d256-3/3s", "d256-4/2s-36rows"])
def test_shapes_vs_oracle(oracle, lib, dev, D, H, bk, bv, body, n_q, n_head):
    S, G = 128, 128
    B = S + 5 * G
    n_pos = B + 333
    OL, PL = make_pair(oracle, lib, D, H, bk, bv, body, 256, 512, n_ctx=n_pos + 64, n_ubatch=512)
    view = lib.sjk_layer_view(C.byref(PL))
    try:
        device_context(oracle, lib, dev, OL, PL, view, n_pos, B, seed=5000 + D + bk)
        q = np.random.default_rng(31).standard_normal((n_q, n_head, D)).astype(np.float32)
        for qpos0 in (n_pos - n_q, B - n_q // 2 - 3):          # rows in the tail; rows across the body's end
            got = attend(lib, dev, view, B, n_pos, qpos0, q, 1.0 / float(np.sqrt(D)))
            rows = [(iq, hq) for iq in range(n_q) for hq in range(n_head)]
            if len(rows) > 64:
                rows = rows[::len(rows) // 48]
            worst, _ = check_rows(got, oracle_rows(oracle, OL, B, n_pos, q, qpos0, 1.0 / float(np.sqrt(D)), rows))
            say("[tiles] D=%d H=%d %d/%d%s qpos0=%d: worst %.4f" % (D, H, bk, bv, "t" if body else "s", qpos0, worst))
    finally:
        oracle.layer_free(C.byref(OL))
        lib.sj_kvarn_layer_free(C.byref(PL))


@pytest.mark.parametrize("bk,bv,body", [(4, 4, 0), (3, 2, 1), (4, 2, 0)], ids=["4/4s", "3/2t", "4/2s"])
def test_wide_gqa_group(oracle, lib, dev, bk, bv, body):
    """32 query heads per KV head: one position's rows span two tiles (a tile boundary inside a position)."""
    D, H, S, G = 256, 2, 128, 128
    B = S + 4 * G
    n_pos = B + 300                                   # the context builder keeps the last 256 positions unsealed
    OL, PL = make_pair(oracle, lib, D, H, bk, bv, body, 256, 512, n_ctx=n_pos + 64, n_ubatch=512)
    view = lib.sjk_layer_view(C.byref(PL))
    try:
        device_context(oracle, lib, dev, OL, PL, view, n_pos, B, seed=6000 + bk)
        n_q, n_head = 3, 64
        q = np.random.default_rng(41).standard_normal((n_q, n_head, D)).astype(np.float32)
        got = attend(lib, dev, view, B, n_pos, n_pos - n_q, q, 0.0625)
        rows = [(iq, hq) for iq in range(n_q) for hq in range(0, n_head, 5)] + [(1, 31), (1, 32), (2, 63)]
        worst, _ = check_rows(got, oracle_rows(oracle, OL, B, n_pos, q, n_pos - n_q, 0.0625, rows))
        say("[tiles] gq=32 %d/%d: worst %.4f" % (bk, bv, worst))
    finally:
        oracle.layer_free(C.byref(OL))
        lib.sj_kvarn_layer_free(C.byref(PL))


@pytest.mark.parametrize("bk,bv,body,D", [(4, 4, 0, 256), (3, 3, 1, 256), (4, 4, 0, 128)], ids=["4/4s", "3/3t", "d128-4/4s"])
def test_small_and_edge_contexts(oracle, lib, dev, bk, bv, body, D):
    """One KV head (GQA 16:1, so 16 rows per position and several tiles at width 4) over contexts at the region
    edges on the matrix-core kernels: a single sink position, a partial sink, the sink exactly full, one tail
    position, a body that ends exactly at N (no tail), queries at the very start (causal prefixes of the sink),
    and part of the stored groups read from the ring instead of the body."""
    H, S, G = 1, 128, 128
    n_pos = S + 2 * G + 37
    OL, PL = make_pair(oracle, lib, D, H, bk, bv, body, 256, 512, n_ctx=n_pos + 64, n_ubatch=512)
    view = lib.sjk_layer_view(C.byref(PL))
    try:
        K, V = inputs.kv_rows(n_pos, H, D, seed=8800 + bk)
        dK, dV = dev.put(K), dev.put(V)
        sjk.check(lib.sjk_hip_layer_store(C.byref(view), 0, n_pos, dK, dV, 1, None), "layer_store")
        sjk.check(lib.sjk_hip_commit(C.byref(view), 1, S, S + 2 * G, 16, None), "commit")
        dev.sync()
        assert n_pos - S <= PL.cap
        for name, nb in (("sink", S * H * D * 4), ("ring", OL.cap * H * 2 * OL.stage_bytes),
                         ("body", 2 * H * OL.lay.bytes)):
            b = dev.get(C.c_void_p(getattr(view, name)), nb, np.uint8)
            C.memmove(getattr(OL, name), b.ctypes.data, nb)
        n_head = 16
        cases = [  # B, N, qpos0, n_q
            (0, 1, 0, 1), (0, 64, 63, 1), (S, S, S - 4, 4), (S, S + 1, S, 1), (S + 2 * G, S + 2 * G, S + 2 * G - 4, 4),
            (S + 2 * G, n_pos, 0, 4), (S + G, n_pos, n_pos - 4, 4), (S + 2 * G, n_pos, n_pos - 4, 4)]
        for B, N, qpos0, n_q in cases:
            q = np.random.default_rng(B + N + qpos0).standard_normal((n_q, n_head, D)).astype(np.float32)
            got = attend(lib, dev, view, B, N, qpos0, q, 0.0625)
            rows = [(iq, hq) for iq in range(n_q) for hq in range(n_head)]
            worst, _ = check_rows(got, oracle_rows(oracle, OL, B, N, q, qpos0, 0.0625, rows))
            say("[tiles] H=1 D=%d %d/%d%s B=%d N=%d qpos0=%d n_q=%d: worst %.4f" % (D, bk, bv, "t" if body else "s", B,
                                                                                   N, qpos0, n_q, worst))
    finally:
        oracle.layer_free(C.byref(OL))
        lib.sj_kvarn_layer_free(C.byref(PL))


WIDE = [
    # D, H, bk, bv, body, n_q, n_head, sealed groups
    (256, 4, 4, 4, 0, 5, 16, 14),   # width 5 at GQA 4:1: 20 rows per KV head, the configs[3] layout
    (128, 4, 4, 4, 0, 4, 32, 14),   # width 4 at GQA 8:1: 32 rows (the common D = 128 shape)
    (128, 4, 4, 4, 0, 4, 32, 0),    # the same with no sealed records: row slots only
    (128, 96, 4, 4, 0, 4, 768, 3),  # 96 KV heads: two CU slots per KV head for two jobs, each share raised to two
    (256, 4, 4, 4, 0, 8, 16, 14),   # 32 rows at D = 256
    (256, 4, 3, 3, 0, 5, 16, 14),   # a scalar body other than 4/4, 20 rows
    (128, 2, 4, 2, 0, 8, 8, 14),    # 4/2 at D = 128, 32 rows
    (256, 4, 3, 3, 1, 5, 16, 14),   # the 3/3 trellis body, 20 rows
]


@pytest.mark.parametrize("D,H,bk,bv,body,n_q,n_head,n_groups", WIDE,
                         ids=["4/4-d256-20rows", "4/4-d128-32rows", "4/4-d128-32rows-tail-only", "4/4-d128-32rows-96heads",
                              "4/4-d256-32rows", "3/3s-d256-20rows", "4/2s-d128-32rows", "3/3t-d256-20rows"])
def test_wide_rows_vs_oracle(oracle, lib, dev, D, H, bk, bv, body, n_q, n_head, n_groups):
    """More than 16 query rows per KV head: the 16-row tiles run side by side as the jobs of one launch, sharing its
    workgroups in proportion to their work (the 4/4 kernel, the other scalar bodies' kernel, the trellis kernel).
    Every row of the call against the oracle, for rows in the tail and rows across the body's (sink's) end; the
    second tile's rows see one position more than the first's at width 5 (the causal end of each row is its own)."""
    S, G = 128, 128
    B = S + n_groups * G
    n_pos = B + 301
    OL, PL = make_pair(oracle, lib, D, H, bk, bv, body, 256, 512, n_ctx=n_pos + 64, n_ubatch=512)
    view = lib.sjk_layer_view(C.byref(PL))
    try:
        device_context(oracle, lib, dev, OL, PL, view, n_pos, B, seed=7100 + D + bk + n_q)
        q = np.random.default_rng(33 + n_q).standard_normal((n_q, n_head, D)).astype(np.float32)
        for qpos0 in (n_pos - n_q, B - 2):                  # rows in the tail; rows across the body's (sink's) end
            got = attend(lib, dev, view, B, n_pos, qpos0, q, 1.0 / float(np.sqrt(D)))
            rows = [(iq, hq) for iq in range(n_q) for hq in range(n_head)]
            worst, l2 = check_rows(got, oracle_rows(oracle, OL, B, n_pos, q, qpos0, 1.0 / float(np.sqrt(D)), rows))
            say("[tiles] wide D=%d H=%d %d/%d %d rows qpos0=%d: worst %.4f, rel L2 %.2e" % (
                D, H, bk, bv, n_q * n_head // H, qpos0, worst, l2))
    finally:
        oracle.layer_free(C.byref(OL))
        lib.sj_kvarn_layer_free(C.byref(PL))


PREFILL = [
    # D, H, gq, n_q, staging, sink_type, sealed groups, tail, first query position before the end, scale
    (256, 4, 4, 64, 0, 0, 9, 301, 64, 0.0625),     # 256 rows of 4 heads (16-row kernels); a tail that is no multiple of 32
    (128, 4, 4, 67, 0, 0, 9, 256, 67, 0.08),       # a last tile of 12 rows
    (256, 1, 16, 17, 0, 0, 0, 0, 128, 0.0625),     # causal in a sink that is all there is
    (256, 2, 8, 33, 0, 1, 3, 470, 300, 0.0625),    # sink in the staging type, rows across the body's end
    (128, 2, 4, 100, 1, 0, 4, 290, 600, -0.05),    # fp16 staging, a negative scale, later records masked
    (256, 4, 4, 64, 1, 1, 2, 257, 64, 0.0),        # fp16 sink in the staging type, scale 0 (plain means)
    (128, 16, 4, 65, 0, 0, 1, 260, 65, 0.08),      # 16 heads: 144 tiles
    (256, 8, 4, 64, 0, 0, 9, 301, 64, 0.0625),     # 256 rows, the fewest that the 32-row kernel takes (from 8 heads on)
    (256, 4, 4, 66, 1, 1, 2, 257, 66, 0.0),        # fp16 sink in the staging type, scale 0, a last tile of 8 rows
    (128, 16, 4, 160, 0, 0, 3, 300, 160, 0.08),    # 320 tiles: some whole in their workgroup, which normalises them
    (128, 4, 8, 300, 0, 1, 3, 450, 400, 0.08),     # 75 tiles a head: past the first 64 of the search for a share's tile
]


@pytest.mark.parametrize("D,H,gq,n_q,staging,sink_type,ngr,tail,back,scale", PREFILL)
def test_prefill_kernel_edges(oracle, lib, dev, D, H, gq, n_q, staging, sink_type, ngr, tail, back, scale):
    """Calls of 256 query rows per KV head and more, most of them on the 32-row kernel: ragged tiles, every region and staging type, causal rows in each
    region, each against the oracle; the descriptor call gives the same bits, and a call whose output lies over its
    queries (which takes the 16-row kernels) agrees with the oracle too."""
    S, G = 128, 128
    B = S + ngr * G
    n_pos = B + tail
    OL, PL = make_pair(oracle, lib, D, H, 4, 4, 0, 256, 512, n_ctx=4096, n_ubatch=512, staging=staging, sink_type=sink_type)
    view = lib.sjk_layer_view(C.byref(PL))
    try:
        K, V = inputs.kv_rows(n_pos, H, D, seed=70 + D + ngr)
        dK, dV = dev.put(K), dev.put(V)
        done = S
        for p in range(0, n_pos, 256):             # the ring holds no more at once
            n = min(256, n_pos - p)
            view_at = lambda d, off: C.c_void_p(d.value + 4 * off * H * D)
            sjk.check(lib.sjk_hip_layer_store(C.byref(view), p, n, view_at(dK, p), view_at(dV, p), 1, None), "layer_store")
            full = min(B, S + (p + n - S) // G * G) if p + n > S else S
            if full > done:
                sjk.check(lib.sjk_hip_commit(C.byref(view), 1, done, full, 16, None), "commit")
                done = full
        assert done == B
        dev.sync()
        sink_b = S * H * (4 * D if sink_type == 0 else 2 * OL.stage_bytes)
        for name, nb in (("sink", sink_b), ("ring", OL.cap * H * 2 * OL.stage_bytes), ("body", ngr * H * OL.lay.bytes)):
            if nb:
                b = dev.get(C.c_void_p(getattr(view, name)), nb, np.uint8)
                C.memmove(getattr(OL, name), b.ctypes.data, nb)
        n_head, qpos0 = H * gq, max(0, n_pos - back)
        q = np.random.default_rng(3 + n_q).standard_normal((n_q, n_head, D)).astype(np.float32)
        q[0] *= 1e-6                               # a row's scale is its own
        got = attend(lib, dev, view, B, n_pos, qpos0, q, scale)
        rng = np.random.default_rng(n_q)
        rows = sorted({(0, 0), (1, n_head - 1), (n_q - 1, 0), (n_q - 1, n_head - 1)} |
                      {(int(a), int(b)) for a, b in zip(rng.integers(0, n_q, 60), rng.integers(0, n_head, 60))})
        want = oracle_rows(oracle, OL, B, n_pos, q, qpos0, scale, rows)
        worst, l2 = check_rows(got, want)
        desc = np.zeros(16, np.int32)
        desc[2], desc[3], desc[4] = B, n_pos, qpos0
        dq, do, dd = dev.put(q), dev.put(q), dev.put(desc)
        sjk.check(lib.sjk_hip_attend(C.byref(view), B, n_pos, qpos0, n_q, n_head, do, scale, do, None), "attend over q")
        check_rows(dev.get(do, q.nbytes, np.float32).reshape(q.shape), want)
        sjk.check(lib.sjk_hip_attend_dyn(C.byref(view), dd, 4096, n_q, n_head, dq, scale, do, None), "attend_dyn")
        assert np.array_equal(dev.get(do, q.nbytes, np.uint32), got.reshape(-1).view(np.uint32))
        desc[2] = 4095                             # no whole number of groups: NaN rows
        bad = dev.put(desc)
        sjk.check(lib.sjk_hip_attend_dyn(C.byref(view), bad, 4096, n_q, n_head, dq, scale, do, None), "attend_dyn")
        assert np.isnan(dev.get(do, q.nbytes, np.float32)).all()
        say("[tiles] prefill D=%d %d rows: worst %.4f of the tolerance, rel L2 %.2e" % (D, n_q * gq, worst, l2))
    finally:
        oracle.layer_free(C.byref(OL))
        lib.sj_kvarn_layer_free(C.byref(PL))


def filled_context(lib, dev, OL, view, K, V, B, rotate=1):
    """K, V rows [n][H][D] stored and [S, B) sealed in windows that fit the ring, the oracle's layer given the bytes"""
    n_pos, H, D = K.shape
    S, G, cfg = view.S, 128, OL.cfg
    dK, dV = dev.put(K), dev.put(V)
    done = S
    for p in range(0, n_pos, 256):
        n = min(256, n_pos - p)
        at = lambda d: C.c_void_p(d.value + 4 * p * H * D)
        sjk.check(lib.sjk_hip_layer_store(C.byref(view), p, n, at(dK), at(dV), rotate, None), "layer_store")
        full = min(B, S + (p + n - S) // G * G) if p + n > S else S
        if full > done:
            sjk.check(lib.sjk_hip_commit(C.byref(view), 1, done, full, 16, None), "commit")
            done = full
    assert done == B
    dev.sync()
    sink_b = S * H * (4 * D if cfg.sink_type == 0 else 2 * OL.stage_bytes)
    for name, nb in (("sink", sink_b), ("ring", OL.cap * H * 2 * OL.stage_bytes), ("body", (B - S) // G * H * OL.lay.bytes)):
        if nb:
            b = dev.get(C.c_void_p(getattr(view, name)), nb, np.uint8)
            C.memmove(getattr(OL, name), b.ctypes.data, nb)


def some_rows(n_q, n_head, n, seed):
    rng = np.random.default_rng(seed)
    return sorted({(0, 0), (1, n_head - 1), (n_q - 1, 0), (n_q - 1, n_head - 1)} |
                  {(int(a), int(b)) for a, b in zip(rng.integers(0, n_q, n), rng.integers(0, n_head, n))})


@pytest.mark.parametrize("D,H,gq,n_q,wide", [(256, 1, 16, 16, False), (256, 4, 4, 64, False), (128, 7, 1, 256, False),
                                             (128, 8, 4, 64, True), (128, 2, 1, 257, True), (256, 1, 4, 65, True),
                                             (256, 8, 1, 255, False)])
def test_which_calls_take_the_32_row_kernel(oracle, lib, dev, D, H, gq, n_q, wide):
    """More than 256 query rows per KV head, or 256 of at least 8 heads: below, the 16-row kernels are the faster ones. Their
    result (a call with its output over the queries takes them) has other last bits than the 32-row kernel's."""
    B = 128 + 4 * 128
    n_pos = B + 301
    OL, PL = make_pair(oracle, lib, D, H, 4, 4, 0, 256, 512, n_ctx=4096, n_ubatch=512)
    view = lib.sjk_layer_view(C.byref(PL))
    try:
        K, V = inputs.kv_rows(n_pos, H, D, seed=90)
        filled_context(lib, dev, OL, view, K, V, B)
        q = np.random.default_rng(5).standard_normal((n_q, H * gq, D)).astype(np.float32)
        got = attend(lib, dev, view, B, n_pos, n_pos - n_q, q, 0.0625)
        dq = dev.put(q)
        sjk.check(lib.sjk_hip_attend(C.byref(view), B, n_pos, n_pos - n_q, n_q, H * gq, dq, 0.0625, dq, None), "attend over q")
        same = np.array_equal(dev.get(dq, q.nbytes, np.uint32), got.reshape(-1).view(np.uint32))
        assert same == (not wide)
        check_rows(got, oracle_rows(oracle, OL, B, n_pos, q, n_pos - n_q, 0.0625, some_rows(n_q, H * gq, 20, 3)))
    finally:
        oracle.layer_free(C.byref(OL))
        lib.sj_kvarn_layer_free(C.byref(PL))


@pytest.mark.parametrize("D", [256, 128])
def test_prefill_query_keeps_its_32_bits(oracle, lib, dev, D):
    """A query row with one channel of 2^15 and the others of about 2^-5 (a ratio of 2^20), against keys that weigh them
    alike: every channel's own relative precision counts, so a query cut to parts that share the row's largest exponent
    loses the small channels (an error of 8e-3 in the values). Bound: the one 16-bit rounding in the path is that of P'
    (2^-11 of a weight), and the code x Vscale it multiplies has about 3.2 times the size of the value it makes (codes 0
    to 15, a zero point in the middle): errors that add up like the values themselves stay below 3.2 x 2^-11 of a row's
    norm. The 16-row kernels' result for the same call (output over the queries) is held to the same."""
    H, gq, n_q, S, ngr = 2, 4, 72, 128, 9
    B = S + 128 * ngr
    n_pos = B + 301
    OL, PL = make_pair(oracle, lib, D, H, 4, 4, 0, 256, 512, n_ctx=4096, n_ubatch=512, staging=1)
    view = lib.sjk_layer_view(C.byref(PL))
    try:
        rng = np.random.default_rng(500 + D)
        K = 32.0 * rng.standard_normal((n_pos, H, D), dtype=np.float32)
        K[:, :, 7] *= np.float32(2.0 ** -20)
        V = rng.standard_normal((n_pos, H, D), dtype=np.float32)
        filled_context(lib, dev, OL, view, K, V, B, rotate=0)
        q = np.float32(2.0 ** -5) * rng.standard_normal((n_q, H * gq, D), dtype=np.float32)
        q[:, :, 7] = np.where(rng.integers(0, 2, (n_q, H * gq)), 40000.0, -36000.0)
        scale = 1.0 / float(np.sqrt(D))
        got = attend(lib, dev, view, B, n_pos, n_pos - n_q, q, scale)
        want = oracle_rows(oracle, OL, B, n_pos, q, n_pos - n_q, scale, some_rows(n_q, H * gq, 60, 8))
        dq = dev.put(q)
        sjk.check(lib.sjk_hip_attend(C.byref(view), B, n_pos, n_pos - n_q, n_q, H * gq, dq, scale, dq, None), "attend over q")
        for name, x in (("32", got), ("16", dev.get(dq, q.nbytes, np.float32).reshape(q.shape))):
            worst, l2 = check_rows(x, want)
            say("[tiles] prefill D=%d, channels 2^20 apart, %s-row kernel: worst %.4f of the tolerance, rel L2 %.2e" % (
                D, name, worst, l2))
            assert l2 <= 3.2 * 2.0 ** -11
    finally:
        oracle.layer_free(C.byref(OL))
        lib.sj_kvarn_layer_free(C.byref(PL))


@pytest.mark.parametrize("D,staging", [(256, 0), (128, 1)])
def test_prefill_tiny_queries_and_scales(oracle, lib, dev, D, staging):
    """Scores that round to zero: subnormal query rows, and a scale whose product with the row is below every float.
    The rows are plain means over what they see, positions that a row does not see stay out of it."""
    H, gq, n_q, S = 2, 4, 72, 128
    B = S + 3 * 128
    n_pos = B + 301
    OL, PL = make_pair(oracle, lib, D, H, 4, 4, 0, 256, 512, n_ctx=4096, n_ubatch=512, staging=staging)
    view = lib.sjk_layer_view(C.byref(PL))
    try:
        K, V = inputs.kv_rows(n_pos, H, D, seed=91)
        filled_context(lib, dev, OL, view, K, V, B)
        for name, amp, scale in (("subnormal rows", 1e-44, 0.0625), ("1e-30 rows", 1e-30, -0.0625),
                                 ("subnormal scale", 0.25, 1e-45), ("rows and scale", 1e-25, 1e-25)):
            q = np.float32(amp) * np.random.default_rng(4).uniform(0.5, 1.0, (n_q, H * gq, D)).astype(np.float32)
            q[3] = 0.0
            for qpos0 in (n_pos - n_q, B - 40, 20):          # rows in the tail, across the body's end, in the sink
                got = attend(lib, dev, view, B, n_pos, qpos0, q, scale)
                assert np.isfinite(got).all(), (name, qpos0)
                worst, _ = check_rows(got, oracle_rows(oracle, OL, B, n_pos, q, qpos0, scale, some_rows(n_q, H * gq, 20, 5)))
                say("[tiles] prefill D=%d %s at %d: worst %.4f of the tolerance" % (D, name, qpos0, worst))
    finally:
        oracle.layer_free(C.byref(OL))
        lib.sj_kvarn_layer_free(C.byref(PL))


@pytest.mark.parametrize("D,staging,sink_type", [(256, 0, 0), (128, 0, 1), (256, 1, 1), (128, 1, 0)])
def test_prefill_unseen_values_stay_out(oracle, lib, dev, D, staging, sink_type):
    """An infinity or a NaN among the values of one position: the rows before it, whose weight for it is zero, keep
    their bits (a product of zero with it would be a NaN); the rows that see it are not finite. The position is in the
    sink, in the tail, or in a record (its value scale or zero point, or a channel's scale, which all tokens share)."""
    H, gq, n_q, S = 2, 4, 72, 128
    B = S + 4 * 128
    n_pos = B + 301
    OL, PL = make_pair(oracle, lib, D, H, 4, 4, 0, 256, 512, n_ctx=4096, n_ubatch=512, staging=staging, sink_type=sink_type)
    view = lib.sjk_layer_view(C.byref(PL))
    lay = OL.lay
    sb = OL.stage_bytes
    try:
        K, V = inputs.kv_rows(n_pos, H, D, seed=92)
        filled_context(lib, dev, OL, view, K, V, B)
        q = np.random.default_rng(6).standard_normal((n_q, H * gq, D)).astype(np.float32)
        scale = 1.0 / float(np.sqrt(D))

        def staged(base, entry):                     # the V row's first half of head 1: a block norm or a value
            return base + entry * H * 2 * sb + 2 * sb + sb

        def sink_at(p):
            return p * H * 4 * D + 4 * D + 2 * D if sink_type == 0 else staged(0, p)

        rec = ((2 * H + 1) * lay.bytes, S + 2 * 128)  # record 2 of head 1, its first position
        cases = []                                   # (name, pointer, offset, qpos0, first position that may differ)
        for bad in (29, 8):
            cases.append(("sink %d" % bad, view.sink, sink_at(bad), 0, bad))
        for qpos0 in (n_pos - n_q, n_pos - 2 * n_q):  # the end of a tile's steps, and not
            p = qpos0 + 29
            cases.append(("tail %d" % p, view.ring, staged(0, (p - S) % OL.cap), qpos0, p))
        for what, off, p in (("scale", lay.v_scale + 2 * 7, rec[1] + 7), ("zero", lay.v_zero + 2 * 7, rec[1] + 7),
                             ("channel", lay.v_ch + 2 * 5, rec[1])):
            cases.append(("record " + what, view.body, rec[0] + off, rec[1] - 30, p))
        for name, ptr, off, qpos0, first in cases:
            good = attend(lib, dev, view, B, n_pos, qpos0, q, scale)
            assert np.isfinite(good).all(), name
            ptr = C.c_void_p(ptr)
            old = dev.get(ptr, 2, np.uint16, off)
            for half in (0x7C00, 0xFE00):
                dev.upload(ptr, np.array([half], np.uint16), off)
                got = attend(lib, dev, view, B, n_pos, qpos0, q, scale)
                n = first - qpos0
                a, b = got.view(np.uint32), good.view(np.uint32)
                bad = [(iq, hq) for iq in range(n) for hq in range(H * gq) if not np.array_equal(a[iq, hq], b[iq, hq])]
                assert not bad, (name, hex(half), len(bad), bad[:4])
                assert np.array_equal(a[:, :gq], b[:, :gq]), name          # the other head
                assert not np.isfinite(got[n:, gq:]).all(axis=-1).any(), (name, hex(half))
            dev.upload(ptr, old, off)
            say("[tiles] prefill D=%d staging %d, %s: %d positions keep their rows" % (D, staging, name, first - qpos0))
    finally:
        oracle.layer_free(C.byref(OL))
        lib.sj_kvarn_layer_free(C.byref(PL))


@pytest.mark.parametrize("D", [256, 128])
def test_prefill_batch_on_a_block_pool(oracle, lib, dev, D):
    """Two sequences of 288 rows per KV head whose records lie in one pool, in another order, behind block tables: one
    call each, a batch, a batch on one shared workspace and a captured batch's graph, replayed, all give the bits of a
    call on the layer that holds the records in order. A batch in which one job's output lies over its queries, and one
    with a workspace below a partial per compute unit, run on the 16-row kernels: the same bits as that job alone."""
    H, gq, n_q, S, G = 4, 4, 72, 128, 128
    n_head, scale = H * gq, 1.0 / float(np.sqrt(D))
    ctx = [(S + 9 * G + 301, 9), (S + 3 * G + 277, 3)]           # (positions, sealed groups)
    pairs = [make_pair(oracle, lib, D, H, 4, 4, 0, 256, 512, n_ctx=n + 64, n_ubatch=512) for n, _ in ctx]
    views = [lib.sjk_layer_view(C.byref(PL)) for _, PL in pairs]
    hip, graph, gexec = dev.hip, C.c_void_p(), C.c_void_p()
    hip.hipStreamBeginCapture.argtypes = [C.c_void_p, C.c_int]
    hip.hipStreamEndCapture.argtypes = [C.c_void_p, C.POINTER(C.c_void_p)]
    hip.hipGraphInstantiate.argtypes = [C.POINTER(C.c_void_p), C.c_void_p, C.c_void_p, C.c_char_p, C.c_size_t]
    hip.hipGraphLaunch.argtypes = [C.c_void_p, C.c_void_p]
    hip.hipGraphExecDestroy.argtypes = [C.c_void_p]
    hip.hipGraphDestroy.argtypes = [C.c_void_p]
    try:
        rb, want, want16 = H * pairs[0][0].lay.bytes, [], []
        order = np.random.default_rng(2).permutation(14)[:12].astype(np.uint32)      # blocks of both, two unused
        pool = np.zeros((14, rb), np.uint8)
        q = np.random.default_rng(17).standard_normal((2, n_q, n_head, D)).astype(np.float32)
        dq, do = [dev.put(q[k]) for k in range(2)], [dev.alloc(q[k].nbytes) for k in range(2)]
        at, paged = 0, []
        for k, ((n_pos, ngr), (OL, PL)) in enumerate(zip(ctx, pairs)):
            K, V = inputs.kv_rows(n_pos, H, D, seed=700 + k)
            filled_context(lib, dev, OL, views[k], K, V, S + ngr * G)
            want.append(attend(lib, dev, views[k], S + ngr * G, n_pos, n_pos - n_q, q[k], scale).view(np.uint32))
            check_rows(want[k].view(np.float32), oracle_rows(oracle, OL, S + ngr * G, n_pos, q[k], n_pos - n_q, scale,
                                                             some_rows(n_q, n_head, 30, k)))
            over = dev.put(q[k])
            sjk.check(lib.sjk_hip_attend(C.byref(views[k]), S + ngr * G, n_pos, n_pos - n_q, n_q, n_head, over, scale, over,
                                         None), "attend over q")
            want16.append(dev.get(over, q[k].nbytes, np.uint32).reshape(q[k].shape))
            assert not np.array_equal(want16[k], want[k])
            ids = order[at:at + ngr]
            pool[ids] = dev.get(C.c_void_p(views[k].body), ngr * rb, np.uint8).reshape(ngr, rb)
            v = sjk.View.from_buffer_copy(bytes(views[k]))
            v.blocks = dev.put(ids).value
            paged.append(v)
            at += ngr
        d_pool = dev.put(pool)
        for v in paged:
            v.body = d_pool.value
        jobs = (sjk.AttendJob * 2)()
        for k, (n_pos, ngr) in enumerate(ctx):
            jobs[k].v, jobs[k].B, jobs[k].N, jobs[k].qpos0 = paged[k], S + ngr * G, n_pos, n_pos - n_q
            jobs[k].d_q, jobs[k].d_out = dq[k].value, do[k].value

        def outputs():
            dev.sync()
            return [dev.get(do[k], q[k].nbytes, np.uint32).reshape(q[k].shape) for k in range(2)]

        def batch(name, expect, stream=None):
            for k in range(2):
                dev.upload(do[k], np.full(q[k].shape, np.nan, np.float32))
            sjk.check(lib.sjk_hip_attend_batch(jobs, 2, n_q, n_head, scale, stream), "attend_batch")
            for k, x in enumerate(outputs()):
                assert np.array_equal(x, expect[k]), (name, k)

        for k, (n_pos, ngr) in enumerate(ctx):
            one = attend(lib, dev, paged[k], S + ngr * G, n_pos, n_pos - n_q, q[k], scale)
            assert np.array_equal(one.view(np.uint32), want[k]), ("single", k)
        batch("batch", want)
        jobs[1].v.work = paged[0].work
        batch("one workspace", want)
        stream = dev.stream()
        dev._ck(hip.hipStreamBeginCapture(stream, 2), "hipStreamBeginCapture")
        rc = lib.sjk_hip_attend_batch(jobs, 2, n_q, n_head, scale, stream)
        dev._ck(hip.hipStreamEndCapture(stream, C.byref(graph)), "hipStreamEndCapture")
        sjk.check(rc, "attend_batch")
        dev._ck(hip.hipGraphInstantiate(C.byref(gexec), graph, None, None, 0), "hipGraphInstantiate")
        for _ in range(3):
            for k in range(2):
                dev.upload(do[k], np.full(q[k].shape, np.nan, np.float32))
            dev._ck(hip.hipGraphLaunch(gexec, stream), "hipGraphLaunch")
            dev._ck(hip.hipStreamSynchronize(stream), "hipStreamSynchronize")
            for k, x in enumerate(outputs()):
                assert np.array_equal(x, want[k]), ("graph", k)
            batch("between replays", want)
        jobs[1].v.work = paged[1].work
        # one partial of 32 rows takes two slots of 16 rows and a little more: three quarters of the workspace hold the
        # 16-row kernels' partials and less than that of every compute unit
        jobs[1].v.work_bytes = paged[1].work_bytes * 3 // 4
        single = attend(lib, dev, jobs[1].v, jobs[1].B, jobs[1].N, jobs[1].qpos0, q[1], scale)
        assert np.array_equal(single.view(np.uint32), want16[1])
        jobs[1].v.work_bytes = paged[1].work_bytes
        over = dev.put(q[1])
        jobs[1].d_q = jobs[1].d_out = over.value
        sjk.check(lib.sjk_hip_attend_batch(jobs, 2, n_q, n_head, scale, None), "attend_batch")
        got = [dev.get(do[0], q[0].nbytes, np.float32), dev.get(over, q[1].nbytes, np.float32)]
        for k, (n_pos, ngr) in enumerate(ctx):       # (tiles of both share launches, so that their split is not the single call's)
            check_rows(got[k].reshape(q[k].shape), oracle_rows(oracle, pairs[k][0], S + ngr * G, n_pos, q[k], n_pos - n_q,
                                                               scale, some_rows(n_q, n_head, 30, k)))
    finally:
        if gexec.value:
            hip.hipGraphExecDestroy(gexec)
        if graph.value:
            hip.hipGraphDestroy(graph)
        for OL, PL in pairs:
            oracle.layer_free(C.byref(OL))
            lib.sj_kvarn_layer_free(C.byref(PL))


@pytest.mark.parametrize("S", [0, 1, 100])
def test_prefill_any_sink_length(oracle, lib, dev, S):
    """A hand-built view whose sink is no whole number of steps (or none): the sink's last step ends early, and the tail
    starts at a position that is no multiple of 16."""
    D, H, gq, n_q = 256, 2, 4, 72
    B = S + 5 * 128
    n_pos = B + 301
    OL, PL = make_pair(oracle, lib, D, H, 4, 4, 0, 256, 512, n_ctx=4096, n_ubatch=512)
    view = lib.sjk_layer_view(C.byref(PL))
    try:
        view.S = OL.cfg.sink = S
        K, V = inputs.kv_rows(n_pos, H, D, seed=93)
        filled_context(lib, dev, OL, view, K, V, B)
        q = np.random.default_rng(9).standard_normal((n_q, H * gq, D)).astype(np.float32)
        for qpos0 in (n_pos - n_q, B - 40, max(0, S - 30)):      # rows in the tail, across the body's end, across the sink's
            got = attend(lib, dev, view, B, n_pos, qpos0, q, 0.0625)
            worst, l2 = check_rows(got, oracle_rows(oracle, OL, B, n_pos, q, qpos0, 0.0625, some_rows(n_q, H * gq, 30, 7)))
            say("[tiles] prefill S=%d at %d: worst %.4f of the tolerance, rel L2 %.2e" % (S, qpos0, worst, l2))
    finally:
        OL.cfg.sink = 128
        oracle.layer_free(C.byref(OL))
        lib.sj_kvarn_layer_free(C.byref(PL))


@pytest.mark.parametrize("D,staging", [(128, 0), (256, 0), (256, 1)])
def test_prefill_staged_rows_against_float64(oracle, lib, dev, D, staging):
    """All positions staged, so that only 32-bit sums and split operands are in the path (about 4e-7): the 32-row kernel is
    no further from float64 attention over the same rows than the 16-row kernels (the call with its output over the
    queries). One KV head, every row."""
    H, gq, n_q, n_pos, S = 2, 4, 300, 4000, 128
    OL, PL = make_pair(oracle, lib, D, H, 4, 4, 0, 4096, 8192, n_ctx=8192, n_ubatch=512, staging=staging)
    view = lib.sjk_layer_view(C.byref(PL))
    try:
        K, V = inputs.kv_rows(n_pos, H, D, seed=94, outlier_scale=1.0)
        filled_context(lib, dev, OL, view, K, V, S)
        q = np.random.default_rng(13).standard_normal((n_q, H * gq, D)).astype(np.float32)
        scale, qpos0 = 1.0 / float(np.sqrt(D)), n_pos - n_q
        got = attend(lib, dev, view, S, n_pos, qpos0, q, scale)
        dq = dev.put(q)
        sjk.check(lib.sjk_hip_attend(C.byref(view), S, n_pos, qpos0, n_q, H * gq, dq, scale, dq, None), "attend over q")
        over = dev.get(dq, q.nbytes, np.float32).reshape(q.shape)
        k64, v64 = (np.zeros((n_pos, D), np.float32) for _ in range(2))
        for p in range(n_pos):
            oracle.layer_kv_row(C.byref(OL), S, p, 0, cabi.ptr(k64[p], cabi.f32p), cabi.ptr(v64[p], cabi.f32p))
        rows = q[:, :gq].reshape(-1, D).astype(np.float64)
        sc = rows @ k64.astype(np.float64).T * scale
        sc[np.arange(n_pos)[None, :] > (qpos0 + np.arange(n_q).repeat(gq))[:, None]] = -np.inf
        pw = np.exp(sc - sc.max(axis=1, keepdims=True))
        want = (pw @ v64.astype(np.float64)) / pw.sum(axis=1, keepdims=True)
        err = [float(np.linalg.norm(x[:, :gq].reshape(-1, D) - want) / np.linalg.norm(want)) for x in (got, over)]
        say("[tiles] staged rows D=%d staging %d: error against float64 %.3e, 16-row kernels %.3e" % (D, staging, *err))
        assert err[0] <= err[1]
    finally:
        oracle.layer_free(C.byref(OL))
        lib.sj_kvarn_layer_free(C.byref(PL))
