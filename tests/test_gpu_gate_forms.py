"""Gate evaluations where a launch changes its form: the both-party kernel's
four and eight waves per SIMD (4096 elements per CU) and the one-lane kernel's
512- and 1024-thread workgroups (2048 per CU, Z_2^64), just below and just past
the line, the last tile of 64 elements whole, short by one, and one over.  The
unmasked outputs are checked against the plaintext gate, whatever the form."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
S = 12


@pytest.fixture(scope="module")
def mp():
    import mpcx
    return mpcx


@pytest.fixture(scope="module")
def num_cu():
    import torch
    return torch.cuda.get_device_properties(0).multi_processor_count


def _signed(v, bw):
    return v.astype(np.uint32).view(np.int32).astype(np.int64) if bw == 32 else v.view(np.int64)


def _inputs(n, bw, span, seed):
    rng = np.random.default_rng(seed)
    x = rng.integers(-span, span, n, dtype=np.int64)
    r = rng.integers(0, 1 << bw, n, dtype=np.uint64)
    m = np.uint64((1 << bw) - 1)
    return x, r, (x.astype(np.uint64) + r) & m


@pytest.mark.parametrize("bw,kind,per_cu,extra", [
    (32, "RELU", 4096, -1), (32, "RELU", 4096, 0), (32, "TRSLACK", 4096, 65), (32, "EXT", 4096, 1),
    (64, "RELU", 2048, -1), (64, "RELU", 2048, 65), (64, "EXT", 2048, 0)])
def test_gate_form_edges(mp, num_cu, bw, kind, per_cu, extra):
    n = per_cu * num_cu + extra
    c = mp.Ctx(bw=bw, scale=S)
    try:
        code = getattr(mp, kind)
        # EXT reads its input and mask modulo 2^(bw-s); TRSLACK wants |x| < 2^(bw-2)
        span = 1 << (bw - S - 1 if kind == "EXT" else bw - 2)
        x, r, xhat = _inputs(n, bw, span, per_cu + extra + code)
        k0, k1, ro = c.tr_keygen(code, r, seed=5, gate=3)
        got = _signed((c.tr_eval(code, k0, k1, xhat).astype(np.uint64) - ro.astype(np.uint64)), bw)
        want = np.maximum(x, 0) if kind == "RELU" else x >> S if kind == "TRSLACK" else x
        assert np.array_equal(got, want)
    finally:
        c.close()


@pytest.mark.parametrize("per_cu,extra", [(65, 0), (128, 0), (128, 1), (192, 0), (192, 1), (256, 1), (512, 0), (512, 1)])
@pytest.mark.parametrize("bw,kind", [(32, "RELU"), (32, "TRSLACK"), (64, "EXT"), (64, "RELU")])
def test_one_lane_instance_edges(mp, num_cu, bw, kind, per_cu, extra):
    """The one-lane kernel's workgroups of 256, 384 and 512 threads, and past 512
    elements per CU the instance with its reads in phases."""
    n = per_cu * num_cu + extra
    c = mp.Ctx(bw=bw, scale=S)
    try:
        code = getattr(mp, kind)
        assert c.tr_eval_form(code, n) == 0
        x, r, xhat = _inputs(n, bw, 1 << (bw - S - 1 if kind == "EXT" else bw - 2), n + code)
        k0, k1, ro = c.tr_keygen(code, r, seed=15, gate=2)
        got = _signed((c.tr_eval(code, k0, k1, xhat).astype(np.uint64) - ro.astype(np.uint64)), bw)
        assert np.array_equal(got, np.maximum(x, 0) if kind == "RELU" else x >> S if kind == "TRSLACK" else x)
    finally:
        c.close()


@pytest.mark.parametrize("bw", [32, 64])
@pytest.mark.parametrize("per_cu,extra", [(128, 0), (128, 1), (256, -1), (512, 0), (512, 1)])
def test_maxpool_instance_edges(mp, num_cu, bw, per_cu, extra):
    """One level of pairs at the same lines."""
    C = per_cu * num_cu + extra
    c = mp.Ctx(bw=bw, scale=S)
    try:
        x, r, xhat = _inputs(2 * C, bw, 1 << (bw - 3), C)
        k0, k1, ro = c.maxpool_keygen(1, 2, C, r, seed=6, gate=2)
        got = _signed(c.maxpool_eval(1, 2, C, k0, k1, xhat).astype(np.uint64) - ro.astype(np.uint64), bw)
        assert np.array_equal(got, x.reshape(2, C).max(0))
    finally:
        c.close()


@pytest.mark.parametrize("extra", [-1, 65])
def test_maxpool_form_edges(mp, num_cu, extra):
    """A first level of pairs at the eight-wave line, its odd last row carried to a
    second one."""
    B, N, C = 1, 3, 4096 * num_cu + extra
    c = mp.Ctx(bw=32, scale=S)
    try:
        x, r, xhat = _inputs(B * N * C, 32, 1 << 29, 9 + extra)
        k0, k1, ro = c.maxpool_keygen(B, N, C, r, seed=6, gate=2)
        got = _signed(c.maxpool_eval(B, N, C, k0, k1, xhat).astype(np.uint64) - ro.astype(np.uint64), 32)
        assert np.array_equal(got, x.reshape(N, C).max(0))
    finally:
        c.close()


@pytest.mark.parametrize("bw,kind,extra", [(32, "EXTRELU", -1), (32, "EXTRELU", 65), (64, "TRMOD", 1),
                                           (64, "TRRELU", -63), (32, "DRELU", 0), (32, "EXTRELU", -64),
                                           (64, "TRRELU", -65), (32, "TR", -127)])
def test_keygen_form_edges(mp, orc, num_cu, bw, kind, extra):
    """The dealer at the line between its 256- and 1024-thread workgroups (512
    elements per CU, in tiles of 64: the last one below is 64 less): both keys and
    the output mask as the oracle's dealer writes them, byte for byte."""
    n = 512 * num_cu + extra
    c = mp.Ctx(bw=bw, scale=S)
    try:
        code = getattr(mp, kind)
        rin = _inputs(n, bw, 1, n)[1]
        k0, k1, ro = c.tr_keygen(code, rin, seed=11, gate=4)
        o0, o1, oro = orc.tr_keygen(11, 4, code, bw, S, rin)
        assert np.array_equal(ro.astype(np.uint64), oro.astype(np.uint64))
        for got, want in ((k0, o0), (k1, o1)):
            assert np.array_equal(mp.from_dev(got, np.uint8), np.asarray(want, np.uint8).reshape(-1))
    finally:
        c.close()
