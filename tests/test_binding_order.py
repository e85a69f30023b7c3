"""Order between torch's stream and a context's: the library launches on a
non-blocking stream of its own, which torch's stream is not ordered with.  The
binding therefore enters the library with no fill of a key or output buffer
still pending on torch's stream, and gives a temporary back to torch's allocator
only once the library's work on it is done.

On the CPU the binding runs against a stand-in library and stand-in streams that
keep track of what is pending; on the GPU it runs behind a torch stream that is
busy for a while."""
import ctypes
import types

import numpy as np
import pytest

import mpcx


class Streams:
    """What is pending on torch's stream and on the context's."""

    def __init__(self):
        self.fills = self.calls = False

    def sync_torch(self):
        self.fills = False

    def sync_all(self):
        self.fills = self.calls = False


class DevTensor:
    """A host array in the place of a device tensor."""

    def __init__(self, st, a):
        self.st, self.a = st, a

    def cuda(self):  # pageable host to device: torch waits for its stream
        self.st.sync_torch()
        return self

    def detach(self):
        return self

    def cpu(self):
        return self

    def numpy(self):
        return self.a

    def data_ptr(self):
        return self.a.ctypes.data

    def numel(self):
        return self.a.size


def _torch_on(st):
    def zeros(n, dtype=None, device=None):
        st.fills = True
        return DevTensor(st, np.zeros(n, np.uint8))

    t = types.SimpleNamespace()
    t.uint8 = np.uint8
    t.zeros = zeros
    t.from_numpy = lambda a: DevTensor(st, a)
    t.cuda = types.SimpleNamespace(
        synchronize=st.sync_all,
        current_stream=lambda: types.SimpleNamespace(synchronize=st.sync_torch))
    return t


# entry points that return with their work enqueued
ENQUEUES = {"mpcx_prg_hash", "mpcx_prf", "mpcx_dcf_keygen", "mpcx_dcf_eval", "mpcx_dcf_eval_ring",
            "mpcx_tr_keygen", "mpcx_mul_keygen", "mpcx_lut8_keygen", "mpcx_reveal_keygen", "mpcx_ring_gemm",
            "mpcx_maxpool_eval_noalloc"}


class Lib:
    def __init__(self, st):
        self.st, self.late = st, []

    def __getattr__(self, name):
        def call(*a):
            if name.endswith("_key_bytes"):
                return 64
            if name == "mpcx_synchronize":
                self.st.calls = False
            elif self.st.fills:
                self.late.append(name)
            if name in ENQUEUES:
                self.st.calls = True
            return 0
        return call


@pytest.fixture
def host(monkeypatch):
    st = Streams()
    monkeypatch.setattr(mpcx, "_torch", lambda: _torch_on(st))
    c = mpcx.Ctx.__new__(mpcx.Ctx)
    c.lib, c.h, c.bw, c.s, c.T = Lib(st), None, 32, 12, np.uint32
    return c, st


V = np.arange(8, dtype=np.uint32)
K = types.SimpleNamespace(data_ptr=lambda: 0)  # a key held from before
PEER = types.SimpleNamespace(h=ctypes.c_void_p(0))
CALLS = {
    "prg_hash": lambda c: c.prg_hash(np.zeros((2, 4), np.uint32)),
    "prf": lambda c: c.prf(1, 2, 3, 4),
    "dcf_keygen": lambda c: c.dcf_keygen(12, V, np.zeros(8, np.uint8)),
    "dcf_eval": lambda c: c.dcf_eval(0, 12, K, V),
    "dcf_eval_ring": lambda c: c.dcf_eval_ring(0, 12, K, V, np.zeros(1, np.uint32)),
    "tr_keygen": lambda c: c.tr_keygen(1, V),
    "tr_eval": lambda c: c.tr_eval(1, K, K, V, V),
    "maxpool_keygen": lambda c: c.maxpool_keygen(1, 4, 2, V),
    "maxpool_eval": lambda c: c.maxpool_eval(1, 4, 2, K, K, V),
    "maxpool_eval_noalloc": lambda c: c.maxpool_eval_noalloc(1, 4, 2, K, K, V),
    "mul_keygen": lambda c: c.mul_keygen(V, V, V, V),
    "mul_eval": lambda c: c.mul_eval(K, K, V, V, V, V),
    "lut8_keygen": lambda c: c.lut8_keygen(V),
    "lut8_eval": lambda c: c.lut8_eval(K, K, np.zeros(256, np.uint32), V),
    "sxs_keygen": lambda c: c.sxs_keygen(1, 2, 4, 2, V, V),
    "sxs_eval": lambda c: c.sxs_eval(1, 2, 4, 2, K, K, V, V),
    "ring_gemm": lambda c: c.ring_gemm(V.reshape(2, 4), V.reshape(4, 2)),
    "reveal_keygen": lambda c: c.reveal_keygen(8),
    "reveal_eval": lambda c: c.reveal_eval(K, K, V, V),
    "party_tr_eval": lambda c: c.party_tr_eval(PEER, 1, K, V),
    "party_mul_eval": lambda c: c.party_mul_eval(PEER, K, V, V, V, V),
    "party_lut8_eval": lambda c: c.party_lut8_eval(PEER, K, np.zeros(256, np.uint32), V),
    "party_sxs_eval": lambda c: c.party_sxs_eval(PEER, 1, 2, 4, 2, K, V, V),
    "party_reveal_eval": lambda c: c.party_reveal_eval(PEER, K, V),
    "adjnorm_keygen": lambda c: c.adjnorm_keygen(1, 2),
    "adjnorm_eval": lambda c: c.adjnorm_eval(1, 2, 3, K, K, V[:4], V[:4]),
}


@pytest.mark.parametrize("name", sorted(CALLS))
def test_no_fill_is_pending_when_the_library_is_entered(host, name):
    c, st = host
    CALLS[name](c)
    assert not c.lib.late, f"entered with a fill pending: {c.lib.late}"
    assert not st.calls, "returned, and freed its temporaries, with the library's work pending"


# ---- the same on the GPU ----
@pytest.fixture
def busy(monkeypatch):
    """Some 20 ms of work on torch's stream before the call, and again after each
    of its copies to the device, so that a fill comes late."""
    import torch
    big = torch.empty(1 << 30, dtype=torch.uint8, device="cuda")

    def queue():
        for k in range(64):
            big.fill_(k)

    copy = mpcx.to_dev

    def to_dev(a):
        t = copy(a)
        queue()
        return t

    monkeypatch.setattr(mpcx, "to_dev", to_dev)
    queue()
    yield queue
    torch.cuda.synchronize()


@pytest.mark.gpu
def test_prg_and_prf_behind_a_busy_torch_stream(orc, busy):
    c = mpcx.Ctx(bw=32, scale=12)
    blocks = np.random.default_rng(3).integers(0, 2**32, size=(4099, 4), dtype=np.uint64).astype(np.uint32)
    for leaf in (False, True):
        assert np.array_equal(c.prg_hash(blocks, leaf), orc.hash_blocks(blocks, leaf))
    busy()
    assert np.array_equal(c.prf(77, 5, 0x30, 1000), orc.prf_blocks(77, 5, 0x30, 1000))
    c.close()


@pytest.mark.gpu
@pytest.mark.parametrize("bw", [32, 64])
def test_reveal_and_relu_behind_a_busy_torch_stream(bw, busy):
    """Keys filled last (reveal) and outputs filled last (both evaluations)."""
    c = mpcx.Ctx(bw=bw, scale=12)
    rng = np.random.default_rng(bw)
    n, m = 3001, np.uint64((1 << bw) - 1)
    v = rng.integers(-(1 << 20), 1 << 20, n).astype(np.int64)
    v0 = rng.integers(0, 1 << 63, n, dtype=np.uint64) & m
    k0, k1, mask = c.reveal_keygen(n, seed=9)
    vh = c.reveal_eval(k0, k1, v0, (v.astype(np.uint64) - v0) & m).astype(np.uint64)
    assert np.array_equal((vh - mask.astype(np.uint64)) & m, v.astype(np.uint64) & m)
    k0, k1, ro = c.tr_keygen(mpcx.RELU, mask, seed=9, gate=2)
    y = c.tr_eval(mpcx.RELU, k0, k1, vh).astype(np.uint64)
    assert np.array_equal((y - ro.astype(np.uint64)) & m, np.maximum(v, 0).astype(np.uint64) & m)
    c.close()
