"""Device memory around a dealer's run: what a model keeps of it afterwards, and
what it gives back when its keys come from elsewhere.  Sizes are differences of the
device's used memory, which the allocator rounds to a few MiB."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
MIB = 1 << 20


def _used():
    import torch
    torch.cuda.synchronize()
    free, total = torch.cuda.mem_get_info()
    return total - free


def _model(mpcx, synth, B, bw):
    wl = synth.workload(B, synth.Dims(bw=bw), seed=4)
    c = mpcx.Ctx(bw=bw, scale=12)
    return c, wl, lambda lanes=1: mpcx.Model(c, wl.dims, wl.W, lanes=lanes)


def _forward(m, wl, B):
    m.set_inputs(B, *wl.shares["x"], *wl.shares["a"], *wl.shares["m"], wl.prot)
    m.forward(B)
    return m.output(B)


@pytest.mark.parametrize("how", ["stream", "import"])
def test_other_keys_give_the_dealing_memory_back(synth, how):
    """A model that dealt, then took its keys from host buffers, holds what one
    holds that never dealt (the masks of a run of 8 samples are 23 MiB)."""
    import mpcx
    B = 8
    c, wl, make = _model(mpcx, synth, B, 32)
    d = make()
    d.keygen(B, 5)
    k0, k1 = d.export_keys(0, B), d.export_keys(1, B)
    want = _forward(d, wl, B)
    d.close()
    held = []
    for dealt in (False, True):
        before = _used()
        m = make()
        if dealt:
            m.keygen(B, 6)
        if how == "stream":
            m.attach_host_keys(B, k0, k1, 256 * MIB)
        else:
            m.import_keys(B, k0, k1)
        assert np.array_equal(_forward(m, wl, B), want)
        held.append(_used() - before)
        m.close()
    assert held[1] - held[0] <= 8 * MIB
    c.close()


def test_dealing_memory_kept_is_bounded(synth):
    """Past 256 MiB of masks (50 samples in Z_2^64) a lane keeps none of them,
    however many runs it has had."""
    import mpcx
    c, wl, make = _model(mpcx, synth, 1, 64)
    m = make()
    for B in (50, 60, 70):
        m.keygen(B, B)
        u = _used()
    arena = 2 * m.key_bytes(70)
    m.release_arena()
    assert u - _used() <= arena + 256 * MIB + 16 * MIB
    m.close()
    c.close()


@pytest.mark.parametrize("bw,B,N,C", [(64, 64, 140, 312), (32, 256, 7, 1024), (64, 4096, 5, 128)])
def test_maxpool_dealing_workspace(bw, B, N, C):
    """At most three times the input's size (all levels' pairs twice, and the two
    planes of running masks)."""
    import mpcx
    import torch
    c = mpcx.Ctx(bw=bw, scale=12)
    t = torch.int32 if bw == 32 else torch.int64
    r = torch.arange(B * N * C, device="cuda").to(t)
    ro = torch.zeros(B * C, dtype=t, device="cuda")
    kb = c.lib.mpcx_maxpool_key_bytes(c.h, B, N, C)
    k0, k1 = mpcx.empty_dev(kb), mpcx.empty_dev(kb)
    p = mpcx.dptr
    # the first level's keys alone: the kernel's own memory (spilled registers) is there
    c.check(c.lib.mpcx_tr_keygen(c.h, mpcx.RELU, B * (N // 2) * C, p(r), p(r), 3, 1, p(k0), p(k1)), "tr_keygen")
    before = _used()
    c.check(c.lib.mpcx_maxpool_keygen(c.h, B, N, C, p(r), p(ro), 3, 1, p(k0), p(k1)), "maxpool_keygen")
    assert _used() - before <= 3 * r.numel() * (bw // 8) + 4 * MIB
    c.close()


@pytest.mark.parametrize("bw,B,lanes,slack,mib", [(32, 2, 1, 0, 0), (32, 3, 2, 1, 0), (32, 2, 1, 2, 0), (32, 2, 1, 3, 0),
                                                  (64, 3, 2, 0, 0), (32, 8, 1, 0, 16), (32, 9, 2, 0, 12)])
def test_gate_by_gate_dealing_writes_the_same_keys(synth, monkeypatch, bw, B, lanes, slack, mib):
    """A lane that may hold no masks at once (0), or fewer than its run needs
    (16 MiB: refused after the first chunk), deals gate by gate."""
    import mpcx
    keys = []
    for limit in (None, str(mib)):
        if limit is not None:
            monkeypatch.setenv("MPCX_DEAL_MIB", limit)
        wl = synth.workload(B, synth.Dims(bw=bw, slack=slack), seed=4)
        c = mpcx.Ctx(bw=bw, scale=12)
        m = mpcx.Model(c, wl.dims, wl.W, lanes=lanes)
        m.keygen(B, 21)
        keys.append([m.export_keys(p, B) for p in (0, 1)])
        m.close()
        c.close()
    for a, b in zip(*keys):
        assert np.array_equal(a, b)
