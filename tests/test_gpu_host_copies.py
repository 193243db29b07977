"""Copies to and from a caller's arrays below and above the sizes from which
they go through the host's loop, plain copies and pinned chunks, with whole
chunks and a rest: state fields set and read back, exactly; both directions of
the network's forward pass against slices small enough for the plain copy.
(Rests of every kind, to one byte: test_host_copies.py.)"""
import time

import numpy as np
import pytest
import torch

from lsd import make_config
from lsd.gpu import Context, Mlp, _p

pytestmark = pytest.mark.gpu


# H = 528 (L = 32) and 4656 (L = 96) coll rows: 2 x 8 x H N bytes a field, from
# 59 KB to 25 MB
@pytest.mark.parametrize("L,N", [(32, 7), (32, 31), (32, 248), (32, 249), (32, 256), (32, 124), (32, 125), (96, 10),
                                 (96, 11), (96, 127), (96, 339)])
def test_state_fields(L, N):
    cfg = make_config(L=L, M=L, N=N, dt=1e-6)
    g = Context(cfg)
    H = cfg.sizes()[0]
    rng = np.random.default_rng(N)
    want = [rng.standard_normal((2, H, N)) for _ in range(6)]
    for k in (0, 1, 2, 4, 5):
        g.set_coll(k, want[k][0], want[k][1])
    for k in (0, 1, 2, 4, 5):
        re, im = g.get_coll(k)
        assert np.array_equal(re, want[k][0]) and np.array_equal(im, want[k][1])
    g.close()


def test_one_array_for_two_results():
    """A caller that wants one of the results passes its array twice: it gets
    the later one."""
    cfg = make_config(L=64, M=64, N=96, dt=1e-6)
    g = Context(cfg)
    H = cfg.sizes()[0]
    re, im = np.random.default_rng(3).standard_normal((2, H, 96))
    g.set_coll(4, re, im)
    buf = np.zeros((H, 96))
    for _ in range(3):
        assert g.lib.lsd_get_coll(g.h, 4, _p(buf), _p(buf)) == 0
        assert np.array_equal(buf, im)
    sre, sim = np.ascontiguousarray(re.T), np.ascontiguousarray(im.T)
    want = g.grad(sre, sim)[1]
    p = np.zeros_like(want)
    for _ in range(3):
        assert g.lib.lsd_tra_grad(g.h, _p(sre), _p(sim), _p(p), _p(p)) == 0
        assert np.array_equal(p, want)
    g.close()


def test_transform_uploads():
    """rtp -> qst and back of 28 MB of pageable arrays, in chunks, and of pinned
    ones, directly: the same bits."""
    cfg = make_config(L=64, M=64, N=65, dt=1e-6)
    g = Context(cfg)
    p = [torch.randn((65, g.Ph, g.Th), dtype=torch.float64, generator=torch.Generator().manual_seed(k)) for k in range(3)]
    assert 3 * p[0].numel() * 8 > 24 << 20
    a = g.rtp2qst(*[x.numpy() for x in p])
    b = g.rtp2qst(*[x.pin_memory().numpy() for x in p])
    for x, y in zip(a, b):
        assert np.array_equal(x[0], y[0]) and np.array_equal(x[1], y[1])
    g.close()


@pytest.mark.parametrize("rows", [1000, 32768, 32769, 70001, 400001])
def test_network_forward(rows):
    net = Mlp(16, 32, 16)
    x = np.random.default_rng(rows).standard_normal((rows, 16)).astype(np.float32)
    y = net.forward(x)
    step = min(300, rows) if rows < 40000 else 5000
    for r in range(0, rows, step):
        assert np.array_equal(y[r:r + step], net.forward(x[r:r + step]))


def test_failed_call_has_read_its_pinned_array():
    """A call that fails after its upload was queued returns when the upload is
    done: 190 MB of pinned memory, which may be read until the stream is waited
    for, take more than 190 MB / 100 GB/s on the link."""
    cfg = make_config(L=260, M=2, N=128, Th=390, Ph=486, dt=1e-6)
    g = Context(cfg)
    p = torch.ones((128, 486, 390), dtype=torch.float64, pin_memory=True).numpy()
    out = np.zeros((2, 128, cfg.sizes()[0]))
    for _ in range(2):
        t = time.perf_counter()
        rc = g.lib.lsd_tra_phys2spec(g.h, _p(p), _p(out[0]), _p(out[1]))
        t = time.perf_counter() - t
        assert rc != 0 and b"too large" in g.lib.lsd_last_error()
        assert t >= p.nbytes / 100e9
    g.close()
