"""Scans whose last round of workgroups is half empty cut its sequences into segments
(``m3s_fwd_ws`` with its workspace): bit for bit the same scan with every sequence in one
workgroup (``m3s_fwd``), which the other files hold to the oracle. The segments' states come
from the chunks' shares by the scan's own operations in the scan's own order."""

import ctypes

import pytest
import torch

from helpers import boundary_inputs, fwd_args
from test_gpu_raw import raw_case, views

pytestmark = pytest.mark.gpu

@pytest.fixture
def whole(m3, monkeypatch):
    """Run a callable with every sequence in one workgroup."""
    K, lib = m3.kernels, m3._lib

    def run(fn):
        def launch(a, dev):
            lib.check(lib.load().m3s_fwd(ctypes.byref(a), lib.stream_handle(dev)), "m3s_fwd")

        with monkeypatch.context() as mp:
            mp.setattr(K, "_launch_fwd", launch)
            return fn()

    return run


def _split_bytes(m3, b, h, L, n, p, chunk):
    return m3._lib.load().m3s_fwd_workspace_bytes(m3._lib.DTYPE_BF16, b, L, h, p, n, chunk)


# (B, H, chunks, chunk, N, P, Nr): one chunk per segment, uneven segments, many chunks, whole
# sequences before the split ones, a rotary block that Nr cuts, phi read by scalars, all of N
SHAPES = [
    (1, 1, 4, 128, 128, 64, 32), (1, 3, 7, 128, 128, 64, 32), (1, 5, 40, 128, 128, 64, 32),
    (2, 64, 9, 128, 128, 64, 32), (3, 24, 5, 128, 128, 64, 32), (1, 258, 5, 128, 128, 64, 32),
    (4, 96, 8, 128, 128, 64, 16), (1, 4, 9, 64, 128, 64, 64), (2, 3, 11, 64, 64, 64, 16),
    (1, 2, 6, 128, 64, 64, 6),
]


@pytest.mark.parametrize("b,h,nc,chunk,n,p,nr", SHAPES)
@pytest.mark.parametrize("seeds", [False, True])
def test_split_scan_equals_whole(m3, dev, whole, b, h, nc, chunk, n, p, nr, seeds):
    L = nc * chunk
    assert _split_bytes(m3, b, h, L, n, p, chunk) > 0, "the shape does not split"
    _, d = boundary_inputs(b, h, L, n, p, nr, "bf16", seed=b + h + nc, seeds=seeds)

    def run():
        return m3.siso_forward(*fwd_args(d), chunk=chunk, save_residuals=True)

    got, ref = run(), whole(run)
    for i, what in enumerate(("y", "final_ssm", "final_k", "final_v")):
        assert torch.equal(got[i], ref[i]), what
    assert torch.equal(got[4].ybar, ref[4].ybar), "ybar"
    assert torch.equal(got[4].chunk_states, ref[4].chunk_states), "chunk_states"


@pytest.mark.parametrize("b,h,nc,chunk,n,p,nr", [s for s in SHAPES if s[6] % 4 == 0])
@pytest.mark.parametrize("phi_init", [False, True])
def test_split_raw_scan_equals_whole(m3, dev, whole, b, h, nc, chunk, n, p, nr, phi_init):
    K, L = m3.kernels, nc * chunk
    _, d = raw_case(b, h, L, n, p, nr, seed=nc, phi_init=phi_init)
    dt, a, trap, ang = views(d, h, nr)
    if not K.raw_forward_ok("bf16", chunk, n, p, nr, L, h):
        pytest.skip("no raw-mode kernel for this shape")
    (k, q), _, angs = K.bcnorm_forward([d["kr"], d["qr"]], [d["wb"], d["wc"]], 1e-5,
                                       theta=(ang, dt, d["bias"], chunk))

    def run():
        return K.siso_forward_raw(q, k, d["v"], dt, a, trap, angs, d["bias"], d["qb"], d["kb"],
                                  d_skip=d["d"], z=d["z"], phi_init=d.get("phi_init"),
                                  chunk=chunk)

    got, ref = run(), whole(run)
    for i, what in enumerate(("y", "final_ssm", "final_k", "final_v", "phi_final")):
        assert torch.equal(got[i], ref[i]), what


def test_split_needs_its_workspace(m3, dev):
    """Full rounds and single chunks ask for none; a short workspace is refused."""
    lib = m3._lib
    assert _split_bytes(m3, 8, 32, 8192, 128, 64, 128) == 0      # 256 sequences
    assert _split_bytes(m3, 1, 200, 1024, 128, 64, 128) == 0     # over half a round
    assert _split_bytes(m3, 1, 4, 128, 128, 64, 128) == 0        # one chunk
    assert _split_bytes(m3, 4, 24, 512, 128, 64, 128) == 0       # two chunks saved
    _, d = boundary_inputs(1, 2, 512, 128, 64, 32, "bf16")
    args = {}

    def keep(a, dev_):
        args["rc"] = lib.load().m3s_fwd_ws(ctypes.byref(a), d["q"].data_ptr(), 64,
                                           lib.stream_handle(dev_))

    K, old = m3.kernels, m3.kernels._launch_fwd
    K._launch_fwd = keep
    try:
        m3.siso_forward(*fwd_args(d))
    finally:
        K._launch_fwd = old
    assert args["rc"] == lib.ERR_INVALID and b"workspace" in lib.load().m3s_last_error()
