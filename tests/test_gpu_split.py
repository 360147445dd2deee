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


# raw mode's own: of SHAPES those whose angle tables fit (a chunk's, for all heads, in 64 KiB),
# and whole sequences before the split ones (256 of 264, 288 and 384; two segments of 128)
RAW_SHAPES = [s for s in SHAPES if s[6] % 4 == 0 and s[1] < 64] + [
    (11, 24, 5, 128, 128, 64, 32), (9, 32, 4, 128, 128, 64, 32), (16, 24, 8, 128, 128, 64, 32),
    (4, 32, 8, 128, 128, 64, 32), (20, 16, 9, 64, 64, 64, 16),
    # more chunks than the angles entering a segment are staged for at once (67 at 64 angles)
    (1, 1, 150, 64, 128, 64, 64)]


@pytest.mark.parametrize("b,h,nc,chunk,n,p,nr", RAW_SHAPES)
@pytest.mark.parametrize("phi_init", [False, True])
def test_split_raw_scan_equals_whole(m3, dev, whole, b, h, nc, chunk, n, p, nr, phi_init):
    K, L = m3.kernels, nc * chunk
    assert _split_bytes(m3, b, h, L, n, p, chunk) > 0, "the shape does not split"
    _, d = raw_case(b, h, L, n, p, nr, seed=nc, phi_init=phi_init)
    dt, a, trap, ang = views(d, h, nr)
    assert K.raw_forward_ok("bf16", chunk, n, p, nr, L, h), "no raw-mode kernel for this shape"
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


# (H, chunks, chunk, N, Nr, without z): heads of one sequence; padded to whole rounds of 256
BWD_SHAPES = [(1, 4, 128, 128, 32, False), (3, 7, 128, 128, 32, True), (24, 5, 128, 128, 32, False),
              (258, 4, 128, 128, 16, False), (4, 9, 64, 128, 64, False), (5, 11, 64, 64, 6, True)]


@pytest.mark.parametrize("h,nc,chunk,n,nr,gate", BWD_SHAPES)
@pytest.mark.parametrize("final", [False, True])
def test_split_backward_equals_whole(m3, dev, h, nc, chunk, n, nr, gate, final):
    """The same heads repeated to a full round, where nothing is split: every per-head
    gradient bit for bit, the bias sums (over the segments, then as before) to f32 rounding."""
    L, p, full = nc * chunk, 64, (h + 255) // 256 * 256
    lib = m3._lib.load()
    rows = lambda hh: 2 * hh * L * n * 2  # noqa: E731
    assert lib.m3s_bwd_workspace_bytes(m3._lib.DTYPE_BF16, 1, L, h, n) > rows(h), "does not split"
    assert lib.m3s_bwd_workspace_bytes(m3._lib.DTYPE_BF16, 1, L, full, n) == rows(full)
    _, d = boundary_inputs(1, h, L, n, p, nr, "bf16", seed=h + nc)
    gen = torch.Generator().manual_seed(nc)
    extra = {k: torch.randn(1, h, *s, generator=gen).cuda() if final else None
             for k, s in (("dfinal_ssm", (p, n)), ("dfinal_v", (p,)))}

    def run(idx):
        pick = lambda t, dim=1: None if t is None else t.index_select(dim, idx).contiguous()  # noqa: E731
        z = pick(d["z"]) if gate else None
        args = [d["q"], d["k"], pick(d["v"]), pick(d["adt"]), pick(d["gamma"]), pick(d["scale"]),
                pick(d["phi"]), pick(d["q_bias"], 0), pick(d["k_bias"], 0)]
        skip = pick(d["d_skip"], 0)
        res = m3.siso_forward(*args, skip, z, chunk=chunk, save_residuals=True)[4]
        return m3.siso_backward_kernel(
            pick(d["dy"]), res.ybar, z, *args, res.chunk_states, d_skip=skip, chunk=chunk,
            **{k: pick(t) for k, t in extra.items()})

    idx = torch.arange(full, device=dev) % h
    got, ref = run(idx[:h]), run(idx)
    for name in ("dv", "dadt", "dqk_diag", "dscale", "dphi", "dz", "uw", "k_final", "dseed_ssm"):
        a, b = getattr(got, name), getattr(ref, name)
        if a is not None:
            assert torch.equal(a, b[:, :h]), name
    for name in ("dq_bias", "dk_bias"):   # at most 16 segments' f32 sums in another order
        a, b = getattr(got, name), getattr(ref, name)[:h]
        assert float((a - b).abs().max()) <= 1e-5 * float(b.abs().max()), name


@pytest.mark.parametrize("entry", ["m3s_bwd", "m3s_bwd_ws"])
def test_backward_with_the_rows_alone_is_not_split(m3, dev, monkeypatch, entry):
    """``m3s_bwd``, and ``m3s_bwd_ws`` with a workspace too small for a split, stay within the
    per-head rows (a guard after them keeps its bytes) and give the split scan's bits,
    the bias sums to f32 rounding."""
    b, h, L, n, p = 1, 3, 896, 128, 64
    lib, K = m3._lib, m3.kernels
    _, d = boundary_inputs(b, h, L, n, p, 32, "bf16", seed=5)
    args = fwd_args(d)
    res = m3.siso_forward(*args, chunk=128, save_residuals=True)[4]

    def run():
        return m3.siso_backward_kernel(d["dy"], res.ybar, d["z"], *args[:9], res.chunk_states,
                                       d_skip=d["d_skip"], chunk=128)

    ref = run()
    rows, need = 2 * h * L * n * 2, lib.load().m3s_bwd_workspace_bytes(lib.DTYPE_BF16, b, L, h, n)
    assert need > rows
    guard = torch.full((need,), 0x5A, dtype=torch.uint8, device=dev)
    launch, seen = lib.launch, []

    def whole(fn, a, dev_, what):
        if what != "m3s_bwd":
            return launch(fn, a, dev_, what)
        seen.append(a.workspace)
        a.workspace = guard.data_ptr()
        if entry == "m3s_bwd":
            return launch(lib.load().m3s_bwd, a, dev_, what)
        return launch(lambda x, s: lib.load().m3s_bwd_ws(x, rows + 4096, s), a, dev_, what)

    monkeypatch.setattr(lib, "launch", whole)
    got = run()
    assert len(seen) == 1 and bool((guard[rows:] == 0x5A).all()) and not bool((guard[:rows] == 0x5A).all())
    for name in got._fields:
        x, y = getattr(got, name), getattr(ref, name)
        if name in ("dq_bias", "dk_bias"):   # at most 16 segments' f32 sums in another order
            assert float((x - y).abs().max()) <= 1e-5 * float(y.abs().max()), name
        else:
            assert torch.equal(x, y), name


def test_no_room_for_the_scratch_runs_whole_sequences(m3, dev, monkeypatch):
    """Where a split's scratch cannot be allocated, forward and backward run unsplit: the same
    bits (the bias sums to f32 rounding)."""
    K, empty, refused = m3.kernels, m3.kernels.empty, []
    _, d = boundary_inputs(1, 3, 896, 128, 64, 32, "bf16", seed=6)
    args = fwd_args(d)

    def run():
        out = m3.siso_forward(*args, chunk=128, save_residuals=True)
        return out[:4], m3.siso_backward_kernel(
            d["dy"], out[4].ybar, d["z"], *args[:9], out[4].chunk_states, d_skip=d["d_skip"], chunk=128)

    ref, gref = run()
    rows = 2 * 3 * 896 * 128 * 2

    def full(*size, **kw):
        if kw.get("dtype") == torch.uint8 and size[0] != rows:
            refused.append(size[0])
            raise torch.cuda.OutOfMemoryError("no room")
        return empty(*size, **kw)

    monkeypatch.setattr(K, "empty", full)
    got, ggot = run()
    assert len(refused) == 2
    for a, b in zip(got, ref):
        assert torch.equal(a, b)
    for name in ggot._fields:
        x, y = getattr(ggot, name), getattr(gref, name)
        if name in ("dq_bias", "dk_bias"):   # at most 16 segments' f32 sums in another order
            assert float((x - y).abs().max()) <= 1e-5 * float(y.abs().max()), name
        else:
            assert torch.equal(x, y), name
