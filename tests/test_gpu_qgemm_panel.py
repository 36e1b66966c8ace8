"""GPU parity: the 2-D tiled q8_0 / q4_0 GEMM (the panel route for M >= 64,
kernels/quantization/qgemm_panel.cpp:234-286 in the reference) through the
C ABI.

Every row is held to the contract |y - y64| <= 1e-4 * ||x_m||_2 * ||w_n||_2
against the f64 oracle over exactly dequantized weights (all rows for small
shapes, sampled rows at prefill sizes), on both K-range settings and the
automatic route; reruns are bit-identical.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-4


def _check(oracle, fmt, packed, x, y, n, k, rows):
    for r in rows:
        y64, wn = oracle.gemv_f64(fmt, packed, x[r], n, k)
        ok, worst = oracle.within_contract(y[r], y64, wn, x[r], TOL)
        assert ok, f"row {r}: normalised error {worst:.3g} > {TOL}"


def _run(qc, dev, fmt, P, x, n, k, mode, x_off=0):
    import torch
    m = x.shape[0]
    X = torch.zeros(m * k + x_off, dtype=torch.float32, device=dev)
    X[x_off:] = torch.from_numpy(x.reshape(-1)).to(dev)
    Y = torch.full((m, n), float("nan"), dtype=torch.float32, device=dev)
    qc.set_qgemm_panel(mode)
    try:
        assert qc.qgemm_raw(fmt, P, X[x_off:], Y, m, n, k) == 0
        torch.cuda.synchronize()
    finally:
        qc.set_qgemm_panel(0)
    return Y.cpu().numpy()


@pytest.fixture(params=[1, 2], ids=["one_k_range", "two_k_ranges"])
def split(request):
    return request.param


@pytest.mark.parametrize("fmt", [0, 1])
@pytest.mark.parametrize("m,n,k", [(64, 256, 256), (100, 300, 512), (128, 128, 64),
                                   (130, 1000, 1024), (2, 200, 128), (257, 513, 192),
                                   (129, 255, 4096)])
def test_panel_shapes(qc, oracle, synth, dev, fmt, m, n, k, split):
    import torch
    print(f"panel fmt={fmt} m={m} n={n} k={k} split={split}", flush=True)
    w = synth.normal_fast(31 + n, n * k, 0.02).reshape(n, k)
    st, packed = oracle.pack(fmt, w)
    assert st == 0
    x = synth.normal_fast(37 + m, m * k).reshape(m, k)
    P = torch.from_numpy(packed).to(dev)
    y = _run(qc, dev, fmt, P, x, n, k, split)
    _check(oracle, fmt, packed, x, y, n, k, range(m))
    # bit-identical rerun (two K ranges add onto zero: order-independent)
    assert np.array_equal(y.view(np.uint32), _run(qc, dev, fmt, P, x, n, k, split).view(np.uint32))


@pytest.mark.parametrize("fmt", [0, 1])
def test_panel_activation_range(qc, oracle, synth, dev, fmt):
    """Activations over 40 decades, zero rows, a misaligned x, and a row of
    subnormal activations alone."""
    import torch
    m, n, k = 96, 160, 512
    w = synth.normal_fast(41, n * k, 0.02).reshape(n, k)
    st, packed = oracle.pack(fmt, w)
    rng = np.random.default_rng(5)
    x = (rng.standard_normal((m, k)) * 10.0 ** rng.uniform(-20, 20, (m, k))).astype(np.float32)
    x[3] = 0.0
    x[7] = (rng.standard_normal(k) * 1e-39).astype(np.float32)      # subnormal row
    x[9, ::5] = np.float32(3e4)
    P = torch.from_numpy(packed).to(dev)
    for mode, off in ((1, 0), (2, 1), (-1, 0)):
        y = _run(qc, dev, fmt, P, x, n, k, mode, off)
        _check(oracle, fmt, packed, x, y, n, k, range(m))


@pytest.mark.parametrize("fmt", [0, 1])
@pytest.mark.parametrize("m,n,k", [(512, 14336, 4096), (2048, 4096, 4096), (384, 4096, 14336)])
def test_panel_prefill_sizes(qc, oracle, dev, fmt, m, n, k):
    """Prefill shapes of a 4096-hidden / 14336-FFN layer on the automatic
    route (sampled rows; GPU-packed weights are byte-identical to the
    oracle's packer)."""
    import torch
    print(f"panel prefill fmt={fmt} m={m} n={n} k={k}", flush=True)
    g = torch.Generator(device=dev).manual_seed(m + n + k)
    W = torch.randn((n, k), generator=g, device=dev) * 0.02
    P = qc.pack(fmt, W)
    del W
    x = torch.randn((m, k), generator=g, device=dev).cpu().numpy()
    y = _run(qc, dev, fmt, P, x, n, k, 0)
    _check(oracle, fmt, P.cpu().numpy(), x, y, n, k, (0, 1, m // 2, m - 1))


# Automatic route: 33 rows (q4_0: 17) are the first 2-D call, and shapes around the edges
# of its tiles (32 / 64 / 128 / 256 rows by 128 / 256 columns), with K of one block
# pair, odd pairs, and K splits; the last six take the re-encoded 6-bit form for
# q4_0 (its three tiles, one and two K ranges).
@pytest.mark.parametrize("fmt", [0, 1])
@pytest.mark.parametrize("m,n,k", [(17, 64, 14336), (25, 333, 8256), (32, 1000, 16448),
                                   (17, 129, 64), (18, 127, 320), (31, 1361, 1088),
                                   (32, 4096, 4096), (32, 14337, 512),
                                   (33, 129, 64), (64, 2048, 4096), (65, 127, 320),
                                   (77, 1361, 1088), (257, 300, 448), (383, 2049, 192),
                                   (384, 2048, 64), (385, 2079, 576), (641, 2305, 128),
                                   (1025, 4097, 192), (2049, 2080, 64),
                                   (2049, 36900, 64), (1025, 24580, 192), (513, 14340, 1088),
                                   (641, 6201, 2112), (385, 6201, 4160), (1025, 2305, 2112)])
def test_wide_tile_edges(qc, oracle, dev, fmt, m, n, k):
    import torch
    print(f"wide fmt={fmt} m={m} n={n} k={k}", flush=True)
    g = torch.Generator(device=dev).manual_seed(m + n + k)
    P = qc.pack(fmt, torch.randn((n, k), generator=g, device=dev) * 0.02)
    x = torch.randn((m, k), generator=g, device=dev)
    x[torch.rand((m, k), generator=g, device=dev) < 0.01] *= 20.0
    Y = [torch.full((m, n), float("nan"), device=dev) for _ in range(2)]
    for y in Y:
        assert qc.qgemm_raw(fmt, P, x, y, m, n, k) == 0
    torch.cuda.synchronize()
    assert torch.equal(Y[0].view(torch.int32), Y[1].view(torch.int32))
    w = torch.from_numpy(oracle.unpack(fmt, P.cpu().numpy(), n, k)).to(dev).double()
    y64 = x.double() @ w.T.contiguous()
    bound = TOL * x.double().norm(dim=1, keepdim=True) * w.norm(dim=1)[None, :]
    err = (Y[0].double() - y64).abs()
    assert bool((err <= bound).all()), float((err / bound).max()) * TOL
    # as a whole the result is far closer than one output's bound: q4_0's
    # 6-bit digits keep at least 2^-19 of a block's largest element, about 7e-7
    # of the result here; the f16 pair keeps 2^-22 of each element
    rel = float((Y[0].double() - y64).norm() / y64.norm())
    assert rel < (4e-6 if fmt == 1 and m >= 384 and n >= 2048 else 1e-6), rel


@pytest.mark.parametrize("m,n,k", [(400, 2050, 320), (700, 4100, 64), (385, 14340, 1088),
                                   (2100, 36000, 64)])
def test_q4_digits_range_and_nonfinite_rows(qc, oracle, dev, m, n, k):
    """The re-encoded q4_0 form with activations over 40 decades, zero,
    subnormal and huge rows, a misaligned x, and rows holding NaN or +-inf:
    those rows' outputs have the class of the exact sum, the others are
    bit-identical to the same call with them zeroed."""
    import torch
    print(f"q4 digits m={m} n={n} k={k}", flush=True)
    g = torch.Generator(device=dev).manual_seed(m + k)
    P = qc.pack(1, torch.randn((n, k), generator=g, device=dev) * 0.02)
    w = torch.from_numpy(oracle.unpack(1, P.cpu().numpy(), n, k)).to(dev).double()
    X = torch.zeros(m * k + 1, device=dev)
    x = X[1:].view(m, k)
    x.copy_(torch.randn((m, k), generator=g, device=dev) *
            10.0 ** (40 * torch.rand((m, k), generator=g, device=dev) - 20))
    x[3] = 0.0
    x[7] = torch.randn(k, generator=g, device=dev) * 1e-39
    x[9] = torch.randn(k, generator=g, device=dev) * 1e37
    x[11] = torch.randn(k, generator=g, device=dev)
    bad = {0: [(5, float("inf"))], m - 1: [(k - 5, float("-inf"))], 33: [(2, float("nan"))],
           130: [(0, float("inf")), (k - 1, float("-inf"))]}
    finite = x.clone()
    for r, items in bad.items():
        finite[r] = 0.0
        for c, v in items:
            x[r, c] = v
    y, z = (torch.full((m, n), float("nan"), device=dev) for _ in range(2))
    assert qc.qgemm_raw(1, P, x, y, m, n, k) == 0
    assert qc.qgemm_raw(1, P, finite, z, m, n, k) == 0
    torch.cuda.synchronize()
    keep = torch.ones(m, dtype=torch.bool, device=dev)
    keep[list(bad)] = False
    assert torch.equal(y[keep].view(torch.int32), z[keep].view(torch.int32))
    y64 = finite.double() @ w.T.contiguous()
    bound = TOL * finite.double().norm(dim=1, keepdim=True) * w.norm(dim=1)[None, :]
    assert bool(((z.double() - y64).abs() <= bound)[keep].all())
    for r in bad:
        want = (w * x[r].double()[None, :]).sum(dim=1)
        assert torch.equal(torch.isnan(y[r]), torch.isnan(want)), r
        inf = ~torch.isnan(want)
        assert bool((y[r][inf].double() == want[inf]).all()), r


@pytest.mark.parametrize("m,n,k", [(1025, 2305, 2112), (385, 6201, 4160), (513, 14340, 1088)])
@pytest.mark.parametrize("kind", ["channels 50", "channels 100", "channels 1e4", "channels 1e6",
                                  "rows 1e3", "every block 1e3", "elements 50", "misaligned 1e3"])
def test_q4_digits_outliers(qc, oracle, dev, kind, m, n, k):
    """Elements far above the rest of their block, where the codes there are
    zero or not: the re-encoded q4_0 form is no further from 64 bits than a
    hi + lo pair of bf16 activations (2^-18 of each element) would be, up to the
    2^-20 of the largest that eight digits are for.  (f32 sums add at most sqrt(K / 32) 2^-25 of the
    result on either: 4e-7 covers it.)  Sizes for its three tiles, with one and
    two K ranges."""
    import torch
    print(f"q4 outliers {kind} m={m} n={n} k={k}", flush=True)
    g = torch.Generator(device=dev).manual_seed(m + n + k)
    ratio = float(kind.split()[-1])
    X = torch.zeros(m * k + 1, device=dev)
    x = (X[1:] if kind.startswith("misaligned") else X[:-1]).view(m, k)
    x.copy_(torch.randn((m, k), generator=g, device=dev))
    channels = torch.arange(0, k, 32, device=dev) + 7 if kind.startswith("every") else \
        torch.tensor([5, k - 40], device=dev)
    if kind.startswith("elements"):
        hit = torch.rand((m, k), generator=g, device=dev) < 0.002
        x[hit] *= ratio
    elif kind.startswith("rows"):
        rows = torch.tensor([3, 40, 41, m - 1], device=dev)
        x[rows[:, None], channels[None, :]] = ratio
    else:
        x[:, channels] = ratio * (1.0 + 0.1 * torch.randn((m, len(channels)), generator=g, device=dev))
    w = torch.randn((n, k), generator=g, device=dev) * 0.02
    w[: n // 2, channels] = 0.0
    P = qc.pack(1, w)
    wd = torch.from_numpy(oracle.unpack(1, P.cpu().numpy(), n, k)).to(dev).double()
    assert bool((wd[: n // 2, channels] == 0).all())
    y = torch.full((m, n), float("nan"), device=dev)
    assert qc.qgemm_raw(1, P, x, y, m, n, k) == 0
    torch.cuda.synchronize()
    hi = x.bfloat16().float()
    pair = hi.double() + (x - hi).bfloat16().double()
    for half in (slice(0, n // 2), slice(n // 2, n)):   # codes of zero in the channels; any
        wt = wd[half].T.contiguous()
        y64 = x.double() @ wt
        old = (pair @ wt - y64).norm(dim=1)
        new = (y[:, half].double() - y64).norm(dim=1)
        size = y64.norm(dim=1)
        assert float(new.norm() / size.norm()) <= float(old.norm() / size.norm()) + 4e-7
        # row by row, a row's own draw of roundings aside
        assert bool((new <= 1.5 * old + 4e-7 * size).all()), float((new / old).max())


@pytest.mark.parametrize("fmt,m,n,k", [
    (1, 4700, 2079, 14336),     # 6-bit form: two chunks of rows, the first in two K ranges
    (1, 400, 18945, 14336),     # two chunks of columns
    (1, 4700, 18945, 14336),    # both
    (1, 4700, 300, 14336), (0, 4700, 300, 14336)])   # f16 form: two chunks of rows
def test_chunks(qc, dev, fmt, m, n, k):
    """Calls whose encoded operands pass the 256 MB of a chunk, with ragged
    remainders in both directions, rows that the 6-bit form gives further
    digits and one that is not finite in each chunk of rows."""
    import torch
    print(f"chunks fmt={fmt} m={m} n={n} k={k}", flush=True)
    g = torch.Generator(device=dev).manual_seed(m + n)
    P = qc.pack(fmt, torch.randn((n, k), generator=g, device=dev) * 0.02)
    x = torch.randn((m, k), generator=g, device=dev)
    x[::50, 77] = 3000.0
    bad = [7, m - 3]
    x[bad, 1234] = float("nan")
    y, z = (torch.full((m, n), float("nan"), device=dev) for _ in range(2))
    for out in (y, z):
        assert qc.qgemm_raw(fmt, P, x, out, m, n, k) == 0
    torch.cuda.synchronize()
    assert torch.equal(y.view(torch.int32), z.view(torch.int32))
    assert bool(torch.isnan(y[bad]).all())
    del z
    w = qc.unpack(fmt, P, n, k).double()
    x[bad] = 0.0
    y[bad] = 0.0
    wt = w.T.contiguous()
    for r in range(0, m, 1024):
        xs = x[r:r + 1024].double()
        y64 = xs @ wt
        err = (y[r:r + 1024].double() - y64).abs()
        assert bool((err <= TOL * xs.norm(dim=1, keepdim=True) * w.norm(dim=1)[None, :]).all()), r
        rel = float(err.norm() / y64.norm())
        assert rel < 2e-6, (r, rel)
