"""GPU parity of the pre-norm projections (sys1hip_fold_norm_weight,
sys1hip_norm_linear_bf16) against the oracle's unfused reference chain:
norm -> bf16 -> projection -> epilogue, as the reference runs it
(ModernBERT: bias-free LayerNorm, src/archs/modernbert.rs:865-868,884,1005-1034;
Qwen3.5: RMSNorm(1+w), src/archs/qwen35_text.rs:178-203,933,939).

Bar: the projection path's parity metrics, relative Frobenius error <= 1e-2
and max-abs error <= 2e-2 * max|ref|, per output.  The fused path folds the
norm weight into the bf16 weight and normalises the f32 accumulators, so it
rounds in different places from the reference (which rounds the normalised
activations); the bar is the tolerance, not bit equality.  The inputs carry
per-row offsets and a few large columns, as residual streams do, so that
the LayerNorm mean term (r_m mu_m colsum_n) is exercised.
"""
import numpy as np
import pytest

from gpu_helpers import assert_parity, to_gpu_bf16, to_np

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from sys1_amd.device import HipDevice
    d = HipDevice(0)
    yield d
    d.set_kernel(-1)
    d.set_grid(0)


def _stream(orc, M, K, seed):
    """Residual-stream-like rows: N(0,1) + a per-row offset, 4 columns x6."""
    x = orc.fill_normal((M, K), seed)
    x += orc.fill_normal((M, 1), seed + 7, 0.7)
    x[:, [1, K // 3, K // 2, K - 2]] *= 6.0
    return orc.round_bf16(x)


def _weights(orc, N, K, seed, kind):
    w = orc.round_bf16(orc.fill_normal((N, K), seed, 0.02))
    g = orc.fill_normal((K,), seed + 3, 0.1)
    g = orc.round_bf16(1.0 + g) if kind == "layer" else orc.round_bf16(g)  # LN weight ~1; RMS w ~0
    return w, g


def _ref(orc, x, w, g, kind, eps, gated):
    if kind == "layer":
        xn = orc.layer_norm_bf16(x, g, eps)
    else:
        xn = orc.round_bf16(orc.rms_norm(x, g, eps))
    proj = orc.linear_f32(xn, w)
    if gated == "gelu":
        return orc.geglu(proj)
    if gated == "silu":
        return orc.swiglu(*np.split(proj, 2, axis=1))
    return orc.round_bf16(proj)


CASES = [
    # (kind, gated, M, N, K): ModernBERT-base Wqkv / Wi, Qwen-small qkv and gate/up shapes
    ("layer", None, 1000, 2304, 768),
    ("layer", "gelu", 1000, 2304, 768),
    ("layer", None, 64, 768, 768),
    ("layer", "gelu", 200, 5248, 1024),
    ("rms", None, 1000, 4608, 2048),
    ("rms", "silu", 700, 2048, 2048),
    ("rms", None, 128, 1024, 2048),
    ("rms", "silu", 33, 1024, 512),
    ("layer", None, 40, 256, 8200),   # rows longer than the register-resident statistics path
    ("rms", None, 40, 256, 8200),
]


@pytest.mark.parametrize("kind,gated,M,N,K", CASES)
def test_norm_linear_matches_unfused_chain(dev, orc, kind, gated, M, N, K):
    from sys1_amd.norm import NormLinear
    eps = 1e-5 if kind == "layer" else 1e-6
    print(f"[gpu] norm={kind} gated={gated} M={M} N={N} K={K}", flush=True)
    x = _stream(orc, M, K, 11 + M)
    w, g = _weights(orc, N, K, 5 + N, kind)
    lin = NormLinear(to_gpu_bf16(w, torch), torch.from_numpy(g), kind, eps, gated, device=dev)
    y = to_np(lin(to_gpu_bf16(x, torch)))
    ref = _ref(orc, x, w, g, kind, eps, gated)
    assert y.shape == ref.shape
    rel, mx = assert_parity(y, ref, f"{kind}/{gated} M={M} N={N} K={K}")
    print(f"[gpu]   rel_fro={rel:.2e} max_abs/max={mx:.2e}", flush=True)


@pytest.mark.parametrize("offset", [4.0, 16.0])
def test_layernorm_rows_with_large_means(dev, orc, offset):
    """Rows whose mean is large against their spread: the epilogue's r (acc -
    mu c) cancels heavily, and the -mu c term (a bf16 hi/lo-split MFMA in
    the kernel) must keep the result within the projection tolerance, on the
    producer-wave 128x128 shape and on the plain one."""
    from sys1_amd import kernel_names
    from sys1_amd.norm import NormLinear
    M, N, K = 600, 2304, 768
    x = orc.fill_normal((M, K), 61)
    x += offset * (1.0 + orc.fill_normal((M, 1), 62, 0.25))
    x = orc.round_bf16(x)
    w, g = _weights(orc, N, K, 63, "layer")
    ref = _ref(orc, x, w, g, "layer", 1e-5, None)
    lin = NormLinear(to_gpu_bf16(w, torch), torch.from_numpy(g), "layer", 1e-5, None, device=dev)
    try:
        for name in ("tile_128x128_s2_w2x2_p4", "tile_128x128_s2_w2x2", None):
            dev.set_kernel(kernel_names().index(name) if name else -1)
            print(f"[gpu] layernorm offset={offset} kernel={name or 'auto'}", flush=True)
            rel, mx = assert_parity(to_np(lin(to_gpu_bf16(x, torch))), ref, f"offset {offset} {name}")
            print(f"[gpu]   rel_fro={rel:.2e} max_abs/max={mx:.2e}", flush=True)
    finally:
        dev.set_kernel(-1)


def test_fold_is_exact_and_colsum_sums_the_folded_rows(dev, orc):
    from sys1_amd.norm import fold_norm_weight
    N, K = 300, 1032
    for kind in ("layer", "rms"):
        w, g = _weights(orc, N, K, 17, kind)
        print(f"[gpu] fold {kind} N={N} K={K}", flush=True)
        wf, cs = fold_norm_weight(to_gpu_bf16(w, torch), torch.from_numpy(g), kind, device=dev)
        a = g if kind == "layer" else 1.0 + g.astype(np.float32)
        expect = orc.round_bf16(w * a[None, :].astype(np.float32))
        np.testing.assert_array_equal(to_np(wf), expect)
        if kind == "layer":
            s64 = expect.astype(np.float64).sum(axis=1)
            got = cs.cpu().numpy().astype(np.float64)
            assert np.abs(got - s64).max() <= 1e-5 * np.abs(expect).sum(axis=1).max()
        else:
            assert cs is None


def test_every_kernel_with_every_norm_epilogue(dev, orc):
    """Force each kernel id (tile and stream-K schedules) through the four
    pre-norm epilogues on a ragged shape."""
    from sys1_amd import kernel_names
    from sys1_amd.norm import NormLinear
    M, N, K = 300, 384, 328
    x = _stream(orc, M, K, 23)
    xg = to_gpu_bf16(x, torch)
    try:
        for kind, gated in (("layer", None), ("layer", "gelu"), ("rms", None), ("rms", "silu")):
            eps = 1e-5 if kind == "layer" else 1e-6
            w, g = _weights(orc, N, K, 29, kind)
            lin = NormLinear(to_gpu_bf16(w, torch), torch.from_numpy(g), kind, eps, gated, device=dev)
            ref = _ref(orc, x, w, g, kind, eps, gated)
            for kid, name in enumerate(kernel_names()):
                # (the gated epilogues need whole 32-row gate/up groups)
                if gated and name.startswith("skinny_") and int(name.split("_")[1].split("x")[1]) % 32:
                    continue
                dev.set_kernel(kid)
                print(f"[gpu] {name} norm={kind} gated={gated}", flush=True)
                assert_parity(to_np(lin(xg)), ref, f"{name} {kind}/{gated}")
    finally:
        dev.set_kernel(-1)


def test_rows_are_independent_and_repeat_bitwise(dev, orc):
    """Row statistics are per row: a permutation of the rows permutes the
    output exactly, and a second call gives the same bits."""
    from sys1_amd.norm import NormLinear
    M, N, K = 513, 768, 768
    x = _stream(orc, M, K, 31)
    w, g = _weights(orc, N, K, 37, "layer")
    lin = NormLinear(to_gpu_bf16(w, torch), torch.from_numpy(g), "layer", 1e-5, device=dev)
    xg = to_gpu_bf16(x, torch)
    y1 = lin(xg)
    y2 = lin(xg)
    assert torch.equal(y1, y2)
    perm = torch.from_numpy(np.random.default_rng(0).permutation(M)).to(xg.device)
    yp = lin(xg[perm].contiguous())
    assert torch.equal(yp, y1[perm])


def test_norm_linear_errors(dev, orc):
    from sys1_amd import _lib
    from sys1_amd.norm import NormLinear
    w = torch.zeros(64, 64, dtype=torch.bfloat16, device="cuda:0")
    g = torch.ones(64)
    with pytest.raises(ValueError):
        NormLinear(w, g, "batch", 1e-5, device=dev)
    with pytest.raises(ValueError):
        NormLinear(w, torch.ones(32), "layer", 1e-5, device=dev)
    lin = NormLinear(w, g, "layer", 1e-5, device=dev)
    with pytest.raises(ValueError):
        lin(torch.zeros(4, 32, dtype=torch.bfloat16, device="cuda:0"))
    # RMSNorm with GeGLU is not a combination the reference has.
    with pytest.raises(_lib.Sys1HipError):
        NormLinear(torch.zeros(64, 64, dtype=torch.bfloat16, device="cuda:0"), g, "rms", 1e-6,
                   "gelu", device=dev)(torch.zeros(4, 64, dtype=torch.bfloat16, device="cuda:0"))


def test_blocked_weight_with_every_norm_epilogue_is_bitwise_row_major(dev, orc):
    """The folded weight in the blocked layout (what ProjectionStack(norms=True,
    blocked=True) and the bench run) gives the row-major folded weight's
    results bit for bit, on a forced kernel of every family (tile, stream-K,
    skinny) and every pre-norm epilogue, with N and K not multiples of the
    32 x 64 block."""
    from sys1_amd import kernel_names
    from sys1_amd.norm import NormLinear
    names = kernel_names()
    picks = [next(i for i, n in enumerate(names) if n.startswith(f)) for f in ("tile_", "stream_", "skinny_")]
    picks += [i for i, n in enumerate(names) if n.startswith("skinny_") and int(n.split("_")[1].split("x")[1]) % 32 == 0][:1]
    M, N, K = 150, 352, 328
    x = _stream(orc, M, K, 41)
    xg = to_gpu_bf16(x, torch)
    try:
        for kind, gated in (("layer", None), ("layer", "gelu"), ("rms", None), ("rms", "silu")):
            eps = 1e-5 if kind == "layer" else 1e-6
            w, g = _weights(orc, N, K, 43, kind)
            wg, gg = to_gpu_bf16(w, torch), torch.from_numpy(g)
            rm = NormLinear(wg, gg, kind, eps, gated, device=dev)
            bl = NormLinear(wg, gg, kind, eps, gated, device=dev, blocked=True)
            ref = _ref(orc, x, w, g, kind, eps, gated)
            for kid in picks:
                name = names[kid]
                if gated and name.startswith("skinny_") and int(name.split("_")[1].split("x")[1]) % 32:
                    continue
                dev.set_kernel(kid)
                print(f"[gpu] blocked norm {name} {kind}/{gated}", flush=True)
                a, b = rm(xg), bl(xg)
                assert torch.equal(a, b), f"{name} {kind}/{gated}"
                assert_parity(to_np(b), ref, f"blocked {name} {kind}/{gated}")
    finally:
        dev.set_kernel(-1)


@pytest.mark.parametrize("name,grid", [("skinny_16x16_w16", 0), ("skinny_128x32_w8", 0), ("skinny_64x48_w8", 0),
                                       ("stream_32x256_s4_w1x4_p4", 7), ("stream_128x256_s3_w2x4", 5),
                                       ("stream_64x256_s4_w2x4_p4", 3)])
@pytest.mark.parametrize("kind", ["layer", "rms"])
def test_row_sums_of_the_multiplying_kernels(dev, orc, name, grid, kind):
    """The skinny and stream-K kernels on rows up to 16 deviations off zero (a
    ragged last tile row, split tiles), and with an infinity in a row, which
    stays that row's alone.  Projection tolerance, as everywhere: the
    statistics themselves are test_row_statistics_on_every_kernel's."""
    from sys1_amd import kernel_names
    from sys1_amd.norm import NormLinear
    N, K = 330, 712
    eps = 1e-5 if kind == "layer" else 1e-6
    w, g = _weights(orc, N, K, 71, kind)
    lin = NormLinear(to_gpu_bf16(w, torch), torch.from_numpy(g), kind, eps, None, device=dev)
    try:
        dev.set_kernel(kernel_names().index(name))
        dev.set_grid(grid)
        for M in (1, 17, 133):
            print(f"[gpu] row sums {name} grid={grid} {kind} M={M}", flush=True)
            x = orc.fill_normal((M, K), 80 + M)
            x += np.array([0.0, 3.0, 6.0, -16.0, 0.1], np.float32)[np.arange(M) % 5][:, None]
            x = orc.round_bf16(x)
            ref = _ref(orc, x, w, g, kind, eps, None)
            assert_parity(to_np(lin(to_gpu_bf16(x, torch))), ref, f"{name} {kind} M={M}")
            if M == 1:
                continue
            x[7, 11] = np.inf
            y = to_np(lin(to_gpu_bf16(x, torch)))
            # LayerNorm: inf - inf; RMSNorm: inf / inf.  NaN throughout the row.
            assert np.isnan(y[7]).all()
            keep = np.arange(M) != 7
            assert_parity(y[keep], ref[keep], f"{name} {kind} M={M} beside an infinity")
    finally:
        dev.set_kernel(-1)
        dev.set_grid(0)


def _readout(orc, M, N, K, kind, seed):
    """Inputs whose products and sums are exact in f32 in any order, so that
    an output shows its row's statistics and nothing else: small integers
    around an offset, a power of two per row, and weight rows with one entry
    (RMSNorm) or a +v, -v pair, whose column sum is zero (LayerNorm)."""
    rng = np.random.default_rng(seed)
    rows = [(0, 1.0), (3, 1.0), (50, 2.0 ** -60), (-100, 1.0), (0, 2.0 ** -12), (120, 2.0 ** 40)]
    if kind == "layer":
        # sigma 4.9 at 130 * 2^52: the squares' sum overflows f32, the deviations' does not
        rows.append((120, 2.0 ** 53))
    off, scale = (np.array(v, np.float64)[np.arange(M) % len(rows)][:, None] for v in zip(*rows))
    x = (rng.integers(-8, 9, (M, K)) + off) * scale
    w = np.zeros((N, K), np.float32)
    v = orc.round_bf16(rng.uniform(0.5, 2.0, N).astype(np.float32))
    cols = np.stack([rng.permutation(K)[:2] for _ in range(N)])
    w[np.arange(N), cols[:, 0]] = v
    if kind == "layer":
        w[np.arange(N), cols[:, 1]] = -v
    return x.astype(np.float32), w


@pytest.mark.parametrize("kind", ["layer", "rms"])
@pytest.mark.parametrize("K", [712, 1032])
def test_row_statistics_on_every_kernel(dev, orc, kind, K):
    """Whoever takes the row statistics (the pass, a skinny kernel's waves for
    LayerNorm up to K = 1024, the sums of the skinny and stream-K kernels for
    RMSNorm): the same outputs bit for bit, each within one bf16 rounding
    (2^-8) of float64, for rows far off zero, scaled down to where eps is
    all, and up to where x^2 summed over the row would overflow."""
    from sys1_amd import kernel_names
    from sys1_amd.norm import NormLinear
    N, eps = 200, 1e-5
    names = kernel_names()
    first = names.index("tile_128x128_s2_w2x2")
    order = [first] + [i for i in range(len(names)) if i != first]
    try:
        for M in (1, 17, 133, 300):
            x, w = _readout(orc, M, N, K, kind, 7 * M + K)
            x64 = x.astype(np.float64)
            mu = x64.mean(1, keepdims=True) if kind == "layer" else 0.0
            # (a LayerNorm's mean term drops out: the weight rows sum to zero)
            ref = x64 @ w.T.astype(np.float64) / np.sqrt(((x64 - mu) ** 2).mean(1, keepdims=True) + eps)
            g = torch.ones(K) if kind == "layer" else torch.zeros(K)
            lin = NormLinear(to_gpu_bf16(w, torch), g, kind, eps, None, device=dev)
            xg = to_gpu_bf16(x, torch)
            for kid in order:
                dev.set_kernel(kid)
                print(f"[gpu] statistics {names[kid]} {kind} M={M} K={K}", flush=True)
                y = to_np(lin(xg))
                if kid == first:
                    expect = y
                    assert (np.abs(y - ref) <= 2.0 ** -8 * np.abs(ref)).all()
                np.testing.assert_array_equal(y, expect, err_msg=f"{names[kid]} M={M}")
    finally:
        dev.set_kernel(-1)


@pytest.mark.parametrize("grid", [0, 7])
def test_rms_row_sums_hold_their_precision(dev, orc, grid):
    """The sums of squares that the skinny and stream-K kernels take: a row of
    ones behind one 2^13, whose square an f32 sum would add no 1 or 2 to (a
    lane's whole share lost: f32 sums were up to 4.8e-6 of 1/rms off).  Read
    off 1/rms to 2^-21 from the column whose product first rounds to bf16's
    1 + 2^-7; bound 1e-6: 3 of the 2^13's fragment's 4 f32 sums round by up to
    4 (0.9e-7 of 1/rms), the mean, root, quotient and product 0.6e-7 each at
    most, the column 4.8e-7."""
    from sys1_amd import kernel_names
    from sys1_amd.norm import NormLinear
    N, K, M = 512, 5120, 40
    x = np.ones((M, K), np.float32)
    x[np.arange(M), (np.arange(M) * 136) % (K - 8)] = 2.0 ** 13  # (row 0: its first element)
    r = 1.0 / np.sqrt((x.astype(np.float64) ** 2).mean(1)[0] + 1e-6)  # the same for every row
    # products v_n around (1 + 2^-8) / r, 2^-21 apart, as three bf16 parts on columns where x = 1
    v = ((1 + 2.0 ** -8) / r * (1 + (np.arange(N) - N // 2) * 2.0 ** -21)).astype(np.float32)
    w = np.zeros((N, K), np.float32)
    rest = v.copy()
    for c in (K - 7, K - 4, K - 1):
        w[:, c] = orc.round_bf16(rest)
        rest = rest - w[:, c]
    assert (rest == 0).all() and (x[:, [K - 7, K - 4, K - 1]] == 1).all()
    lin = NormLinear(to_gpu_bf16(w, torch), torch.zeros(K), "rms", 1e-6, None, device=dev)
    xg = to_gpu_bf16(x, torch)
    try:
        dev.set_grid(grid)
        for kid, name in enumerate(kernel_names()):
            if not name.startswith(("skinny_", "stream_")):
                continue
            dev.set_kernel(kid)
            print(f"[gpu] rms row sums {name} grid={grid}", flush=True)
            y = to_np(lin(xg))
            assert np.isin(y, [1.0, 1.0 + 2.0 ** -7]).all()
            first = (y > 1.0).argmax(axis=1)
            err = -(first - N // 2) * 2.0 ** -21
            assert np.abs(err).max() <= 1e-6, f"{name}: {np.abs(err).max():.1e}"
    finally:
        dev.set_kernel(-1)
        dev.set_grid(0)
