"""GPU parity of the INT4 group-128 projections (engine.cu:83-109, launched
at 626-630, 792-797, 858-859) through the C-ABI, against the oracle.

The GPU sums in fp32 in its own order, the oracle in fp64; the tolerance is
written against the scale of the summation error:
    |y_gpu - y_ref| <= 1e-5 * sum_k |x[k] * w[n][k]|
(fp32 sums of a few thousand terms stay orders of magnitude inside it; one
dropped or doubled term of typical size is ~1/K of the sum of magnitudes,
about 50x the bound at K = 2048)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

REL = 1e-5


def _weights(rng, N, K, orc, kind="normal"):
    if kind == "normal":
        w = (rng.standard_normal((N, K)) * 0.02).astype(np.float32)
        w[rng.integers(0, N, 8), rng.integers(0, K, 8)] *= 30.0  # outliers set their groups' scales
        return orc.quant_int4_g128(w)
    if kind == "extreme":  # nibbles 0 (-8) and 15 (+7), zero-scale groups
        packed = rng.choice(np.array([0x00, 0xFF, 0x0F, 0xF0, 0x88], np.uint8), (N, K // 2))
        scales = rng.uniform(0.001, 0.5, (N, K // 128)).astype(np.float16).view(np.uint16)
        scales[:, ::3] = 0
        return packed, scales
    raise ValueError(kind)


def _t(a, dev):
    a = np.ascontiguousarray(a)
    if a.dtype == np.uint16:
        a = a.view(np.int16)
    return torch.from_numpy(a).to(dev)


def _check(got, ref, ab, what, extra=0.0):
    err = np.abs(got.astype(np.float64) - ref.astype(np.float64))
    bound = REL * ab.astype(np.float64) + extra + 1e-30
    bad = err > bound
    if bad.any():
        i = np.unravel_index(np.argmax(err - bound), err.shape)
        raise AssertionError(f"{what}: {bad.sum()} of {bad.size} outside; worst at {i}: "
                             f"got {got[i]} ref {ref[i]} absum {ab[i]}")


CASES = [
    (2048, 2048, 1, "normal", 0),   # q_proj / out_proj at decode
    (512, 2048, 1, "normal", 1),    # k_proj / v_proj
    (96, 128, 1, "normal", 2),      # one group per row
    (100, 384, 3, "normal", 3),     # ragged rows, K < 2048, three rows of x
    (33, 2176, 5, "normal", 4),     # K = 17 groups: a second, partial lane pass
    (2048, 4096, 2, "normal", 5),
    (64, 2048, 1, "extreme", 6),
    (512, 2048, 9, "normal", 7),
    (2048, 2048, 96, "normal", 8),
    (100, 384, 200, "normal", 9),    # ragged tiles in both directions
    (520, 2048, 300, "extreme", 13),
    # the K-split GEMM's edges: first M, one row past a tile, rows of W that end
    # inside a tile, fewer groups than waves (K = 128, 384), a second and a
    # partial third pass over the groups (K = 1152, 2176), the largest K
    (100, 128, 3, "normal", 20),
    (130, 384, 16, "normal", 21),
    (47, 1152, 17, "normal", 22),
    (200, 2176, 33, "normal", 23),
    (48, 4096, 65, "normal", 24),
    (2000, 256, 130, "normal", 26),
    (2048, 128, 300, "normal", 27),
    (2050, 384, 511, "normal", 28),
    (33, 256, 768, "normal", 29),
    # its multi-pass forms at wider tiles, and the tile GEMM beyond its K
    (2048, 2176, 130, "normal", 31),
    (2048, 4096, 300, "normal", 32),
    (2048, 2176, 511, "normal", 33),
    (48, 4224, 40, "normal", 25),    # (the GEMV: 55 rows and fewer)
    (48, 4224, 60, "normal", 34),
    (200, 4096, 2100, "normal", 30),
]


@pytest.mark.parametrize("N,K,M,kind,seed", CASES)
def test_gemv_int4(orc, cia, dev, N, K, M, kind, seed):
    from cuda_inf_amd import kernels as KK
    rng = np.random.default_rng(seed)
    packed, scales = _weights(rng, N, K, orc, kind)
    x = rng.standard_normal((M, K)).astype(np.float16)
    ref, ab = orc.gemv_int4(x, packed, scales, want_absum=True)
    print(f"gemv_int4 N={N} K={K} M={M} {kind}", flush=True)
    y = torch.full((M, N), float("nan"), dtype=torch.float32, device=dev)
    KK.gemv_int4(_t(x, dev), _t(packed, dev), _t(scales, dev), y, N, K, M)
    torch.cuda.synchronize()
    _check(y.cpu().numpy(), ref, ab, "y")
    # out_proj + residual: y += x W^T
    y0 = rng.standard_normal((M, N)).astype(np.float32)
    yd = torch.from_numpy(y0).to(dev)
    KK.gemv_int4(_t(x, dev), _t(packed, dev), _t(scales, dev), yd, N, K, M, add=True)
    torch.cuda.synchronize()
    _check(yd.cpu().numpy(), y0.astype(np.float64) + ref, ab, "y + residual",
           extra=2 * np.finfo(np.float32).eps * (np.abs(y0) + np.abs(ref)))


@pytest.mark.parametrize("M,seed", [(1, 10), (2, 31), (3, 11), (6, 12), (16, 32), (40, 33), (130, 14),
                                    (300, 34), (600, 37)])
def test_qkv_proj_int4(orc, cia, dev, M, seed):
    """q/k/v in one launch with the fp16 conversion fused: each output is
    the fp16 rounding of the same kernel's fp32 sum (compared with the fp32
    GEMV bit for bit) and within tolerance of the oracle."""
    from cuda_inf_amd import kernels as KK
    rng = np.random.default_rng(seed)
    K = 2048
    W = {n: _weights(rng, N, K, orc) for n, N in (("q", 2048), ("k", 512), ("v", 512))}
    x = (rng.standard_normal((M, K)) * 0.5).astype(np.float16)
    xd = _t(x, dev)
    Wd = {n: (_t(p, dev), _t(s, dev)) for n, (p, s) in W.items()}
    out = {n: torch.zeros((M, N), dtype=torch.float16, device=dev)
           for n, N in (("q", 2048), ("k", 512), ("v", 512))}
    print(f"qkv_proj_int4 M={M}", flush=True)
    KK.qkv_proj_int4(xd, Wd["q"], Wd["k"], Wd["v"], out["q"], out["k"], out["v"], M, K)
    torch.cuda.synchronize()
    for n in ("q", "k", "v"):
        N = out[n].shape[1]
        y = torch.zeros((M, N), dtype=torch.float32, device=dev)
        KK.gemv_int4(xd, Wd[n][0], Wd[n][1], y, N, K, M)
        torch.cuda.synchronize()
        want16 = y.cpu().numpy().astype(np.float16)
        got16 = out[n].cpu().numpy()
        assert np.array_equal(got16.view(np.uint16), want16.view(np.uint16)), n
        ref, ab = orc.gemv_int4(x, *W[n], want_absum=True)
        _check(got16.astype(np.float32), ref, ab, n,
               extra=np.abs(ref) * 2.0 ** -11 + 2.0 ** -25)


# Every matrix-core kernel and tile shape adds a row's groups in the same order
# from 56 rows of x on: launches over the first M rows, one M for each shape that
# the rule of a size takes, have the bits of one launch of the 128 x 128 tiles.
# (K above 2048: three and four passes of the K-split kernel, no 256-row tiles.)
@pytest.mark.parametrize("N,K,shapes,seed", [
    (64, 2048, {0, 1}, 60), (512, 2048, {0, 1, 2, 3, 4, 5}, 61), (2048, 2048, {1, 2, 3, 4, 5, 7}, 62),
    (8192, 2048, {5, 2, 7, 8}, 63), (2050, 384, {2, 3, 4, 5, 7}, 64),
    (2048, 2176, {1, 2, 3, 4, 5}, 65), (512, 4096, {0, 1, 2, 3, 4, 5}, 66)])
def test_kernels_have_the_tile_kernels_bits(orc, cia, dev, int4_choose, N, K, shapes, seed):
    from cuda_inf_amd import kernels as KK
    rng = np.random.default_rng(seed)
    rows = np.arange(56, 2400)
    chosen = np.array([c[0] for c in int4_choose([(int(m), N, K) for m in rows])])
    first = {}  # shape -> a ragged M that takes it, its first one and its last
    for i in sorted(set(chosen)):
        at = rows[chosen == i]
        first[i] = sorted({int(at[0]), int(at[len(at) // 2]) | 1, int(at[-1])} & set(at.tolist()))
    assert shapes <= set(first) - {6}
    M, most = first[6][-1], max(m for ms in first.values() for m in ms)
    packed, scales = _weights(rng, N, K, orc)
    x = rng.standard_normal((most, K)).astype(np.float16)
    xd, pd, sd = _t(x, dev), _t(packed, dev), _t(scales, dev)
    for add in (False, True):
        y0 = torch.full((most, N), 0.5 if add else float("nan"), dtype=torch.float32, device=dev)
        y = y0[:M].clone()
        KK.gemv_int4(xd[:M], pd, sd, y, N, K, M, add=add)
        for i, ms in first.items():
            for m in ms:
                z = y0[:m].clone()
                print(f"N={N} K={K} shape {i} M={m} add={add}", flush=True)
                KK.gemv_int4(xd[:m], pd, sd, z, N, K, m, add=add)
                torch.cuda.synchronize()
                n = min(m, M)
                assert torch.equal(z[:n], y[:n]) and not z.isnan().any(), (i, m)


@pytest.mark.parametrize("N,K,shapes,seed", [
    (64, 2048, {0}, 70), (3072, 2048, {0, 1, 2}, 71), (9000, 2176, {1, 3, 4}, 72), (12300, 4096, {1, 2, 5}, 73)])
def test_few_rows_have_the_same_bits(orc, cia, dev, int4_choose, N, K, shapes, seed):
    """Below 56 rows of x the sums take another order (four chains a pass), the
    same in every tile shape: 55 rows against slices of them, and against the
    same rows of a narrow matrix (its own shapes)."""
    from cuda_inf_amd import kernels as KK
    rng = np.random.default_rng(seed)
    M, lo = 55, 3 + 2 * int4_choose([(3, N, K)])[0][1]
    assert {c[0] for c in int4_choose([(m, N, K) for m in (lo, 16, 17, 33, 40, 55)])} == shapes
    packed, scales = _weights(rng, N, K, orc)
    xd = _t(rng.standard_normal((M, K)).astype(np.float16), dev)
    pd, sd = _t(packed, dev), _t(scales, dev)
    y = torch.full((M, N), float("nan"), dtype=torch.float32, device=dev)
    KK.gemv_int4(xd, pd, sd, y, N, K, M)
    for m in (lo, 16, 17, 33, 40):
        z = torch.full((m, N), float("nan"), dtype=torch.float32, device=dev)
        print(f"N={N} K={K} M={m}", flush=True)
        KK.gemv_int4(xd[:m], pd, sd, z, N, K, m)
        torch.cuda.synchronize()
        assert torch.equal(z, y[:m]), m
    n = 40  # the first 40 rows of W alone
    z = torch.full((M, n), float("nan"), dtype=torch.float32, device=dev)
    KK.gemv_int4(xd, pd, sd, z, n, K, M)
    torch.cuda.synchronize()
    assert torch.equal(z, y[:, :n])


# The 256-row tiles: 128 and 192 columns a tile, each with ragged last rows and
# columns and tiles past the end of the grid; one, two, three and sixteen groups.
# The rows have the bits of launches over slices of them, whatever those take;
# the first and last rows are checked against the oracle.
BIG_TILES = [(2080, 128, 2060, 2, 40), (2080, 384, 2060, 2, 41), (4100, 256, 2561, 3, 42),
             (1100, 2048, 4000, 4, 43), (3072, 2048, 2700, 3, 44)]


@pytest.mark.parametrize("N,K,M,parts,seed", BIG_TILES)
def test_gemm_big_tiles(orc, cia, dev, int4_choose, N, K, M, parts, seed):
    from cuda_inf_amd import kernels as KK
    assert int4_choose([(M, N, K)])[0][0] >= 7
    rng = np.random.default_rng(seed)
    packed, scales = _weights(rng, N, K, orc, "normal")
    x = rng.standard_normal((M, K)).astype(np.float16)
    xd, pd, sd = _t(x, dev), _t(packed, dev), _t(scales, dev)
    print(f"big tiles N={N} K={K} M={M}", flush=True)
    for add in (False, True):
        y0 = torch.full((M, N), 0.5 if add else float("nan"), dtype=torch.float32, device=dev)
        y, z = y0.clone(), y0.clone()
        KK.gemv_int4(xd, pd, sd, y, N, K, M, add=add)
        for r in torch.arange(M).tensor_split(parts):
            r0, n = int(r[0]), len(r)
            KK.gemv_int4(xd[r0:r0 + n], pd, sd, z[r0:r0 + n], N, K, n, add=add)
        torch.cuda.synchronize()
        assert torch.equal(y, z)
        if not add:
            ends = np.r_[0:3, M - 3:M]
            ref, ab = orc.gemv_int4(x[ends], packed, scales, want_absum=True)
            _check(y.cpu().numpy()[ends], ref, ab, "y")


@pytest.mark.parametrize("M,seed", [(1600, 35), (2700, 36)])
def test_qkv_big_tiles_bits(orc, cia, dev, M, seed):
    """The same for the 256-row tiles of 128 and 192 columns: the fp16
    rounding of each matrix's own fp32 sums, bit for bit."""
    from cuda_inf_amd import kernels as KK
    rng = np.random.default_rng(seed)
    K, rows = 2048, {"q": 2048, "k": 512, "v": 512}
    W = {n: tuple(_t(a, dev) for a in _weights(rng, N, K, orc)) for n, N in rows.items()}
    x = _t((rng.standard_normal((M, K)) * 0.5).astype(np.float16), dev)
    out = {n: torch.zeros((M, N), dtype=torch.float16, device=dev) for n, N in rows.items()}
    print(f"qkv big tiles M={M}", flush=True)
    KK.qkv_proj_int4(x, W["q"], W["k"], W["v"], out["q"], out["k"], out["v"], M, K)
    for n, N in rows.items():
        y = torch.zeros((M, N), dtype=torch.float32, device=dev)
        KK.gemv_int4(x, *W[n], y, N, K, M)
        torch.cuda.synchronize()
        assert torch.equal(out[n].view(torch.int16), y.half().view(torch.int16)), n


@pytest.mark.parametrize("M,seed", [(3, 50), (5, 53), (23, 51), (55, 52)])
def test_few_rows_no_further_off_than_gemv(orc, cia, dev, M, seed):
    """out_proj into the residual for the rows that the GEMV would take too: the
    2-norm distance from 64 bits is no larger than that of the GEMV, which runs
    for two rows at a time (its trees of sums have fewer roundings in a row than
    a sum over the 16 groups in order)."""
    from cuda_inf_amd import kernels as KK
    rng = np.random.default_rng(seed)
    N = K = 2048
    packed, scales = _weights(rng, N, K, orc)
    x = rng.standard_normal((M, K)).astype(np.float16)
    y0 = rng.standard_normal((M, N)).astype(np.float32)
    nib = np.stack((packed & 15, packed >> 4), -1).reshape(N, K).astype(np.float64) - 8.0
    w = nib * np.repeat(scales.view(np.float16).astype(np.float64), 128, axis=1)
    ref = y0.astype(np.float64) + x.astype(np.float64) @ w.T
    xd, pd, sd, y, z = _t(x, dev), _t(packed, dev), _t(scales, dev), _t(y0, dev), _t(y0, dev)
    print(f"few rows M={M}", flush=True)
    KK.gemv_int4(xd, pd, sd, y, N, K, M, add=True)
    for r in range(0, M, 2):
        n = min(2, M - r)
        KK.gemv_int4(xd[r:r + n], pd, sd, z[r:r + n], N, K, n, add=True)
    torch.cuda.synchronize()
    err, gemv = (np.linalg.norm(t.cpu().numpy() - ref) / np.linalg.norm(ref) for t in (y, z))
    assert err <= gemv, (err, gemv)
