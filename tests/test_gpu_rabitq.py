"""GPU parity of the one-bit RaBitQ quantizer against the oracle.

The device computes P^T x on the matrix cores in fp32 with a different
summation order than the oracle (the reference's cuBLAS order is
unspecified as well), so:
  * a code bit must match wherever |r_i| > 1e-5 * ||r|| (a sign can only
    differ where rounding moves r_i across zero);
  * f_rescale within 2e-5 relative; f_add within 2e-5 of the magnitude of
    its terms (||r||^2, 2||r||^2 s_cx / s_rx, <r, c'>, 1).
"""

import numpy as np
import pytest
import torch

import oracle

pytestmark = pytest.mark.gpu


def _check(jasper, x, m, c, metric, f16):
    n, dim = x.shape
    xt = torch.from_numpy(x.astype(np.float16 if f16 else np.float32)).cuda()
    rot = torch.from_numpy(np.asarray(m, dtype=np.float32)).cuda()
    cen = None if c is None else torch.from_numpy(c).cuda()
    got = jasper.rabitq_quantize(xt, rotation=rot, centroid=cen, distance=metric)
    torch.cuda.synchronize()
    nodes = got.nodes.cpu().numpy()
    xin = x.astype(np.float16).astype(np.float32) if f16 else x.astype(np.float32)
    ref, codes, f_add, f_rescale, r = oracle.rabitq_quantize(xin, m, c, metric=metric, return_residuals=True)
    assert nodes.shape == ref.shape
    cb = codes.shape[1]
    gb = np.unpackbits(nodes[:, :cb], axis=1, bitorder="little")[:, :dim]
    rb = np.unpackbits(codes, axis=1, bitorder="little")[:, :dim]
    nrm = np.sqrt((r.astype(np.float64) ** 2).sum(1))
    clear = np.abs(r) > 1e-5 * nrm[:, None]
    assert np.array_equal(gb[clear], rb[clear]), f"{(gb != rb)[clear].sum()} clear bits differ"
    assert not np.unpackbits(nodes[:, :cb], axis=1, bitorder="little")[:, dim:].any()
    ga = nodes[:, cb:cb + 4].copy().view(np.float32).ravel()
    gr = nodes[:, cb + 4:].copy().view(np.float32).ravel()
    np.testing.assert_allclose(gr, f_rescale, rtol=2e-5)
    rc = np.zeros(dim) if c is None else (np.asarray(m, np.float64).reshape(dim, dim).T @ c)
    s_cx = np.abs(rc).sum() * 0.5
    scale = nrm ** 2 * (1 + 2 * s_cx / np.maximum(0.5 * np.abs(r).sum(1), 1e-30)) + nrm * np.abs(rc).sum() + 1
    assert np.all(np.abs(ga - f_add) <= 2e-5 * scale), np.abs(ga - f_add).max()
    return got


@pytest.mark.parametrize("dim", [8, 32, 96, 100, 128, 200, 256])
@pytest.mark.parametrize("metric", ["l2", "ip"])
def test_rabitq_matches_oracle(jasper, oracle_lib, dim, metric):
    rng = np.random.default_rng(dim)
    n = 1000 + dim
    x = (rng.normal(size=(n, dim)) * 3).astype(np.float32)
    m, _ = oracle.rotation_matrix(dim, 42)
    c = (rng.normal(size=dim) * 0.5).astype(np.float32)
    _check(jasper, x, m, c, metric, f16=True)
    _check(jasper, x, m, None, metric, f16=False)


def test_rabitq_identity_closed_form(jasper, oracle_lib):
    rng = np.random.default_rng(7)
    x = rng.normal(size=(333, 64)).astype(np.float32)
    got = _check(jasper, x, np.eye(64, dtype=np.float32).ravel(), None, "l2", f16=False)
    sq = (x.astype(np.float64) ** 2).sum(1)
    np.testing.assert_allclose(got.f_add.cpu().numpy(), sq, rtol=1e-5)
    assert torch.equal(got.bits().cpu(), torch.from_numpy((x >= 0).astype(np.uint8)))


def test_rabitq_default_rotation_and_sizes(jasper, oracle_lib):
    x = torch.randn(5, 97, device="cuda", dtype=torch.float16)
    got = jasper.rabitq_quantize(x)
    assert got.nodes.shape == (5, 24) and got.code_bytes == 16
    assert torch.isfinite(got.f_add).all() and (got.f_rescale < 0).all()
    empty = jasper.rabitq_quantize(x[:0])
    assert empty.nodes.shape == (0, 24)


# fp16 rows: the smallest dims, a last output tile of one coordinate, the edge
# between P held in LDS whole (up to 160) and staged per K step, partial tiles
# of vectors; and a matrix whose columns differ by ten orders of magnitude,
# each split against its own largest entry.
@pytest.mark.parametrize("dim,n", [(1, 33), (16, 1), (17, 31), (144, 500), (160, 4097), (161, 47), (177, 300),
                                   (240, 129)])
@pytest.mark.parametrize("metric", ["l2", "ip"])
def test_rabitq_split_edges(jasper, oracle_lib, dim, n, metric):
    rng = np.random.default_rng(dim)
    x = rng.normal(size=(n, dim)).astype(np.float32)
    m, _ = oracle.rotation_matrix(dim, 5)
    c = (rng.normal(size=dim) * 0.5).astype(np.float32)
    _check(jasper, x, m, c, metric, f16=True)


def test_rabitq_columns_of_any_scale(jasper, oracle_lib):
    """r_i = sum_k P[k + i*dim] x_k for P's column i scaled by 10^(i % 11 - 5):
    the signs of every column's outputs are those of the 64-bit product."""
    dim, n = 96, 2000
    rng = np.random.default_rng(3)
    x = rng.normal(size=(n, dim)).astype(np.float16)
    p = (rng.normal(size=(dim, dim)) * 10.0 ** (np.arange(dim) % 11 - 5)[:, None]).astype(np.float32)  # row i = column i
    got = jasper.rabitq_quantize(torch.from_numpy(x).cuda(), rotation=torch.from_numpy(p).cuda())
    r = x.astype(np.float64) @ p.astype(np.float64).T
    clear = np.abs(r) > 1e-5 * np.sqrt((p.astype(np.float64) ** 2).sum(1))[None, :]
    bits = got.bits().cpu().numpy()
    assert np.array_equal(bits[clear], (r >= 0)[clear].astype(np.uint8))


# The code bits of fp16 rows are those of the fp32 product, also where nearly
# every output is a small rest of large sums (so that the two products' rounding
# decides its sign unless it is taken again): pairs that cancel, and a first half
# that the second half cancels; at any scale of the matrix's columns.
@pytest.mark.parametrize("dim", [24, 128, 160, 176, 256])
@pytest.mark.parametrize("scale", [1e-36, 1e-25, 1.0, 1e25])
@pytest.mark.parametrize("halves", [False, True])
def test_rabitq_cancelling_sums_take_the_fp32_bits(jasper, dim, scale, halves):
    rng = np.random.default_rng(dim)
    n, h = 4000, dim // 2
    pos = np.abs(rng.normal(size=(n, h))) + 0.1 if halves else rng.normal(size=(n, h))
    col = np.abs(rng.normal(size=(dim, h))) + 0.1 if halves else rng.normal(size=(dim, h))  # row i = column i
    near = col * (1 + rng.normal(size=(dim, h)) * 2.0**-19)
    x, p = np.empty((n, dim)), np.empty((dim, dim))
    at = (slice(0, h), slice(h, dim)) if halves else (slice(0, dim, 2), slice(1, dim, 2))
    x[:, at[0]], x[:, at[1]] = pos, -pos
    p[:, at[0]], p[:, at[1]] = col, near
    rows = torch.from_numpy(x.astype(np.float16)).cuda()
    matrix = torch.from_numpy((p * scale).astype(np.float32)).cuda()
    got = jasper.rabitq_quantize(rows, rotation=matrix)
    ref = jasper.rabitq_quantize(rows.float(), rotation=matrix)
    assert 0.2 < got.bits().float().mean() < 0.8
    assert torch.equal(got.codes, ref.codes), f"{(got.bits() != ref.bits()).sum()} of {n * dim} bits"


@pytest.mark.parametrize("dim", [200, 256])
def test_short_calls_on_fp16_rows_take_no_longer_than_on_fp32_rows(jasper, dim):
    """10,000 rows are one turn of the chip, in which a tile that takes the fp32
    product again must not wait out a cold read per K step: that cost fp16 rows
    1.2 to 1.3 times the time of the same rows in fp32, where they take 0.8."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(dim)
    x = torch.randn((10_000, dim), generator=gen, device="cuda").half()
    wide = x.float()
    p = torch.linalg.qr(torch.randn((dim, dim), generator=gen, device="cuda"))[0].contiguous()
    c = wide.mean(dim=0)

    def once(rows):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        for _ in range(40):
            jasper.rabitq_quantize(rows, rotation=p, centroid=c)
        b.record()
        torch.cuda.synchronize()
        return a.elapsed_time(b)

    times = [(once(x), once(wide)) for _ in range(6)]
    ratio = min(t[0] for t in times) / min(t[1] for t in times)
    print(f"fp16 rows against fp32 rows: {ratio:.2f}")
    assert ratio <= 1.1


def test_fp32_rows_of_200_values_take_their_share(jasper):
    """300,000 fp32 rows of 200 values take 1.38 times the multiplications of 176
    (both padded to whole tiles); with two waves per SIMD instead of three they
    took 1.46 times as long, with three 1.31."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(5)

    def setup(dim):
        x = torch.randn((300_000, dim), generator=gen, device="cuda")
        return x, torch.linalg.qr(torch.randn((dim, dim), generator=gen, device="cuda"))[0].contiguous(), x.mean(dim=0)

    def once(x, p, c):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        for _ in range(10):
            jasper.rabitq_quantize(x, rotation=p, centroid=c)
        b.record()
        torch.cuda.synchronize()
        return a.elapsed_time(b)

    small, large = setup(176), setup(200)
    times = [(once(*small), once(*large)) for _ in range(6)]
    ratio = min(t[1] for t in times) / min(t[0] for t in times)
    print(f"200 values against 176: {ratio:.2f}")
    assert ratio <= 1.39
