"""Parity of the hand-written gfx950 kernels against the CPU oracle, through the
C ABI (ctypes -> liborion_kernels.so).  Triad: bit-exact.  GEMM: fp32 output
within 1e-3 of the exact result's RMS (the tolerance the job description names
for floating point); bf16 output equal to the nearest-even rounding of the fp32
output."""

import numpy as np
import pytest
import torch

from oracle import kernels_oracle as ko
from orion_amd import kernels

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
GEMM_RTOL = 1e-3


def _uniform(n, seed):
    return (np.random.default_rng(seed).random(n, dtype=np.float32) * 2 - 1)


@pytest.mark.parametrize("n", [0, 1, 3, 4, 5, 255, 1023, 4096, 65537, (1 << 22) + 3])
def test_triad_bit_exact(n):
    b, c = _uniform(n, 1), _uniform(n, 2)
    s = 1.7
    a = torch.full((n,), 7.0, device=DEV)
    kernels.triad(a, torch.from_numpy(b).to(DEV), torch.from_numpy(c).to(DEV), s)
    torch.cuda.synchronize()
    assert np.array_equal(a.cpu().numpy().view(np.uint32), ko.triad(b, c, s).view(np.uint32))


@pytest.mark.parametrize("grid", [1, 7, 256, 4096])
def test_triad_any_grid_gives_the_same_bits(grid):
    n = 1_000_003
    b, c = _uniform(n, 3), _uniform(n, 4)
    a = torch.empty(n, device=DEV)
    kernels.triad(a, torch.from_numpy(b).to(DEV), torch.from_numpy(c).to(DEV), -0.3,
                  grid_blocks=grid)
    torch.cuda.synchronize()
    assert np.array_equal(a.cpu().numpy(), ko.triad(b, c, -0.3))


# The loop over a caller's grid changes at eight tiles of 2048 16-byte accesses a
# workgroup (two from 1024 workgroups on); last tiles whole, partial and of one
# access; 0 to 3 elements past the last 16 bytes.
@pytest.mark.parametrize("grid", [1, 3, 64, 1024])
@pytest.mark.parametrize("half_tiles, more", [(3, 7), (4, -4), (4, 0), (4, 5), (5, 4093),
                                              (16, -4), (16, 0), (16, 1), (17, 1026)])
def test_triad_loops_at_the_edges_of_tiles(grid, half_tiles, more):
    n = half_tiles * grid * 4096 + more
    rng = np.random.default_rng(n)
    b, c = (rng.standard_normal(n).astype(np.float32) for _ in range(2))
    a = torch.full((n + 64,), 7.0, device=DEV)
    kernels.triad(a[:n], torch.from_numpy(b).to(DEV), torch.from_numpy(c).to(DEV), 0.9,
                  grid_blocks=grid)
    assert np.array_equal(a[:n].cpu().numpy().view(np.uint32),
                          ko.triad(b, c, 0.9).view(np.uint32))
    assert (a[n:] == 7.0).all()


def test_triad_special_values_and_in_place():
    b = np.array([0.0, -0.0, np.inf, 1.0, np.nan, 1e38, -1e38, 1e-45], dtype=np.float32)
    c = np.array([0.0, 0.0, 1.0, np.inf, 1.0, 1e38, 1e38, 1e-45], dtype=np.float32)
    tb, tc = torch.from_numpy(b).to(DEV), torch.from_numpy(c).to(DEV)
    kernels.triad(tb, tb, tc, 2.0)              # a aliases b
    torch.cuda.synchronize()
    want = ko.triad(b, c, 2.0)
    assert np.array_equal(tb.cpu().numpy().view(np.uint32), want.view(np.uint32))


def test_triad_full_size_linearity():
    # 1 GiB arrays (the benchmark's size): triad(b, c, s) with c = 0 is the
    # identity on b, bit for bit, and with b = 0, s = 1 the identity on c.
    n = 1 << 28
    b = torch.rand(n, device=DEV) * 2 - 1
    z = torch.zeros(n, device=DEV)
    a = torch.empty(n, device=DEV)
    kernels.triad(a, b, z, 3.0)
    assert torch.equal(a, b)
    kernels.triad(a, z, b, 1.0)
    assert torch.equal(a, b)
    # and a sampled window against the oracle
    kernels.triad(a, b, b, 0.5)
    torch.cuda.synchronize()
    lo = n - 100_003
    hb = b[lo:].cpu().numpy()
    assert np.array_equal(a[lo:].cpu().numpy(), ko.triad(hb, hb, 0.5))


def test_triad_rejects_misaligned_and_mismatched():
    b = torch.zeros(64, device=DEV)
    with pytest.raises(kernels.KernelError) as e:
        kernels.triad(b[1:], b[1:], b[1:], 1.0)
    assert e.value.code == 3
    with pytest.raises(ValueError):
        kernels.triad(b, b[:8], b, 1.0)
    with pytest.raises(ValueError):
        kernels.triad(b.cpu(), b.cpu(), b.cpu(), 1.0)


def _gemm_case(m, n, k, seed):
    rng = np.random.default_rng(seed)
    a = ko.f32_to_bf16_bits(rng.random((m, k), dtype=np.float32) * 2 - 1)
    b = ko.f32_to_bf16_bits(rng.random((n, k), dtype=np.float32) * 2 - 1)
    ta = torch.from_numpy(a.view(np.int16)).view(torch.bfloat16).to(DEV)
    tb = torch.from_numpy(b.view(np.int16)).view(torch.bfloat16).to(DEV)
    return a, b, ta, tb


@pytest.mark.parametrize("shape", [(256, 256, 64), (256, 256, 128), (256, 256, 192), (256, 512, 256), (512, 256, 1024),
                                   (768, 1024, 512), (1024, 1024, 2048)])
def test_gemm_against_exact_product(shape):
    m, n, k = shape
    a, b, ta, tb = _gemm_case(m, n, k, sum(shape))
    ref = ko.gemm_bf16_nt(a, b)
    out = kernels.gemm_bf16_nt(ta, tb, out_dtype=torch.float32)
    torch.cuda.synchronize()
    got = out.cpu().numpy().astype(np.float64)
    rms = np.sqrt(np.mean(ref ** 2))
    assert np.max(np.abs(got - ref)) <= GEMM_RTOL * rms
    out16 = kernels.gemm_bf16_nt(ta, tb)
    torch.cuda.synchronize()
    bits = out16.view(torch.int16).cpu().numpy().view(np.uint16)
    assert np.array_equal(bits, ko.f32_to_bf16_bits(out.cpu().numpy()))


def test_gemm_exact_on_small_integers():
    # integer inputs: every partial sum is exact in fp32, so the result is exact
    rng = np.random.default_rng(5)
    a = rng.integers(-4, 5, (256, 256)).astype(np.float32)
    b = rng.integers(-4, 5, (512, 256)).astype(np.float32)
    ta = torch.from_numpy(a).to(torch.bfloat16).to(DEV)
    tb = torch.from_numpy(b).to(torch.bfloat16).to(DEV)
    out = kernels.gemm_bf16_nt(ta, tb, out_dtype=torch.float32)
    torch.cuda.synchronize()
    assert np.array_equal(out.cpu().numpy(), a @ b.T)


def test_gemm_full_size_sampled_rows_and_identity():
    m = n = k = 8192
    g = torch.Generator(device=DEV).manual_seed(11)
    ta = (torch.rand(m, k, device=DEV, generator=g) * 2 - 1).to(torch.bfloat16)
    tb = (torch.rand(n, k, device=DEV, generator=g) * 2 - 1).to(torch.bfloat16)
    out = kernels.gemm_bf16_nt(ta, tb, out_dtype=torch.float32)
    torch.cuda.synchronize()
    rows = [0, 1, 255, 256, 4097, 8191]
    a_bits = ta[rows].view(torch.int16).cpu().numpy().view(np.uint16)
    b_bits = tb.view(torch.int16).cpu().numpy().view(np.uint16)
    ref = ko.gemm_bf16_nt(a_bits, b_bits)
    got = out[rows].cpu().numpy().astype(np.float64)
    assert np.max(np.abs(got - ref)) <= GEMM_RTOL * np.sqrt(np.mean(ref ** 2))
    # size-independent property: B = identity returns A (in fp32) exactly
    eye = torch.eye(k, device=DEV, dtype=torch.bfloat16)
    out = kernels.gemm_bf16_nt(ta, eye, out_dtype=torch.float32)
    assert torch.equal(out, ta.float())


def test_gemm_rejects_bad_shapes_without_launching():
    for k in (80, 96):                                # K not a multiple of 64
        a = torch.zeros(256, k, device=DEV, dtype=torch.bfloat16)
        b = torch.zeros(256, k, device=DEV, dtype=torch.bfloat16)
        with pytest.raises(kernels.KernelError) as e:
            kernels.gemm_bf16_nt(a, b)
        assert e.value.code == 2
    a = torch.zeros(100, 64, device=DEV, dtype=torch.bfloat16)
    with pytest.raises(kernels.KernelError) as e:
        kernels.gemm_bf16_nt(a, torch.zeros(256, 64, device=DEV, dtype=torch.bfloat16))
    assert e.value.code == 2
    with pytest.raises(ValueError):
        kernels.gemm_bf16_nt(torch.zeros(256, 64, device=DEV), b)


@pytest.mark.parametrize("shape", [
    # one shape for each tile of the kernel at odd, smallest and pipeline-edge depths
    (256, 256, 320), (256, 256, 384), (512, 512, 704), (1024, 1024, 192), (1024, 1024, 448),
    (1024, 2048, 64), (1024, 2048, 576), (2048, 2048, 128), (2048, 2048, 320),
    (2304, 2304, 1088), (2816, 3328, 192), (4096, 4096, 256)])
def test_gemm_every_tile_exact_on_small_integers(shape):
    # integers and depths at which every partial sum is exact in fp32: any order of
    # the sums gives the same bits, and a fragment out of place does not
    m, n, k = shape
    g = torch.Generator(device=DEV).manual_seed(sum(shape))
    ta, tb = (torch.randint(-4, 5, (rows, k), device=DEV, generator=g).to(torch.bfloat16)
              for rows in (m, n))
    want = (ta.float() @ tb.float().t())
    for dtype in (torch.float32, torch.bfloat16):
        out = torch.full((m, n), float("nan"), device=DEV, dtype=dtype)
        for _ in range(3):
            kernels.gemm_bf16_nt(ta, tb, out=out)
            assert torch.equal(out, want.to(dtype))


@pytest.mark.parametrize("cus", [0, 32, 64])
def test_gemm_on_a_limited_stream_and_captured(cus):
    # the tile depends on the compute units that the stream may use, which are asked for
    # while the stream is being captured too
    m, n, k = 1024, 1024, 192
    g = torch.Generator(device=DEV).manual_seed(cus)
    ta, tb = (torch.randint(-4, 5, (rows, k), device=DEV, generator=g).to(torch.bfloat16)
              for rows in (m, n))
    out = torch.empty((m, n), device=DEV)
    stream = kernels.cu_masked_stream(cus)
    torch.cuda.synchronize()
    kernels.gemm_bf16_nt(ta, tb, out=out, stream=stream)
    stream.synchronize()
    assert torch.equal(out, ta.float() @ tb.float().t())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        kernels.gemm_bf16_nt(ta, tb, out=out)
    for _ in range(3):
        ta.copy_(torch.randint(-4, 5, (m, k), device=DEV, generator=g))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ta.float() @ tb.float().t())


# the 32 x 64 tile's two groups of waves: 1 to 8 and 64 k-tiles each, about its four stages
@pytest.mark.parametrize("k", [128, 256, 384, 512, 640, 768, 896, 1024, 8192])
def test_gemm_two_wave_groups_exact_on_small_integers(k):
    # as above: every partial sum is exact in fp32
    g = torch.Generator(device=DEV).manual_seed(k)
    ta, tb = (torch.randint(-4, 5, (rows, k), device=DEV, generator=g).to(torch.bfloat16)
              for rows in (256, 512))
    want = (ta.float() @ tb.float().t())
    for dtype in (torch.float32, torch.bfloat16):
        assert torch.equal(kernels.gemm_bf16_nt(ta, tb, out_dtype=dtype), want.to(dtype))


# one group has a k-tile less: 4 to 8 and 63 of them; test_kernel_launches.py holds them to the tile
UNEVEN_DEPTHS = [576, 704, 832, 960, 1088, 8128]


@pytest.mark.parametrize("k", UNEVEN_DEPTHS)
def test_gemm_two_wave_groups_of_uneven_depth_exact_on_small_integers(k):
    """As above; what lies around the operands is infinite and reaches no result."""
    g = torch.Generator(device=DEV).manual_seed(k)
    around = [torch.full((rows + 512, k), float("inf"), device=DEV, dtype=torch.bfloat16)
              for rows in (256, 512)]
    ta, tb = (t[256:-256] for t in around)
    for t in (ta, tb):
        t.copy_(torch.randint(-4, 5, t.shape, device=DEV, generator=g))
    want = ta.float() @ tb.float().t()
    for dtype in (torch.float32, torch.bfloat16):
        assert torch.equal(kernels.gemm_bf16_nt(ta, tb, out_dtype=dtype), want.to(dtype))


# Depths around the stages of the tiles by k-steps, and partial last tiles of those that do
# not divide 256; test_kernel_launches.py holds each shape to its tile.
EDGE_TILES = [
    ("256x128", (1280, 3328, 64)), ("256x128", (1280, 3328, 128)), ("256x128", (1280, 3328, 192)),
    ("256x128", (1280, 3328, 256)), ("256x128", (1024, 5632, 576)),
    ("192x128", (1280, 3328, 320)), ("192x128", (1280, 3328, 448)), ("192x128", (1280, 3328, 576)),
    ("128x128", (768, 2816, 64)), ("128x128", (768, 2816, 128)), ("128x128", (768, 2816, 192)),
    ("128x128", (768, 2816, 256)), ("128x128", (512, 5632, 320)),
    ("96x128", (3072, 1024, 2560)), ("96x128", (3072, 1024, 2624)),
    # 32 and 64 of the last tile's 96 rows
    ("96x128", (512, 4352, 2112)), ("96x128", (1280, 1792, 2176)), ("96x128", (1024, 2304, 2176)),
    ("96x128", (2560, 1024, 2240)),
    # from 18 k-tiles on
    ("96x128", (512, 4352, 1152)), ("96x128", (1280, 1792, 1216)), ("96x128", (3072, 1024, 1152)),
    ("128x128", (512, 4352, 1088)), ("128x128", (3072, 1024, 1024))]


@pytest.mark.parametrize("tile,shape", EDGE_TILES)
def test_gemm_tiles_past_the_edges_exact_on_small_integers(tile, shape):
    """Tiles that do not divide 256 and tiles by k-steps, at depths around their stages; as
    above, every partial sum is exact in fp32.  A row past the last one would land in the
    guard behind the result."""
    m, n, k = shape
    g = torch.Generator(device=DEV).manual_seed(sum(shape))
    ta, tb = (torch.randint(-4, 5, (rows, k), device=DEV, generator=g).to(torch.bfloat16)
              for rows in (m, n))
    want = ta.float() @ tb.float().t()
    for dtype in (torch.float32, torch.bfloat16):
        guarded = torch.full((m + 256, n), 7.0, device=DEV, dtype=dtype)
        out = guarded[:m]
        torch.cuda.synchronize()
        kernels.gemm_bf16_nt(ta, tb, out=out)
        torch.cuda.synchronize()
        assert torch.equal(out, want.to(dtype))
        assert bool((guarded[m:] == 7.0).all())


@pytest.mark.filterwarnings("ignore:Named tensors")
def test_gemm_takes_tensors_with_named_dimensions():
    g = torch.Generator(device=DEV).manual_seed(2)
    ta, tb = (torch.randint(-4, 5, (256, 128), device=DEV, generator=g).to(torch.bfloat16)
              for _ in range(2))
    want = kernels.gemm_bf16_nt(ta, tb)
    assert torch.equal(kernels.gemm_bf16_nt(ta.rename("m", "k"), tb.rename("n", "k")), want)
