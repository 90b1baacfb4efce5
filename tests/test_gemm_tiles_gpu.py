"""Every GEMM block-tile variant (the general kernels of gemm.hip and
gemm_dma.hip, and the pipelined kernels: register-staged and direct-to-LDS,
128- and 256-row) against the oracle, forced through MUNET_HIP_GEMM_TILE (read
by the library at every GEMM call), on shapes with ragged M / N tails,
N % 4 != 0 (general epilogue), K from one to seven 64-wide slabs and ragged K
(short first slab; the direct-to-LDS tiles fall back to the register-staged
kernel there)."""
import pytest

from munet_amd import synth
from munet_amd.backend import empty
from util import assert_close, rand

pytestmark = pytest.mark.gpu

SHAPES = [(300, 192, 200), (257, 128, 129), (64, 64, 64), (520, 256, 264), (96, 200, 72),
          (130, 320, 96), (70, 448, 136), (33, 40, 48), (530, 136, 392)]
TILES = [0, 1, 2, 3, 4, 5, 6, 100, 101, 102, 103, 104, 105, 106, 107, 200, 201, 202, 203, 207, 208, 209,
         210, 211, 212, 216, 217, 219]


@pytest.mark.parametrize("tile", TILES)
def test_forced_tile(tile, hip, orc, monkeypatch):
    from munet_amd.backend import empty, to_device, to_host
    monkeypatch.setenv("MUNET_HIP_GEMM_TILE", str(tile))
    for dt in (synth.BF16, synth.F16):
        for (M, K, N) in SHAPES:
            x, w, b = rand((M, K), dt, 1), rand((K, N), dt, 2, 0.2), rand((N,), dt, 3)
            r = rand((M, N), dt, 4)
            ref = orc.add(r, orc.gelu(orc.linear(x, w, b, dt), dt), dt)
            wt = empty((N, K), dt)
            hip.pack_linear_weight(to_device(w, dt), wt, K, N)
            out = empty((M, N), dt)
            hip.linear(to_device(x, dt), wt, to_device(b, dt), out, M, K, N, 2, to_device(r, dt))
            assert_close(to_host(out, dt), ref, dt, what=f"tile={tile} dt={dt} {M}x{K}x{N}")


@pytest.mark.parametrize("tile", [207, 208, 209, 210, 211, 212, 216, 217, 219])
def test_tiles_bit_identical_to_128(tile, hip, monkeypatch):
    """The 256-row and direct-to-LDS tiles accumulate every output in the
    same K order as the register-staged 128x128 tile (64-wide slabs, two
    32-wide MFMA halves), so their outputs are bit-identical, for every fused
    epilogue kind and the head split (K = 320: five slabs, so every stage
    count takes its unrolled loop and its tail)."""
    import torch
    from munet_amd.backend import empty
    g = torch.Generator(device="cuda").manual_seed(7)
    M, K, N = 520, 320, 392
    bf = torch.bfloat16
    x = torch.randn(M, K, device="cuda", generator=g).to(bf)
    wt = (torch.randn(N, K, device="cuda", generator=g) * 0.1).to(bf)
    bias = (torch.randn(N, device="cuda", generator=g) * 0.1).to(bf)
    r = torch.randn(M, N, device="cuda", generator=g).to(bf)
    for act, resid, use_bias in [(0, None, False), (0, None, True), (2, None, True), (1, None, True),
                                 (0, r, True), (0, r, False)]:
        outs = []
        for t in (200, tile):
            monkeypatch.setenv("MUNET_HIP_GEMM_TILE", str(t))
            out = empty((M, N), 2)
            hip.linear(x, wt, bias if use_bias else None, out, M, K, N, act, resid)
            torch.cuda.synchronize()
            outs.append(out.view(torch.int16).clone())
        assert torch.equal(outs[0], outs[1]), f"tile {tile} act={act} resid={resid is not None} bias={use_bias}"
    # head split: [B*T, 3E] -> q, k, v [B, H, T, hd]
    Bq, Tq, E, Hq = 2, 136, 192, 3
    xq = torch.randn(Bq * Tq, E, device="cuda", generator=g).to(bf)
    wq = (torch.randn(3 * E, E, device="cuda", generator=g) * 0.1).to(bf)
    bqk = (torch.randn(3 * E, device="cuda", generator=g) * 0.1).to(bf)
    res = []
    for t in (200, tile):
        monkeypatch.setenv("MUNET_HIP_GEMM_TILE", str(t))
        q, k, v = (empty((Bq * Tq * E,), 2) for _ in range(3))
        hip.qkv_projection(xq, wq, bqk, q, k, v, Bq, Tq, E, Hq)
        torch.cuda.synchronize()
        res.append(torch.cat([q, k, v]).view(torch.int16).clone())
    assert torch.equal(res[0], res[1]), f"tile {tile} head split"


@pytest.mark.parametrize("tile", [None, 200, 203, 208, 209, 216, 217])
def test_xcd_tile_enumeration_bit_identical(tile, hip, monkeypatch):
    """The per-XCD tile enumeration (row groups, or column groups of any width,
    a ragged last group included) only reorders the tiles: every output is
    computed by the same tile code, so the outputs are bit-identical.  Shapes
    have tile counts divisible by 8 and not (the last XCDs walk one tile less);
    None is the automatic tile."""
    import torch
    from munet_amd.backend import empty
    if tile is not None:
        monkeypatch.setenv("MUNET_HIP_GEMM_TILE", str(tile))
    g = torch.Generator(device="cuda").manual_seed(9)
    bf = torch.bfloat16
    for (M, K, N) in [(1024, 192, 768), (512, 128, 1536), (256, 320, 3072), (2048, 64, 384), (900, 64, 1032)]:
        x = torch.randn(M, K, device="cuda", generator=g).to(bf)
        wt = (torch.randn(N, K, device="cuda", generator=g) * 0.1).to(bf)
        bias = (torch.randn(N, device="cuda", generator=g) * 0.1).to(bf)
        r = torch.randn(M, N, device="cuda", generator=g).to(bf)
        for act, resid in [(2, None), (0, r)]:
            outs = []
            for gn in ("0", "1", "3", "8", "16", "64"):
                monkeypatch.setenv("MUNET_HIP_XCD_GN", gn)
                out = empty((M, N), 2)
                hip.linear(x, wt, bias, out, M, K, N, act, resid)
                torch.cuda.synchronize()
                outs.append(out.view(torch.int16).clone())
            for gn, o in zip(("1", "3", "8", "16", "64"), outs[1:]):
                assert torch.equal(outs[0], o), f"tile {tile} gn {gn} {M}x{K}x{N} act={act}"


@pytest.mark.parametrize("tile", [200, 201, 202, 203, 208, 209, 216, 217])
def test_f16_fixed_programs_bit_identical_to_general(tile, hip, monkeypatch):
    """fp16 runs the fixed epilogue programs (plain, bias, bias+GELU,
    bias+ReLU, bias+residual) when the destination is 8-byte aligned; an
    output one element off that alignment takes the general program on the
    same tile.  Both round every step with MuNet's half-away fp16 codec, so the
    outputs are bit-identical."""
    import torch
    from munet_amd.backend import empty
    monkeypatch.setenv("MUNET_HIP_GEMM_TILE", str(tile))
    g = torch.Generator(device="cuda").manual_seed(11)
    M, K, N = 512, 320, 384
    h = torch.float16
    x = torch.randn(M, K, device="cuda", generator=g).to(h)
    wt = (torch.randn(N, K, device="cuda", generator=g) * 0.1).to(h)
    bias = (torch.randn(N, device="cuda", generator=g) * 0.1).to(h)
    r = torch.randn(M, N, device="cuda", generator=g).to(h)
    for act, resid, use_bias in [(0, None, False), (0, None, True), (2, None, True), (1, None, True), (0, r, True)]:
        outs = []
        for shift in (0, 1):
            buf = empty((M * N + 1,), 1)
            out = buf[shift:shift + M * N]
            hip.linear(x, wt, bias if use_bias else None, out, M, K, N, act, resid)
            torch.cuda.synchronize()
            outs.append(out.view(torch.int16).clone())
        assert torch.equal(outs[0], outs[1]), f"tile {tile} act={act} resid={resid is not None} bias={use_bias}"


@pytest.mark.parametrize("tile", [None, 300, 301, 302, 104])
@pytest.mark.parametrize("M,K,N", [(65, 32, 64), (64, 36, 68), (31, 4, 33), (130, 100, 200), (1, 64, 5), (300, 516, 31)])
@pytest.mark.parametrize("batched", [False, True])
def test_f32_tiles(hip, monkeypatch, tile, M, K, N, batched):
    """The fp32 kernel's tiles, and the general kernel's chunked loader (104),
    at their edges: one slab, an odd and an even
    number of 32-wide slabs, K tails of 4 values, ragged rows and columns, batch
    slices.  Against float64; a sum of K products rounds at most K times, each
    by 2^-24 of a partial sum, and M N outputs of standard normal operands stay
    below 6 sqrt(K): bound 6 sqrt(K) K 2^-24."""
    import torch
    if tile is not None:
        monkeypatch.setenv("MUNET_HIP_GEMM_TILE", str(tile))
    nb = 3 if batched else 1
    g = torch.Generator().manual_seed(M * 7 + K)
    a, b = torch.randn(nb, M, K, generator=g), torch.randn(nb, N, K, generator=g)
    out = empty((nb, M, N), synth.F32)
    hip.batched_matmul(a.cuda(), b.cuda(), out, nb, M, K, N, False, True, M * K, N * K, M * N)
    ref = a.double() @ b.double().transpose(1, 2)
    assert float((out.cpu().double() - ref).abs().max()) <= 6 * K ** 1.5 * 2.0 ** -24


@pytest.mark.parametrize("B,iC,H,W,oC,k,s,p", [(2, 4, 9, 7, 33, 3, 1, 1), (1, 12, 8, 8, 64, 5, 2, 2), (3, 36, 5, 6, 20, 3, 2, 1),
                                               (1, 64, 16, 16, 128, 3, 1, 1), (2, 32, 4, 4, 8, 1, 1, 0), (1, 8, 7, 7, 8, 7, 1, 3),
                                               (40, 8, 3, 2, 70, 3, 2, 1), (2, 16, 40, 37, 100, 3, 1, 1), (2, 4, 6, 1, 9, 1, 3, 2)])
def test_f32_conv_columns(hip, B, iC, H, W, oC, k, s, p, monkeypatch):
    """The fp32 implicit-GEMM convolution's stepped (tap, channel) columns:
    channel counts below, at and above a 32-wide slab that divide it or not,
    1x1 to 7x7 taps, strides, padding, tiles that cross image borders.  Against
    float64, bound as in test_f32_tiles with K = k k iC, on every tile, which
    all sum in one order: the same bits; and on the general kernel's chunked
    loader."""
    import torch
    g = torch.Generator().manual_seed(iC * 10 + k)
    x, w, b = torch.randn(B, iC, H, W, generator=g), torch.randn(oC, iC, k, k, generator=g), torch.randn(oC, generator=g)
    ref = torch.nn.functional.conv2d(x.double(), w.double(), b.double(), stride=s, padding=p).permute(0, 2, 3, 1)
    K = iC * k * k
    args = x.permute(0, 2, 3, 1).contiguous().cuda(), w.permute(0, 2, 3, 1).contiguous().cuda(), b.cuda()
    outs = {}
    for tile in (None, "300", "301", "302", "general"):
        monkeypatch.delenv("MUNET_HIP_CONV_TILE", raising=False)
        monkeypatch.delenv("MUNET_HIP_CONV_KERNEL", raising=False)
        if tile:
            monkeypatch.setenv("MUNET_HIP_CONV_KERNEL" if tile == "general" else "MUNET_HIP_CONV_TILE", tile)
        out = empty(tuple(ref.shape), synth.F32)
        hip.conv2d_nhwc(*args, out, B, iC, H, W, oC, k, k, s, p)
        outs[tile] = out.cpu()
        assert float((outs[tile].double() - ref).abs().max()) <= 6 * K ** 1.5 * 2.0 ** -24 + 1e-6, tile
    assert all(torch.equal(outs["300"], outs[t]) for t in (None, "301", "302"))


def test_f32_conv_large_image(hip):
    """An image of 1 GiB (its offsets are taken from the tile's first input
    row): rows at both ends and in the middle against float64."""
    import torch
    C, H, W, oC = 64, 2048, 2048, 8
    g = torch.Generator(device="cuda").manual_seed(1)
    x = torch.randn(1, H, W, C, device="cuda", generator=g)
    w, b = torch.randn(oC, 3, 3, C, device="cuda", generator=g), torch.randn(oC, device="cuda", generator=g)
    out = empty((1, H, W, oC), synth.F32)
    hip.conv2d_nhwc(x, w, b, out, 1, C, H, W, oC, 3, 3, 1, 1)
    wd, K = w.cpu().double().permute(0, 3, 1, 2), 9 * C
    for r in (0, 1, 1023, 1024, H - 2, H - 1):
        lo, hi = max(r - 1, 0), min(r + 2, H)
        xs = torch.nn.functional.pad(x[:, lo:hi].cpu().double().permute(0, 3, 1, 2), (1, 1, lo - (r - 1), r + 2 - hi))
        ref = torch.nn.functional.conv2d(xs, wd, b.cpu().double())[0, :, 0].T
        assert float((out[0, r].cpu().double() - ref).abs().max()) <= 6 * K ** 1.5 * 2.0 ** -24 + 1e-6, r


@pytest.mark.parametrize("tile", list(range(220, 228)))
def test_deep_tiles(tile, hip, orc, monkeypatch):
    """The small many-stage tiles (up to 16 stages: products of fewer slabs
    than stages re-load the last one) at the edges of test_forced_tile's shapes
    against the oracle, and bit for bit against the 128x128 kernel."""
    test_forced_tile(tile, hip, orc, monkeypatch)
    test_tiles_bit_identical_to_128(tile, hip, monkeypatch)


@pytest.mark.parametrize("M,N,K", [(1, 64, 64), (33, 96, 128), (256, 1024, 64), (257, 1024, 64), (500, 2048, 192), (512, 768, 256),
                                   (2048, 768, 64), (2049, 768, 64), (300, 4096, 64), (1900, 2056, 128), (4096, 1024, 192), (1500, 2048, 768), (600, 4096, 2048),
                                   (1100, 5000, 64), (1536, 4096, 128), (2048, 3072, 192), (2100, 4040, 320),
                                   (2000, 516, 64), (500, 2044, 192), (33, 97, 64), (500, 2049, 192), (4000, 250, 64), (1100, 2501, 256), (1000, 2501, 1024), (2000, 2050, 64), (1100, 8193, 512), (1100, 8195, 2048), (1100, 2048, 64), (8192, 768, 256), (8100, 864, 448)])
def test_deep_tile_choice_bits(M, N, K, hip, monkeypatch):
    """Both sides of each border of the small-tile choice (at most one tile per
    CU) give the 128x128 kernel's bits, bias + GELU, bias + residual and ReLU."""
    from munet_amd.backend import to_device, to_host
    for dt in (synth.BF16, synth.F16):
        x, w, b, r = (to_device(rand(s, dt, i, c), dt) for i, (s, c) in
                      enumerate([((M, K), 1.0), ((N, K), 0.2), ((N,), 1.0), ((M, N), 1.0)]))
        for act, resid in ((2, None), (0, r), (1, None)):
            outs = []
            for t in (None, 200):
                if t is None:
                    monkeypatch.delenv("MUNET_HIP_GEMM_TILE", raising=False)
                else:
                    monkeypatch.setenv("MUNET_HIP_GEMM_TILE", str(t))
                out = empty((M, N), dt)
                hip.linear(x, w, b, out, M, K, N, act, resid)
                hip.synchronize()
                outs.append(to_host(out, dt))
            assert (outs[0] == outs[1]).all()
