"""The fp32 matrix kernels of the GEMM and attention operators at the edges of their tiles, against float64 arithmetic."""
import pytest
import torch

from gpu_util import M
from sd3_c_amd import lib as L
from sd3_c_amd.params import block_param_shapes

pytestmark = pytest.mark.gpu
U = 2.0 ** -24  # unit roundoff of fp32


@pytest.fixture(autouse=True)
def _automatic_tile_afterwards():
    yield
    L.call("sd3_tune", b"gemm_f32_tile", -1)


@pytest.mark.parametrize("m,k,n", [(1, 4, 4), (33, 36, 68), (128, 32, 128), (129, 64, 132), (154, 1536, 1540), (257, 100, 64), (65, 2052, 36)])
def test_gemm_f32_every_tile_shape(m, k, n):
    """Rows, columns and depths on and beside the multiples of the tiles (32, 64, 128 and 32 k values). The bound is that of a sum of k
    products in any order, (k + 2) u (|x| |W| + |b|) element by element; the tile shapes agree bit for bit (same order of k)."""
    g = torch.Generator(device="cuda").manual_seed(m * 31 + k)
    x, W, b = (torch.randn(s, device="cuda", generator=g) for s in ((m, k), (k, n), (n,)))
    want = x.double() @ W.double() + b.double()
    bound = (k + 2) * U * (x.double().abs() @ W.double().abs() + b.double().abs())
    first = None
    for tile in (-1, 0, 1, 2, 3, 4):
        L.call("sd3_tune", b"gemm_f32_tile", tile)
        y = M.linear(x, W, b)
        assert ((y.double() - want).abs() <= bound).all(), tile
        first = y if first is None else first
        assert torch.equal(y, first), tile


def test_gemm_f32_column_window_and_unaligned_rows():
    """Columns n0.. of a wider weight (whole 16-byte chunks), and strides that are not made of such chunks (the element-wise kernel)."""
    g = torch.Generator(device="cuda").manual_seed(5)
    for m, k, nmax, n0, n in ((40, 96, 200, 100, 68), (40, 95, 201, 3, 77)):
        x, W, b = (torch.randn(s, device="cuda", generator=g) for s in ((m, k), (k, nmax), (nmax,)))
        y = M.partial_linear(x, W, b, n0, n)
        xd, Wd, bd = x.double(), W[:, n0:n0 + n].double(), b[n0:n0 + n].double()
        assert ((y.double() - (xd @ Wd + bd)).abs() <= (k + 2) * U * (xd.abs() @ Wd.abs() + bd.abs())).all()


@pytest.mark.parametrize("m,k,n", [(33, 36, 68), (154, 96, 132)])
def test_gemm_f32_output_at_any_float(m, k, n):
    """The output may begin at any float: the same kernel, hence the same bits, for every tile shape, and nothing beside it is written."""
    g = torch.Generator(device="cuda").manual_seed(m)
    x, W, b = (torch.randn(s, device="cuda", generator=g) for s in ((m, k), (k, n), (n,)))
    want = M.linear(x, W, b)
    for tile in (-1, 0, 1, 2, 3, 4):
        L.call("sd3_tune", b"gemm_f32_tile", tile)
        for off in (1, 2, 3):
            buf = torch.full((m * n + 8,), 7.0, device="cuda")
            L.call("sd3_linear", x.data_ptr(), W.data_ptr(), b.data_ptr(), buf.data_ptr() + 4 * off, m, k, n, None)
            torch.cuda.synchronize()
            assert torch.equal(buf[off:off + m * n].view(m, n), want) and bool((buf[:off] == 7).all()) and bool((buf[off + m * n:] == 7).all()), (tile, off)


@pytest.mark.parametrize("B,Tc,Tx,C,discard", [(2, 5, 33, 192, False), (3, 77, 70, 128, False), (1, 0, 65, 64, True)])
def test_block_f32_every_tile_shape_and_streams_at_any_float(B, Tc, Tx, C, discard):
    """The gated epilogue (a gate row per batch element, residual in place) in a block with dual attention: every tile shape gives equal bits,
    also on streams that begin one float after a 16-byte boundary. Those go through another LayerNorm, whose sums have another order: a
    few u sqrt(K) of relative difference (K <= 384 terms, 1e-6) in each of the six layers behind one another."""
    g = torch.Generator(device="cuda").manual_seed(Tx)
    P = {k: 0.1 * torch.randn(s, device="cuda", generator=g) for k, s in block_param_shapes(C, 2, True, True, discard, 64).items()}
    y, c, x = (torch.randn(s, device="cuda", generator=g) for s in ((B, C), (B, Tc, C), (B, Tx, C)))

    def at(t, off):
        buf = torch.empty(t.numel() + 4, device="cuda")
        return buf[off:off + t.numel()].view(t.shape).copy_(t)

    results = []
    for off in (0, 1):
        first = None
        for tile in (-1, 0, 1, 2, 3, 4):
            L.call("sd3_tune", b"gemm_f32_tile", tile)
            got = M.Dit_block(y, at(c, off), at(x, off), P, B, Tc, Tx, C, C // 64, 2, True, True, discard)
            torch.cuda.synchronize()
            assert torch.isfinite(got[1]).all()
            first = got if first is None else first
            assert torch.equal(got[0], first[0]) and torch.equal(got[1], first[1]), (tile, off)
        results.append(first)
    for a, b in zip(*results):
        assert float((a - b).norm()) <= 1e-5 * float(b.norm())


def test_forward_f32_every_tile_shape():
    """The row-table epilogue (patch embedding, 63 positions per batch element) in a forward: every tile shape gives equal bits."""
    from sd3_c_amd.config import reference_dit_test
    from sd3_c_amd.params import dit_param_shapes

    cfg = reference_dit_test()
    g = torch.Generator(device="cuda").manual_seed(3)
    P = {k: 0.05 * torch.randn(s, device="cuda", generator=g) for k, s in dit_param_shapes(cfg).items()}
    inputs = [torch.randn(s, device="cuda", generator=g) for s in ((2, cfg.pooled_dim), (2, 5, cfg.captions_dim), (2, cfg.in_channels, 14, 18))]
    first = None
    for tile in (-1, 0, 1, 2, 3, 4):
        L.call("sd3_tune", b"gemm_f32_tile", tile)
        out = M.DiT(*inputs, torch.tensor([3.0, 700.0], device="cuda"), P, cfg.num_layers, cfg.dual_attention_layers, cfg.pooled_dim, cfg.captions_dim, cfg.in_channels,
                    cfg.emb_dim, cfg.attn_heads, cfg.mlp_expand, cfg.patch_size, cfg.pos_embed_max_size, cfg.base_height, True)
        assert torch.isfinite(out).all()
        first = out if first is None else first
        assert torch.equal(out, first), tile


@pytest.mark.parametrize("B,NH,hs,Tq,Tk", [(1, 1, 64, 1, 1), (2, 3, 64, 15, 17), (1, 2, 64, 33, 65), (1, 24, 64, 300, 129), (1, 2, 128, 17, 16),
                                           (2, 1, 128, 100, 1000), (1, 12, 128, 530, 47), (1, 2, 40, 20, 30)])
def test_attention_f32(B, NH, hs, Tq, Tk):
    """One query, one key, partly empty tiles, wavefronts without keys, both shapes of either head size and a head size of the general
    kernel. Bound: a score carries (hs + 3) u sum|q k| / sqrt(hs), a weighted mean of values twice the largest score error (to first order)
    plus the rounding of sums over Tk keys, the exponential's included."""
    g = torch.Generator(device="cuda").manual_seed(Tq * 7 + Tk)
    q, k, v = (torch.randn((B, t, NH * hs), device="cuda", generator=g) for t in (Tq, Tk, Tk))
    out = M.mha(q, k, v, NH)
    heads = [t.double().view(B, -1, NH, hs).transpose(1, 2).contiguous() for t in (q, k, v)]
    kt = heads[1].transpose(2, 3).contiguous()
    want = torch.softmax(heads[0] @ kt / hs ** 0.5, -1) @ heads[2]
    score_err = (hs + 3) * U * float((heads[0].abs() @ kt.abs()).max()) / hs ** 0.5
    bound = (2 * score_err + (Tk + 8) * U) * float(v.abs().max())
    assert float((out.double() - want.transpose(1, 2).reshape(B, Tq, -1)).abs().max()) <= bound


@pytest.mark.parametrize("NH", [2, 100])
@pytest.mark.parametrize("hs", [64, 128])
@pytest.mark.parametrize("Tk", [16, 63, 64, 65, 127, 128, 129, 193, 257])
def test_attention_f32_by_the_key_tiles_of_a_wavefront(NH, hs, Tk):
    """A wavefront's last key tile is its only one, its second or its third, for some wavefronts of a workgroup and not for others, and whole or not:
    16 and 32 queries per workgroup (few and many heads)."""
    test_attention_f32(1, NH, hs, 40, Tk)


@pytest.mark.parametrize("NH,hs", [(65536, 64), (98304, 64), (32768, 128)])
def test_attention_f32_of_long_rows(NH, hs):
    """Rows of 2^22 floats and more: the heads have the bits that they have in calls of a quarter as many, partly empty tile and query block included."""
    g = torch.Generator(device="cuda").manual_seed(NH)
    q, k, v = (torch.randn((1, t, NH * hs), device="cuda", generator=g) for t in (3, 21, 21))
    out = M.mha(q, k, v, NH)
    for part, want in zip(zip(*(t.chunk(4, 2) for t in (q, k, v))), out.chunk(4, 2)):
        assert torch.equal(M.mha(*(t.contiguous() for t in part), NH // 4), want)


@pytest.mark.parametrize("m,k,n", [(1, 32, 4), (31, 96, 36), (130, 160, 132), (65, 192, 68)])
def test_gemm_f32_depths_of_whole_k_tiles(m, k, n):
    """Depths of one to six whole K tiles of 32 (fewer than, as many as and more than the rings hold), whose operands are addressed by one scalar and a
    32-bit offset: for every tile shape the bound of a sum of k products in any order, and the bits of the same product 4 deeper with zeros behind it
    (the path of all other depths)."""
    g = torch.Generator(device="cuda").manual_seed(m + k)
    x, W, b = (torch.randn(s, device="cuda", generator=g) for s in ((m, k), (k, n), (n,)))
    want = x.double() @ W.double() + b.double()
    bound = (k + 2) * U * (x.double().abs() @ W.double().abs() + b.double().abs())
    deeper = M.linear(torch.cat([x, torch.zeros(m, 4, device="cuda")], 1).contiguous(), torch.cat([W, torch.zeros(4, n, device="cuda")]).contiguous(), b)
    for tile in (-1, 0, 1, 2, 3, 4):
        L.call("sd3_tune", b"gemm_f32_tile", tile)
        y = M.linear(x, W, b)
        assert ((y.double() - want).abs() <= bound).all() and torch.equal(y, deeper), tile
