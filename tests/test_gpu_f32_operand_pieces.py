"""fp32 blocks whose operands are written as bf16 pieces by what produces them: the same bits as from products that split fp32 operands themselves.

`sd3_dit_block_static` has a fixed 64 MiB for its intermediates and goes without the pieces where these, six bytes a value instead of four, do not fit; the
context's workspace grows. Blocks between the two sizes are computed both ways, and the context tells which of its products had operands in pieces."""
import numpy as np
import pytest
import torch

from gpu_util import M, dev, dev_params, host
from sd3_c_amd import lib as L
from sd3_c_amd.config import DiTConfig
from sd3_c_amd.params import block_param_shapes, dit_param_shapes, synthetic_params_numpy

pytestmark = pytest.mark.gpu


def _plain_and_pieces_bytes(B, Tc, Tx, C, E, dual):
    """The block's activations (fp32; pieces of LayerNorm's outputs, and from 1.7e6 values on of attention's and the first MLP layer's too)."""
    rows = B * (Tc + Tx)
    qkv = 12 * C * (rows + (B * Tx if dual else 0))
    wide = rows * C >= 1.7e6
    plain = qkv + 4 * C * (rows + B * Tx) + 4 * C * rows + 4 * E * C * rows
    return plain, qkv + 6 * C * (rows + B * Tx) + (6 if wide else 4) * (C * rows + E * C * rows)


def _products(B, Tc, Tx, C, dual):
    """How many of a block's products have operands in pieces: q|k|v and the first MLP layers; attention's outputs and the second MLP layers too"""
    values = B * (Tc + Tx) * C
    return 0 if values < 1.0e6 else 2 if values < 1.7e6 else 4 + dual


def _at(a, off):
    """`a` on the GPU, `off` floats behind a multiple of 16 bytes"""
    t = torch.empty(a.size + off, device="cuda")[off:].view(a.shape)
    t.copy_(torch.from_numpy(a))
    assert t.data_ptr() % 16 == 4 * off
    return t


def _both_ways(B, Tc, Tx, C, NH, E, dual, discard, spoil=None, off=0):
    plain, pieces = _plain_and_pieces_bytes(B, Tc, Tx, C, E, dual)
    limit = 64 << 20
    assert plain + (1 << 19) < limit < pieces  # (room for the modulation vectors, and the case tells the two apart)
    rng = np.random.Generator(np.random.Philox(Tx))
    P = synthetic_params_numpy(block_param_shapes(C, E, dual, True, discard, C // NH), 11, 0.05, 0.05)
    y, c, x = (rng.standard_normal(s, dtype=np.float32) for s in ((B, C), (B, Tc, C), (B, Tx, C)))
    if spoil:
        spoil(P, c, x)
    ctx = M.Context()
    try:
        ctx.bind(dev_params(P))
        out = []
        for run, products in ((ctx.block, _products(B, Tc, Tx, C, dual)), (ctx.block_static, 0)):
            cg, xg = _at(c, off), _at(x, off)
            before = ctx.operand_pieces_launches()
            run(dev(y), cg, xg, B, Tc, Tx, C, NH, E, dual, True, discard, precision="fp32")
            assert ctx.operand_pieces_launches() - before == products
            out.append((host(cg), host(xg)))
        return out
    finally:
        ctx.close()


@pytest.mark.parametrize("B,Tc,Tx,C,NH,E,dual,discard", [
    (1, 77, 1100, 1536, 24, 2, False, False),   # all three, heads of 64, rows that are no whole blocks of 16
    (3, 50, 351, 1536, 12, 2, False, False),    # heads of 128, several elements
    (1, 20, 930, 1536, 24, 2, True, False),     # LayerNorm's outputs only; two of them
    (1, 33, 1090, 1536, 24, 2, False, True),    # no context behind attention
    (5, 1, 500, 768, 12, 2, False, False),      # 768 deep
    (2, 15, 1701, 512, 8, 2, False, False),     # the least depth of the kernel
])
def test_the_same_bits_with_operands_in_pieces(B, Tc, Tx, C, NH, E, dual, discard):
    (ca, xa), (cb, xb) = _both_ways(B, Tc, Tx, C, NH, E, dual, discard)
    assert np.isfinite(xa).all()
    assert np.array_equal(xa, xb) and np.array_equal(ca, cb)


@pytest.mark.parametrize("tile", range(6))
def test_the_same_bits_for_every_tile_shape(tile):
    L.check(L.load().sd3_tune(b"gemm_f32_tile", tile))
    try:
        (ca, xa), (cb, xb) = _both_ways(1, 37, 3361, 512, 8, 2, False, False)
    finally:
        L.check(L.load().sd3_tune(b"gemm_f32_tile", -1))
    assert np.array_equal(xa, xb) and np.array_equal(ca, cb)


@pytest.mark.parametrize("B,Tc,Tx,C,NH,E,dual", [(1, 77, 1100, 1536, 24, 2, False), (1, 20, 930, 1536, 24, 2, True), (2, 15, 1701, 512, 8, 2, False)])
def test_the_same_bits_with_streams_at_any_float(B, Tc, Tx, C, NH, E, dual):
    """Rows of x and c that are not on 16 bytes go through the LayerNorm that writes its pieces value by value."""
    (ca, xa), (cb, xb) = _both_ways(B, Tc, Tx, C, NH, E, dual, False, off=1)
    assert np.isfinite(xa).all()
    assert np.array_equal(xa, xb) and np.array_equal(ca, cb)


@pytest.mark.parametrize("off", [0, 3])
@pytest.mark.parametrize("what", ["scales", "tokens"])
def test_values_without_pieces(what, off):
    """Infinities, NaNs and values from 2^112 on in LayerNorm's, attention's and the MLP's outputs are formed anew by the fp32 instruction, from the bits that stand in the pieces' place."""
    C = 1536

    def spoil(P, c, x):
        if what == "tokens":
            x[0, 5, 3] = np.inf
            x[0, 700, 8] = np.nan
            return
        for n, q in P.items():
            if "ada" in n and n.endswith(".bias"):
                q[1 * C + 7] = 2.0 ** 115   # the scale of LayerNorm's channel 7 in front of q|k|v: values, too, and what attention makes of them
                q[4 * C + 9] = -2.0 ** 115  # ... in front of the MLP: some of the hidden values
    (ca, xa), (cb, xb) = _both_ways(1, 77, 1100, C, 24, 2, False, False, spoil, off)
    assert np.isfinite(xa).all() == (what == "scales")
    assert np.array_equal(xa, xb, equal_nan=True) and np.array_equal(ca, cb, equal_nan=True)


@pytest.mark.parametrize("warm", ["pieces", "plain"])
def test_captured_forwards_and_eager_ones_of_the_same_sizes(warm):
    """A captured forward with operands in pieces, and one in a workspace that holds the layout without them only (as it is after a call that there was no memory for
    more for), replayed behind eager calls of the same sizes: these leave the workspace where it is, with the bits of an eager forward throughout."""
    cfg = DiTConfig(num_layers=2, dual_attention_layers=(0,), pooled_dim=64, captions_dim=64, in_channels=16, emb_dim=512, attn_heads=8, mlp_expand=2, patch_size=2,
                    pos_embed_max_size=64, base_height=32, use_qk_norm=True)
    g = torch.Generator(device="cuda").manual_seed(41)
    P = {n: (1 if "rmsnorm" in n else 0) + 0.02 * torch.randn(s, device="cuda", generator=g) for n, s in dit_param_shapes(cfg).items()}
    B, Tc, H, W = 2, 9, 80, 84   # 3378 rows of 512
    lat = torch.randn((B, cfg.in_channels, H, W), device="cuda", generator=g)
    captions = torch.randn((B, Tc, cfg.captions_dim), device="cuda", generator=g)
    args = (torch.randn((B, cfg.pooled_dim), device="cuda", generator=g), captions, lat, torch.full((B,), 300.0, device="cuda"))
    want = M.Denoiser(P, cfg, "fp32")(*args)
    torch.cuda.synchronize()
    den, out, eager = M.Denoiser(P, cfg, "fp32"), torch.empty_like(lat), torch.empty_like(lat)
    L.check(L.load().sd3_tune(b"gemm_f32_no_pieces", int(warm == "plain")))
    try:
        den(*args, out=out)
    finally:
        L.check(L.load().sd3_tune(b"gemm_f32_no_pieces", 0))
    graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=side):
        den(*args, out=out)
    launched = den.ctx.operand_pieces_launches()
    assert launched == (4 * 2 + 1) * 2 if warm == "pieces" else launched == 0   # (the warm call and the captured one, a dual block and a plain one)
    eager.zero_()   # (the runtime takes memory of its own at first launches)
    graph.replay()
    torch.cuda.synchronize()
    assert torch.equal(out, want)
    free = torch.cuda.mem_get_info()[0]
    for _ in range(3):
        out.zero_()
        eager.zero_()
        den(*args, out=eager)
        torch.cuda.synchronize()
        assert torch.cuda.mem_get_info()[0] == free and torch.equal(eager, want)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
    assert (den.ctx.operand_pieces_launches() > launched) == (warm == "pieces")


@pytest.mark.parametrize("norm_off", [0, 1])
@pytest.mark.parametrize("B,Tc,Tx,C,NH,E,dual,qk", [
    (2, 30, 400, 1536, 24, 2, False, True),    # 0.66e6 values alone, 1.3e6 together: LayerNorm's outputs in pieces
    (3, 41, 471, 1536, 24, 2, True, True),     # 0.79e6 and 2.4e6: all of them; attention by pieces, 288 workgroups of 128 queries one after the other
    (5, 10, 390, 1024, 16, 4, False, True),    # attention on the fp32 instruction
    (4, 25, 300, 1536, 12, 2, False, True),    # heads of 128
    (4, 25, 300, 1536, 24, 2, False, False),   # no norms
])
def test_an_element_alone_and_in_a_batch(norm_off, B, Tc, Tx, C, NH, E, dual, qk):
    """Whether operands come in pieces depends on the rows of the whole batch, an element's bits do not, also where a norm's weights lie at any float."""
    rng = np.random.Generator(np.random.Philox(Tx))
    P = dev_params(synthetic_params_numpy(block_param_shapes(C, E, dual, qk, False, C // NH), 13, 0.05, 0.05))
    if norm_off and qk:
        for n in [n for n in P if "rmsnorm" in n][:1]:
            moved = torch.empty(P[n].numel() + norm_off, device="cuda")[norm_off:]
            moved.copy_(P[n].flatten())
            P[n] = moved.view(P[n].shape)
            assert P[n].data_ptr() % 16
    y, c, x = (rng.standard_normal(s, dtype=np.float32) for s in ((B, C), (B, Tc, C), (B, Tx, C)))
    assert (Tc + Tx) * C < 1.0e6 < B * (Tc + Tx) * C

    def run(b0, b1):
        cg, xg = M.Dit_block(dev(y[b0:b1]), dev(c[b0:b1].copy()), dev(x[b0:b1].copy()), P, b1 - b0, Tc, Tx, C, NH, E, dual, qk, False, precision="fp32")
        return host(cg), host(xg)

    launched = M.shared_context(torch.device("cuda:0")).operand_pieces_launches
    before = launched()
    cg, xg = run(0, B)
    assert launched() - before == _products(B, Tc, Tx, C, dual)
    for b in range(B):
        before = launched()
        c1, x1 = run(b, b + 1)
        assert launched() == before
        assert np.array_equal(cg[b:b + 1], c1) and np.array_equal(xg[b:b + 1], x1)
