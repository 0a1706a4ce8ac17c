"""Product over stored block values at the edges of its tiles and segments, and the block transpose that feeds dX."""
import numpy as np
import pytest
import torch

from mortar_amd import ops, synth
from mortar_amd.pack import BcsrTopology

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Rb,Cb,M", [(1, 1, 1), (33, 5, 63), (97, 79, 65), (160, 3, 15), (257, 48, 1030), (70, 155, 31),   # all of K in one tile
                                     (49, 156, 65), (5, 390, 130), (12, 191, 4097), (200, 228, 16)])                     # K segments, whole and ragged
@pytest.mark.parametrize("density", [0.0, 0.04, 0.5])
def test_values_product_edges(dev, Rb, Cb, M, density):
    rng = np.random.default_rng(Rb * 1000 + Cb)
    mask = rng.random((Rb, Cb)) < density
    mask[::3] = False                                     # whole rows without blocks
    if density == 0.5:
        mask[Rb // 2] = True                              # and one full row
    offsets = np.concatenate([[0], np.cumsum(mask.sum(1))]).astype(np.int32)
    col = np.nonzero(mask)[1].astype(np.int16)
    T = BcsrTopology(offsets, col, Rb * 16, Cb * 16, dev)
    g = torch.Generator(device=dev).manual_seed(M)
    data = (torch.randn(T.nnz, 16, 16, device=dev, generator=g) * 0.5).bfloat16()
    x = torch.randn(M, Cb * 16, device=dev, generator=g).bfloat16()
    dense = torch.zeros(Rb, Cb, 16, 16, device=dev, dtype=torch.float64)
    rows = np.repeat(np.arange(Rb), mask.sum(1))
    dense[torch.from_numpy(rows).to(dev), torch.from_numpy(col.astype(np.int64)).to(dev)] = data.double()
    dense = dense.permute(0, 2, 1, 3).reshape(Rb * 16, Cb * 16)
    out = torch.full((M + 1, Rb * 16), 7.0, device=dev, dtype=torch.bfloat16)
    y = ops.dds_values(x, data, T, out=out[:M])
    ref, bound = x.double() @ dense.t(), x.double().abs() @ dense.abs().t()
    assert ((y.double() - ref).abs() <= ref.abs() * 2.0 ** -8 + bound * 2.0 ** -20).all()
    assert (out[M] == 7.0).all()                          # nothing past the last token
    if T.nnz:
        _, src = T.transposed()
        assert torch.equal(ops.transpose_blocks(data, src), data[src.long()].transpose(1, 2))


@pytest.mark.parametrize("Rb,Cb,M", [(131, 5, 16400), (129, 80, 8161), (256, 3, 8137)])      # units of four rows (64-token tiles), of two in the same range of 32-token ones; rows and tokens left over
@pytest.mark.parametrize("density", [0.04, 0.5])
def test_values_product_four_rows_at_a_time(dev, Rb, Cb, M, density):
    test_values_product_edges(dev, Rb, Cb, M, density)


@pytest.mark.parametrize("Rb,Cb,M", [(34, 5, 130), (256, 3, 8200), (30, 80, 97), (128, 80, 8161),      # units of two and of four rows (64-token tiles), of two (32-token ones)
                                     (26, 200, 70), (50, 160, 4100), (12, 200, 16389)])               # K segments, one to four rows per wave
@pytest.mark.parametrize("pad", [4, 32, 64])
def test_values_product_has_the_same_bits_whatever_the_pitch(dev, Rb, Cb, M, pad):
    """Rows of y that start on lines, on half lines and on neither (the stores differ), and a base off the lines."""
    rng = np.random.default_rng(Rb)
    mask = rng.random((Rb, Cb)) < 0.2
    T = BcsrTopology(np.concatenate([[0], np.cumsum(mask.sum(1))]).astype(np.int32), np.nonzero(mask)[1].astype(np.int16), Rb * 16, Cb * 16, dev)
    g = torch.Generator(device=dev).manual_seed(pad)
    data = torch.randn(T.nnz, 16, 16, device=dev, generator=g).bfloat16()
    x = torch.randn(M, Cb * 16, device=dev, generator=g).bfloat16()
    want = ops.dds_values(x, data, T)
    for base in (0, 4):
        ld = Rb * 16 + pad
        buf = torch.full((base + M * ld,), 7.0, device=dev, dtype=torch.bfloat16)
        out = buf[base:].view(M, ld)
        ops.dds_values(x, data, T, out=out[:, :Rb * 16])
        assert torch.equal(out[:, :Rb * 16], want)
        assert (out[:, Rb * 16:] == 7.0).all() and (buf[:base] == 7.0).all()


@pytest.mark.parametrize("Rb,Cb", [(5, 3), (33, 170)])                 # all of K in one tile, K segments
@pytest.mark.parametrize("ld,M", [(2 ** 23 + 8, 70), (2 ** 26, 19), (2 ** 30, 3)])      # 64 rows of y in 31 bits; 16 of them; one
def test_values_product_into_rows_far_apart(dev, Rb, Cb, ld, M):
    rng = np.random.default_rng(7)
    mask = rng.random((Rb, Cb)) < 0.4
    T = BcsrTopology(np.concatenate([[0], np.cumsum(mask.sum(1))]).astype(np.int32), np.nonzero(mask)[1].astype(np.int16), Rb * 16, Cb * 16, dev)
    data = torch.randn(T.nnz, 16, 16, device=dev).bfloat16()
    x = torch.randn(M, Cb * 16, device=dev).bfloat16()
    buf = torch.empty((M - 1) * ld + Rb * 16 + 16, device=dev, dtype=torch.bfloat16)
    out = buf.as_strided((M, Rb * 16 + 16), (ld, 1))
    out.fill_(7.0)
    ops.dds_values(x, data, T, out=out[:, :Rb * 16])
    # other tiles pair the blocks of a row differently: one bf16 step apart, and 2^-20 of at most 2720 * 0.4 products of size 1
    assert torch.allclose(out[:, :Rb * 16].float(), ops.dds_values(x, data, T).float(), rtol=2.0 ** -7, atol=1e-3)
    assert (out[:, Rb * 16:] == 7.0).all()


@pytest.mark.parametrize("lda,ldb", [(2 ** 26 + 8, None), (None, 2 ** 26 + 8)])
def test_weight_gradient_of_rows_far_apart(dev, lda, ldb):
    """Leading dimensions beyond 2^26 values, where 32 tokens no longer fit a 32-bit offset; a whole step and a part of one."""
    W = synth.to_pack(synth.synth_matrix(16 * 9, 16 * 50, 0.3, seed=8), dev)
    M = 37

    def far(t, ld):
        if ld is None:
            return t
        out = torch.empty((M - 1) * ld + t.shape[1], device=dev, dtype=torch.bfloat16).as_strided(t.shape, (ld, 1))
        return out.copy_(t)

    a, b = (torch.randn(M, n, device=dev).bfloat16() for n in (W.out_features, W.in_features))
    assert torch.equal(ops.sdd(far(a, lda), far(b, ldb), W), ops.sdd(a, b, W))


@pytest.mark.parametrize("Rb,Cb,M", [(33, 78, 65), (12, 77, 130), (70, 155, 97), (17, 156, 33), (49, 157, 65)])   # the widest tiles of all K (64 tokens, 32), the first K segments
@pytest.mark.parametrize("density", [0.04, 0.5])
def test_values_product_of_the_widest_whole_tiles(dev, Rb, Cb, M, density):
    test_values_product_edges(dev, Rb, Cb, M, density)
