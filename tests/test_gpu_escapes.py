"""Blocks that the 80-bit code has no window for (one coordinate 16 below the others' window), which the batch-1 products make
up for from a tile's list: none, a few, as many as the list holds and more, in every row or in one, against the oracle's
decoded matrix; and through the batched products, which read the code itself."""
import numpy as np
import pytest

from llvq_amd import artifact, synth
from test_gpu_gemm import _check, _reference, _x16

pytestmark = pytest.mark.gpu


def _far(orc, cap):
    """Ranks of points whose coordinates span more than 14: no window of eight values holds them."""
    rng = synth.SplitMix64(cap)
    got = []
    while sum(g.size for g in got) < 300:
        idx = rng.take(200_000) % np.uint64((orc.N12 if cap == 12 else orc.N13) + 1)
        pts = orc.decode_many(idx).astype(np.int64)
        got.append(idx[pts.max(axis=1) - pts.min(axis=1) > 14])
    return np.concatenate(got)


# nb, tail: one step, several, a wavefront's second step (past 512 blocks); share: of a row's blocks that are such points
# (0.02 of 16 x 40 fills the list of eight and more; 1.0 is every block).
@pytest.mark.parametrize("nb,tail,d_out,cap,share", [(1, 0, 33, 12, 1.0), (3, 5, 16, 12, 0.1), (40, 8, 40, 12, 0.02), (40, 8, 40, 12, 1.0), (106, 16, 70, 13, 0.05),
                                                     (170, 16, 33, 12, 0.004), (530, 3, 20, 13, 0.01), (530, 0, 20, 12, 0.3)])
def test_points_without_a_window(gpu_rt, orc, nb, tail, d_out, cap, share):
    import torch

    d_in = nb * 24 + tail
    raw = synth.make_matrix(f"model.layers.0.far.{d_out}x{d_in}.weight", d_out, d_in, seed=nb, shell_cap=cap)
    rng = np.random.default_rng(nb + d_out)
    far = _far(orc, cap)
    idx, gains = raw.unpack()
    idx = np.array(idx, np.uint64)
    at = rng.random(idx.size) < share
    at[nb:2 * nb] |= d_out > 16  # a row full of them, in a tile of its neighbours' few
    idx[at] = rng.choice(far, int(at.sum()))
    raw = artifact.RawMatrix(raw.name, d_out, d_in, cap, raw.centroids, raw.row_scales, raw.tail, artifact.pack_codes(idx, gains, artifact.index_bits(cap)))
    X = synth.make_activation(d_in, seed=nb, rows=20)
    Y_ref, A_ref = _reference(orc, raw, X)
    proj = gpu_rt.upload(raw)
    other = gpu_rt.upload(raw)
    try:
        x = _x16(X)
        y32 = gpu_rt.forward(proj, x[0], out_dtype=torch.float32).reshape(1, -1)
        y16 = gpu_rt.forward(proj, x[0]).reshape(1, -1)
        again = gpu_rt.forward(other, x[0], out_dtype=torch.float32).reshape(1, -1)
        seq = gpu_rt.plan_sequence([([proj], x[0], False)], out_dtype=torch.float32)
        seq.run()
        seq.status()
        in_sequence = seq.outputs[0][0].reshape(1, -1).clone()
        seq.close()
        rows = [gpu_rt.forward_batched(proj, x[:m], out_dtype=torch.float32) for m in (2, 20)]
        wide = gpu_rt.forward_batched(proj, x.repeat(5, 1), out_dtype=torch.float32)
    finally:
        gpu_rt.free(proj)
        gpu_rt.free(other)
    assert _check(y32.cpu().numpy(), Y_ref[:1], A_ref[:1]) < 1e-5
    _check(y16.float().cpu().numpy(), Y_ref[:1], A_ref[:1], out_rounding=2.0 ** -11)
    assert torch.equal(y32, again) and torch.equal(y32, in_sequence)  # the list is in order whatever order it was filled in
    bar = 1e-5 if cap == 13 else 3e-4  # (cap 13: row by row; else weights are rounded to binary16)
    for y in rows + [wide]:
        n = y.shape[0]
        assert _check(y.cpu().numpy(), np.resize(Y_ref, (n, d_out)), np.resize(A_ref, (n, d_out))) < bar


# Tiles of 384 weight rows by 128 activation rows (which 10 000 rows at 1000 take: 27 x 8 workgroups): a step and a half, several
# with tail columns; a last tile of 16 rows, 104 activation rows in the last column.  share: a wavefront's list holds 64 of its 96
# rows' escapes and places 16 in a step; 0.05 and 1.0 are more, whose codes are read.
@pytest.mark.parametrize("nb,tail,share,out", [(3, 0, 0.001, "f32"), (17, 8, 0.001, "f16"), (17, 16, 0.05, "f32"), (5, 8, 1.0, "f32")])
def test_tall_tiles(gpu_rt, orc, nb, tail, share, out):
    import torch

    d_out, d_in, M = 10000, nb * 24 + tail, 1000
    raw = synth.make_matrix(f"model.layers.0.tall.{d_out}x{d_in}.weight", d_out, d_in, seed=nb + tail)
    rng = np.random.default_rng(nb + tail)
    idx, gains = raw.unpack()
    idx = np.array(idx, np.uint64)
    at = rng.random(idx.size) < share
    idx[at] = rng.choice(_far(orc, 12), int(at.sum()))
    raw = artifact.RawMatrix(raw.name, d_out, d_in, 12, raw.centroids, raw.row_scales, raw.tail, artifact.pack_codes(idx, gains, artifact.index_bits(12)))
    X = synth.make_activation(d_in, seed=nb, rows=M)
    Y_ref, A_ref = _reference(orc, raw, X)
    proj = gpu_rt.upload(raw)
    try:
        y = gpu_rt.forward_batched(proj, _x16(X), out_dtype=torch.float32 if out == "f32" else torch.float16)
    finally:
        gpu_rt.free(proj)
    # weights are rounded to binary16, 2^-11 of each at the most (the sums in binary32 take 2^-24 of a few hundred terms beside
    # that), and so may the results be
    bound = 1.05 * 2.0 ** -11 * A_ref + (2.0 ** -11 * np.abs(Y_ref) if out == "f16" else 0.0) + 1e-7
    assert np.all(np.abs(y.double().cpu().numpy() - Y_ref) <= bound)
