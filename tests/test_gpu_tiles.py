"""The products over unranked tiles at the sizes where their split of the work turns: against the oracle's
decoded matrix in f64, and (batch 1) against the other ways to the same rows."""
import numpy as np
import pytest

from llvq_amd import synth
from test_gpu_gemm import _check, _reference, _x16

pytestmark = pytest.mark.gpu


# Columns: a record's blocks go to 4, 8 or 16 wavefronts (past 128 and 256 blocks), to the eight-step
# variant past 512 and are refused past 1024; rows: eight to a record.
@pytest.mark.parametrize("nb,tail,d_out", [(1, 0, 1), (7, 23, 9), (8, 1, 8), (9, 0, 17), (31, 5, 64), (32, 0, 7), (33, 16, 40), (128, 0, 24),
                                           (129, 3, 4099), (256, 7, 16), (257, 0, 31), (512, 23, 8), (513, 1, 33), (1024, 0, 9)])
def test_single_row_products(gpu_rt, orc, nb, tail, d_out):
    import torch

    d_in = nb * 24 + tail
    raw = synth.make_matrix(f"model.layers.0.tiles.{d_out}x{d_in}.weight", d_out, d_in, seed=nb + tail)
    X = synth.make_activation(d_in, seed=nb, rows=1)
    Y_ref, A_ref = _reference(orc, raw, X)
    proj = gpu_rt.upload(raw)
    try:
        x = _x16(X)[0]
        y32 = gpu_rt.forward(proj, x, out_dtype=torch.float32).reshape(1, -1)
        y16 = gpu_rt.forward(proj, x).reshape(1, -1)
        grouped = gpu_rt.forward_group([proj, proj], x, out_dtype=torch.float32)
        again = gpu_rt.forward(proj, x, out_dtype=torch.float32).reshape(1, -1)
    finally:
        gpu_rt.free(proj)
    assert _check(y32.cpu().numpy(), Y_ref, A_ref) < 1e-5  # integer products: f32 sums are all that rounds
    _check(y16.float().cpu().numpy(), Y_ref, A_ref, out_rounding=2.0 ** -11)
    assert torch.equal(again, y32)
    for y in grouped:
        assert torch.equal(y.reshape(1, -1), y32)  # the same split, whatever shares the launch


# Rows of activations: 16, 64 and 128 close a variant or a tile; columns: products of four blocks, of two, steps of
# the last split that are short, a block beyond them, tails and row strides of any parity; few rows split the columns.
@pytest.mark.parametrize("nb,tail,d_out,M", [(1, 0, 1, 2), (5, 7, 31, 16), (63, 0, 33, 17), (64, 1, 16, 64), (65, 23, 70, 65), (170, 16, 255, 128),
                                             (171, 3, 257, 129), (34, 0, 4100, 256), (16, 5, 200, 257), (512, 0, 64, 1024), (33, 1, 24, 1025)])
def test_batched_products(gpu_rt, orc, nb, tail, d_out, M):
    import torch

    d_in = nb * 24 + tail
    raw = synth.make_matrix(f"model.layers.0.tiles.{d_out}x{d_in}.weight", d_out, d_in, seed=nb + M)
    X = synth.make_activation(d_in, seed=M, rows=M)
    Y_ref, A_ref = _reference(orc, raw, X)
    proj = gpu_rt.upload(raw)
    try:
        Y32 = gpu_rt.forward_batched(proj, _x16(X), out_dtype=torch.float32)
        Y16 = gpu_rt.forward_batched(proj, _x16(X))
        again = gpu_rt.forward_batched(proj, _x16(X), out_dtype=torch.float32)
    finally:
        gpu_rt.free(proj)
    assert _check(Y32.cpu().numpy(), Y_ref, A_ref) < 3e-4  # weights are rounded to binary16
    _check(Y16.float().cpu().numpy(), Y_ref, A_ref, out_rounding=2.0 ** -11)
    assert torch.equal(again, Y32)


# Rotations: octets that span groups (m < 8), groups of an octet up to one run of 512, levels above it in one pass of 2, 4
# or 8 and in two, blocks of every depth; rows whose last run is short.  Bound: a rounding per level and per term of the
# k x k block, at most 2^-24 of the row's norm each.
@pytest.mark.parametrize("n", [5, 6, 12, 8, 16, 24, 31 * 8, 31 * 32, 1024, 3 * 1024, 29 * 512, 17 * 1024, 7 * 2048, 3 * 4096, 16384, 32768])
def test_rotations(gpu_rt, orc, n):
    import torch

    raw = synth.make_matrix(f"model.layers.0.rot{n}.weight", 9, n, seed=n)
    raw.rotation_seed = 77 + n
    X = synth.make_activation(n, seed=n, rows=3)
    want = np.stack([orc.Rotation(n, 77 + n).apply(x.astype(np.float64)) for x in X])
    proj = gpu_rt.upload(raw)
    try:
        xr = np.stack([gpu_rt.rotate(proj, x).cpu().numpy().reshape(-1) for x in _x16(X)])
        levels = (n & -n).bit_length() + n // (n & -n) + 1
        assert np.linalg.norm(xr - want, axis=1).max() <= levels * 2.0 ** -24 * np.linalg.norm(want, axis=1).max()
        if 24 <= n <= 24 * 1024:
            one = gpu_rt.forward(proj, _x16(X)[0], out_dtype=torch.float32).reshape(-1)
            two = gpu_rt.forward_rotated(proj, gpu_rt.rotate(proj, _x16(X)[0]), out_dtype=torch.float32).reshape(-1)
            assert torch.equal(one, two)
    finally:
        gpu_rt.free(proj)
