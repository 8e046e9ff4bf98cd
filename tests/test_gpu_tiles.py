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


# Rows past sixteen steps, whose steps go to the wavefronts across the ends of tiles: the fewest and the most of them, one tile to a workgroup
# and one more, as many as are finished together (fourteen and eight of them) and one more.
@pytest.mark.parametrize("nb,tail,tiles", [(513, 1, 257), (513, 0, 256 * 14 + 1), (725, 8, 320), (1024, 0, 256), (1024, 0, 256 * 8 + 3)])
def test_tiles_of_a_large_launch_are_those_of_a_small_one(gpu_rt, nb, tail, tiles):
    import torch

    from llvq_amd import artifact

    d_in, d_out = nb * 24 + tail, tiles * 16
    rng = np.random.default_rng(nb + tiles)
    codes = rng.integers(0, 2 * (artifact.N12 + 1), size=(d_out, nb), dtype=np.uint64).astype(">u8").view(np.uint8).reshape(d_out, nb, 8)[:, :, 2:]
    scales = np.exp(-4.0 + 0.3 * rng.standard_normal(d_out))
    tails = (0.02 * rng.standard_normal((d_out, tail))).astype(np.float32)
    few = np.unique([t for t in (0, 1, 255, 256, 256 * 8 - 1, 256 * 8, 256 * 13 + 5, tiles - 2, tiles - 1) if t < tiles])
    rows = (few[:, None] * 16 + np.arange(16)).ravel()

    def matrix(name, r):
        return artifact.RawMatrix(name, len(r), d_in, 12, (0.8, 1.25), scales[r], tails[r].ravel(), codes[r].reshape(-1))

    x = _x16(synth.make_activation(d_in, seed=nb)[:1])[0]
    projs = [gpu_rt.upload(matrix("model.layers.0.all.weight", np.arange(d_out))), gpu_rt.upload(matrix("model.layers.0.few.weight", rows))]
    try:
        for dtype in (torch.float32, torch.float16):
            whole, some = (gpu_rt.forward(p, x, out_dtype=dtype).reshape(-1) for p in projs)
            assert torch.equal(whole[torch.from_numpy(rows).to(whole.device)], some)
    finally:
        for p in projs:
            gpu_rt.free(p)


# Rows of activations: 16, 64 and 128 close a variant or a tile; columns: products of four blocks, of two, steps of
# the last split that are short, a block beyond them, tails and row strides of any parity; few rows split the columns.
# (Tails of 8 and 16 columns keep the rows on 16-byte boundaries: weights of one term.  Other tails: of two.)
@pytest.mark.parametrize("nb,tail,d_out,M", [(1, 0, 1, 2), (5, 7, 31, 16), (63, 0, 33, 17), (64, 1, 16, 64), (65, 23, 70, 65), (170, 16, 255, 128),
                                             (171, 3, 257, 129), (34, 0, 4100, 256), (16, 5, 200, 257), (512, 0, 64, 1024), (33, 1, 24, 1025),
                                             (5, 8, 31, 16), (64, 16, 16, 64), (65, 8, 70, 65), (171, 16, 257, 129), (16, 8, 200, 257), (33, 16, 24, 1025)])
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


# Rows that do not start on 16-byte boundaries: widths that are no multiple of 8 (every tail length's parity, blocks that
# end inside a quad and inside a step), or a first row one value past a boundary (`off`).  Sizes: the edges of the three
# kernels (16, 64, 128 rows), row tiles with something over, column splits, more rows than a launch takes.
# Bar: what rounds is a weight's block scale (twice), its two terms, the row scale and the sums, 2^-24 of the weight each:
# eight of those.  (A weight rounded to binary16 once is 2e-4 off.)
@pytest.mark.parametrize("nb,tail,d_out,M,off", [
    (1, 1, 9, 2, 0), (16, 17, 1024, 3, 0), (41, 19, 33, 16, 0), (63, 23, 100, 17, 0), (170, 17, 70, 64, 0), (65, 5, 257, 65, 0), (106, 17, 1000, 129, 0),
    (541, 15, 300, 200, 0), (3, 4, 70, 700, 0), (20, 2, 31, 1030, 0), (684, 3, 24, 515, 0), (32, 0, 40, 5, 1), (64, 8, 70, 40, 3), (85, 16, 300, 300, 1)])
def test_batched_rows_off_their_boundaries_are_as_good_as_single_rows(gpu_rt, orc, nb, tail, d_out, M, off):
    import torch

    d_in = nb * 24 + tail
    raw = synth.make_matrix(f"model.layers.0.tiles.{d_out}x{d_in}.weight", d_out, d_in, seed=nb + M)
    X = synth.make_activation(d_in, seed=M, rows=M)
    Y_ref, _ = _reference(orc, raw, X)
    proj = gpu_rt.upload(raw)
    try:
        buf = torch.empty(M * d_in + 8, dtype=torch.float16, device="cuda")
        x = buf[off:off + M * d_in].view(M, d_in)
        x.copy_(_x16(X))
        Y32, again = (torch.empty((M, d_out), dtype=torch.float32, device="cuda") for _ in range(2))
        Y16 = torch.empty((M, d_out), dtype=torch.float16, device="cuda")
        gpu_rt.forward_batched_into(proj, x, Y32)
        gpu_rt.forward_batched_into(proj, x, again)
        gpu_rt.forward_batched_into(proj, x, Y16)
        rows = sorted({0, 1, M // 2, M - 1})
        single = torch.stack([gpu_rt.forward(proj, x[r], out_dtype=torch.float32) for r in rows])
    finally:
        gpu_rt.free(proj)

    def error(Y, want):
        return np.linalg.norm(Y.double().cpu().numpy() - want) / np.linalg.norm(want)

    print(f"OBSERVED {d_out}x{d_in} M={M} off={off}: {error(Y32, Y_ref):.2e}, single rows {error(single, Y_ref[rows]):.2e}")
    assert error(single, Y_ref[rows]) < 8 * 2.0 ** -24
    assert error(Y32, Y_ref) < 8 * 2.0 ** -24
    assert torch.equal(Y32, again)
    # the same sums to the nearest binary16: half a unit in the last place, 2^-11 of the value (and 2^-25 below the normal
    # range), and a rounding of the f32 sum itself, which a conversion fused with the last operation does not have
    off16 = (Y16.double() - Y32.double()).abs()
    assert bool((off16 <= (2.0 ** -11 + 2.0 ** -23) * Y32.double().abs() + 2.0 ** -25).all())


# In a rotated basis such rows go one by one, as they always have: rotated in f32, the bits of the single-row product.
@pytest.mark.parametrize("n,M,off", [(100, 5, 0), (124, 70, 0), (26, 3, 0), (256, 17, 1), (960, 3, 1)])
def test_rotated_rows_off_their_boundaries_go_one_by_one(gpu_rt, n, M, off):
    import torch

    raw = synth.make_matrix(f"model.layers.0.tiles.rot{n}.weight", 40, n, seed=n)
    raw.rotation_seed = n
    proj = gpu_rt.upload(raw)
    try:
        buf = torch.empty(M * n + 8, dtype=torch.float16, device="cuda")
        x = buf[off:off + M * n].view(M, n)
        x.copy_(_x16(synth.make_activation(n, seed=M, rows=M)))
        for dt in (torch.float32, torch.float16):
            y = torch.empty((M, 40), dtype=dt, device="cuda")
            gpu_rt.forward_batched_into(proj, x, y)
            assert torch.equal(y, torch.stack([gpu_rt.forward(proj, x[r], out_dtype=dt) for r in range(M)]))
    finally:
        gpu_rt.free(proj)


# A row that is not finite spoils itself and no other, whatever repeats or pads it: the last row of a batch and one inside,
# in a block's column and in the last tail column (odd and even tails), through each of the kernels.
@pytest.mark.parametrize("nb,tail,d_out,M", [(9, 8, 40, 5), (9, 7, 40, 5), (70, 16, 50, 60), (70, 1, 50, 60), (9, 16, 300, 300), (9, 23, 300, 300),
                                             (65, 8, 257, 70), (65, 5, 257, 70)])
def test_rows_that_are_not_finite_spoil_no_others(gpu_rt, nb, tail, d_out, M):
    import torch

    d_in = nb * 24 + tail
    raw = synth.make_matrix(f"model.layers.0.tiles.{d_out}x{d_in}.weight", d_out, d_in, seed=nb)
    X = _x16(synth.make_activation(d_in, seed=M, rows=M))
    proj = gpu_rt.upload(raw)
    try:
        for dt in (torch.float32, torch.float16):
            clean = gpu_rt.forward_batched(proj, X, out_dtype=dt)
            assert bool(torch.isfinite(clean).all())
            for column, value in ((nb * 24 - 1, float("inf")), (3, float("nan")), (d_in - 1, float("-inf")), (d_in - 1, float("nan"))):
                bad = [M // 3, M - 1]
                x = X.clone()
                x[bad, column] = value
                y = gpu_rt.forward_batched(proj, x, out_dtype=dt)
                good = [r for r in range(M) if r not in bad]
                assert torch.equal(y[good], clean[good]), (column, value)
                if column == d_in - 1 and value < 0:  # an infinite value in f32 columns: infinite by the weight's sign
                    want = -np.sign(raw.tail.reshape(d_out, tail)[:, -1]) * np.inf
                    assert np.array_equal(y[bad].double().cpu().numpy(), np.broadcast_to(want, (2, d_out)))
                else:
                    assert not bool(torch.isfinite(y[bad]).any())
    finally:
        gpu_rt.free(proj)
