"""Wide batched products whose escapes (block codes that say kBlockEscape or more) are not all in what a wavefront keeps of its tiles'
lists: lists that overflow, more than 64 in a wavefront's share, more than sixteen in a step, beside tiles and steps with few or
none.  Against the oracle's decoded matrix, through every form of the kernel; and that such matrices are not many times as slow."""
import numpy as np
import pytest

from llvq_amd import artifact, synth
from test_gpu_escapes import _far
from test_gpu_gemm import _reference, _x16

pytestmark = pytest.mark.gpu


def _with_escapes(orc, d_out, nb, tail, share, full=()):
    """share: of all blocks that are escapes by hand, besides 0.08 % by chance; full: rows of nothing else."""
    raw = synth.make_matrix(f"model.layers.0.lists.{d_out}x{nb}.weight", d_out, nb * 24 + tail, seed=nb + tail)
    rng = np.random.default_rng(nb + d_out)
    idx, gains = raw.unpack()
    idx = np.array(idx, np.uint64)
    at = rng.random(idx.size) < share
    for row in full:
        at[row * nb:(row + 1) * nb] = True
    far = _far(orc, 12)
    idx[at] = rng.choice(far, int(at.sum()))
    return artifact.RawMatrix(raw.name, d_out, raw.d_in, 12, raw.centroids, raw.row_scales, raw.tail, artifact.pack_codes(idx, gains, artifact.index_bits(12)))


# Forms: 384 x 128 (10000 by 1000, 12000 by 1000), 256 x 256 (16384 by 700), 256 x 128 split over the columns (2560 by 500), both terms
# of the weights split (tail 1) and whole (rows off their boundary).  nb: 17 and 25 blocks, lists of eight, 0.01 is some three a
# tile and overflows one in thirty; 200 (lists of 16, 96 rows of them) and 541 (lists of 24, 64 rows): 0.004 and 0.0027 are more than 64
# for most wavefronts, in lists that hold and lists that do not; rows full of them: more than sixteen of a step in one wavefront.
@pytest.mark.parametrize("d_out,nb,tail,M,off,share,full", [
    (10000, 17, 8, 1000, 0, 0.01, ()), (12000, 200, 0, 1000, 0, 0.004, range(96, 130)), (16384, 25, 16, 700, 0, 0.01, range(40, 60)),
    (2560, 405, 0, 500, 0, 0.003, range(7)), (1000, 541, 0, 1024, 0, 0.0027, ()), (700, 200, 1, 130, 0, 0.004, range(70, 90)), (500, 541, 8, 100, 1, 0.0027, range(9))])
def test_escapes_past_the_lists(gpu_rt, orc, d_out, nb, tail, M, off, share, full):
    import torch

    raw = _with_escapes(orc, d_out, nb, tail, share, full)
    X = synth.make_activation(raw.d_in, seed=nb, rows=M)
    pick = sorted({0, 1, 31, 32, M // 2, M - 2, M - 1})
    Y_ref, A_ref = _reference(orc, raw, X[pick])
    proj = gpu_rt.upload(raw)
    try:
        buf = torch.empty(M * raw.d_in + 8, dtype=torch.float16, device="cuda")
        x = buf[off:off + M * raw.d_in].view(M, raw.d_in)
        x.copy_(_x16(X))
        y, again = (torch.empty((M, d_out), dtype=torch.float32, device="cuda") for _ in range(2))
        gpu_rt.forward_batched_into(proj, x, y)
        gpu_rt.forward_batched_into(proj, x, again)
    finally:
        gpu_rt.free(proj)
    assert torch.equal(y, again)
    y = y[pick].double().cpu().numpy()
    if off or tail % 8:  # both terms: the bar of test_gpu_tiles.py's rows off their boundaries
        assert np.linalg.norm(y - Y_ref) / np.linalg.norm(Y_ref) < 8 * 2.0 ** -24
    else:  # weights are rounded to binary16, 2^-11 of each at the most; the sums in binary32 beside that
        assert np.all(np.abs(y - Y_ref) <= 1.05 * 2.0 ** -11 * A_ref + 1e-7)


def test_one_escape_in_a_hundred_blocks_does_not_double_the_time(gpu_rt, orc):
    """Gate and up of a 4B layer at 512 rows, 81 us with the escapes of uniform codes: with twelve times as many, which no tile's list
    holds, it took 192 us when every step of such a tile was read by every lane, and 124 where a lane reads each."""
    import torch

    def time(share):
        proj = gpu_rt.upload(_with_escapes(orc, 9728, 106, 16, share))
        x = torch.randn(512, 2560, device="cuda").half()
        ys = [torch.empty((512, 9728), dtype=torch.float16, device="cuda") for _ in range(2)]
        took = []
        try:
            for _ in range(8):
                begin, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
                begin.record()
                for _ in range(10):
                    gpu_rt.forward_batched_group_into([proj, proj], x, ys)
                end.record()
                torch.cuda.synchronize()
                took.append(begin.elapsed_time(end))
        finally:
            gpu_rt.free(proj)
        return sorted(took)[3]

    usual, many = time(0.0), time(0.01)
    print(f"OBSERVED {usual * 100:.1f} us, {many * 100:.1f} us with one escape in a hundred blocks")
    assert many < 1.95 * usual


@pytest.mark.parametrize("extra", [25, 60])
def test_lists_of_more_than_a_lane_each(gpu_rt, orc, extra):
    """The widest rows of shells up to 13: 88 places, in which 25 escapes a tile besides the 50 by chance are more than 64; 60 are too many
    for some tiles and not for others."""
    import torch

    nb, tail, d_out = 1000, 8, 36
    raw = synth.make_matrix("model.layers.0.lists13.weight", d_out, nb * 24 + tail, seed=extra, shell_cap=13)
    rng = np.random.default_rng(extra)
    idx, gains = raw.unpack()
    idx = np.array(idx, np.uint64)
    at = rng.random(idx.size) < extra / (16 * nb)
    idx[at] = rng.choice(_far(orc, 13), int(at.sum()))
    raw = artifact.RawMatrix(raw.name, d_out, raw.d_in, 13, raw.centroids, raw.row_scales, raw.tail, artifact.pack_codes(idx, gains, artifact.index_bits(13)))
    X = synth.make_activation(raw.d_in, seed=1, rows=1)
    Y_ref, A_ref = _reference(orc, raw, X)
    proj = gpu_rt.upload(raw)
    try:
        x = _x16(X)[0]
        y = gpu_rt.forward(proj, x, out_dtype=torch.float32).reshape(-1)
        seq = gpu_rt.plan_sequence([([proj], x, False)], out_dtype=torch.float32)
        seq.run()
        seq.status()
        assert torch.equal(y, seq.outputs[0][0].reshape(-1))
        seq.close()
    finally:
        gpu_rt.free(proj)
    assert np.max(np.abs(y.double().cpu().numpy() - Y_ref[0]) / A_ref[0]) < 1e-5


def test_a_list_that_overflows_is_not_many_times_a_batch1_launch(gpu_rt, orc):
    """One tile of a 9728 x 2560 product with twenty escapes, where its list has eight places: the launch of 5.6 us took 30 when each row of
    the tile was walked 64 blocks at a time, and takes 10.5 (twice it, and a quarter more for the runs' differences)."""
    import torch

    raw = synth.make_matrix("model.layers.0.lists1.weight", 9728, 2560, seed=3)
    idx, gains = raw.unpack()
    idx = np.array(idx, np.uint64)
    idx[106 * np.arange(20) % (16 * 106) + np.arange(20)] = _far(orc, 12)[:20]  # (rows 0 to 15, each a block or two)
    many = artifact.RawMatrix(raw.name, 9728, 2560, 12, raw.centroids, raw.row_scales, raw.tail, artifact.pack_codes(idx, gains, artifact.index_bits(12)))
    x = torch.randn(2560, device="cuda").half()
    projs = [gpu_rt.upload(m) for m in (raw, many)]
    took = [[], []]
    try:
        for _ in range(8):
            for (launch, _), t in zip([gpu_rt.plan_group([proj], x) for proj in projs], took):
                begin, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
                begin.record()
                for _ in range(100):
                    launch()
                end.record()
                torch.cuda.synchronize()
                t.append(begin.elapsed_time(end))
    finally:
        for proj in projs:
            gpu_rt.free(proj)
    usual, one = (sorted(t)[3] for t in took)
    print(f"OBSERVED {usual * 10:.2f} us, {one * 10:.2f} us with a list that overflows")
    assert one < 2.5 * usual


@pytest.mark.parametrize("M", [2, 65])
def test_rows_of_more_blocks_than_an_entry_has_bits_for(gpu_rt, orc, M):
    """Past 2^19 blocks (12.6 M columns) a tile has no list: its codes are read.  With lists, the escapes past that block were added to
    other rows."""
    import torch

    nb, d_out = (1 << 19) + 300, 2
    rng = np.random.default_rng(3)
    few = synth.make_matrix("model.layers.0.widest.weight", d_out, 24, seed=2)
    codes = artifact.pack_codes(rng.integers(0, orc.N12 + 1, d_out * nb).astype(np.uint64), rng.integers(0, 2, d_out * nb).astype(np.uint8), artifact.index_bits(12))
    raw = artifact.RawMatrix(few.name, d_out, nb * 24, 12, few.centroids, few.row_scales, few.tail, codes)
    X = rng.standard_normal((2, raw.d_in), dtype=np.float32).astype(np.float16)
    Y_ref, _ = _reference(orc, raw, X)
    proj = gpu_rt.upload(raw)
    try:
        x = _x16(X)[torch.arange(M, device="cuda") % 2]
        y = gpu_rt.forward_batched(proj, x, out_dtype=torch.float32).double().cpu().numpy()
    finally:
        gpu_rt.free(proj)
    # weights are rounded to binary16 one by one: 2^-12 of each on average, whose sum over 12.6 M columns goes with the root of their number
    for m in range(M):
        assert np.linalg.norm(y[m] - Y_ref[m % 2]) < 1e-3 * np.linalg.norm(Y_ref[m % 2])
