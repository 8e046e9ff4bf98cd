"""Rotated artifacts on the device: the activation rotation kernel against the
oracle's Rotation, and the product y = W'(Q x) against the oracle's dense arm
(decode_matrix un-rotates to the natural basis) — the identity of
llvq-artifact/tests/fused_path_matches_dense.rs."""
import numpy as np
import pytest

from llvq_amd import artifact, decoder, synth

pytestmark = pytest.mark.gpu
TOL = 1e-3


def _x16(x):
    import torch

    return torch.from_numpy(x.view(np.int16).copy()).view(torch.float16).cuda()


def _rotated(name, d_out, d_in, seed, rot_seed):
    raw = synth.make_matrix(name, d_out, d_in, seed=seed)
    raw.rotation_seed = rot_seed
    return raw


# widths of fused.rs:1274 (k = 15, 5, 19, 1, 3) plus the 8B/14B hidden sizes (k = 1, 5)
@pytest.mark.parametrize("n,seed", [(240, 1), (2560, 2), (9728, 3), (4096, 4), (96, 5), (5120, 6), (24, 7)])
def test_rotate_kernel_matches_oracle(gpu_rt, orc, n, seed):
    raw = _rotated(f"model.layers.0.r{n}.weight", 8, n, 1, seed)
    x = synth.make_activation(n, seed=seed)[0]
    proj = gpu_rt.upload(raw)
    xr = gpu_rt.rotate(proj, _x16(x)).cpu().numpy().reshape(-1)
    gpu_rt.free(proj)
    want = orc.Rotation(n, seed).apply(x.astype(np.float64))
    dev = np.linalg.norm(xr - want) / np.linalg.norm(want)
    assert dev < 1e-5, f"relative deviation {dev:.3e}"   # f32 butterflies
    assert np.abs(xr - want).max() < 1e-4 * np.abs(want).max()


def test_natural_basis_rotate_only_widens(gpu_rt):
    raw = synth.make_matrix("model.layers.0.plain.weight", 8, 240, seed=1)
    x = synth.make_activation(240, seed=3)[0]
    proj = gpu_rt.upload(raw)
    xr = gpu_rt.rotate(proj, _x16(x)).cpu().numpy().reshape(-1)
    gpu_rt.free(proj)
    assert np.array_equal(xr, x.astype(np.float32))


@pytest.mark.parametrize("d_out,d_in", [(8, 240), (16, 2560), (8, 9728), (24, 4096), (8, 96), (5, 256), (7, 104)])
def test_rotated_gemv_matches_dense_arm(gpu_rt, orc, d_out, d_in):
    import torch

    raw = _rotated(f"model.layers.0.rot.{d_out}x{d_in}.weight", d_out, d_in, seed=d_in, rot_seed=0xA5 + d_in)
    x = synth.make_activation(d_in, seed=d_in + 1)[0]
    om, _ = orc.read_matrix_raw(artifact.write_matrix_raw(raw))
    y_ref, a_ref = om.fused_product(x.astype(np.float64))        # rotates the activation, f64
    W = om.decode_matrix().astype(np.float64)                      # un-rotated weights
    assert np.abs(W @ x.astype(np.float64) - y_ref).max() < 1e-6 * a_ref.max()
    proj = gpu_rt.upload(raw)
    try:
        y = gpu_rt.forward(proj, _x16(x), out_dtype=torch.float32).cpu().numpy().astype(np.float64)
        y2 = gpu_rt.forward_rotated(proj, gpu_rt.rotate(proj, _x16(x)), out_dtype=torch.float32).cpu().numpy().reshape(-1)
    finally:
        gpu_rt.free(proj)
    e = np.abs(y - y_ref) / np.maximum(a_ref, 1e-30)
    assert e.max() < 1e-5, f"max |dy|/sum|wx| = {e.max():.3e}"
    assert np.array_equal(y.astype(np.float32), y2)  # the two-call form is the same computation


def test_wide_odd_factor_is_refused_at_upload(gpu_rt):
    from llvq_amd import LlvqError

    raw = _rotated("model.layers.0.odd.weight", 8, 2568, 1, 5)  # 2568 = 8 * 321 (fused.rs:698-704)
    with pytest.raises(LlvqError) as e:
        gpu_rt.upload(raw)
    assert e.value.kind == "Unsupported" and "321" in str(e.value)


def test_group_with_mixed_bases(gpu_rt, orc):
    """q rotated with one seed, k with another, v in the natural basis: three bases, one call."""
    import torch

    mats = [_rotated("model.layers.1.self_attn.q_proj.weight", 32, 2560, 3, 11),
            _rotated("model.layers.1.self_attn.k_proj.weight", 16, 2560, 3, 12),
            synth.make_matrix("model.layers.1.self_attn.v_proj.weight", 16, 2560, seed=3),
            _rotated("model.layers.1.self_attn.x_proj.weight", 8, 2560, 4, 11)]
    x = synth.make_activation(2560, seed=8)[0]
    projs = [gpu_rt.upload(m) for m in mats]
    ys = gpu_rt.forward_group(projs, _x16(x), out_dtype=torch.float32)
    for p, raw, y in zip(projs, mats, ys):
        om, _ = orc.read_matrix_raw(artifact.write_matrix_raw(raw))
        y_ref, a_ref = om.fused_product(x.astype(np.float64))
        assert (np.abs(y.cpu().numpy() - y_ref) / a_ref).max() < 1e-5
        gpu_rt.free(p)


def test_rotated_batched_rows(gpu_rt, orc):
    import torch

    raw = _rotated("model.layers.2.mlp.up_proj.weight", 128, 2560, 4, 99)
    X = synth.make_activation(2560, seed=21, rows=24)
    om, _ = orc.read_matrix_raw(artifact.write_matrix_raw(raw))
    W = om.decode_matrix().astype(np.float64)
    Y_ref = X.astype(np.float64) @ W.T
    # the normaliser in the rotated basis, where the kernel sums
    rot = orc.Rotation(2560, 99)
    Wr = np.stack([rot.apply(r) for r in W])
    Xr = np.stack([rot.apply(r) for r in X.astype(np.float64)])
    A_ref = np.abs(Xr) @ np.abs(Wr).T
    proj = gpu_rt.upload(raw)
    Y = gpu_rt.forward_batched(proj, _x16(X), out_dtype=torch.float32).cpu().numpy()
    gpu_rt.free(proj)
    assert (np.abs(Y - Y_ref) / A_ref).max() < TOL


def test_decoder_with_rotated_projections(gpu_rt, orc):
    """The decode loop over an artifact whose projections are all stored rotated
    (one seed per activation site, as the reference's rotation keys are)."""
    from oracle import qwen3_oracle

    cfg = decoder.Qwen3Config(num_hidden_layers=2, hidden_size=192, num_attention_heads=4, num_key_value_heads=2,
                              head_dim=32, intermediate_size=320, vocab_size=300, rope_theta=1e4, rms_norm_eps=1e-6,
                              max_positions=32, tie_word_embeddings=True)
    raws = decoder.synthetic_projections(cfg, 5)
    for L, layer in enumerate(raws):
        for j, m in enumerate(layer):
            m.rotation_seed = 1000 + 10 * L + (0 if j < 3 else 1 if j == 3 else 2 if j < 6 else 3)
    weights = decoder.synthetic_weights(cfg, 5)
    dense = [[orc.read_matrix_raw(artifact.write_matrix_raw(m))[0].decode_matrix() for m in layer] for layer in raws]
    ref = qwen3_oracle.Qwen3Oracle(cfg, dense, weights)
    dec = decoder.Decoder(gpu_rt, cfg, raws, weights)
    try:
        worst = 0.0
        for t in np.random.default_rng(5).integers(0, cfg.vocab_size, size=12):
            want = ref.forward_token(int(t))
            got, _ = dec.forward_token(int(t))
            worst = max(worst, float(np.abs(got - want).max() / np.abs(want).max()))
        assert worst < 2e-2
    finally:
        dec.close()


@pytest.mark.parametrize("k", [-40, -64, -75, -90, 60])
@pytest.mark.parametrize("d_in", [248, 13000])  # 13 000: rows past 512 blocks
def test_a_power_of_two_goes_through_a_rotated_product_unchanged(gpu_rt, k, d_in):
    """The activation is quantised per block relative to the block's largest value, so a power of two in front of an f32
    activation is one in front of an f32 result, bit for bit, as long as nothing leaves the normal range (|k| <= 90)."""
    import torch

    proj = gpu_rt.upload(synth.make_matrix(f"model.layers.0.scaled.{d_in}.weight", 40, d_in, seed=4))
    try:
        xr = torch.from_numpy(synth.make_activation(d_in, seed=9)[0].astype(np.float32)).cuda().reshape(1, -1)
        one = gpu_rt.forward_rotated(proj, xr, out_dtype=torch.float32).double()
        got = gpu_rt.forward_rotated(proj, xr * 2.0 ** k, out_dtype=torch.float32)
        assert torch.equal(got.double(), one * 2.0 ** k)
    finally:
        gpu_rt.free(proj)


def test_rows_too_wide_to_be_rotated_in_the_launch(gpu_rt, orc):
    """24 576 columns with f32 results do not fit LDS beside their digit planes: the activation is rotated by a kernel of its own,
    into memory that belongs to the rotation.  An upload between two products (which brings another such rotation) changes
    nothing about the first, nor about rows that are rotated in their launch."""
    import torch

    first = _rotated("model.layers.0.wide.0.weight", 9, 20480, 3, 41)
    x = {n: _x16(synth.make_activation(n, seed=n)[0]) for n in (20480, 24576)}
    projs = [gpu_rt.upload(first)]
    try:
        one = gpu_rt.forward(projs[0], x[20480], out_dtype=torch.float32)
        projs += [gpu_rt.upload(_rotated("model.layers.0.wide.1.weight", 9, 24576, 4, 42)),
                  gpu_rt.upload(_rotated("model.layers.0.wide.2.weight", 9, 20480, 5, 43))]
        for p in projs:
            for dt in (torch.float32, torch.float16):
                y = gpu_rt.forward(p, x[p.d_in], out_dtype=dt).reshape(-1)
                assert torch.equal(y, gpu_rt.forward_rotated(p, gpu_rt.rotate(p, x[p.d_in]), out_dtype=dt).reshape(-1))
        assert torch.equal(gpu_rt.forward(projs[0], x[20480], out_dtype=torch.float32), one)
        om, _ = orc.read_matrix_raw(artifact.write_matrix_raw(first))
        y_ref, a_ref = om.fused_product(synth.make_activation(20480, seed=20480)[0].astype(np.float64))
        assert (np.abs(one.cpu().numpy().reshape(-1) - y_ref) / a_ref).max() < 1e-5
    finally:
        for p in projs:
            gpu_rt.free(p)


# The widest rows that are rotated in their product's launch (f32 up to 20480, binary16 up to 24576 columns), whose partial sums lie
# where the rotated row was, with more tiles than a round of a launch has; and past them, between uploads of another such rotation.
@pytest.mark.parametrize("n,out", [(19456, "f32"), (20480, "f32"), (23552, "f16"), (24576, "f16"), (24576, "f32")])
def test_widest_rotated_rows(gpu_rt, orc, n, out):
    import torch

    d_out = 16 * 256 + 9 if n == 20480 or out == "f16" else 40
    raw = _rotated(f"model.layers.0.widest.{n}.weight", d_out, n, 3, 51)
    x = synth.make_activation(n, seed=n)[0]
    proj = gpu_rt.upload(raw)
    dt = torch.float32 if out == "f32" else torch.float16
    try:
        one = gpu_rt.forward(proj, _x16(x), out_dtype=dt).reshape(-1)
        other = gpu_rt.upload(_rotated("model.layers.0.widest.other.weight", 9, n, 4, 52))
        gpu_rt.forward(other, _x16(x), out_dtype=dt)
        again = gpu_rt.forward(proj, _x16(x), out_dtype=dt).reshape(-1)
        gpu_rt.free(other)
        apart = gpu_rt.forward_rotated(proj, gpu_rt.rotate(proj, _x16(x)), out_dtype=dt).reshape(-1)
    finally:
        gpu_rt.free(proj)
    assert torch.equal(one, again) and torch.equal(one, apart)
    om, _ = orc.read_matrix_raw(artifact.write_matrix_raw(raw))
    y_ref, a_ref = om.fused_product(x.astype(np.float64))
    err = np.abs(one.double().cpu().numpy() - y_ref)
    # (binary16 results: the activation to 2^-15 of its block's largest value, which is less than five times their mean, and the result's rounding)
    assert np.all(err <= (1e-5 * a_ref if out == "f32" else 5 * 2.0 ** -15 * a_ref + 2.0 ** -11 * np.abs(y_ref)))


# Rows that are rotated straight to the products' octets, in a call of its own, against the rotated rows of a group too large for
# one launch (five matrices): the same values, so the same bits.  m = 8 (the narrowest with octets), tails of 8 and 16 columns;
# rows around the padding of 16, 64 and 128 and around 256, from where both calls take the second way.
@pytest.mark.parametrize("n,rows", [(31 * 8, 2), (31 * 8, 17), (1024, 16), (1024, 65), (3 * 1024, 64), (3 * 1024, 130), (4096, 256), (4096, 257)])
def test_rotated_rows_to_octets(gpu_rt, n, rows):
    import torch

    projs = [gpu_rt.upload(_rotated(f"model.layers.3.mlp.p{i}.weight", 48, n, 5 + i, 77)) for i in range(5)]
    try:
        x = _x16(synth.make_activation(n, seed=n + rows, rows=rows))
        ys = [torch.empty((rows, 48), dtype=torch.float32, device="cuda") for _ in projs]
        gpu_rt.forward_batched_group_into(projs, x, ys)
        junk = torch.full((rows, n), float("nan"), dtype=torch.float16, device="cuda")  # what the octets' padding must not keep
        gpu_rt.forward_batched(projs[0], junk)
        alone = [gpu_rt.forward_batched(p, x, out_dtype=torch.float32) for p in projs]
    finally:
        for p in projs:
            gpu_rt.free(p)
    for y, z in zip(ys, alone):
        assert torch.isfinite(z).all() and torch.equal(y, z)


# around what the lane moves reach (columns of 32 values, m = 64 .. 1024), above and below it; k up to 9 as scalars (whole columns to a lane,
# parts of a column to the wavefronts), above on the matrix cores
@pytest.mark.parametrize("m,k", [(32, 9), (64, 1), (64, 3), (64, 9), (64, 11), (128, 5), (256, 7), (256, 31), (512, 1), (512, 9), (512, 11), (1024, 1), (1024, 3),
                                 (1024, 9), (1024, 17), (2048, 1), (2048, 5), (4096, 3), (8192, 1)])
def test_rotation_of_every_kind_of_width(gpu_rt, orc, m, k):
    import torch

    n = m * k
    raw = _rotated(f"model.layers.0.rw{n}.weight", 16, n, 1, n)
    x = synth.make_activation(n, seed=n)[0]
    proj = gpu_rt.upload(raw)
    try:
        xr = gpu_rt.rotate(proj, _x16(x))
        got = xr.cpu().numpy().reshape(-1)
        want = orc.Rotation(n, n).apply(x.astype(np.float64))
        # f32: a rounding for each of log2 m levels, for the k terms of a sum and for the two factors
        assert np.linalg.norm(got - want) <= (np.log2(m) + k + 2) * 2.0**-24 * np.linalg.norm(want)
        assert np.array_equal(gpu_rt.forward(proj, _x16(x), out_dtype=torch.float32).cpu().numpy().reshape(-1),
                              gpu_rt.forward_rotated(proj, xr, out_dtype=torch.float32).cpu().numpy().reshape(-1))
        # one value that is not finite is in all of them
        for value in (float("nan"), float("inf"), float("-inf")):
            bad = _x16(x)
            bad[n // 2] = value
            for dtype in (torch.float16, torch.float32):
                assert not torch.isfinite(gpu_rt.forward(proj, bad, out_dtype=dtype)).any()
    finally:
        gpu_rt.free(proj)


# up to the rows of a launch every batch's rotation writes octets: past 256, off and on the padding of 128 and 256 rows, and the last count
# (widths whose columns no plan splits: the same sums)
@pytest.mark.parametrize("n,rows", [(31 * 8, 300), (31 * 8, 700), (1024, 512), (3 * 128, 1000), (31 * 8, 1024), (31 * 8, 1025)])
def test_many_rotated_rows_to_octets(gpu_rt, n, rows):
    test_rotated_rows_to_octets(gpu_rt, n, rows)


# widths whose rotation goes to many workgroups (rot_split_pays): every m, few and many groups, one and several tiles a wavefront
@pytest.mark.parametrize("m,k", [(512, 17), (512, 31), (1024, 11), (1024, 23), (2048, 7), (2048, 11), (4096, 3), (4096, 5)])
def test_rotation_by_many_workgroups(gpu_rt, orc, m, k):
    test_rotation_of_every_kind_of_width(gpu_rt, orc, m, k)


# rows wider than a batch-1 product takes, rotated by themselves: as many tiles as the wavefronts' last turn begins with, and nearly all of it
@pytest.mark.parametrize("m,k", [(4096, 7), (1024, 31)])
def test_rotation_of_rows_past_the_products(gpu_rt, orc, m, k):
    n = m * k
    proj = gpu_rt.upload(_rotated(f"model.layers.0.rw{n}.weight", 16, n, 1, n))
    x = synth.make_activation(n, seed=n)[0]
    try:
        got = gpu_rt.rotate(proj, _x16(x)).cpu().numpy().reshape(-1)
        want = orc.Rotation(n, n).apply(x.astype(np.float64))
        assert np.linalg.norm(got - want) <= (np.log2(m) + k + 2) * 2.0**-24 * np.linalg.norm(want)  # (as above)
    finally:
        gpu_rt.free(proj)
