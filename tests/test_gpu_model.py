"""Device pipeline (vocalarc_hip.h model entry points) vs the oracle.

Stage tests compare one stage at a time on identical inputs; the forward and
chunked tests compare whole waveforms at the fp32 parity bar: per-sample
max |delta| <= 1e-4 and SNR >= 80 dB.
"""

import numpy as np
import pytest

from helpers import assert_close, empty_dev, from_dev, gpu_available, snr_db, to_dev

pytestmark = pytest.mark.gpu

if gpu_available():
    import torch
    import oracle as O
    from vocalarc_hip import audio, native, pack
    from vocalarc_hip.dims import CONFIG_DIMS, REFERENCE_DIMS, ModelDims


@pytest.fixture(scope="module")
def ctx():
    if not gpu_available():
        pytest.skip("no GPU")
    c = native.Context()
    yield c
    c.close()


@pytest.fixture(scope="module")
def cfg2():
    """Config shape (dim 384, 62 bands, hop 441, GELU-GLU) at depth 2."""
    d = CONFIG_DIMS.with_depth(2)
    return d, pack.synthetic_pack(d, 77)


@pytest.fixture(scope="module")
def cfg2_models(ctx, cfg2):
    d, blob = cfg2
    return O.Model(d, blob), native.Model(ctx, d, blob)


@pytest.fixture(scope="module")
def ref_models(ctx, ref_pack):
    return O.Model(REFERENCE_DIMS, ref_pack), native.Model(ctx, REFERENCE_DIMS, ref_pack)


@pytest.mark.parametrize("axis,S,L", [(0, 4, 62), (1, 3, 130), (0, 2, 801)])
def test_transformer_block_config(cfg2_models, rng, axis, S, L):
    om, dm = cfg2_models
    x = rng.standard_normal((S, L, om.d.dim), dtype=np.float32)
    ref = om.transformer(1, axis, x, S, L)
    dx = to_dev(x)
    dm.transformer(1, axis, dx, S, L)
    out = from_dev(dx)
    assert_close(ref, out, rtol=1e-4, atol=1e-4, min_snr=100, what="transformer (config)")


@pytest.mark.parametrize("axis,S,L", [(0, 4, 62), (1, 3, 801), (1, 2, 161)])
def test_transformer_block_kv_prescale_bit_identical(cfg2_models, rng, monkeypatch, axis, S, L):
    """The fused block's QKV GEMM writes k and v times the attention's piece
    scales (2^ek, 2^ev: one ldexp exponent per 32-column tile) and the
    attention stages them unscaled; VOCALARC_KV_PRESCALE=0 keeps the
    unscaled projection and the scaling multiplies in the attention.  Both
    must give the same bits (powers of two commute with the rotation and the
    splits), on both axes and on a ragged length (64 < L <= 128 never scales
    them).  The band axis runs its projection and attention as the two kernels
    here (VOCALARC_BAND_FUSED=0: the fused kernel always scales k and v in its
    epilogue).  A block alone norms x as a pass; the norm inside the projection
    is test_forward_kv_prescale_bit_identical's."""
    om, dm = cfg2_models
    x = rng.standard_normal((S, L, om.d.dim), dtype=np.float32)
    monkeypatch.setenv("VOCALARC_BAND_FUSED", "0")
    outs = []
    for env in (None, "0"):
        if env is None:
            monkeypatch.delenv("VOCALARC_KV_PRESCALE", raising=False)
        else:
            monkeypatch.setenv("VOCALARC_KV_PRESCALE", env)
        dx = to_dev(x)
        dm.transformer(1, axis, dx, S, L)
        outs.append(from_dev(dx))
    monkeypatch.delenv("VOCALARC_KV_PRESCALE", raising=False)
    monkeypatch.delenv("VOCALARC_BAND_FUSED", raising=False)
    assert np.array_equal(outs[0].view(np.uint32), outs[1].view(np.uint32))


@pytest.mark.parametrize("pieces", [None, "0"])
def test_forward_kv_prescale_bit_identical(cfg2_models, monkeypatch, pieces):
    """Two layers on 201 frames: from the second block on the attention's norm runs inside the QKV GEMM, whose k and v
    leave scaled (with VOCALARC_KV_PIECES=0 as fp32, else split) or, with VOCALARC_KV_PRESCALE=0, as they are: the same
    bits.  The band axis on the two kernels, as above."""
    om, dm = cfg2_models
    x = audio.sine_mix(2.0, 16)
    monkeypatch.setenv("VOCALARC_BAND_FUSED", "0")
    if pieces is not None:
        monkeypatch.setenv("VOCALARC_KV_PIECES", pieces)
    outs = []
    for env in (None, "0"):
        if env is not None:
            monkeypatch.setenv("VOCALARC_KV_PRESCALE", env)
        dx = empty_dev(x.shape)
        dm.forward(to_dev(x), x.shape[1], dx)
        outs.append(from_dev(dx))
    assert np.all(np.isfinite(outs[0]))
    assert np.array_equal(outs[0].view(np.uint32), outs[1].view(np.uint32))


@pytest.mark.parametrize("S,L", [(4, 62), (23, 62), (5, 64), (7, 17), (3, 1)])
def test_band_attention_fused(cfg2_models, rng, monkeypatch, S, L):
    """The band axis's pre-norm projection and attention in one kernel
    (sequences of L <= 64 consecutive rows; q, k, v and the gate logits stay
    on chip), against the oracle and against the two kernels it replaces
    (VOCALARC_BAND_FUSED=0).  The fused kernel splits x and norms the products;
    a block alone on the two kernels norms x as a pass and splits the normed
    rows.  The gate logit is an fp32 dot product instead of the split GEMM's
    column.  So the two paths agree to a few fp32 roundings, not bit for bit.  Odd S leaves a tile with one sequence, L = 64
    fills a tile's 64 positions, L = 1 is a single key."""
    om, dm = cfg2_models
    x = rng.standard_normal((S, L, om.d.dim), dtype=np.float32)
    outs = []
    for env in (None, "0"):
        if env is None:
            monkeypatch.delenv("VOCALARC_BAND_FUSED", raising=False)
        else:
            monkeypatch.setenv("VOCALARC_BAND_FUSED", env)
        dx = to_dev(x)
        dm.transformer(1, 1, dx, S, L)
        outs.append(from_dev(dx))
    monkeypatch.delenv("VOCALARC_BAND_FUSED", raising=False)
    ref = om.transformer(1, 1, x, S, L)
    assert_close(ref, outs[0], rtol=1e-4, atol=1e-4, min_snr=100, what="fused band attention (oracle)")
    scale = float(np.max(np.abs(outs[1])))
    assert float(np.max(np.abs(outs[0] - outs[1]))) <= 1e-5 * scale
    assert snr_db(outs[1], outs[0]) >= 120.0


@pytest.mark.parametrize("axis,S,L", [(0, 3, 129), (1, 5, 160), (0, 2, 801), (0, 31, 191)])
def test_kv_pieces_consecutive_rows_bit_identical(cfg2_models, monkeypatch, axis, S, L):
    """A block on sequences of consecutive rows (vh_transformer's order): the QKV GEMM rotates k by one position
    per row, sequences ending inside a wave's 32 rows, and a ragged last row tile; the same bits as the attention's own
    rotation and split (VOCALARC_KV_PIECES=0)."""
    rng = np.random.default_rng(L)
    om, dm = cfg2_models
    x = rng.standard_normal((S, L, om.d.dim), dtype=np.float32)
    outs = []
    for env in (None, "0"):
        if env is None:
            monkeypatch.delenv("VOCALARC_KV_PIECES", raising=False)
        else:
            monkeypatch.setenv("VOCALARC_KV_PIECES", env)
        dx = to_dev(x)
        dm.transformer(1, axis, dx, S, L)
        outs.append(from_dev(dx))
    monkeypatch.delenv("VOCALARC_KV_PIECES", raising=False)
    assert np.array_equal(outs[0].view(np.uint32), outs[1].view(np.uint32))


@pytest.mark.parametrize("axis,S,L", [(0, 3, 129), (1, 5, 160), (0, 2, 801), (0, 31, 191), (0, 0, 0)])
def test_bf16_rotated_k_bit_identical(cfg2_models, monkeypatch, axis, S, L):
    """The bf16 variant: k leaves the projection rotated (consecutive rows, and with S = 0 a 2 s forward's
    [frame][band] rows, 201 frames) and the attention copies k and v into LDS by DMA; the same bits as the rotation
    and transposition in the attention (VOCALARC_KV_PIECES=0)."""
    rng = np.random.default_rng(L)
    om, dm = cfg2_models
    x = rng.standard_normal((S, L, om.d.dim), dtype=np.float32) if S else audio.sine_mix(2.0, 15)
    dm.set_precision(native.PRECISION_BF16)
    outs = []
    try:
        for env in (None, "0"):
            if env is None:
                monkeypatch.delenv("VOCALARC_KV_PIECES", raising=False)
            else:
                monkeypatch.setenv("VOCALARC_KV_PIECES", env)
            if S:
                dx = to_dev(x)
                dm.transformer(1, axis, dx, S, L)
            else:
                dx = empty_dev(x.shape)
                dm.forward(to_dev(x), x.shape[1], dx)
            outs.append(from_dev(dx))
    finally:
        dm.set_precision(native.PRECISION_FP32)
        monkeypatch.delenv("VOCALARC_KV_PIECES", raising=False)
    assert np.all(np.isfinite(outs[0]))
    assert np.array_equal(outs[0].view(np.uint32), outs[1].view(np.uint32))


@pytest.mark.parametrize("windows", [1, 3])
def test_kv_pieces_bit_identical(cfg2_models, monkeypatch, windows):
    """On the pipeline's time axis (L > 64, [chunk][frame][band] rows) the
    fused QKV GEMM writes k, rotated, and v as the attention's fp16 pieces
    and the attention copies them into LDS by DMA, reading V^T through the
    transpose load; VOCALARC_KV_PIECES=0 keeps the fp32 projection and the
    attention's own rotation and splits.  Both must give the same bits: one
    2 s window (T = 201: ragged query and key blocks) and three 2 s windows
    in one pass (M = 37386 rows: a ragged last row tile, waves whose 32 rows
    straddle two frames, and frames that wrap to the next window)."""
    om, dm = cfg2_models
    chunk, step = 88200, 66150
    x = audio.sine_mix(2.0 if windows == 1 else 5.0, 15)
    length = x.shape[1]
    assert O.chunk_count(length, chunk, step) == windows
    outs = []
    for env in (None, "0"):
        if env is None:
            monkeypatch.delenv("VOCALARC_KV_PIECES", raising=False)
        else:
            monkeypatch.setenv("VOCALARC_KV_PIECES", env)
        dv = empty_dev(x.shape)
        if windows == 1:
            dm.forward(to_dev(x), length, dv)
        else:
            dm.separate(to_dev(x), length, chunk, step, windows, dv)
        outs.append(from_dev(dv))
    monkeypatch.delenv("VOCALARC_KV_PIECES", raising=False)
    assert np.all(np.isfinite(outs[0]))
    assert np.array_equal(outs[0].view(np.uint32), outs[1].view(np.uint32))


@pytest.mark.parametrize("axis,S,L", [(0, 90, 23), (1, 23, 90)])
def test_transformer_block_reference_shape(ref_models, rng, axis, S, L):
    om, dm = ref_models
    x = rng.standard_normal((S, L, om.d.dim), dtype=np.float32)
    ref = om.transformer(5, axis, x, S, L)
    dx = to_dev(x)
    dm.transformer(5, axis, dx, S, L)
    assert_close(ref, from_dev(dx), rtol=1e-4, atol=1e-4, min_snr=100, what="transformer (reference)")


def _to_layout(spec: np.ndarray, layout: int) -> np.ndarray:
    """[F][C][T][2] -> the device layout (frame-major: [C][T][F][2])."""
    return spec if layout == native.SPEC_REFERENCE else np.ascontiguousarray(spec.transpose(1, 2, 0, 3))


def _from_layout(spec: np.ndarray, layout: int) -> np.ndarray:
    return spec if layout == native.SPEC_REFERENCE else np.ascontiguousarray(spec.transpose(2, 0, 1, 3))


LAYOUTS = [0, 1]  # SPEC_REFERENCE, SPEC_FRAME_MAJOR


@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("which", ["config", "reference"])
def test_stft_istft(ctx, cfg2_models, ref_models, which, layout):
    om, dm = cfg2_models if which == "config" else ref_models
    d = om.d
    x = audio.sine_mix(0.5, 3)
    length = x.shape[1]
    T = d.frames(length)
    src = O.stft(d, x)
    dsrc = empty_dev(_to_layout(src, layout).shape)
    dm.stft(to_dev(x), length, dsrc, layout)
    gsrc = _from_layout(from_dev(dsrc), layout)
    assert_close(src, gsrc, rtol=1e-6, atol=2e-6, min_snr=120, what="stft")
    rng = np.random.default_rng(5)
    mask = rng.standard_normal(src.shape).astype(np.float32)
    ref = O.istft(d, src, mask, length)
    dout = empty_dev((d.channels, length))
    dm.istft(to_dev(_to_layout(src, layout)), to_dev(_to_layout(mask, layout)), length, dout, layout)
    assert_close(ref, from_dev(dout), rtol=1e-5, atol=1e-6, min_snr=120, what="istft")
    assert T == src.shape[2]


@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("length", [1200, 2049, 3969, 4410])
def test_stft_istft_edges(cfg2_models, length, layout):
    """Signals of a few frames (3, 5, 9 or 11: the kernels take four at a time), reflected at both ends, digital
    silence in the first half of one channel, and a mask that makes bins 0 and 1024 complex (only their real parts
    reach the signal)."""
    rng = np.random.default_rng(length)
    om, dm = cfg2_models
    d = om.d
    x = rng.standard_normal((d.channels, length)).astype(np.float32)
    x[0, :length // 2] = 0.0
    src = O.stft(d, x)
    dsrc = empty_dev(_to_layout(src, layout).shape)
    dm.stft(to_dev(x), length, dsrc, layout)
    got = _from_layout(from_dev(dsrc), layout)
    assert_close(src, got, rtol=1e-6, atol=4e-6, min_snr=120, what="stft")
    silent = [t for t in range(src.shape[2]) if not np.any(src[:, 0, t])]
    assert np.all(got[:, 0, silent] == 0.0)  # an exactly silent frame stays exactly zero
    mask = rng.standard_normal(src.shape).astype(np.float32)
    ref = O.istft(d, src, mask, length)
    dout = empty_dev((d.channels, length))
    dm.istft(to_dev(_to_layout(src, layout)), to_dev(_to_layout(mask, layout)), length, dout, layout)
    assert_close(ref, from_dev(dout), rtol=1e-5, atol=4e-6, min_snr=120, what="istft")


def test_istft_perfect_reconstruction(ctx, cfg2_models):
    """A unit mask reproduces the input (closed form: Hann OLA normalised by
    the summed squared window)."""
    om, dm = cfg2_models
    d = om.d
    x = audio.sine_mix(0.4, 9)
    length = x.shape[1]
    dsrc = empty_dev((d.freq_bins, d.channels, d.frames(length), 2))
    dm.stft(to_dev(x), length, dsrc)
    ones = np.zeros((d.freq_bins, d.channels, d.frames(length), 2), np.float32)
    ones[..., 0] = 1.0
    dout = empty_dev((d.channels, length))
    dm.istft(dsrc, to_dev(ones), length, dout)
    assert_close(x, from_dev(dout), rtol=0, atol=2e-6, what="istft(stft(x))")


@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("which", ["config", "reference"])
def test_band_split_and_mask(ctx, cfg2_models, ref_models, which, rng, layout):
    om, dm = cfg2_models if which == "config" else ref_models
    d = om.d
    x = audio.sine_mix(0.3, 4)
    src = O.stft(d, x)
    T = src.shape[2]
    ref = om.band_split(src)
    dout = empty_dev(ref.shape)
    dm.band_split(to_dev(_to_layout(src, layout)), T, dout, layout)
    assert_close(ref, from_dev(dout), rtol=1e-4, atol=2e-5, min_snr=110, what="band split")
    feats = rng.standard_normal((T, d.bands, d.dim), dtype=np.float32)
    mref = om.mask_estimate(feats)
    dmask = empty_dev(_to_layout(mref, layout).shape)
    dm.mask_estimate(to_dev(feats), T, dmask, layout)
    assert_close(mref, _from_layout(from_dev(dmask), layout), rtol=1e-4, atol=1e-5, min_snr=110,
                 what="mask estimator")


@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("T", [1, 31, 33, 65, 130])
@pytest.mark.parametrize("which", ["config", "reference"])
def test_band_split_and_mask_row_tiles(cfg2_models, ref_models, which, T, layout):
    """Frames around the kernels' 32 and 64 row tiles, of very different level (the rows are normalised before
    they are split into fp16 pieces, so quiet frames keep their precision) and one of zeros; the mask's GLU and
    scatter on ragged row tiles, bands of 8 to 516 inputs (16-wide value and gate groups)."""
    rng = np.random.default_rng(T)
    om, dm = cfg2_models if which == "config" else ref_models
    d = om.d
    src = rng.standard_normal((d.freq_bins, d.channels, T, 2)).astype(np.float32)
    src *= (10.0 ** rng.uniform(-5, 4, T)).astype(np.float32)[None, None, :, None]
    src[:, :, T // 2] = 0.0
    ref = om.band_split(src)
    dout = empty_dev(ref.shape)
    dm.band_split(to_dev(_to_layout(src, layout)), T, dout, layout)
    assert_close(ref, from_dev(dout), rtol=1e-4, atol=2e-5, min_snr=110, what="band split")
    feats = rng.standard_normal((T, d.bands, d.dim), dtype=np.float32)
    mref = om.mask_estimate(feats)
    dmask = empty_dev(_to_layout(mref, layout).shape)
    dm.mask_estimate(to_dev(feats), T, dmask, layout)
    assert_close(mref, _from_layout(from_dev(dmask), layout), rtol=1e-4, atol=1e-5, min_snr=110, what="mask")


@pytest.mark.parametrize("which", ["config", "reference"])
def test_band_split_error_within_fp32_mfma(cfg2_models, ref_models, cfg2, ref_pack, which):
    """The pieces' products against float64: no further off than the same bands on the fp32 MFMA instruction, on normal
    spectra, on a tone mix's and on bins of very different level (the operands' 22 bits cost less than the fp32
    accumulation's roundings saved by 16-wide products)."""
    om, dm = cfg2_models if which == "config" else ref_models
    d, blob = om.d, cfg2[1] if which == "config" else ref_pack
    views, rng = pack.tensor_views(d, blob), np.random.default_rng(12)
    normal = rng.standard_normal((d.freq_bins, d.channels, 70, 2)).astype(np.float32)
    levels = (10.0 ** rng.uniform(-6, 0, normal.shape[:3])).astype(np.float32)[..., None]
    for name, src in (("normal", normal), ("tones", O.stft(d, audio.sine_mix(0.8, 5))), ("levels", normal * levels)):
        T = src.shape[2]
        ref = np.empty((d.bands, T, d.dim))
        for b, (f0, w) in enumerate(zip(d.first_frequencies(), d.band_widths)):
            v = src[f0:f0 + w].astype(np.float64).transpose(2, 0, 1, 3).reshape(T, -1)
            v *= np.sqrt(v.shape[1]) / np.sqrt((v * v).sum(1, keepdims=True) + 1e-12)
            wm = pack.unpack_matrix(views[f"bands.{b}.weight"], d.dim, v.shape[1]).astype(np.float64)
            ref[b] = (v * views[f"bands.{b}.gamma"]) @ wm.T + views[f"bands.{b}.bias"]
        err = {}
        for precision in (native.PRECISION_FP32, native.PRECISION_FP32_MFMA):
            dm.set_precision(precision)
            out = empty_dev(ref.shape)
            dm.band_split(to_dev(src), T, out)
            err[precision] = np.linalg.norm(from_dev(out) - ref) / np.linalg.norm(ref)
        dm.set_precision(native.PRECISION_FP32)
        assert err[native.PRECISION_FP32] <= err[native.PRECISION_FP32_MFMA], (name, err)


# Shapes that neither model has: other n_fft (the workgroup-per-frame transforms), 1, 3 and 8 channels, features that
# are no multiple of 32 or 16, a mask width that is no multiple of 32, bands of 2 to 640 inputs (some no multiple of 4
# or 16) and more than 96 bands (three launches of the mask's second layer).
SHAPES = {
    "mono": dict(dim=48, n_fft=1024, hop=200, channels=1, mask_hidden=80,
                 band_widths=(1,) * 9 + (2,) * 20 + (17, 33, 64, 50, 300)),
    "three": dict(dim=40, n_fft=512, hop=128, channels=3, mask_hidden=48, band_widths=(1,) * 20 + (5,) * 10 + (106, 81)),
    "eight": dict(dim=112, n_fft=128, hop=50, channels=8, mask_hidden=64, band_widths=(1,) * 25 + (40,)),
    "many": dict(dim=64, n_fft=4096, hop=700, channels=2, mask_hidden=64, band_widths=(10,) * 151 + (11,) * 49),
    "tiny": dict(dim=36, n_fft=2, hop=1, channels=2, mask_hidden=16, band_widths=(1, 1)),
}


@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("shape", sorted(SHAPES))
def test_front_and_back_end_other_shapes(ctx, shape, layout):
    d = ModelDims(depth=0, heads=1, ff_dim=64, model_frames=0, **SHAPES[shape])
    blob = pack.synthetic_pack(d, 79)
    om, dm = O.Model(d, blob), native.Model(ctx, d, blob)
    rng = np.random.default_rng(len(shape))
    length = 36 * d.hop + min(5, d.hop - 1)
    T = d.frames(length)  # 37: a whole row tile and a ragged one
    x = rng.standard_normal((d.channels, length)).astype(np.float32)
    src = O.stft(d, x)
    dsrc = empty_dev(_to_layout(src, layout).shape)
    dm.stft(to_dev(x), length, dsrc, layout)
    assert_close(src, _from_layout(from_dev(dsrc), layout), rtol=1e-6, atol=4e-6, min_snr=120, what="stft")
    mask = rng.standard_normal(src.shape).astype(np.float32)
    dout = empty_dev((d.channels, length))
    dm.istft(to_dev(_to_layout(src, layout)), to_dev(_to_layout(mask, layout)), length, dout, layout)
    assert_close(O.istft(d, src, mask, length), from_dev(dout), rtol=1e-5, atol=4e-6, min_snr=120, what="istft")
    ref = om.band_split(src)
    dout = empty_dev(ref.shape)
    dm.band_split(to_dev(_to_layout(src, layout)), T, dout, layout)
    assert_close(ref, from_dev(dout), rtol=1e-4, atol=2e-5, min_snr=110, what="band split")
    feats = rng.standard_normal((T, d.bands, d.dim), dtype=np.float32)
    ref = om.mask_estimate(feats)
    dmask = empty_dev(_to_layout(ref, layout).shape)
    dm.mask_estimate(to_dev(feats), T, dmask, layout)
    assert_close(ref, _from_layout(from_dev(dmask), layout), rtol=1e-4, atol=1e-5, min_snr=110, what="mask")
    dm.close()


@pytest.mark.parametrize("name,power", [("weight", 121), ("weight", -110), ("gamma", 118), ("gamma", -118)])
def test_band_split_outside_scale_range(ctx, name, power):
    """One band's weights or gains so large or so small that their power-of-two scale would be clamped: the fp16 pieces
    would overflow or lose bits, so the band split runs on the fp32 MFMA instruction."""
    d = CONFIG_DIMS.with_depth(0)
    blob = pack.synthetic_pack(d, 78)
    views = pack.tensor_views(d, blob)
    band = 50  # 96 inputs
    views[f"bands.{band}.{name}"] *= np.float32(2.0 ** power)
    views[f"bands.{band}.bias"] *= 0
    src = np.random.default_rng(9).standard_normal((d.freq_bins, d.channels, 40, 2)).astype(np.float32)
    ref = O.Model(d, blob).band_split(src)
    dm = native.Model(ctx, d, blob)
    dout = empty_dev(ref.shape)
    dm.band_split(to_dev(src), 40, dout)
    out = from_dev(dout)
    dm.close()
    scale = np.abs(ref).max(axis=(1, 2), keepdims=True).astype(np.float64)
    assert_close(ref / scale, out / scale, rtol=1e-4, atol=2e-5, min_snr=110, what="band split")


@pytest.mark.parametrize("precision", [0, 1, 2])
def test_stream_switch_keeps_order(ctx, cfg2_models, precision):
    """A context's calls share its scratch, so after a change of stream one waits for the last mask estimate: the end of a
    call on B implies that of one on A behind a long product, also from and to the null stream, over a block that leaves
    no end of its own, and mask estimates issued in turn on two streams give what they give on one."""
    om, dm = cfg2_models
    d, T = om.d, 301
    g = torch.Generator("cuda:0").manual_seed(31 + precision)
    feats = [torch.randn(T, d.bands, d.dim, device="cuda:0", generator=g) * s for s in (1.0, 3.0, 0.1, 2.0)]
    shape = (d.freq_bins, d.channels, T, 2)
    big = torch.randn(8192, 8192, device="cuda:0", generator=g)
    home = torch.cuda.current_stream().cuda_stream
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    dm.set_precision(precision)
    try:
        want = []
        for f in feats:
            want.append(empty_dev(shape))
            dm.mask_estimate(f, T, want[-1])
        torch.cuda.synchronize()
        out, x = empty_dev(shape), torch.randn(130, d.dim, device="cuda:0", generator=g)
        torch.cuda.synchronize()
        for first, second in ((a, b), (torch.cuda.default_stream(), b), (a, torch.cuda.default_stream())):
            ctx.set_stream(first.cuda_stream)
            with torch.cuda.stream(first):
                for _ in range(4):
                    big @ big
            dm.mask_estimate(feats[0], T, out)
            done = first.record_event()
            if first is a:
                dm.transformer(0, 0, x, 2, 65)
            ctx.set_stream(second.cuda_stream)
            dm.mask_estimate(feats[0], T, out)
            second.synchronize()
            assert done.query()  # the second call ended after the first
            assert torch.equal(out, want[0])
        got = [empty_dev(shape) for _ in feats]
        torch.cuda.synchronize()
        for i, (f, o) in enumerate(zip(feats, got)):
            ctx.set_stream((a, b)[i % 2].cuda_stream)
            dm.mask_estimate(f, T, o)
        torch.cuda.synchronize()
    finally:
        ctx.set_stream(home)
        dm.set_precision(native.PRECISION_FP32)
    for w, o in zip(want, got):
        assert torch.equal(w, o)


def test_stream_destroyed_before_the_switch(ctx, cfg2_models):
    """A stream whose work has ended may be gone when the context leaves it."""
    import ctypes
    om, dm = cfg2_models
    hip = ctypes.CDLL(next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line))
    home = torch.cuda.current_stream().cuda_stream
    feats = torch.randn(40, om.d.bands, om.d.dim, device="cuda:0", generator=torch.Generator("cuda:0").manual_seed(7))
    outs = [empty_dev((om.d.freq_bins, om.d.channels, 40, 2)) for _ in range(3)]
    dm.mask_estimate(feats, 40, outs[0])
    torch.cuda.synchronize()
    stream = ctypes.c_void_p()
    assert hip.hipStreamCreateWithFlags(ctypes.byref(stream), 1) == 0
    ctx.set_stream(stream.value)
    dm.mask_estimate(feats, 40, outs[1])
    torch.cuda.synchronize()  # not vh_synchronize: the context does not know
    assert hip.hipStreamDestroy(stream) == 0
    ctx.set_stream(home)
    dm.mask_estimate(feats, 40, outs[2])
    torch.cuda.synchronize()
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])


def test_short_windows_share_row_tiles(cfg2_models):
    """Windows of 11 frames, up to nine in a pass: a row tile of the band split and of the mask's second layer, and a
    wave of the projection, span several windows.  Against the same windows one at a time: the values differ only by
    the operand scales, which follow the pass's largest value."""
    om, dm = cfg2_models
    x = audio.sine_mix(0.5, 21)
    length, chunk, step = x.shape[1], 4410, 2205
    outs = []
    for batch in (9, 1):
        dv = empty_dev(x.shape)
        dm.separate(to_dev(x), length, chunk, step, batch, dv)
        outs.append(from_dev(dv))
    assert_close(outs[1], outs[0], rtol=1e-4, atol=1e-6, min_snr=110, what="windows together")


def test_forward_config_shape(cfg2_models):
    om, dm = cfg2_models
    x = audio.sine_mix(0.5, 11)
    ref = om.forward(x)
    dv, di = empty_dev(x.shape), empty_dev(x.shape)
    dm.forward(to_dev(x), x.shape[1], dv, di)
    out = from_dev(dv)
    err = float(np.max(np.abs(out.astype(np.float64) - ref)))
    print(f"forward (dim 384, depth 2, 0.5 s): max|d| {err:.3e}, SNR {snr_db(ref, out):.1f} dB")
    assert err <= 1e-4, err
    assert snr_db(ref, out) >= 80
    # instrumental = mix - vocals, computed on the device from the same vocals
    assert np.array_equal(from_dev(di), x - out)


def test_forward_band_unfused(cfg2_models, monkeypatch):
    """The whole forward with the band axis on the two separate kernels
    (VOCALARC_BAND_FUSED=0: the QKV GEMM, then attention_short_h2_kernel)
    against the oracle and against the default, fused path: the path the
    pipeline no longer takes by default stays at the parity bar."""
    om, dm = cfg2_models
    x = audio.sine_mix(0.5, 13)
    ref = om.forward(x)
    outs = []
    for env in ("0", None):
        if env is None:
            monkeypatch.delenv("VOCALARC_BAND_FUSED", raising=False)
        else:
            monkeypatch.setenv("VOCALARC_BAND_FUSED", env)
        dv = empty_dev(x.shape)
        dm.forward(to_dev(x), x.shape[1], dv)
        outs.append(from_dev(dv))
    monkeypatch.delenv("VOCALARC_BAND_FUSED", raising=False)
    for out in outs:
        assert float(np.max(np.abs(out.astype(np.float64) - ref))) <= 1e-4
        assert snr_db(ref, out) >= 80
    assert snr_db(outs[0], outs[1]) >= 110


def test_forward_reference_shape(ref_models):
    om, dm = ref_models
    x = audio.sine_mix(0.2, 12)
    ref = om.forward(x)
    dv = empty_dev(x.shape)
    dm.forward(to_dev(x), x.shape[1], dv)
    out = from_dev(dv)
    err = float(np.max(np.abs(out.astype(np.float64) - ref)))
    print(f"forward (reference shape, depth 16, 0.2 s): max|d| {err:.3e}, SNR {snr_db(ref, out):.1f} dB")
    assert err <= 1e-4, err
    assert snr_db(ref, out) >= 80


def test_chunked_separation(ctx):
    d = CONFIG_DIMS.with_depth(1)
    blob = pack.synthetic_pack(d, 91)
    om, dm = O.Model(d, blob), native.Model(ctx, d, blob)
    x = audio.sine_mix(1.0, 13)
    chunk, step = 13230, 8820  # 0.3 s windows every 0.2 s -> 5 chunks
    ref = om.separate_chunked(x, chunk, step)
    dv, di = empty_dev(x.shape), empty_dev(x.shape)
    dm.separate(to_dev(x), x.shape[1], chunk, step, 2, dv, di)
    out = from_dev(dv)
    assert O.chunk_count(x.shape[1], chunk, step) == 5
    assert np.array_equal(from_dev(di), x - out)
    err = float(np.max(np.abs(out.astype(np.float64) - ref)))
    print(f"chunked separation (5 windows, batch 2): max|d| {err:.3e}, SNR {snr_db(ref, out):.1f} dB")
    assert err <= 1e-4, err
    assert snr_db(ref, out) >= 80
