"""The native vocoder frame step against the CPU oracle and against vectors written from the
reference's own classes (through the C ABI, fp32)."""
import dataclasses
import os

import numpy as np
import pytest
import torch

from oracle import codec_oracle as O

pytestmark = pytest.mark.gpu
GOLD = os.path.join(os.path.dirname(__file__), "golden")
TOL = 2e-4  # absolute, on audio in [-1, 1] (fp32 sums in another order through ~60 layers)


def small_dims():
    return O.CodecDims(n_codebooks=4, codebook_size=32, codebook_dim=16, vq_dim=32, latent_dim=64, d_model=32,
                       n_layers=2, n_heads=2, head_dim=16, mlp_dim=64, max_seq=40, up_ratios=(2, 2),
                       decoder_dim=128, rates=(3, 2))


def native(d, sd):
    from vui_amd.codec import CodecConfig, QwenCodecDecoder

    return QwenCodecDecoder(sd, CodecConfig(**dataclasses.asdict(d)), device="cuda")


@pytest.fixture(scope="module")
def small():
    d = small_dims()
    sd = O.synthetic_codec_state_dict(d, seed=4)
    return d, O.CodecDecoderOracle(d, sd), native(d, sd)


@pytest.fixture(scope="module")
def full():
    d = O.CodecDims()
    sd = O.synthetic_codec_state_dict(d, seed=0)
    fx = {k: torch.from_numpy(v) for k, v in np.load(os.path.join(GOLD, "codec_full.npz")).items()}
    return d, sd, native(d, sd), fx


def err(a, b):
    return float((a.detach().cpu().float() - b.float()).abs().max())


def test_small_stream_frame_by_frame(small):
    d, ora, dec = small
    g = torch.Generator().manual_seed(1)
    codes = torch.randint(0, d.codebook_size, (1, d.n_codebooks, 14), generator=g)
    ora.open_stream()
    with dec.streaming(1):
        for t in range(codes.shape[2]):
            ref = ora.forward(codes[:, :, t:t + 1])
            got = dec(codes[:, :, t:t + 1].cuda())
            assert got.shape == (1, 1, d.hop)
            assert err(got, ref) < TOL, (t, err(got, ref))
        assert dec.frames_since_reset() == 14
    ora.close_stream()
    assert float(ref.abs().max()) > 0.05  # the comparison is not about silence


def test_small_offline_chunk_and_fewer_codebooks(small):
    d, ora, dec = small
    g = torch.Generator().manual_seed(2)
    codes = torch.randint(0, d.codebook_size, (1, d.n_codebooks, 9), generator=g)
    assert err(dec(codes.cuda()), ora.forward(codes)) < TOL
    assert err(dec(codes[:, :2].cuda()), ora.forward(codes[:, :2])) < TOL
    assert err(dec(codes[:, :1].cuda()), ora.forward(codes[:, :1])) < TOL
    # an offline call leaves the state cold: the same call again gives the same audio
    a = dec(codes.cuda()).clone()
    assert err(dec(codes.cuda()), a.cpu()) == 0.0
    with dec.streaming(1):
        with pytest.raises(AssertionError):
            dec.streaming(1)


def test_small_reset_restarts_cold(small):
    d, ora, dec = small
    g = torch.Generator().manual_seed(3)
    codes = torch.randint(0, d.codebook_size, (1, d.n_codebooks, 5), generator=g).cuda()
    with dec.streaming(1):
        first = torch.cat([dec(codes[:, :, t:t + 1]).clone() for t in range(5)], dim=-1)
        dec.reset_streaming()
        again = torch.cat([dec(codes[:, :, t:t + 1]).clone() for t in range(5)], dim=-1)
    assert err(first, again.cpu()) == 0.0


def test_small_graph_replays_equal_eager(small):
    d, ora, dec = small
    g = torch.Generator().manual_seed(5)
    codes = torch.randint(0, d.codebook_size, (1, d.n_codebooks, 7), generator=g).cuda()
    with dec.streaming(1):
        eager = [dec(codes[:, :, t:t + 1]).clone() for t in range(7)]
    dec.setup_streaming_graph(1)
    try:
        with dec.streaming(1):
            for t in range(7):
                got = dec(codes[:, :, t:t + 1])
                torch.cuda.synchronize()
                assert err(got, eager[t].cpu()) == 0.0, t
    finally:
        dec._graphs.clear()


def test_persistent_trunk_equals_kernel_sequence(small):
    """The one-column steps run as one persistent kernel by default; switched off they are separate
    launches.  Same sums in another order."""
    d, ora, dec = small
    assert dec.persistent()
    g = torch.Generator().manual_seed(8)
    codes = torch.randint(0, d.codebook_size, (1, d.n_codebooks, 12), generator=g).cuda()
    a = dec(codes).clone()
    try:
        assert not dec.persistent(0)
        b = dec(codes).clone()
        assert err(a, b.cpu()) < 2e-5
        assert err(dec(codes[:, :2]), ora.forward(codes[:, :2].cpu())) < TOL
    finally:
        assert dec.persistent(1)


@pytest.mark.parametrize("nwg", [96, 128, 40])
def test_persistent_trunk_on_fewer_workgroups(small, full, nwg):
    """vui_codec_workgroups: the persistent kernel on part of the GPU (more rows of every matrix per workgroup, the
    row plan of its second instantiation) against the oracle at reduced dims and against the reference's own vectors
    at the real dims; 40 workgroups cannot hold the real model's rows and are refused there."""
    d, ora, dec = small
    g = torch.Generator().manual_seed(9)
    codes = torch.randint(0, d.codebook_size, (1, d.n_codebooks, 12), generator=g).cuda()
    try:
        dec.workgroups(nwg)
        assert dec.persistent()
        assert err(dec(codes), ora.forward(codes.cpu())) < TOL
    finally:
        dec.workgroups(256)
    df, sdf, decf, fx = full
    try:
        if nwg < 96:
            with pytest.raises(RuntimeError, match="rows per wave"):
                decf.workgroups(nwg)
            return
        decf.workgroups(nwg)
        codes = fx["codes"].cuda()
        with decf.streaming(1):
            st = torch.cat([decf(codes[:, :, t:t + 1]).clone() for t in range(codes.shape[2])], dim=-1)
        assert err(st, fx["stream"]) < TOL, err(st, fx["stream"])
    finally:
        decf.workgroups(256)


def test_errors_are_reported(small):
    d, ora, dec = small
    bad = torch.full((1, d.n_codebooks, 1), d.codebook_size, dtype=torch.long).cuda()
    with dec.streaming(1):
        dec(bad)
        with pytest.raises(RuntimeError, match="outside"):
            dec.frames_since_reset()
    with pytest.raises(ValueError):
        dec(torch.zeros(1, d.n_codebooks + 1, 1, dtype=torch.long).cuda())
    with pytest.raises(ValueError, match="window"):
        dec(torch.zeros(1, d.n_codebooks, d.max_seq + 1, dtype=torch.long).cuda())
    # a stream longer than the cache: flagged, nothing out of bounds
    with dec.streaming(1):
        z = torch.zeros(1, d.n_codebooks, 1, dtype=torch.long).cuda()
        for _ in range(d.max_seq + 1):
            dec(z)
        with pytest.raises(RuntimeError, match="max_seq"):
            dec.frames_since_reset()


def test_unsupported_dims_raise():
    from vui_amd.codec import CodecConfig, QwenCodecDecoder

    with pytest.raises(ValueError, match="multiple of 32"):
        QwenCodecDecoder({}, CodecConfig(latent_dim=24), device="cuda")


def test_full_dims_against_reference_vectors(full):
    d, sd, dec, fx = full
    codes = fx["codes"].cuda()
    with dec.streaming(1):
        st = torch.cat([dec(codes[:, :, t:t + 1]).clone() for t in range(codes.shape[2])], dim=-1)
    assert err(st, fx["stream"]) < TOL, err(st, fx["stream"])
    assert err(dec(codes), fx["offline"]) < TOL
    assert err(dec(codes[:, :8, :2]), fx["offline_q8"]) < TOL
    assert st.shape[-1] == 4 * 1920


@pytest.mark.parametrize("T", [33, 65, 250])
def test_clips_in_one_pass(full, T, monkeypatch):
    """A clip of more frames than a block, up to the decoder's window, against the same frames streamed in portions of 32; where
    its memory cannot be had, in shorter passes.  Each is within 6e-6 to 9e-6 of 64 bits at 93 frames (2 seeds); 5e-5 is three times
    what two of them can differ by."""
    d, sd, dec, _ = full
    codes = torch.randint(0, d.codebook_size, (1, d.n_codebooks, T), generator=torch.Generator().manual_seed(T)).cuda()
    whole = dec(codes).clone()
    with dec.streaming(1):
        parts = torch.cat([dec(codes[:, :, i:i + 32]).clone() for i in range(0, T, 32)], dim=-1)
    assert float(whole.abs().max()) > 0.05 and err(whole, parts.cpu()) < 5e-5
    empty, refused = torch.empty, []

    def short(*size, **kw):
        if kw.get("dtype") == torch.uint8 and size[0] > 260e6:
            refused.append(size[0])
            raise torch.OutOfMemoryError("no room")
        return empty(*size, **kw)

    monkeypatch.setattr(torch, "empty", short)
    assert err(dec(codes), parts.cpu()) < 5e-5 and refused


def test_memory_of_clips_that_grow(full):
    """Clips of growing lengths share the scratch memory of 64 and of 128 frames (8 MB each, 1.6 GB) instead of leaving one buffer per length
    behind (7 GB for these)."""
    d, sd, dec, fx = full
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    before = torch.cuda.memory_reserved()
    for T in range(40, 121, 8):
        dec(torch.zeros(1, d.n_codebooks, T, dtype=torch.long, device="cuda"))
    torch.cuda.synchronize()
    assert torch.cuda.memory_reserved() - before < 1.8e9


def _digest(a):
    a = a.detach().cpu().reshape(-1).double()
    return np.array([a.sum().item(), a.abs().sum().item(), *a[:4].tolist(), *a[-4:].tolist()])


def test_full_dims_codec_ctx_session(full):
    """The reference's CodecCtx session: prompt 30 + 10 added, prefill seeds 40 frames, 90 streamed
    frames with the cold restart after 125."""
    from vui_amd.codec import CodecCtx

    d, sd, dec, fx = full
    ctx = CodecCtx(dec)
    ctx.set_prompt(fx["ctx_prompt"])
    ctx.add(fx["ctx_extra"])
    ctx.prefill()
    assert ctx._frames_since_prefill == 40
    frames = fx["ctx_frames"].cuda()
    for t in range(frames.shape[0]):
        a = ctx.decode_frame(frames[t].view(1, -1, 1))
        assert ctx._frames_since_prefill == int(fx["ctx_fsp"][t])
        got, ref = _digest(a), fx["ctx_digest"][t].numpy()
        assert abs(got[0] - ref[0]) < 0.1 and abs(got[1] - ref[1]) < 0.1, (t, got[:2], ref[:2])
        assert np.abs(got[2:] - ref[2:]).max() < 5e-4, t
    assert ctx.n_frames == 130
    ctx.reset()
    assert not dec.is_streaming


@pytest.mark.parametrize("T", [2, 3, 31, 32, 33, 40])
def test_blocks_of_frames_equal_single_frames(small, T):
    """Offline calls take their frames in one pass here (up to the decoder's window of 40): against the oracle, and against the same
    frames one at a time (fp32 sums in another order through ~60 layers: 2e-5, measured 2e-6), whatever is in the rings from before."""
    d, ora, dec = small
    codes = torch.randint(0, d.codebook_size, (1, d.n_codebooks, T), generator=torch.Generator().manual_seed(T))
    ref = ora.forward(codes)
    got = dec(codes.cuda())
    with dec.streaming(1):
        one = torch.cat([dec(codes[:, :, t:t + 1].cuda()).clone() for t in range(T)], dim=-1)
    assert err(got, ref) < TOL and err(got, one.cpu()) < 2e-5


@pytest.mark.parametrize("T", [33, 40])
def test_offline_calls_of_several_passes(small, T, monkeypatch):
    """Calls of more frames than a pass takes: two passes of 17 and 16 or of 20 frames, with the bounds of the test above."""
    d, ora, dec = small
    monkeypatch.setattr(dec, "_clip", dec._block)
    codes = torch.randint(0, d.codebook_size, (1, d.n_codebooks, T), generator=torch.Generator().manual_seed(T))
    got = dec(codes.cuda())
    with dec.streaming(1):
        one = torch.cat([dec(codes[:, :, t:t + 1].cuda()).clone() for t in range(T)], dim=-1)
    assert err(got, ora.forward(codes)) < TOL and err(got, one.cpu()) < 2e-5


def test_block_entry(small):
    """vui_codec_decode_block, which callers of the C ABI have beside the clip's: as many frames as a block takes are decoded to the
    same samples, more are refused, and too little scratch memory is."""
    import ctypes as C

    d, ora, dec = small
    lib, st = dec.lib, torch.cuda.current_stream().cuda_stream
    codes = torch.randint(0, d.codebook_size, (1, d.n_codebooks, 33), generator=torch.Generator().manual_seed(12)).cuda()
    rows = codes[0].t().contiguous()
    size = [int(lib.vui_codec_block_scratch_bytes(C.byref(dec._cc), n)) for n in (2, 32)]
    scratch = torch.empty(2 * size[1], dtype=torch.uint8, device="cuda")

    def block(n, room):
        audio = torch.empty(n * d.hop, device="cuda")
        dec.reset_streaming()
        return lib.vui_codec_decode_block(dec.handle, rows.data_ptr(), n, d.n_codebooks, audio.data_ptr(), scratch.data_ptr(), room, st), audio

    for n, room in zip((2, 32), size):
        rc, audio = block(n, room)
        assert rc == 0 and torch.equal(audio, dec(codes[:, :, :n].contiguous()).view(-1)), n
    assert block(33, scratch.numel())[0] == block(0, scratch.numel())[0] == -22 and block(32, size[1] - 1)[0] == -12
    dec.reset_streaming()


def test_blocks_and_single_frames_in_one_stream(small):
    """A stream may change between blocks and single frames anywhere; past max_seq frames only the flag is raised."""
    d, ora, dec = small
    codes = torch.randint(0, d.codebook_size, (1, d.n_codebooks, d.max_seq + 2), generator=torch.Generator().manual_seed(6)).cuda()
    with dec.streaming(1):
        one = torch.cat([dec(codes[:, :, t:t + 1]).clone() for t in range(d.max_seq)], dim=-1)
        assert dec.frames_since_reset() == d.max_seq
    with dec.streaming(1):
        parts, t = [], 0
        for n in (1, 2, 5, 1, 1, 16, 3, 9, 2):
            parts.append(dec(codes[:, :, t:t + n]).clone())
            t += n
        assert t == d.max_seq and dec.frames_since_reset() == t
    assert err(torch.cat(parts, dim=-1), one.cpu()) < 2e-5
    with dec.streaming(1):
        got = dec(codes)  # two frames more than fit
        assert err(got[..., :one.shape[-1]], one.cpu()) < 2e-5
        with pytest.raises(RuntimeError, match="max_seq"):
            dec.frames_since_reset()


def test_full_dims_blocks_equal_single_frames(full):
    d, sd, dec, fx = full
    codes = torch.randint(0, d.codebook_size, (1, d.n_codebooks, 45), generator=torch.Generator().manual_seed(7)).cuda()
    got = dec(codes)
    for n in (True, False):
        try:
            dec.persistent(int(n))
            with dec.streaming(1):
                one = torch.cat([dec(codes[:, :, t:t + 1]).clone() for t in range(codes.shape[2])], dim=-1)
        finally:
            dec.persistent(1)
        assert err(got, one.cpu()) < 5e-5  # measured 1e-5


def scaled(sd, power):
    """The last product of both upsampling blocks' feed-forwards times a power of two, its scale by the inverse."""
    other = dict(sd)
    for i in range(2):
        for k in ("pwconv2.weight", "pwconv2.bias"):
            other[f"upsample.{i}.1.{k}"] = sd[f"upsample.{i}.1.{k}"] * 2.0 ** power
        other[f"upsample.{i}.1.gamma"] = sd[f"upsample.{i}.1.gamma"] * 2.0 ** -power
    return other


@pytest.mark.parametrize("power", [-104, -60, -20, 20, 60, 120])
def test_wide_products_of_any_magnitude(full, power):
    """Parts of an operand keep its exponent: scaled weights give the same audio from blocks of frames, bit by bit as long as the least
    products are above fp32's least normal number (power-of-two factors pass through every sum of the three parts).  Weights of 2^-110
    keep their three parts; the products' last bits are subnormal (the limit: other orders of the sums differ by 1e-5)."""
    d, sd, dec, fx = full
    codes = torch.randint(0, d.codebook_size, (1, d.n_codebooks, 35), generator=torch.Generator().manual_seed(9)).cuda()
    got, want = native(d, scaled(sd, power))(codes), dec(codes)
    assert err(got, want.cpu()) < 5e-5 if power < -90 else torch.equal(got, want)


def test_wide_products_near_the_largest_number(full):
    """Weights between bf16's largest number and fp32's (1.998 and -1.9999 x 2^127) are finite and count as what they are."""
    d, sd, dec, fx = full
    sd = dict(sd)
    for i in range(2):
        for k in ("pwconv1.weight", "pwconv1.bias"):  # small hidden values: no product reaches infinity
            sd[f"upsample.{i}.1.{k}"] = sd[f"upsample.{i}.1.{k}"] * 2.0 ** -6
        sd[f"upsample.{i}.1.gamma"] = sd[f"upsample.{i}.1.gamma"] * 16  # ... and 2^-127 of it is normal
        w = sd[f"upsample.{i}.1.pwconv2.weight"].clone()
        w[::3, ::7], w[1::3, 1::5] = 1.998, -1.9999
        sd[f"upsample.{i}.1.pwconv2.weight"] = w
    codes = torch.randint(0, d.codebook_size, (1, d.n_codebooks, 35), generator=torch.Generator().manual_seed(9)).cuda()
    want, big = native(d, sd)(codes), scaled(sd, 127)
    assert float(big["upsample.0.1.pwconv2.weight"].abs().max()) > float(torch.finfo(torch.bfloat16).max)
    got = native(d, big)(codes)
    assert err(got, want.cpu()) < 5e-5  # measured 1e-5: the parts of the planted weights are others


@pytest.mark.parametrize("powers", [(0, 6, -6, 11, -2), (-12, 2, 3, 0, -1), (9,)])
def test_wide_products_of_groups_of_different_size(full, powers):
    """The feed-forwards' inputs times a power of two per group of 32 channels and their weights by the inverse give the same audio (the bound is
    that of other orders of the sums)."""
    d, sd, dec, fx = full
    sd = dict(sd)
    for i in range(2):
        p = f"upsample.{i}.1."
        n = sd[p + "norm.weight"].shape[0]
        f = 2.0 ** torch.tensor([powers[c // 32 % len(powers)] for c in range(n)], dtype=torch.float32)
        for k in ("norm.weight", "norm.bias"):
            sd[p + k] = sd[p + k] * f
        sd[p + "pwconv1.weight"] = sd[p + "pwconv1.weight"] / f
    codes = torch.randint(0, d.codebook_size, (1, d.n_codebooks, 35), generator=torch.Generator().manual_seed(9)).cuda()
    assert err(native(d, sd)(codes), dec(codes).cpu()) < 5e-5


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_a_frame_that_is_not_finite_leaves_those_before_it(full, bad):
    """What is not finite does not count in the scale of the columns beside it.  (The last layer's clamp makes a NaN -1.)"""
    d, sd, dec, fx = full
    sd = dict(sd)
    key = "quantizer.semantic.codebooks.0.embed"
    sd[key] = sd[key].clone()
    sd[key][5] = bad
    codes = torch.randint(6, d.codebook_size, (1, d.n_codebooks, 35), generator=torch.Generator().manual_seed(9)).cuda()
    want = dec(codes)
    codes[0, 0, 17] = 5
    got = native(d, sd)(codes)
    n = 17 * (want.shape[-1] // 35)
    assert err(got[..., :n], want[..., :n].cpu()) < 5e-5 and bool((got[..., n:] == -1).all())


def by_channel(sd, powers):
    """The same network with the columns of the wide products' inputs times powers of two, their weights by the inverse: both feed-forwards' inputs, and
    the second upsampling block's output, which the first 7-tap convolution reads."""
    sd = dict(sd)
    n = sd["upsample.0.1.norm.weight"].shape[0]
    f = 2.0 ** torch.tensor([powers[c % len(powers)] for c in range(n)], dtype=torch.float32)
    for i in range(2):
        p = f"upsample.{i}.1."
        for k in ("norm.weight", "norm.bias"):
            sd[p + k] = sd[p + k] * f
        sd[p + "pwconv1.weight"] = sd[p + "pwconv1.weight"] / f
    sd["upsample.1.0.conv.weight"] = sd["upsample.1.0.conv.weight"] * f[:, None]
    sd["upsample.1.0.conv.bias"] = sd["upsample.1.0.conv.bias"] * f
    sd["upsample.1.1.dwconv.conv.weight"] = sd["upsample.1.1.dwconv.conv.weight"] / f[:, None, None]
    sd["upsample.1.1.gamma"] = sd["upsample.1.1.gamma"] * f
    sd["decoder.0.conv.weight"] = sd["decoder.0.conv.weight"] / f[:, None]
    return sd


@pytest.mark.parametrize("powers", [(20, -20), (0, 0, 0, 30, 0, 0, -30)])
def test_wide_products_of_channels_of_different_size(full, powers):
    """Every operand keeps an exponent of its own: channels of any magnitude beside each other give the same bits."""
    d, sd, dec, fx = full
    codes = torch.randint(0, d.codebook_size, (1, d.n_codebooks, 35), generator=torch.Generator().manual_seed(9)).cuda()
    assert torch.equal(native(d, by_channel(sd, powers))(codes), dec(codes))


@pytest.mark.parametrize("power", [20, 30])
def test_wide_products_of_rows_of_different_size(full, power):
    """Rows of a matrix times powers of two, the inverse in the scale behind the product: the same bits."""
    d, sd, dec, fx = full
    other = dict(sd)
    for i in range(2):
        p = f"upsample.{i}.1."
        f = 2.0 ** torch.tensor([(power, -power, 0, 0, 0)[m % 5] for m in range(sd[p + "gamma"].shape[0])], dtype=torch.float32)
        other[p + "pwconv2.weight"] = sd[p + "pwconv2.weight"] * f[:, None]
        other[p + "pwconv2.bias"] = sd[p + "pwconv2.bias"] * f
        other[p + "gamma"] = sd[p + "gamma"] / f
    codes = torch.randint(0, d.codebook_size, (1, d.n_codebooks, 35), generator=torch.Generator().manual_seed(9)).cuda()
    assert torch.equal(native(d, other)(codes), dec(codes))


@pytest.mark.parametrize("power, bound", [(30, 5e-5), (48, 5e-5), (62, 1e-2)])
def test_wide_products_of_two_small_operands(full, power, bound):
    """Inputs and weights of the second upsampling product times 2^-power each.  At 48 the least of the six products that count, 2^-16 of 2^-96, are
    normal numbers: the bound is that of other orders of the sums.  At 62 products themselves are below 2^-126, where bits go from the parts' products on
    (2^-8 of a product and less), while the sums, 2^-122, are normal numbers."""
    d, sd, dec, fx = full
    sd = dict(sd)
    small, least, large = 2.0 ** -power, 2.0 ** (-2 * power), 2.0 ** (2 * power)
    for k, f in (("upsample.0.0.conv.weight", small), ("upsample.0.0.conv.bias", small), ("upsample.0.1.dwconv.conv.weight", 1 / small),
                 ("upsample.0.1.gamma", small), ("upsample.1.0.conv.weight", small), ("upsample.1.0.conv.bias", least),
                 ("upsample.1.1.dwconv.conv.weight", large), ("upsample.1.1.gamma", least), ("decoder.0.conv.weight", large)):
        sd[k] = sd[k] * f
    codes = torch.randint(0, d.codebook_size, (1, d.n_codebooks, 35), generator=torch.Generator().manual_seed(9)).cuda()
    assert err(native(d, sd)(codes), dec(codes).cpu()) < bound


@pytest.mark.parametrize("power", [0, 4, 30, 40])
def test_a_loud_frame_leaves_those_before_it(full, power):
    """A code that alone reaches one channel of the trunk, which its norm takes times 2^power: not a bit of the frames before it changes."""
    d, sd, dec, fx = full
    sd = {k: v.clone() for k, v in sd.items()}
    for k, v in sd.items():  # feature 0 of the first codebook goes through row 0 of each layer alone
        if k.startswith("quantizer.") and k.endswith("embed"):
            v[:, 0] = 0
        elif k.endswith(("output_proj.weight", "pre_conv.conv.weight", "pre_transformer.input_proj.weight")) and "pre_transformer.output" not in k:
            v[0], v[:, 0] = 0, 0
        elif k in ("pre_conv.conv.bias", "pre_transformer.input_proj.bias") or k.endswith(("attn_scale", "mlp_scale")):
            v[0] = 0
    sd["quantizer.semantic.codebooks.0.embed"][5, 0] = 100
    sd["quantizer.semantic.output_proj.weight"][0, 0] = 1
    sd["pre_conv.conv.weight"][0, 0, -1] = 1
    sd["pre_transformer.input_proj.weight"][0, 0] = 1
    sd["pre_transformer.norm.weight"][0] = 2.0 ** power
    dec = native(d, sd)
    codes = torch.randint(6, d.codebook_size, (1, d.n_codebooks, 35), generator=torch.Generator().manual_seed(9)).cuda()
    want = dec(codes)
    codes[0, 0, 17] = 5
    got = dec(codes)
    n = 17 * (want.shape[-1] // 35)
    assert torch.equal(got[..., :n], want[..., :n]) and not torch.equal(got[..., n:], want[..., n:])


def test_snake_activations_of_large_arguments(small):
    """Arguments on both sides of where the activation's own sine ends, up to where a float has no fraction left: channels that a bias alone makes, each with
    a scale that shows its sine; a clip and a stream against the oracle."""
    d, _, _ = small
    sd = {k: v.clone() for k, v in O.synthetic_codec_state_dict(d, seed=4).items()}
    t = torch.tensor([24999.0, 24999.998, 25000.0, 25000.002, -24999.5, -25001.5, 3.1e4, -4.7e5, 2.6e7, 5.3e7, -1.0e8, 7.0])
    n, block = len(t), "decoder.1.block."
    sd["decoder.0.conv.weight"][:n], sd["decoder.0.conv.bias"][:n] = 0, t
    sd[block + "0.alpha"][:n], sd[block + "0.beta"][:n] = 0, -t.abs().log()
    sd[block + "1.conv.weight"][:n] /= t.abs()[:, None, None]
    ora, dec = O.CodecDecoderOracle(d, sd), native(d, sd)
    codes = torch.randint(0, d.codebook_size, (1, d.n_codebooks, 33), generator=torch.Generator().manual_seed(3))
    ref = ora.forward(codes)
    assert err(dec(codes.cuda()), ref) < TOL
    with dec.streaming(1):
        one = torch.cat([dec(codes[:, :, i:i + 1].cuda()).clone() for i in range(33)], dim=-1)
    assert err(one, ref) < TOL


@pytest.mark.parametrize("d_model", [1024, 1312, 2048])
def test_blocks_of_wide_pre_transformers(d_model):
    """Widths whose normed products take eight waves (25-48 units of 32 channels from 17 frames on, 33-64 below) or split
    units: every block length around the 16-column tiles against the oracle and against single frames (2e-5 as above)."""
    d = dataclasses.replace(small_dims(), d_model=d_model)
    sd = O.synthetic_codec_state_dict(d, seed=5)
    ora, dec = O.CodecDecoderOracle(d, sd), native(d, sd)
    for T in (2, 16, 17, 32):
        codes = torch.randint(0, d.codebook_size, (1, d.n_codebooks, T), generator=torch.Generator().manual_seed(T))
        got = dec(codes.cuda())
        with dec.streaming(1):
            one = torch.cat([dec(codes[:, :, t:t + 1].cuda()).clone() for t in range(T)], dim=-1)
        assert err(got, ora.forward(codes)) < TOL and err(got, one.cpu()) < 2e-5, T


@pytest.mark.parametrize("latent, dim, rates", [(96, 1408, (5, 3)), (64, 128, (16, 5)), (1120, 256, (2, 2))])
def test_tiles_of_few_columns(latent, dim, rates):
    """Channel groups that do not divide into the workgroups' shares or chunks (44, 22, 11, 35 of 32 channels), tiles of one to
    four blocks of columns with the last one cut short, single frames and blocks of two and three."""
    d = dataclasses.replace(small_dims(), latent_dim=latent, decoder_dim=dim, rates=rates)
    sd = O.synthetic_codec_state_dict(d, seed=6)
    ora, dec = O.CodecDecoderOracle(d, sd), native(d, sd)
    codes = torch.randint(0, d.codebook_size, (1, d.n_codebooks, 7), generator=torch.Generator().manual_seed(3))
    ref = ora.forward(codes)
    with dec.streaming(1):
        got = [dec(codes[:, :, t:t + 1].cuda()).clone() for t in range(2)] + [dec(codes[:, :, 2:4].cuda()).clone(), dec(codes[:, :, 4:].cuda()).clone()]
    assert err(torch.cat(got, dim=-1), ref) < TOL


def test_memory_of_a_call_follows_its_frames(full):
    """A call of a few frames allocates scratch memory for those (8 MB each), not for the longest block; a call of one none."""
    d, sd, dec, fx = full
    codes = torch.randint(0, d.codebook_size, (1, d.n_codebooks, 3), generator=torch.Generator().manual_seed(8)).cuda()
    torch.cuda.synchronize()
    for T, most in ((1, 2 ** 20), (2, 17e6), (3, 26e6)):
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        dec(codes[:, :, :T].contiguous())
        assert torch.cuda.max_memory_allocated() - before < most
