"""Prompt ingestion in one pass per layer (vui_prefill) against the oracle's bf16 regime and against the
position-by-position path of the same library.  Reference: Decoder.forward_flash with T > 1 /
Engine._prefill_emb (src/vui/model.py:534-549, engine.py:674-694)."""
import pytest
import torch

from oracle import vui_oracle as O
from tests.util import TINY_SD, make_model, rel_err

pytestmark = pytest.mark.gpu
BF, F32 = torch.bfloat16, torch.float32
BF16_TOL = 2.0 ** -5  # 8 bf16 ulps of the largest value, as for the decode step


def _dims(kv):
    # head_dim 32 (the pass needs multiples of 32), ffn 512
    return O.Dims(d_model=128, n_layers=3, n_heads=4, n_kv_heads=kv, n_quantizers=4, codebook_size=32, rq_d_model=64,
                  rq_n_layers=1, rq_n_heads=2, vocab_size=50, max_seqlen=256)


@pytest.mark.parametrize("kv", [4, 2])
def test_prefill_pass_vs_oracle_and_stepwise(kv):
    d = _dims(kv)
    sd = O.synthetic_state_dict(d, **TINY_SD)
    sdb = {k: O.rnd(v, BF) for k, v in sd.items()}
    o = O.OracleModel(d, sdb, BF, n_slots=2, max_seqlen=256)
    of = O.OracleModel(d, sdb, F32, n_slots=2, max_seqlen=256)
    m = make_model(d, sd, BF, max_seqlen=256)
    m.decoder.allocate_flash_kv_cache(2, m.device, BF)
    seq = m.decoder.flash_kv_caches[0].seq_lens
    g = torch.Generator().manual_seed(11)
    blocks = [O.rnd(torch.randn(T, d.d_model, generator=g) * 0.5, BF) for T in (37, 70, 5)]  # 70 crosses a 64-row tile
    slot = torch.tensor([1], dtype=torch.int32, device="cuda")
    pos = 0
    for emb in blocks:
        ref = o.prefill(emb, slot=1)
        ref32 = of.prefill(emb, slot=1)
        got = m.decoder.forward_flash(emb[None].to(BF).cuda(), None, slot_idx=slot)[0]
        pos += emb.shape[0]
        assert int(seq[1]) == pos and int(seq[0]) == 0
        assert rel_err(got, ref) <= BF16_TOL, rel_err(got, ref)
        assert rel_err(got, ref32) <= 1.3 * rel_err(ref, ref32) + 2.0 ** -8
    # cache rows written by the pass: in layer 0 only the summation order inside the dot products differs from
    # the oracle (a bf16 rounding flips here and there, by one ulp), deeper layers within the tolerance
    for l in range(d.n_layers):
        for mine, theirs in ((m.decoder._k, o.k_cache), (m.decoder._v, o.v_cache)):
            a, b = mine[l, 1, :pos].float().cpu(), theirs[l, 1, :pos]
            if l == 0:
                assert float((a != b).float().mean()) < 0.01
                assert float(((a - b).abs() / b.abs().clamp_min(1e-3)).max()) <= 2.0 ** -7
            assert rel_err(a, b) <= BF16_TOL
    assert float(m.decoder._k[:, 0].abs().sum()) == 0  # the other slot is untouched

    # the same blocks position by position through the decode step
    m2 = make_model(d, sd, BF, max_seqlen=256)
    m2.decoder.allocate_flash_kv_cache(2, m2.device, BF)
    m2.decoder.PREFILL_MIN = 10 ** 9
    outs = [m2.decoder.forward_flash(e[None].to(BF).cuda(), None, slot_idx=slot)[0] for e in blocks]
    m.decoder.flash_kv_caches[0].seq_lens[1] = 0
    m.decoder.PREFILL_CHUNK = 32  # several chunks per block
    for e, want in zip(blocks, outs):
        got = m.decoder.forward_flash(e[None].to(BF).cuda(), None, slot_idx=slot)[0]
        assert rel_err(got, want) <= BF16_TOL, rel_err(got, want)
    # a decode step after either prefill sees equivalent caches
    codes = torch.randint(0, d.codebook_size, (1, d.n_quantizers), generator=g).cuda()
    res = []
    for mm in (m, m2):
        cb0 = torch.empty(1, d.codebook_size, dtype=BF, device="cuda")
        mm.decoder._step(codes=codes, emb=None, slot_idx=slot, seq_inc=None, B=1, hidden_out=None, cb0_out=cb0, eos_out=None,
                         n_splits=4, stream=torch.cuda.current_stream().cuda_stream)
        res.append(cb0.float().cpu())
    assert rel_err(res[0], res[1]) <= BF16_TOL


def test_prefill_window_and_errors():
    d = _dims(4)
    sd = O.synthetic_state_dict(d, **TINY_SD)
    from tests.util import dims_to_config
    from vui_amd.model import Vui

    cfg = dims_to_config(d, 256)
    cfg.model.window_size = 16
    m = Vui(cfg, sd, device="cuda", dtype=BF)
    m.decoder.allocate_flash_kv_cache(1, m.device, BF)
    g = torch.Generator().manual_seed(2)
    emb = O.rnd(torch.randn(1, 50, d.d_model, generator=g) * 0.5, BF).to(BF).cuda()
    a = m.decoder.forward_flash(emb, None)
    m.decoder.flash_kv_caches[0].seq_lens.zero_()
    m.decoder.PREFILL_MIN = 10 ** 9
    b = m.decoder.forward_flash(emb, None)
    assert rel_err(a, b) <= BF16_TOL  # sliding window: same visible range as the decode step
    m.decoder.PREFILL_MIN = 4
    with pytest.raises(ValueError):
        m.decoder.forward_flash(torch.zeros(1, 300, d.d_model, dtype=BF, device="cuda"), None)


@pytest.mark.parametrize("window,kv", [(0, 2), (33, 4), (70, 2), (130, 1)])
def test_prefill_attention_masks(window, kv):
    """Steps of 32 keys that no query, some queries and all queries of a tile see, from both ends of a sliding window and
    from a second portion that starts inside a step; grouped KV heads.  Against the position-by-position path."""
    from tests.util import dims_to_config
    from vui_amd.model import Vui

    d = _dims(kv)
    cfg = dims_to_config(d, 256)
    cfg.model.window_size = window or None
    m = Vui(cfg, O.synthetic_state_dict(d, **TINY_SD), device="cuda", dtype=BF)
    m.decoder.allocate_flash_kv_cache(1, m.device, BF)
    emb = (torch.randn(1, 234, d.d_model, generator=torch.Generator().manual_seed(6)) * 0.5).to(BF).cuda()
    outs = []
    for minimum in (4, 10 ** 9):
        m.decoder.PREFILL_MIN = minimum
        m.decoder.flash_kv_caches[0].seq_lens.zero_()
        outs.append(torch.cat([m.decoder.forward_flash(emb[:, a:b].contiguous(), None) for a, b in ((0, 173), (173, 234))], dim=1))
    assert rel_err(outs[0], outs[1]) <= BF16_TOL, rel_err(outs[0], outs[1])


@pytest.mark.parametrize("int8", [False, True])
def test_prefill_nano_576_positions(int8):
    """The benchmark's prompt (512 audio frames + 64 text tokens) at Vui Nano dims, with bf16 and with weight-only
    int8 matrices: the pass against the oracle (which evaluates the same int8 weights) on the first 96 positions,
    its last hidden state and the cache it leaves against the position-by-position path."""
    d = O.Dims()
    sd = O.synthetic_state_dict(d, seed=0)
    m = make_model(d, sd, BF, int8=int8, max_seqlen=1408)
    m.decoder.allocate_flash_kv_cache(1, m.device, BF, max_seqlen=1408)
    assert m.decoder._prefill_available()
    g = torch.Generator().manual_seed(0)
    emb = O.rnd(torch.randn(1, 576, d.d_model, generator=g) * 0.02 * 4, BF).to(BF).cuda()
    o = O.OracleModel(d, sd, BF, n_slots=1, max_seqlen=128, int8=int8)
    ref96 = o.prefill(emb[0, :96].float().cpu(), slot=0)
    got96 = m.decoder.forward_flash(emb[:, :96].contiguous(), None)[0]
    assert rel_err(got96, ref96) <= BF16_TOL, rel_err(got96, ref96)
    m.decoder.flash_kv_caches[0].seq_lens.zero_()
    a = m.decoder.forward_flash(emb, None)
    ka = m.decoder._k[:, 0, :576].clone()
    m.decoder.flash_kv_caches[0].seq_lens.zero_()
    m.decoder.PREFILL_MIN = 10 ** 9
    b = m.decoder.forward_flash(emb, None)
    assert int(m.decoder.flash_kv_caches[0].seq_lens[0]) == 576
    assert rel_err(a[0, -1], b[0, -1]) <= BF16_TOL, rel_err(a[0, -1], b[0, -1])
    assert rel_err(a, b) <= 2 * BF16_TOL
    assert rel_err(ka, m.decoder._k[:, 0, :576]) <= BF16_TOL
    k0a, k0b = ka[0].float(), m.decoder._k[0, 0, :576].float()  # layer 0 keys: only the summation order differs
    assert float((k0a != k0b).float().mean()) < 0.01


@pytest.mark.parametrize("heads,kv,rope_dim", [(4, 2, 64), (2, 1, 64), (2, 2, 128)])
def test_prefill_other_head_dims(heads, kv, rope_dim):
    """head_dim 64 and 128 (other instantiations of the attention kernel; 128 runs four waves per workgroup), grouped
    KV heads, a rotation that covers only part of the head: the pass against the oracle's bf16 regime, and the
    cache it leaves against the position-by-position path, across a block boundary of the staged keys."""
    d = O.Dims(d_model=256, n_layers=2, n_heads=heads, n_kv_heads=kv, n_quantizers=4, codebook_size=32, rq_d_model=64,
               rq_n_layers=1, rq_n_heads=2, vocab_size=50, max_seqlen=192, rope_dim=rope_dim)
    assert d.head_dim in (64, 128)
    sd = O.synthetic_state_dict(d, **TINY_SD)
    sdb = {k: O.rnd(v, BF) for k, v in sd.items()}
    o = O.OracleModel(d, sdb, BF, n_slots=1, max_seqlen=192)
    m = make_model(d, sd, BF, max_seqlen=192)
    m.decoder.allocate_flash_kv_cache(1, m.device, BF)
    assert m.decoder._prefill_available()
    m2 = make_model(d, sd, BF, max_seqlen=192)
    m2.decoder.allocate_flash_kv_cache(1, m2.device, BF)
    m2.decoder.PREFILL_MIN = 10 ** 9
    g = torch.Generator().manual_seed(3)
    pos = 0
    for T in (45, 83):  # 45 + 83 = 128 positions: the second block starts inside a staged block of 32 keys
        emb = O.rnd(torch.randn(T, d.d_model, generator=g) * 0.5, BF)
        ref = o.prefill(emb, slot=0)
        got = m.decoder.forward_flash(emb[None].to(BF).cuda(), None)[0]
        want = m2.decoder.forward_flash(emb[None].to(BF).cuda(), None)[0]
        pos += T
        assert int(m.decoder.flash_kv_caches[0].seq_lens[0]) == pos
        assert rel_err(got, ref) <= BF16_TOL, rel_err(got, ref)
        assert rel_err(got, want) <= BF16_TOL, rel_err(got, want)
    for mine, theirs in ((m.decoder._k, m2.decoder._k), (m.decoder._v, m2.decoder._v)):
        assert rel_err(mine[:, 0, :pos], theirs[:, 0, :pos]) <= BF16_TOL


@pytest.mark.parametrize("width,heads", [(512, 8), (576, 6), (1088, 17), (1600, 25), (2048, 32), (2112, 33)])
def test_prefill_norms_of_every_width(width, heads):
    """A norm keeps one to four pieces of eight columns per lane, whole and with lanes that have none, and reads rows of more than
    2048 columns twice: rows in order (70 positions) and in operand blocks (5)."""
    d = O.Dims(d_model=width, n_layers=1, n_heads=heads, n_kv_heads=heads, intermediate_size=128, n_quantizers=4, codebook_size=32, rq_d_model=64,
               rq_n_layers=1, rq_n_heads=2, vocab_size=50, max_seqlen=96)
    sd = O.synthetic_state_dict(d, **TINY_SD)
    o = O.OracleModel(d, {k: O.rnd(v, BF) for k, v in sd.items()}, BF, n_slots=1, max_seqlen=96)
    m = make_model(d, sd, BF, max_seqlen=96)
    m.decoder.allocate_flash_kv_cache(1, m.device, BF)
    assert m.decoder._prefill_available()
    g = torch.Generator().manual_seed(9)
    for T in (70, 5):
        emb = O.rnd(torch.randn(T, width, generator=g) * 0.5, BF)
        ref = o.prefill(emb, slot=0)
        got = m.decoder.forward_flash(emb[None].to(BF).cuda(), None)[0]
        assert rel_err(got, ref) <= BF16_TOL, (T, rel_err(got, ref))


@pytest.mark.parametrize("int8", [False, True])
def test_prefill_tiles_of_every_size(int8):
    """Block lengths that choose every form of the products (16- and 32-row tiles of 8 to 16 waves, 32 x 32 tiles, large
    tiles) and end inside one, at Vui Nano dims on two layers: against the position-by-position path, or in portions of
    290 positions for the longest.  Two bf16 evaluations: the tolerance of the test above."""
    d = O.Dims(n_layers=2)
    sd = O.synthetic_state_dict(d, seed=1)
    m = make_model(d, sd, BF, int8=int8, max_seqlen=1216)
    m.decoder.allocate_flash_kv_cache(1, m.device, BF, max_seqlen=1216)
    seq = m.decoder.flash_kv_caches[0].seq_lens
    emb = (torch.randn(1, 1187, d.d_model, generator=torch.Generator().manual_seed(4)) * 0.08).to(BF).cuda()

    def run(x, portion, minimum=4):
        seq.zero_()
        m.decoder.PREFILL_MIN = minimum
        h = torch.cat([m.decoder.forward_flash(x[:, i:i + portion].contiguous(), None) for i in range(0, x.shape[1], portion)], dim=1)
        return h, m.decoder._k[:, 0, :x.shape[1]].clone(), m.decoder._v[:, 0, :x.shape[1]].clone()

    for T in (5, 16, 17, 45, 130, 251, 777, 1187):
        x = emb[:, :T].contiguous()
        got = run(x, T)
        want = run(x, T, 10 ** 9) if T < 300 else run(x, 290)
        for a, b in zip(got, want):
            assert rel_err(a, b) <= BF16_TOL, (T, rel_err(a, b))


@pytest.mark.parametrize("T", [32, 33, 64])
def test_more_tiles_than_compute_units(T):
    """Two layers at Vui Nano dims: from 33 positions on a short block's QKV product is 288 tiles and takes eight waves per tile,
    up to 32 it is 144 of twelve.  Against the position-by-position path, with the tolerance of the test above."""
    d = O.Dims(n_layers=2)
    m = make_model(d, O.synthetic_state_dict(d, seed=3), BF, int8=T == 64, max_seqlen=128)
    m.decoder.allocate_flash_kv_cache(1, m.device, BF, max_seqlen=128)
    x = (torch.randn(1, T, d.d_model, generator=torch.Generator().manual_seed(6)) * 0.08).to(BF).cuda()
    outs = []
    for minimum in (4, 10 ** 9):
        m.decoder.flash_kv_caches[0].seq_lens.zero_()
        m.decoder.PREFILL_MIN = minimum
        outs.append((m.decoder.forward_flash(x, None), m.decoder._k[:, 0, :T].clone(), m.decoder._v[:, 0, :T].clone()))
    for a, b in zip(*outs):
        assert rel_err(a, b) <= BF16_TOL, rel_err(a, b)


@pytest.mark.parametrize("int8", [False, True])
def test_large_tiles_add_as_the_small_ones_do(int8):
    """Passes whose products take large tiles (the lengths choose all three for QKV and the pair, two for the others), some
    ending inside one, against portions of 576 positions, which take 32 x 32 tiles: all add the same four parts of K in the
    same order, and a query's attention does not depend on its portion, so every bit is the same."""
    d = O.Dims(n_layers=2)
    m = make_model(d, O.synthetic_state_dict(d, seed=2), BF, int8=int8, max_seqlen=1792)
    m.decoder.allocate_flash_kv_cache(1, m.device, BF, max_seqlen=1792)
    x = (torch.randn(1, 1728, d.d_model, generator=torch.Generator().manual_seed(5)) * 0.08).to(BF).cuda()

    def run(T, portion):
        m.decoder.flash_kv_caches[0].seq_lens.zero_()
        h = torch.cat([m.decoder.forward_flash(x[:, i:i + portion].contiguous(), None) for i in range(0, T, portion)], dim=1)
        return h, m.decoder._k[:, 0, :T].clone(), m.decoder._v[:, 0, :T].clone()

    want = run(1728, 576)
    for T in (397, 700, 1000, 1233, 1600):
        h, k, v = run(T, T)
        assert torch.equal(h, want[0][:, :T]) and torch.equal(k, want[1][:, :T]) and torch.equal(v, want[2][:, :T]), T


@pytest.mark.parametrize("heads,kv,window", [(4, 2, 0), (8, 8, 70), (2, 1, 0), (2, 2, 300)])
def test_short_blocks_behind_a_cache(heads, kv, window):
    """Short blocks at their edges (one position, tiles of 16 rows, the longest) and the next longer block, behind caches that are
    empty, end inside a step of 32 keys or inside a workgroup's range of keys, and are long enough for every number of ranges and
    more; heads of 64, 32 and 128, a window.  The block's outputs and what it appends, against the position-by-position path behind
    the same cache.  Embeddings start at an odd address."""
    from tests.util import dims_to_config
    from vui_amd.model import Vui

    d = O.Dims(d_model=256, n_layers=2, n_heads=heads, n_kv_heads=kv, n_quantizers=4, codebook_size=32, rq_d_model=64, rq_n_layers=1,
               rq_n_heads=2, vocab_size=50, max_seqlen=1280)
    cfg = dims_to_config(d, 1280)
    cfg.model.window_size = window or None
    m = Vui(cfg, O.synthetic_state_dict(d, **TINY_SD), device="cuda", dtype=BF)
    m.decoder.allocate_flash_kv_cache(1, m.device, BF)
    seq = m.decoder.flash_kv_caches[0].seq_lens
    x = (torch.randn(1, 1200, d.d_model, generator=torch.Generator().manual_seed(8)) * 0.5).to(BF).cuda()
    m.decoder.forward_flash(x, None)
    for pos in (0, 3, 126, 129, 257, 640, 1130):
        for T in (1, 16, 17, 33, 64, 65):
            block = torch.empty(T * d.d_model + 1, dtype=BF, device="cuda")[1:].view(1, T, d.d_model)
            block.copy_(x[:, :T])
            outs = []
            for minimum in (1, 10 ** 9):
                seq.fill_(pos)
                m.decoder.PREFILL_MIN = minimum
                h = m.decoder.forward_flash(block, None)
                outs.append((h, m.decoder._k[:, 0, pos:pos + T].clone(), m.decoder._v[:, 0, pos:pos + T].clone()))
                assert int(seq[0]) == pos + T
            for a, b in zip(*outs):
                assert rel_err(a, b) <= BF16_TOL, (pos, T, rel_err(a, b))
            m.decoder.PREFILL_MIN = 4
            if pos == 0:  # the cache the other offsets stand on
                seq.fill_(0)
                m.decoder.forward_flash(x, None)


@pytest.mark.parametrize("heads,kv,window", [(8, 2, 0), (8, 1, 70), (16, 4, 300)])
def test_short_blocks_of_a_multiple_of_eight_heads(heads, kv, window):
    """Cached positions are read ahead by the heads that an XCD attends to, a group's once."""
    test_short_blocks_behind_a_cache(heads, kv, window)


@pytest.mark.parametrize("window,every,heads,dim", [(128, 3, 4, 64), (300, 2, 4, 64), (300, 4, 4, 64), (40, 2, 4, 64), (300, 2, 2, 96)])
def test_short_blocks_of_layers_with_and_without_a_window(window, every, heads, dim):
    """Windowed and global layers in one model, behind caches where the ranges of keys that a layer's attention is dealt in are
    unequal in number (1 to 3 with the window, 2 to 8 without): outputs and every layer's appended keys and values, each position
    against the decode step behind the same cache, and the same bits in a second pass.  Two evaluations in bf16 move apart by 0.007
    of a position's norm per layer where all layers are of one kind (five layers: 0.036); the limit is 2^-6 per layer.  Attention is
    sharp with these weights (logits of tens), so a range that is left out moves a position by its own size."""
    from tests.util import dims_to_config
    from vui_amd.model import Vui

    L = 5
    d = O.Dims(d_model=heads * dim, n_layers=L, n_heads=heads, n_kv_heads=heads // 2, n_quantizers=4, codebook_size=32, rq_d_model=64, rq_n_layers=1,
               rq_n_heads=2, vocab_size=50, max_seqlen=1280, window_size=window, global_every=every)
    m = Vui(dims_to_config(d, 1280), O.synthetic_state_dict(d, **TINY_SD), device="cuda", dtype=BF)
    dec = m.decoder
    assert len(set(dec.block_is_global)) == 2
    dec.allocate_flash_kv_cache(1, m.device, BF)
    seq = dec.flash_kv_caches[0].seq_lens
    x = (torch.randn(1, 1200, d.d_model, generator=torch.Generator().manual_seed(9)) * 0.5).to(BF).cuda()
    dec.forward_flash(x, None)

    def block(pos, T, minimum):
        seq.fill_(pos)
        dec.PREFILL_MIN = minimum
        h = dec.forward_flash(x[:, :T], None)
        # keys and values (L, T, features), outputs (1, T, features)
        return [t[:, 0, pos:pos + T].flatten(2).float() for t in (dec._k, dec._v)] + [h.float()]

    for pos in (200, 300, 640, 1130):
        for T in (4, 16, 33, 64):
            got, again, want = block(pos, T, 1), block(pos, T, 1), block(pos, T, 10 ** 9)
            for a, b, c in zip(got, again, want):
                assert torch.equal(a, b), (pos, T)
                off = ((a - c).norm(dim=-1) / c.norm(dim=-1)).amax(1)  # the worst position
                for l, e in enumerate(off.tolist(), 1 if len(off) == L else L):
                    assert e <= l * 2.0 ** -6, (pos, T, l, e)
            seq.fill_(pos)
            dec.PREFILL_MIN = 4
            dec.forward_flash(x[:, pos:pos + T], None)  # the cache that later positions stand on
