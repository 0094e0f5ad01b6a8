"""Host-side bounds that keep kernels inside their tables, checked against the kernels'
own arithmetic redone in Python."""
import numpy as np
import pytest

from litinfer_amd.kernels import ops


def pages_touched_by_a_split(p, window, nsplit, page_size, split, given=None, max_blocks=None):
    """As paged_attention_decode_mfma_kernel cuts the keys of the query at position p; `given`: the run
    length a batch of unequal contexts brings (never shorter than this token needs, never longer than
    the table's width would need)."""
    lo = p - window + 1 if window > 0 and p - window + 1 > 0 else 0
    nkeys = p - lo + 1
    per = (-(-nkeys // nsplit) + 31) & ~31
    if given is not None:
        widest = max_blocks * page_size
        if 0 < window < widest:
            widest = window
        cap = (-(-widest // nsplit) + 31) & ~31
        per = max(per, min((given + 31) & ~31, cap))
    k_begin = lo + split * per
    k_end = min(k_begin + per, p + 1)
    if k_begin >= k_end:
        return 0
    return (k_end - 1) // page_size - k_begin // page_size + 1


def test_decode_split_bound_covers_every_split_of_every_context():
    rng = np.random.default_rng(0)
    for _ in range(3000):
        page = int(rng.choice([1, 2, 7, 8, 16, 32, 128]))
        max_blocks = int(rng.integers(1, 5000))
        window = int(rng.choice([0, 0, rng.integers(1, 4000)]))
        nsplit = int(rng.integers(1, 65))
        bound = ops.decode_split_blocks(max_blocks, page, window, nsplit)
        for ctx in {max_blocks * page, int(rng.integers(1, max_blocks * page + 1)), max(1, max_blocks * page - 31)}:
            worst = max(pages_touched_by_a_split(ctx - 1, window, nsplit, page, s) for s in range(nsplit))
            assert worst <= bound, (page, max_blocks, window, nsplit, ctx)
            given = int(rng.integers(0, 2 * max_blocks * page + 64))
            worst = max(pages_touched_by_a_split(ctx - 1, window, nsplit, page, s, given, max_blocks) for s in range(nsplit))
            assert worst <= bound, (page, max_blocks, window, nsplit, ctx, given)
    # pages of one token: 64 splits of 1,024 keys fill the kernel's table exactly, one key more does not fit
    assert ops.decode_split_blocks(64 * 1024, 1, 0, 64) == ops.DECODE_TABLE_CAP
    assert ops.decode_split_blocks(64 * 1024 + 1, 1, 0, 64) > ops.DECODE_TABLE_CAP


def test_the_decode_kernels_float_quotient_is_the_page_of_every_key():
    """paged_attention_decode_mfma_kernel finds a key's page as int((key + 0.5f) * (1.0f / page_size)) in
    float32; redone here with numpy's float32 for every key the host lets through, at page sizes of every kind."""
    keys = np.arange(0, (1 << 21) + 1, dtype=np.int64)
    half = np.float32(0.5)
    for page in (1, 2, 3, 5, 7, 12, 16, 17, 48, 64, 100, 127, 128, 255, 1000, 4097, 65535, 65536):
        inv = np.float32(1.0) / np.float32(page)
        blk = ((keys.astype(np.float32) + half) * inv).astype(np.int64)
        assert np.array_equal(blk, keys // page), page


def test_prompt_attention_is_planned_once_a_step(monkeypatch):
    """A step's layers share what the library says of its portions; another window or step asks again."""
    from types import SimpleNamespace
    import torch
    from litinfer_amd.engine.batch import AttentionMeta
    asked = []
    for name, says in (("_prefill_runs", 1), ("_prefill_heads", 2), ("_prefill_tail", (3, 2, 64, 64))):
        monkeypatch.setattr(ops, name, lambda *a, name=name, says=says: (asked.append(name), says)[1])
    sent = []
    monkeypatch.setattr(ops, "_gpu", lambda *a: None)
    monkeypatch.setattr(ops, "_run", lambda *a: sent.append(a))
    ints = lambda *v: torch.tensor(v, dtype=torch.int32)
    t, nh, nkv, dh, page = 70, 6, 2, 64, 16

    def step():
        return AttentionMeta(block_table=torch.zeros(1, 5, dtype=torch.int32), max_blocks=5, seg_of_token=torch.zeros(t, dtype=torch.int32),
                             q_start=ints(0), q_len=ints(t), ctx_len=ints(t), num_segments=1, num_tokens=t, max_q_len=t, max_ctx_len=t,
                             host_q_start=np.zeros(1, np.int32), host_q_len=np.full(1, t, np.int32), host_ctx_len=np.full(1, t, np.int32),
                             num_single=0, num_multi=t, tiles=torch.zeros(3, 4, dtype=torch.int32), num_tiles=3, tile_rows=32)
    cache = torch.zeros(8, nkv, page, dh, dtype=torch.bfloat16)
    q = torch.zeros(t, nh * dh, dtype=torch.bfloat16)
    ws = SimpleNamespace(buffer=lambda name, shape, dt, zero=False: torch.zeros(shape, dtype=dt))
    call = lambda meta, window: ops.paged_attention(q, torch.empty_like(q), cache, cache.clone(), meta, nh, nkv, dh, page, window, 0.1, ws=ws)
    first = step()
    for _ in range(28):
        call(first, 0)
    assert asked == ["_prefill_runs", "_prefill_heads", "_prefill_tail"]
    assert len(sent) == 28 and all(s[1] == "li_paged_attention_prefill" and s[-7] == 3 and s[-3:] == (64, 2, 2) for s in sent)
    call(first, 40)
    call(step(), 0)
    assert len(asked) == 9


def test_decoding_is_planned_once_a_step(monkeypatch):
    """A step's layers share the cut of their keys; another window, layout or step asks again."""
    import torch
    from litinfer_amd.engine.batch import AttentionMeta
    asked, sent = [], []
    cut = ops._decode_cut
    monkeypatch.setattr(ops, "_decode_cut", lambda *a: (asked.append(a), cut(*a))[1])
    monkeypatch.setattr(ops, "_gpu", lambda *a: None)
    monkeypatch.setattr(ops, "_simd_count", lambda device: 1024)
    monkeypatch.setattr(ops, "_run", lambda *a: sent.append(a))
    n, page, width = 3, 16, 64
    ints = lambda *v: torch.tensor(v, dtype=torch.int32)

    def step(longest):
        ctx = np.array([200, longest, 5], np.int32)
        return AttentionMeta(block_table=torch.zeros(n, width, dtype=torch.int32), max_blocks=width, seg_of_token=ints(0, 1, 2), q_start=ints(0, 1, 2),
                             q_len=ints(1, 1, 1), ctx_len=torch.from_numpy(ctx), num_segments=n, num_tokens=n, max_q_len=1, max_ctx_len=longest,
                             host_q_start=np.arange(n, dtype=np.int32), host_q_len=np.ones(n, np.int32), host_ctx_len=ctx, num_single=n, max_single_ctx=width * page)

    def call(meta, nh, nkv, window):
        cache = torch.zeros(8, nkv, page, 64, dtype=torch.bfloat16)
        q = torch.zeros(n, nh * 64, dtype=torch.bfloat16)
        ops.paged_attention(q, torch.empty_like(q), cache, cache.clone(), meta, nh, nkv, 64, page, window, 0.1)
    first = step(1000)
    for _ in range(28):
        call(first, 14, 2, 0)
    assert len(asked) == 1 and len({s[-2] for s in sent if s[1] == "li_paged_attention_decode"}) == 1
    call(first, 14, 2, 100)
    call(first, 8, 4, 0)
    call(step(900), 14, 2, 0)
    assert len(asked) == 4


def _segments(segs):
    return np.array([q for _, q in segs], dtype=np.int32), np.array([c for c, _ in segs], dtype=np.int32)      # (context, new tokens)


def test_heads_a_block_where_segments_differ_and_where_heads_are_short():
    """The longest segment's blocks in a last round of their own: four heads a block there, one or two (by the mean block alone) were
    30 to 45 % slower; heads of 64 gain nothing by fewer heads a block."""
    heads = lambda segs, nh, nkv, *dh: ops._prefill_heads(*_segments(segs), nh, nkv, 1500, 0, *dh)
    assert heads([(4174, 4174), (13230, 660), (10439, 318)], 24, 8) == 4
    assert heads([(111, 111), (3764, 3764), (389, 389), (14028, 294), (3298, 195)], 32, 16) == 4
    assert heads([(1934, 1934), (104, 104), (5919, 438), (798, 798), (385, 125)], 40, 8) == 4
    assert heads([(2048, 2048)], 10, 2, 64) == heads([(4123, 4123), (4448, 4292)], 10, 2, 64) == 4
    assert heads([(17999, 1999)], 40, 8) == 1 and heads([(2048, 2048)], 32, 32) < 4


def test_keys_of_the_first_tiles_are_cut_only_where_the_last_block_is_done_earlier():
    tail = lambda segs, nh, nkv, heads: ops._prefill_tail(*_segments(segs), nh, nkv, 128, 2000, 0, heads)
    assert tail([(17999, 1999)], 40, 8, 1) == (3, 16, 512, 512)
    # a few long tiles and a second segment's first, whose keys are few; long tiles that end before the others do
    assert tail([(5074, 73), (4253, 4253)], 32, 16, 2)[0] == 1 and tail([(2454, 477), (1757, 1757)], 32, 16, 2)[0] == 1
    assert tail([(16418, 1599), (725, 725), (1936, 1936)], 32, 32, 1)[0] == 1
    # (the same library function with lengths at their bounds)
    for segs in ([(2, 2)], [(1, 1)] * 3, [(64, 64)] * 700, [(1 << 20, 1 << 15)]):
        for heads in (4, 2, 1):
            runs, tiles, tokens, upto = tail(segs, 6, 2, heads)
            assert runs == 1 or (0 < tokens <= upto <= sum(q for _, q in segs) and tiles % (4 // heads) == 0)


def test_groups_of_keys_of_the_32_bit_prompt_attention():
    """Heads x groups of a block (1: one head in four groups ... 4: four heads in one): no further groups for a single block of keys, nor
    two rounds of blocks for two."""
    import ctypes
    f = ops._lib_fn("attention", "li_paged_attention_prefill_f32_form", [ctypes.c_int] * 5, ctypes.c_int)
    assert [f(1, 28, 4, 128, keys) for keys in (2, 32, 33, 200, 0)] == [4, 4, 1, 1, 1]
    assert [f(8, 40, 8, 128, keys) for keys in (2, 64, 65, 0)] == [4, 4, 1, 1]          # 320 blocks of one head: more than units
    assert [f(6, 40, 8, 128, keys) for keys in (2, 64)] == [4, 1]                       # 240: not more
    assert [f(8, 40, 8, 64, keys) for keys in (32, 64)] == [4, 1]                       # two blocks of 64 columns share a unit
    assert [f(13, 28, 4, 128, 400), f(32, 28, 4, 128, 1000), f(63, 28, 4, 128, 2000)] == [2, 3, 4]
    assert f(13, 28, 4, 128, 20) == f(32, 28, 4, 128, 20) == 4


@pytest.mark.parametrize("gated,m,n,k,result_bytes,tile", [
    # wide matrices of a few hundred rows (97 -> 128 us without these tiles, 48 -> 61), narrow gated ones (148 -> 169)
    (0, 257, 17472, 8000, 2, (128, 224, False)), (0, 380, 18944, 3584, 2, (128, 224, False)), (1, 2012, 2304, 896, 1, (128, 192, False)),
    (1, 1699, 2688, 16768, 1, (128, 192, False)),
    # a single step of 64 k-values, which a tile in pieces doubles (26 -> 43)
    (1, 3330, 12288, 64, 1, (256, 256, False)),
    # the layers' products of a prompt
    (1, 2048, 37888, 3584, 1, (256, 256, True)), (0, 8192, 8192, 8192, 8, (256, 256, True)),
])
def test_tiles_of_products(gated, m, n, k, result_bytes, tile):
    import ctypes
    f = ops._lib_fn("gemm", "li_linear_tile", [ctypes.c_int] * 5, ctypes.c_int)
    got = f(gated, m, n, k, result_bytes)
    assert (abs(got) >> 16, abs(got) & 65535, got < 0) == tile


@pytest.mark.parametrize("units", [1, 32, 64, 128, 256, 304])
def test_columns_a_block_of_the_kernel_of_one_to_four_rows(units):
    """A block of that kernel writes one tile of 16 columns, however many compute units the device has: with more columns a block
    some would never be written.  A sum takes as many blocks as its shares of the rows' squares are counted by."""
    f = ops._lib_fn("gemm", "li_rows_kernel_cols", [ops.c_int] * 5, ops.c_int)
    taken = 0
    for n in [1, 15, 16, 17, 896, 1152, 1536, 2048, 3072, 3584, 4095, 4096, 4097, 4608, 4864, 4865, 8240, 17920, 151936, 16 * units, 16 * units + 1]:
        for k in (64, 896, 2048, 2112, 11008, 100):
            for m in (1, 2, 4, 5):
                for into_sum in (0, 1):
                    cols = f(m, n, k, into_sum, units)
                    fits = m <= 4 and k % 64 == 0 and (k <= 2048 or n <= 2048) and (n <= 16 * units or not into_sum)
                    assert (1 <= cols <= 16) if fits else cols == 0, (m, n, k, into_sum, units, cols)
                    if fits and n <= 16 * units:
                        assert cols == max(4, -(-n // units))
                    taken += fits
    assert taken


def test_products_are_cut_into_no_more_parts_than_are_added_up():
    """The kernels that add up the parts of K hold sixteen, and eight above 64 rows; a rope or plain sum counts as far as it is told."""
    most = {True: 0, False: 0}
    for m in (17, 33, 48, 64, 65, 128, 300, 1000):
        for n in (8, 64, 128, 896, 1536, 2048, 3584, 4608, 8192):
            for k in (64, 512, 1024, 1536, 4096, 8960, 18944, 65536):
                need = ops._work_bytes(m, n, k, ops._DT[ops.torch.bfloat16])
                assert need % (4 * m * n) == 0
                most[m <= 64] = max(most[m <= 64], need // (4 * m * n))
    assert most[True] == ops.SPLITK_MAX_PARTS == 16 and most[False] == 8


@pytest.mark.parametrize("aligned,dtype", [(False, ops.torch.bfloat16), (True, ops.torch.float32)])
def test_many_equal_contexts_that_fill_the_simds_keep_one_run(aligned, dtype):
    for n, keys, runs in ((100, 1500, 1), (100, 1024, 1), (64, 1500, None)):
        ns, waves, planned = ops._decode_cut(8 * n, keys, 64, dtype, 1024, aligned, _decode_batch([keys] * n), 0)
        assert ns == planned and (ns == 1) == (runs == 1), (n, keys, ns)
    assert ops._decode_cut(800, 1500, 64, dtype, 1024, aligned, _decode_batch([1500] + [200] * 99), 0)[0] > 1


@pytest.mark.parametrize("pairs,dh,block,ends", [(2, 64, 256, 1024), (32, 64, 256, 1024), (32, 128, 128, 1024), (33, 64, 256, 320), (64, 128, 128, 1008),
                                                 (65, 128, 0, 0), (65, 64, 0, 0)])
def test_float32_decoding_is_cut_shorter_only_where_that_was_measured(pairs, dh, block, ends):
    """One block of four runs, then runs of 32 keys and the kernel that joins them; beyond, the ordinary cut was the faster."""
    for keys in range(16, 8192, 16):
        want = None if keys <= 96 or keys > ends else ops.DECODE_QUAD if keys <= block else (32, 64)
        assert ops._short_runs(pairs, keys, dh, ops.torch.float32, 4) == want, keys


def _decode_batch(ctx, padded=False):
    from types import SimpleNamespace
    ctx = np.asarray(ctx, np.int32)
    return SimpleNamespace(host_q_len=np.ones(len(ctx), np.int32), host_ctx_len=ctx, padded=padded)


def _decode_plan_of(ctx, nkv, dh=128, table=0, padded=False):
    """What `_decode_cut` says, and the keys of the longest wave: with a list, at the run length that the device chooses."""
    keys = max(table, max(ctx))
    ns, waves, planned = ops._decode_cut(len(ctx) * nkv, keys, dh, ops.torch.bfloat16, 1024, True, _decode_batch(ctx, padded), 0)
    up = lambda a, b: (-(-a // b) + 31) & ~31
    longest = max(ctx)
    if ns <= planned:
        return (ns, waves), up(longest, ns)
    keys_of, lower, cap = np.asarray(ctx), up(longest, ns), up(keys, ns)
    cost = {c: -(-int(nkv * np.sum(-(-keys_of // c))) // 1024) * (c + 24) for c in range(lower, max(cap, lower) + 1, 32)}
    return (ns, waves), min(cost, key=lambda c: (cost[c], c))


@pytest.mark.parametrize("pairs,dh,ends", [(1, 64, 263), (8, 64, 312), (36, 64, 508), (37, 64, 515), (65, 64, 711), (85, 64, 851), (86, 64, 860), (128, 64, 1280), (191, 64, 1280),
                                           (192, 64, None), (256, 64, None), (257, 64, 1024), (383, 64, 1024), (384, 64, None), (512, 64, None), (1, 128, 256), (32, 128, 256), (48, 128, 256),
                                           (49, 128, 490), (64, 128, 640), (128, 128, 1280), (160, 128, 1280), (192, 128, None), (320, 128, 640)])
def test_a_block_takes_all_runs_only_where_that_was_measured(pairs, dh, ends):
    """Of contexts that are alike, or that the host does not know."""
    for keys in range(1, 20000, 7):
        for spread in (None, (float(keys), float(keys)), (keys / 1.14, float(keys))):
            assert ops._one_block(pairs, keys, dh, 1024, spread) == (keys > 128 and (ends is None or keys <= ends)), keys


@pytest.mark.parametrize("ctx,nkv,dh,most", [
    ([30000] + [200] * 63, 4, 128, 480), ([8000] + [300] * 63, 4, 128, 128), ([16000] + [500] * 47, 4, 128, 256), ([30000] + [200] * 119, 2, 128, 480),
    (np.linspace(16, 4600, 64).astype(int), 4, 128, 672), (np.linspace(16, 4600, 128).astype(int), 2, 64, 672), ([30000] + [200] * 99, 2, 128, 480),
    ([20000] * 4 + [100] * 252, 2, 128, 480)])
@pytest.mark.parametrize("padded", [False, True])
def test_a_long_context_beside_short_ones_is_shared_out_among_the_waves(ctx, nkv, dh, most, padded):
    """One long document beside many short requests: no block of four waves takes it alone, whether the step is recorded or not."""
    ctx = [int(c) for c in ctx]
    table = 1 << (max(ctx) - 1).bit_length() if padded else 0
    (ns, waves), longest = _decode_plan_of(ctx, nkv, dh, table, padded)
    assert waves == 1 and longest <= most, (ns, waves, longest)


@pytest.mark.parametrize("n,nkv,table", [(64, 4, 4096), (48, 4, 16384), (120, 2, 8192), (256, 2, 4096), (128, 2, 32768)])
def test_a_recording_of_contexts_that_differ_does_not_take_blocks_of_four(n, nkv, table):
    """Its replays' contexts may be others of the same tables, as spread as they like; of contexts that are alike it does."""
    for low in (1.5, 2, 8, 100):
        assert _decode_plan_of([int(c) for c in np.linspace(table * 0.9 / low, table * 0.9, n)], nkv, 128, table, True)[0][1] == 1, low
    assert _decode_plan_of([int(table * 0.9)] * n, nkv, 128, table, True)[0] == (4, 4)


@pytest.mark.parametrize("ctx,nkv,table,listed", [(np.linspace(260, 500, 4), 2, 512, False), (np.linspace(600, 1000, 48), 2, 1024, False), ([512] + [100] * 3, 2, 512, True),
                                                  (np.linspace(2047, 4090, 8), 4, 4096, False), (np.linspace(100, 2001, 64), 2, 2048, True),
                                                  (np.linspace(500, 1900, 80), 2, 2048, True)])
def test_runs_are_listed_only_where_they_can_be_shared_out(ctx, nkv, table, listed):
    """Not where all of them are at work at one time, short and of contexts that are not far apart."""
    ctx = [int(c) for c in ctx]
    ns, waves, planned = ops._decode_cut(len(ctx) * nkv, table, 128, ops.torch.bfloat16, 1024, True, _decode_batch(ctx, True), 0)
    assert waves == 1 and (ns > planned) == listed
    if not listed:
        assert len(ctx) * nkv * ns <= 1024 and -(-table // ns) <= 128


def test_every_decoding_step_is_cut_into_runs_that_the_kernels_take():
    """One run, one block of four, or up to DECODE_MAX_SPLITS single waves, whatever the step (the first number) and its contexts."""
    from types import SimpleNamespace
    for dtype in (ops.torch.bfloat16, ops.torch.float32):
        for pairs in (1, 2, 8, 31, 64, 65, 150, 192, 256, 320, 512, 513, 1000, 3000):
            for keys in (1, 32, 96, 97, 128, 129, 256, 500, 1024, 4096, 30000):
                for dh in (64, 128):
                    for aligned in (True, False):
                        for low in (keys, max(1, keys // 8)):
                            ctx = np.linspace(low, keys, max(2, pairs)).astype(np.int32)
                            meta = SimpleNamespace(host_q_len=np.ones(len(ctx), np.int32), host_ctx_len=ctx)
                            ns, waves, planned = ops._decode_cut(pairs, keys, dh, dtype, 1024, aligned, meta, 0)
                            assert 1 <= planned <= ns <= ops.DECODE_MAX_SPLITS and (waves == 1 or ns == planned == waves == ops.DECODE_QUAD)


@pytest.mark.parametrize("pairs,dh,ends", [(2, 128, 384), (32, 128, 384), (2, 64, 448), (64, 128, 640), (512, 64, 896), (512, 128, 896)])
def test_bfloat16_decoding_over_other_pages_takes_one_block_only_where_that_was_measured(pairs, dh, ends):
    """A window, or pages of no multiple of 8 keys (else `_one_block` is asked)."""
    for keys in range(16, 8192, 16):
        assert (ops._short_runs(pairs, keys, dh, ops.torch.bfloat16, 0, False) == ops.DECODE_QUAD) == (128 < keys <= ends), keys


@pytest.mark.parametrize("pairs,dh,differ,begins,ends", [(512, 64, False, 128, 1280), (513, 64, True, 128, 1280), (513, 64, False, 320, 1280), (640, 128, False, 320, 1280),
                                                         (641, 64, False, 0, 0), (2047, 128, True, 128, 1280), (2048, 128, True, 255, 1280), (2048, 64, True, 128, 1280)])
def test_many_equal_contexts_are_not_decoded_in_blocks(pairs, dh, differ, begins, ends):
    for keys in range(1, 4096):
        assert (ops._short_runs(pairs, keys, dh, ops.torch.bfloat16, 0, True, differ) == ops.DECODE_QUAD) == (begins < keys <= ends), keys
