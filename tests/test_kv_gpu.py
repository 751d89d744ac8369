"""GPU parity of the paged KV cache and its attention (dcq_kv_*), through the C ABI, against the
CPU oracle (oracle/kv.py). Slot bytes and the gather are bit-exact; the attention output is
within |out - ref| <= A * (1e-4 + 1e-5 * B), A = sum_t p_t |v_t|, B = max_t scale sum |q k_t|."""
import numpy as np
import pytest

import densecore_amd as dc
from densecore_amd import synth

pytestmark = pytest.mark.gpu

Q8_0, F16, F32 = 8, 1, 0
CACHE_TYPES = [Q8_0, F16, F32]


@pytest.fixture(scope="module")
def KV(O):
    from oracle import kv
    return kv


def to_dev(a, dev):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).to(dev)


def to_host(t):
    import torch
    torch.cuda.synchronize()
    return t.cpu().numpy()


def make_table(n_pos, n_blocks, seed, holes=()):
    rng = np.random.default_rng(seed)
    need = (n_pos + 15) // 16
    table = rng.permutation(n_blocks)[:need].astype(np.int32)
    for h in holes:
        table[h] = -1
    return table


@pytest.mark.parametrize("ct", CACHE_TYPES)
def test_kv_write_bytes(KV, dev, ct):
    """Rows written at positions pos0 .. into a pre-filled arena: every byte equals the
    oracle's (including the slots left alone, and a table entry of -1 that is skipped)."""
    import torch
    n_layer, layer, row, n_blocks = 3, 1, 4 * 64, 9
    sb = KV.slot_bytes(ct, row)
    rng = np.random.default_rng(3)
    arena = rng.integers(0, 256, n_blocks * n_layer * 16 * sb, dtype=np.uint8)
    table = make_table(70, n_blocks, 4, holes=(2,))
    rows = synth.normal(45 * row, 5).reshape(45, row)
    synth.set_outliers(rows.reshape(-1), 30, 25.0, 6)
    rows[3, :64] = 0.0  # an all-zero Q8_0 block
    want = arena.copy()
    KV.write(ct, want, n_layer, layer, table, 25, rows)
    cache = dc.PagedKVCache(ct, n_blocks, n_layer, 4, 64, device=dev)
    cache.k.copy_(to_dev(arena, dev))
    cache.write("k", layer, to_dev(table, dev), 25, to_dev(rows, dev))
    assert np.array_equal(to_host(cache.k), want)
    assert not to_host(cache.v).any()
    del torch


@pytest.mark.parametrize("ct", CACHE_TYPES)
def test_kv_gather_exact(KV, dev, ct):
    """History decoded bit-exactly, missing blocks (short table, -1 entry) as zeros, the current
    rows appended as given."""
    n_layer, layer, row, n_blocks, n_past = 2, 0, 2 * 128, 8, 75
    sb = KV.slot_bytes(ct, row)
    arena = np.zeros(n_blocks * n_layer * 16 * sb, np.uint8)
    table = make_table(64, n_blocks, 8, holes=(1,))  # covers 4 of the 5 history blocks
    hist = synth.normal(n_past * row, 9).reshape(n_past, row)
    KV.write(ct, arena, n_layer, layer, table, 0, hist[:64])
    cur = synth.normal(3 * row, 10).reshape(3, row)
    want = KV.gather(ct, arena, n_layer, layer, table, n_past, cur)
    cache = dc.PagedKVCache(ct, n_blocks, n_layer, 2, 128, device=dev)
    cache.v.copy_(to_dev(arena, dev))
    got = cache.gather("v", layer, to_dev(table, dev), n_past, to_dev(cur, dev))
    assert np.array_equal(to_host(got).view(np.uint32), want.view(np.uint32))


ATTN = [
    # (cache type, n_tokens, n_past, n_head, n_head_kv, head_dim)
    (Q8_0, 1, 4095, 32, 8, 128),   # Qwen3-4B decode at a 4k context: keys split over workgroups
    (Q8_0, 1, 5, 32, 8, 128),      # a short history
    (Q8_0, 1, 0, 32, 8, 128),      # the first token: only its own row
    (Q8_0, 7, 100, 32, 8, 128),    # a chunk of prefill on top of history
    (Q8_0, 130, 0, 8, 8, 64),      # prefill, MHA, current rows over several chunks
    (Q8_0, 3, 300, 8, 1, 256),     # head_dim 256, multi-query (8 heads per KV head)
    (Q8_0, 2, 77, 32, 1, 128),     # 32 query heads per KV head: the group split over workgroups
    (Q8_0, 2, 50, 8, 4, 128),      # the 4-row workgroup with two tokens of two heads each
    (F16, 4, 20, 4, 4, 64),        # the 4-row workgroup with four tokens of one head
    (F16, 1, 4095, 32, 8, 128),
    # the split merge's forms: 17..64 splits, 97..128 (32 lanes per output), over 128 (a workgroup
    # per row)
    (Q8_0, 1, 2000, 32, 8, 128),   # 33 splits
    (Q8_0, 1, 7000, 32, 8, 128),   # 111 splits
    (Q8_0, 1, 300, 32, 8, 128),    # 6 splits of 1024 quads: lanes
    (Q8_0, 1, 500, 32, 8, 128),    # 9 splits
    (F16, 16, 600, 16, 1, 64),     # 6 splits of 4096 quads
    (F16, 33, 700, 16, 2, 64),     # 7 splits of 8448 quads: a thread per quad
    (F16, 34, 1300, 16, 2, 128),   # more of them
    (F16, 1, 20000, 4, 4, 64),     # 158 splits
    (F16, 5, 33, 16, 4, 64),
    (F32, 1, 200, 8, 2, 128),
    (F32, 17, 40, 4, 2, 256),
    # prompts on the MFMA kernel (>= 64 tokens, query-head groups of 4k): two exact 32-token
    # tiles; a ragged last tile over a history that is not a multiple of 32 keys; head_dim 64
    # with 8 query heads per KV head; one KV head; a Qwen3-4B-sized prompt chunk
    (Q8_0, 64, 0, 32, 8, 128),
    (Q8_0, 100, 37, 8, 2, 128),
    (F16, 96, 50, 16, 2, 64),
    (F32, 70, 20, 4, 1, 128),
    (Q8_0, 256, 300, 32, 8, 128),
    # the MFMA kernel with its keys split over workgroups (few tokens over a long history)
    (Q8_0, 32, 700, 8, 2, 128),
    (F16, 40, 1000, 16, 4, 64),
]


@pytest.mark.parametrize("ct,n,n_past,n_head,n_kv,hd", ATTN)
def test_kv_attention(KV, dev, ct, n, n_past, n_head, n_kv, hd):
    n_layer, layer = 2, 1
    row = n_kv * hd
    n_blocks = (n_past + 15) // 16 + 3
    sb = KV.slot_bytes(ct, row)
    arena_k = np.zeros(n_blocks * n_layer * 16 * sb, np.uint8)
    arena_v = np.zeros_like(arena_k)
    table = make_table(max(n_past, 1), n_blocks, 11 + n)
    seed = 100 + n + n_past + hd
    hist_k = synth.normal(n_past * row, seed).reshape(n_past, row)
    hist_v = synth.normal(n_past * row, seed + 1).reshape(n_past, row)
    KV.write(ct, arena_k, n_layer, layer, table, 0, hist_k)
    KV.write(ct, arena_v, n_layer, layer, table, 0, hist_v)
    q = synth.normal(n * n_head * hd, seed + 2, 0.0, 2.0).reshape(n, n_head * hd)
    k_cur = synth.normal(n * row, seed + 3).reshape(n, row)
    v_cur = synth.normal(n * row, seed + 4).reshape(n, row)
    scale = 1.0 / np.sqrt(hd)
    k_all = KV.gather(ct, arena_k, n_layer, layer, table, n_past, k_cur).reshape(-1, n_kv, hd)
    v_all = KV.gather(ct, arena_v, n_layer, layer, table, n_past, v_cur).reshape(-1, n_kv, hd)
    ref, parts = KV.attention(q.reshape(n, n_head, hd), k_all, v_all, n_past, np.float32(scale))

    cache = dc.PagedKVCache(ct, n_blocks, n_layer, n_kv, hd, device=dev)
    cache.k.copy_(to_dev(arena_k, dev))
    cache.v.copy_(to_dev(arena_v, dev))
    out = cache.attention(layer, to_dev(table, dev), to_dev(q, dev), to_dev(k_cur, dev), to_dev(v_cur, dev),
                          n_past, float(np.float32(scale)))
    KV.assert_close_attention(to_host(out).reshape(n, n_head, hd), ref, parts,
                              what=f"attention ct={ct} n={n} n_past={n_past} heads={n_head}/{n_kv} hd={hd}")


@pytest.mark.parametrize("n", [2, 80])  # the VALU kernel with key splits; the MFMA prompt kernel
def test_kv_attention_missing_blocks_read_as_zero_keys(KV, dev, n):
    """A history block absent from the table (-1, or past the table's end) is a zero K/V row,
    as in the reference's gathered K_all: score 0, value 0."""
    ct, n_past, n_head, n_kv, hd, n_layer = Q8_0, 90, 8, 2, 128, 1
    row = n_kv * hd
    n_blocks = 8
    sb = KV.slot_bytes(ct, row)
    arena_k = np.zeros(n_blocks * n_layer * 16 * sb, np.uint8)
    arena_v = np.zeros_like(arena_k)
    table = make_table(64, n_blocks, 12, holes=(2,))  # 4 entries for 6 history blocks
    KV.write(ct, arena_k, n_layer, 0, table, 0, synth.normal(64 * row, 13).reshape(64, row))
    KV.write(ct, arena_v, n_layer, 0, table, 0, synth.normal(64 * row, 14).reshape(64, row))
    q = synth.normal(n * n_head * hd, 15).reshape(n, n_head * hd)
    k_cur = synth.normal(n * row, 16).reshape(n, row)
    v_cur = synth.normal(n * row, 17).reshape(n, row)
    k_all = KV.gather(ct, arena_k, n_layer, 0, table, n_past, k_cur).reshape(-1, n_kv, hd)
    v_all = KV.gather(ct, arena_v, n_layer, 0, table, n_past, v_cur).reshape(-1, n_kv, hd)
    ref, parts = KV.attention(q.reshape(n, n_head, hd), k_all, v_all, n_past, 0.125)
    cache = dc.PagedKVCache(ct, n_blocks, n_layer, n_kv, hd, device=dev)
    cache.k.copy_(to_dev(arena_k, dev))
    cache.v.copy_(to_dev(arena_v, dev))
    out = cache.attention(0, to_dev(table, dev), to_dev(q, dev), to_dev(k_cur, dev), to_dev(v_cur, dev), n_past,
                          0.125)
    KV.assert_close_attention(to_host(out).reshape(n, n_head, hd), ref, parts, what="missing blocks")


def test_kv_decode_steps_write_then_attend(KV, dev):
    """Decode loop: each step attends with its own row in fp32, then writes that row into the
    cache for the next step (the reference's write-then-gather order within one call gives the
    same attention input). Eight steps against the oracle doing the same."""
    ct, n_head, n_kv, hd, n_layer, layer = Q8_0, 16, 4, 128, 2, 0
    row = n_kv * hd
    n_blocks = 6
    sb = KV.slot_bytes(ct, row)
    arena_k = np.zeros(n_blocks * n_layer * 16 * sb, np.uint8)
    arena_v = np.zeros_like(arena_k)
    table = make_table(80, n_blocks, 20)
    n_past0 = 60
    KV.write(ct, arena_k, n_layer, layer, table, 0, synth.normal(n_past0 * row, 21).reshape(n_past0, row))
    KV.write(ct, arena_v, n_layer, layer, table, 0, synth.normal(n_past0 * row, 22).reshape(n_past0, row))
    cache = dc.PagedKVCache(ct, n_blocks, n_layer, n_kv, hd, device=dev)
    cache.k.copy_(to_dev(arena_k, dev))
    cache.v.copy_(to_dev(arena_v, dev))
    tdev = to_dev(table, dev)
    for step in range(8):
        n_past = n_past0 + step
        q = synth.normal(n_head * hd, 30 + step).reshape(1, -1)
        kc = synth.normal(row, 40 + step).reshape(1, -1)
        vc = synth.normal(row, 50 + step).reshape(1, -1)
        k_all = KV.gather(ct, arena_k, n_layer, layer, table, n_past, kc).reshape(-1, n_kv, hd)
        v_all = KV.gather(ct, arena_v, n_layer, layer, table, n_past, vc).reshape(-1, n_kv, hd)
        ref, parts = KV.attention(q.reshape(1, n_head, hd), k_all, v_all, n_past, 0.08838834764831845)
        kd, vd = to_dev(kc, dev), to_dev(vc, dev)
        out = cache.attention(layer, tdev, to_dev(q, dev), kd, vd, n_past, 0.08838834764831845)
        cache.write("k", layer, tdev, n_past, kd)
        cache.write("v", layer, tdev, n_past, vd)
        KV.write(ct, arena_k, n_layer, layer, table, n_past, kc)
        KV.write(ct, arena_v, n_layer, layer, table, n_past, vc)
        KV.assert_close_attention(to_host(out).reshape(1, n_head, hd), ref, parts, what=f"decode step {step}")
    assert np.array_equal(to_host(cache.k), arena_k) and np.array_equal(to_host(cache.v), arena_v)


def prompt_case(KV, dev, ct, hd, n_head, n_kv, k_past, v_past, q, k_cur, v_cur, scale, holes=()):
    """One call over a history written to the cache (with `holes` in its block table): the output
    [n, n_head, hd] in float64, and the oracle's (ref, (A, B)) for the same rows."""
    n, n_past, row = q.shape[0], k_past.shape[0], n_kv * hd
    n_blocks = (n_past + 15) // 16 + 2
    arena_k = np.zeros(n_blocks * 16 * KV.slot_bytes(ct, row), np.uint8)
    arena_v = np.zeros_like(arena_k)
    table = make_table(max(n_past, 1), n_blocks, 5 + n, holes)
    KV.write(ct, arena_k, 1, 0, table, 0, k_past)
    KV.write(ct, arena_v, 1, 0, table, 0, v_past)
    k_all = KV.gather(ct, arena_k, 1, 0, table, n_past, k_cur).reshape(-1, n_kv, hd)
    v_all = KV.gather(ct, arena_v, 1, 0, table, n_past, v_cur).reshape(-1, n_kv, hd)
    with np.errstate(invalid="ignore"):
        ref, parts = KV.attention(q.reshape(n, n_head, hd), k_all, v_all, n_past, np.float32(scale))
    cache = dc.PagedKVCache(ct, n_blocks, 1, n_kv, hd, device=dev)
    cache.k.copy_(to_dev(arena_k, dev))
    cache.v.copy_(to_dev(arena_v, dev))
    out = cache.attention(0, to_dev(table, dev), to_dev(q, dev), to_dev(k_cur, dev), to_dev(v_cur, dev), n_past,
                          float(scale))
    return to_host(out).astype(np.float64).reshape(ref.shape), ref, parts


def prompt_rows(hd, n_head, n_kv, n_past, n, seed):
    """k_past, v_past, q, k_cur, v_cur of normal values."""
    return [synth.normal(m * h * hd, seed + i, 0.0, std).reshape(m, h * hd)
            for i, (m, h, std) in enumerate(((n_past, n_kv, 1.0), (n_past, n_kv, 1.0), (n, n_head, 2.0),
                                             (n, n_kv, 1.0), (n, n_kv, 1.0)))]


def assert_rows(out, ref, parts):
    """Every row of every head by itself: |out - ref| <= (2e-6 + 2^-22 B) |A| in the 2-norm. A score of
    magnitude up to B carries a few units of 2^-24 of B and moves its weight by as much; the weighted sums
    and the operands' two f16 pieces (22 bits) add a few of 2^-23 of A = sum_t p_t |v_t|."""
    a, b = parts
    err = np.linalg.norm(out - ref, axis=2)
    bound = (2e-6 + 2.0 ** -22 * b) * np.linalg.norm(a, axis=2)
    bad = ~(err <= bound)
    assert not bad.any(), (f"{int(bad.sum())} of {err.size} rows, first {np.argwhere(bad)[0]}, "
                           f"worst {np.nanmax(err / bound):.3g}")


PROMPT = [
    # (cache type, n_tokens, n_past, n_head, n_head_kv, head_dim, K scale, V scale): the prompt kernel's
    # tiles hold 128 (token, head of the group) rows, 32 a wave, and 32 keys a block
    (Q8_0, 16, 3, 1, 1, 128, 1, 1),        # the fewest rows it takes; one head; three empty waves
    (Q8_0, 15, 3, 1, 1, 128, 1, 1),        # one fewer: the VALU kernel
    (F32, 129, 0, 2, 2, 64, 1, 1),         # one row past a tile, no history
    (F16, 43, 31, 12, 4, 128, 1, 1),       # groups of 3 (129 rows): tokens straddle waves and tiles
    (Q8_0, 19, 290, 28, 4, 64, 1, 1),      # groups of 7, the keys split over workgroups
    (F16, 64, 960, 4, 2, 256, 1, 1),       # head_dim 256 in few rounds: the VALU kernel
    (Q8_0, 33, 990, 8, 8, 256, 1, 1),      # 33 rows over 1023 keys: the VALU kernel
    (F32, 9, 1300, 8, 1, 256, 1, 1),
    (F32, 70, 20, 4, 1, 128, 3e-7, 2e5),   # magnitudes past f16's range on either side
    (F32, 70, 20, 4, 1, 64, 1e-20, 1e20),
    (F32, 200, 0, 4, 1, 128, 1, 1e-12),
    (F16, 40, 24, 4, 1, 128, 1, 1),        # two blocks: one for each wave group
    (Q8_0, 90, 700, 6, 2, 128, 1, 1),      # key splits with odd numbers of blocks
    (F32, 700, 0, 3, 1, 64, 1, 1),         # a causal prompt with key splits that early tiles do not reach
    (F16, 64, 2752, 4, 2, 256, 1, 1),      # head_dim 256, past the VALU kernel's few rounds: exact blocks and tiles
    (Q8_0, 64, 1153, 4, 2, 256, 1, 1),     # Q8_0 earlier
    (F32, 9, 8400, 8, 1, 256, 1, 1),       # 72 rows, the keys split
    (Q8_0, 19, 300, 14, 2, 128, 1, 1),     # 133 rows, few workgroups of the VALU kernel: that one
    (Q8_0, 19, 1500, 14, 2, 128, 1, 1),    # ... and more of them: the prompt kernel
]


@pytest.mark.parametrize("ct,n,n_past,n_head,n_kv,hd,ks,vs", PROMPT)
def test_kv_attention_prompt(KV, dev, ct, n, n_past, n_head, n_kv, hd, ks, vs):
    """The prompt kernel at its edges. Relative 2-norm error against the float64 oracle at most 4e-6:
    four times what fp32 products and sums measure at these lengths (0.9e-6); one missing f16 piece of
    any operand costs 2^-12 = 2.4e-4."""
    n_layer, layer, row = 2, 1, n_kv * hd
    n_blocks = (n_past + 15) // 16 + 3
    sb = KV.slot_bytes(ct, row)
    arena_k = np.zeros(n_blocks * n_layer * 16 * sb, np.uint8)
    arena_v = np.zeros_like(arena_k)
    table = make_table(max(n_past, 1), n_blocks, 11 + n)
    seed = 900 + n + n_past + hd
    ks, vs = np.float32(ks), np.float32(vs)
    KV.write(ct, arena_k, n_layer, layer, table, 0, ks * synth.normal(n_past * row, seed).reshape(n_past, row))
    KV.write(ct, arena_v, n_layer, layer, table, 0, vs * synth.normal(n_past * row, seed + 1).reshape(n_past, row))
    q = synth.normal(n * n_head * hd, seed + 2, 0.0, 2.0).reshape(n, n_head * hd)
    k_cur = ks * synth.normal(n * row, seed + 3).reshape(n, row)
    v_cur = vs * synth.normal(n * row, seed + 4).reshape(n, row)
    k_cur[n // 2] *= np.float32(8)  # one key of another magnitude among its neighbours
    v_cur[n // 3] *= np.float32(64)
    scale = np.float32(1.0 / (np.sqrt(hd) * ks))
    k_all = KV.gather(ct, arena_k, n_layer, layer, table, n_past, k_cur).reshape(-1, n_kv, hd)
    v_all = KV.gather(ct, arena_v, n_layer, layer, table, n_past, v_cur).reshape(-1, n_kv, hd)
    ref, parts = KV.attention(q.reshape(n, n_head, hd), k_all, v_all, n_past, scale)

    cache = dc.PagedKVCache(ct, n_blocks, n_layer, n_kv, hd, device=dev)
    cache.k.copy_(to_dev(arena_k, dev))
    cache.v.copy_(to_dev(arena_v, dev))
    args = (layer, to_dev(table, dev), to_dev(q, dev), to_dev(k_cur, dev), to_dev(v_cur, dev), n_past, float(scale))
    out = to_host(cache.attention(*args)).astype(np.float64).reshape(ref.shape)
    assert np.linalg.norm(out - ref) <= 4e-6 * np.linalg.norm(ref)
    assert_rows(out, ref, parts)  # one row of outliers does not stand in for the others


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("n_past,least,most", [(1500, 7, 13), (100, 1, 2)])
def test_kv_attention_prompt_takes_the_splits_its_workspace_holds(KV, dev, n_past, least, most, hd):
    """64 tokens of 8/2 heads: a call is accepted with the partial results of `least` key splits (1: none)
    and told to bring those of `most`. With either, and with room between them, the result holds row by row
    and nothing is written past the workspace; with less it is refused."""
    import torch
    n, n_head, n_kv = 64, 8, 2
    cache = dc.PagedKVCache(F16, n_past // 16 + 2, 1, n_kv, hd, device=dev)
    rows = prompt_rows(hd, n_head, n_kv, n_past, n, 40)
    table = np.random.default_rng(3).permutation(n_past // 16 + 1).astype(np.int32)
    k_past, v_past, q, k, v = (to_dev(r, dev) for r in rows)
    cache.write("k", 0, to_dev(table, dev), 0, k_past)
    cache.write("v", 0, to_dev(table, dev), 0, v_past)
    half = [KV.decode_row(F16, KV.encode_row(F16, r.reshape(-1)), r.size).reshape(r.shape) for r in rows[:2]]
    k_all, v_all = (np.concatenate([h, c]).reshape(-1, n_kv, hd) for h, c in zip(half, rows[3:]))
    scale = np.float32(1.0 / np.sqrt(hd))
    ref, parts = KV.attention(rows[2].reshape(n, n_head, hd), k_all, v_all, n_past, scale)

    def partials(splits):
        o, ml = splits * n * n_head * hd * 4, splits * n * n_head * 8
        return 0 if splits == 1 else (o + 255) // 256 * 256 + (ml + 255) // 256 * 256

    assert dc.kv_attention_workspace_size(n_head, n_kv, hd, n, n_past) == partials(most)
    for nbytes in (partials(least), partials(min(least + 2, most)) - 256, partials(most)):
        buf = torch.full((nbytes + 4096,), 255, dtype=torch.uint8, device=dev)
        out = to_host(cache.attention(0, to_dev(table, dev), q, k, v, n_past, float(scale), workspace=buf[:nbytes]))
        assert_rows(out.astype(np.float64).reshape(ref.shape), ref, parts)
        assert bool((buf[nbytes:] == 255).all())
    if least > 1:
        with pytest.raises(dc.DcqError):
            cache.attention(0, to_dev(table, dev), q, k, v, n_past, float(scale), workspace=buf[:partials(least) - 256])


@pytest.mark.parametrize("ct", [F32, F16])
def test_kv_attention_prompt_infinite_elements_leave_their_neighbours(dev, ct):
    """An infinity in one V element changes that dim alone, and one in a K row only the tokens that see
    the key: the finite elements staged beside them keep their exponents. Against the call without them,
    to fp32 rounding (4e-6, as above; an element's exponent may move with its neighbours' maximum)."""
    n, n_past, hd = 48, 40, 64
    cache = dc.PagedKVCache(ct, 4, 1, 1, hd, device=dev)
    rows = [to_dev(synth.normal(m * hd * h, 70 + i).reshape(m, -1), dev)
            for i, (m, h) in enumerate(((n_past, 1), (n_past, 1), (n, 4), (n, 1), (n, 1)))]
    k_past, v_past, q, k, v = rows
    table = to_dev(np.array([2, 0, 1], np.int32), dev)
    outs = []
    for inf in (False, True):
        if inf:
            v_past[5, 3] = float("inf")
            k[31, 7] = float("inf")
        cache.write("k", 0, table, 0, k_past)
        cache.write("v", 0, table, 0, v_past)
        outs.append(to_host(cache.attention(0, table, q, k, v, n_past, 0.125)).astype(np.float64).reshape(n, 4, hd))
    dims = [d for d in range(hd) if d != 3]
    clean, got = outs[0][:31][..., dims], outs[1][:31][..., dims]
    assert np.linalg.norm(got - clean) <= 4e-6 * np.linalg.norm(clean)
    assert not np.isfinite(outs[1][:31, :, 3]).any()


@pytest.mark.parametrize("scale", [None, 0.0])
@pytest.mark.parametrize("ct,n,n_past,n_head,n_kv,hd", [
    (F32, 33, 0, 4, 1, 64),       # 1 key past a block of 32, 31 padded ones beside it
    (F16, 56, 0, 4, 2, 128),      # 24: one padded group of 8 keys
    (Q8_0, 40, 17, 4, 1, 64),     # 25: no padded group
    (F32, 48, 16, 2, 1, 128),     # 0: no padding
    (F16, 16, 1024, 4, 1, 128),   # 16, the keys split over workgroups
    (Q8_0, 20, 3757, 8, 1, 256),  # 1, split
    (F32, 160, 1200, 16, 8, 256),  # 16, many tiles
])
def test_kv_attention_prompt_zero_rows(KV, dev, ct, n, n_past, n_head, n_kv, hd, scale):
    """Query rows of zeros (and of 1e-9, and a scale of 0) weigh every visible key alike, also beside
    keys that are padding: zero rows at the end of the batch, hidden from the rows before them."""
    k_past, v_past, q, k_cur, v_cur = prompt_rows(hd, n_head, n_kv, n_past, n, 300 + n)
    q[::3] = 0.0
    q[1::6] *= np.float32(1e-9)
    q[-5:], k_cur[-5:], v_cur[-5:] = 0.0, 0.0, 0.0
    scale = 1.0 / np.sqrt(hd) if scale is None else scale
    assert_rows(*prompt_case(KV, dev, ct, hd, n_head, n_kv, k_past, v_past, q, k_cur, v_cur, scale))


@pytest.mark.parametrize("past,cur", [(0.0, 1.0), (0.0, 1e25), (0.0, 1e-30), (1e-30, 1.0), (1.0, 1e30), (1e30, 1e-30),
                                      (1e-4, 1.0), (1e-36, 1e-36), (1e35, 1e36)])
@pytest.mark.parametrize("n_past,hd", [(300, 64), (300, 128), (3800, 256)])
def test_kv_attention_prompt_value_magnitudes(KV, dev, n_past, hd, past, cur):
    """Values of one magnitude in the history and another in the batch: no key's weight is lost from
    the sum of weights, whatever its values are beside the others'."""
    k_past, v_past, q, k_cur, v_cur = prompt_rows(hd, 4, 1, n_past, 40, 400 + hd)
    v_past, v_cur = v_past * np.float32(past), v_cur * np.float32(cur)
    assert_rows(*prompt_case(KV, dev, F32, hd, 4, 1, k_past, v_past, q, k_cur, v_cur, 1.0 / np.sqrt(hd)))


@pytest.mark.parametrize("n_kv,hd", [(512, 64), (256, 128), (256, 256),  # a workgroup per CU: the keys unsplit
                                     (2, 64), (2, 128), (4, 256)])       # the keys split
def test_kv_attention_prompt_missing_history(dev, n_kv, hd):
    """8200 history positions without a block read as zero rows: score 0, value 0, in the sum of weights."""
    import torch
    n, n_past = 33, 8200
    _, _, q, k, v = prompt_rows(hd, n_kv, n_kv, 0, n, 500)
    k *= np.float32(3)  # batch keys that outweigh the history for some rows and not for others
    cache = dc.PagedKVCache(F16, 1, 1, n_kv, hd, device=dev)
    table = torch.full((n_past // 16 + 1,), -1, dtype=torch.int32, device=dev)
    scale = np.float32(1.0 / np.sqrt(hd))
    out = to_host(cache.attention(0, table, to_dev(q, dev), to_dev(k, dev), to_dev(v, dev), n_past, float(scale)))
    qh, kh, vh = (x.astype(np.float64).reshape(n, n_kv, hd).transpose(1, 0, 2) for x in (q, k, v))
    s = qh @ kh.transpose(0, 2, 1) * np.float64(scale)
    sa = np.abs(qh) @ np.abs(kh).transpose(0, 2, 1) * np.float64(scale)
    hidden = np.triu(np.ones((n, n), bool), 1)
    s, sa = np.where(hidden, -np.inf, s), np.where(hidden, 0.0, sa)
    m = np.maximum(s.max(2, keepdims=True), 0.0)
    p = np.exp(s - m)
    p /= n_past * np.exp(-m) + p.sum(2, keepdims=True)
    ref, a = (p @ vh).transpose(1, 0, 2), (p @ np.abs(vh)).transpose(1, 0, 2)
    assert_rows(out.astype(np.float64).reshape(ref.shape), ref, (a, sa.max(2).T))


@pytest.mark.parametrize("bits", [10, 20, 30, 40])
@pytest.mark.parametrize("n_past,hd", [(41, 64), (300, 128), (2040, 256)])
def test_kv_attention_prompt_outlier_keys(KV, dev, n_past, hd, bits):
    """A key 2^bits times its neighbours, hidden from a row (a later token) or of no weight for it, costs
    the keys staged beside it no bits: each row by itself."""
    n, n_kv, n_head = 37, 2, 8
    k_past, v_past, q, k_cur, v_cur = prompt_rows(hd, n_head, n_kv, n_past, n, 600 + bits)
    big = np.float32(2.0 ** bits)
    q.reshape(n, n_head, hd)[:, :, 5] = 2.0
    for k, v, t in ((k_past, v_past, 11), (k_past, v_past, n_past - 2), (k_cur, v_cur, 20)):
        k.reshape(-1, n_kv, hd)[t, :, 5] = -60.0 * np.sqrt(hd)  # score about -173 in base 2
        v[t] *= big
    k_cur[29] *= big   # hidden from the rows before
    v_cur[33] *= big
    out, ref, (a, b) = prompt_case(KV, dev, F32, hd, n_head, n_kv, k_past, v_past, q, k_cur, v_cur, 1.0 / np.sqrt(hd))
    b = np.minimum(b, 64.0)  # the scores that weigh anything; those of the outliers are far below them
    assert_rows(out[:29], ref[:29], (a[:29], b[:29]))


@pytest.mark.parametrize("ct", [F32, F16])
@pytest.mark.parametrize("hd,n_past", [(64, 40), (128, 300), (256, 3130)])
def test_kv_attention_prompt_infinities(KV, dev, ct, hd, n_past):
    """As in fp32 arithmetic: a score of minus infinity has no weight, one of plus infinity makes its row
    NaN, and an infinite value makes its dim infinite for the rows that see it, and leaves the others."""
    n, n_head = 48, 4
    k_past, v_past, q, k_cur, v_cur = prompt_rows(hd, n_head, 1, n_past, n, 700 + hd)
    q.reshape(n, n_head, hd)[:, :, 7] = 0.5 + np.abs(q.reshape(n, n_head, hd)[:, :, 7])
    k_past[9, 7] = -np.inf   # no weight for any row
    k_cur[12, 7] = -np.inf
    out, ref, parts = prompt_case(KV, dev, ct, hd, n_head, 1, k_past, v_past, q, k_cur, v_cur, 1.0 / np.sqrt(hd))
    a, b = parts
    finite = np.where(np.isfinite(b), b, 64.0)  # B without the infinite products
    assert_rows(out, ref, (a, finite))
    v_past[5, 3] = np.inf
    v_past[6, 4] = -np.inf
    k_cur[41, 7] = np.inf    # rows from 41 on
    got, _, _ = prompt_case(KV, dev, ct, hd, n_head, 1, k_past, v_past, q, k_cur, v_cur, 1.0 / np.sqrt(hd))
    assert np.isnan(got[41:]).all()
    assert (got[:41, :, 3] == np.inf).all() and (got[:41, :, 4] == -np.inf).all()
    dims = [d for d in range(hd) if d not in (3, 4)]
    assert_rows(got[:41][..., dims], ref[:41][..., dims], (a[:41][..., dims], finite[:41]))


@pytest.mark.parametrize("ct,n,n_past,n_head,n_kv,hd", [
    (Q8_0, 4, 4095, 32, 8, 128), (F32, 2, 8000, 16, 2, 128), (Q8_0, 8, 1000, 28, 4, 128), (F32, 21, 3000, 7, 1, 64),
    (Q8_0, 8, 4800, 16, 4, 256), (F32, 40, 3800, 4, 2, 256), (F16, 150, 900, 4, 2, 256)])
def test_kv_attention_prompt_precision(KV, dev, ct, n, n_past, n_head, n_kv, hd):
    """Shapes that the VALU kernel would serve in fp32: its relative 2-norm error on them is 3.6e-7 to 4.6e-7,
    that of one chain of MFMAs for all of a score's products 4.9e-7 to 9.0e-7. At most 5e-7."""
    rows = prompt_rows(hd, n_head, n_kv, n_past, n, 800 + n)
    out, ref, _ = prompt_case(KV, dev, ct, hd, n_head, n_kv, *rows, 1.0 / np.sqrt(hd))
    err = np.linalg.norm(out - ref) / np.linalg.norm(ref)
    print(f"{ct} {n} tokens over {n_past}, {n_head}/{n_kv} x {hd}: {err:.3g}")
    assert err <= 5e-7
