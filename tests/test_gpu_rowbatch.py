"""The row-batch kernels at the row counts where their tiles, K splits and dispatch rules change: a
prompt prefilled at once against the same positions decoded one by one (other kernels, themselves
checked against the oracle), at the 270M block shape with a small vocabulary."""
import ctypes
import os

import numpy as np
import pytest

import oracle
import synth
import vrt

pytestmark = pytest.mark.gpu

# Both paths hold activations to 22 bits or better and sum in fp32: 2^-22 per block and projection, a few
# times that after the two blocks' norms; a lost low half or a dropped tile shows as 1e-4 or more.
TOL = 5e-6
SHAPE = dict(n_layers=2, d_model=640, n_heads=4, head_dim=256, ffn=2048, vocab=1000, context=8800, window=512)
ROWS = (1, 2, 15, 16, 17, 33, 64, 65, 129, 255, 300, 513, 700, 1025, 1500, 2047, 2049, 4200, 8192, 8193, 8700)   # past 8192: a second segment, over the first one's cache


def _rel(a, b):
    return float(np.linalg.norm(a.astype(np.float64) - b) / np.linalg.norm(b.astype(np.float64)))


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    path = os.path.join(str(tmp_path_factory.mktemp("rowbatch")), "two_blocks.gguf")
    synth.write_gemma3_gguf(path, seed=21, **SHAPE)
    return path


@pytest.fixture(scope="module")
def narrow(tmp_path_factory):
    """Three heads of 96: key ranges shared by the heads of two query tiles, a short last group."""
    path = os.path.join(str(tmp_path_factory.mktemp("rowbatch")), "narrow.gguf")
    synth.write_gemma3_gguf(path, seed=22, **dict(SHAPE, n_layers=6, d_model=288, n_heads=3, head_dim=96, ffn=160, window=70,
                                                  context=1200))
    return path


@pytest.mark.parametrize("rows", ROWS)
def test_prefill_matches_decode(ctx, model, rows):
    _compare(ctx, model, rows, TOL)


@pytest.mark.parametrize("rows", (1, 31, 32, 33, 100, 333, 1187))
def test_prefill_matches_decode_three_heads(ctx, narrow, rows):
    _compare(ctx, narrow, rows, TOL)


def _compare(ctx, path, rows, tol, kv="f32"):
    g = vrt.Gemma3(ctx, path)
    try:
        if kv != "f32":
            g.set_kv_format(kv)
        ids = synth.uniform_ids(900 + rows, rows, 2, 1000)
        print(f"[rowbatch] {rows} rows", flush=True)
        _, hp = g.prefill(ids, top_k=2, hidden=True)
        lp = g.logits()
        g.reset()
        if rows > 1:
            g.forced(ids[:-1], 0)
        _, hd = g.decode(int(ids[-1]), rows - 1, top_k=2, hidden=True)
        ld = g.logits()
        assert _rel(hp, hd) <= tol
        assert _rel(lp, ld) <= tol
    finally:
        g.close()


def _span(buf, offset, nbytes):
    class At:
        ptr, nbytes_ = buf.ptr + offset, nbytes
        keep = buf
    a = At()
    a.nbytes = nbytes
    return a


@pytest.mark.parametrize("blocks", (1, 2, 7, 127, 128, 129, 300))
@pytest.mark.parametrize("x_off,q_off", ((0, 0), (4, 0), (0, 2), (16, 32), (12, 1)))
def test_codec_runs_and_alignments(ctx, blocks, x_off, q_off):
    """Runs of 128 blocks and what is left of them, on arrays that are 16-byte aligned and not: the bytes and
    values of the oracle, and nothing written past the end."""
    _codec(ctx, blocks, x_off, q_off)


@pytest.mark.parametrize("blocks", (20479, 20480, 20481, 20487, 20607, 20609))
@pytest.mark.parametrize("x_off,q_off", ((0, 0), (16, 32), (4, 0), (0, 2)))
def test_codec_many_blocks(ctx, blocks, x_off, q_off):
    """Both sides of the number of blocks from which aligned arrays pass through LDS, 128 to a workgroup, with last
    runs of 1, 7, 127 and 128 blocks."""
    _codec(ctx, blocks, x_off, q_off)


def _codec(ctx, blocks, x_off, q_off):
    x = synth.normal_f32(33 + blocks, 32 * blocks + blocks % 2, 0.7)[:32 * blocks]
    x[:32] = 0.0   # an all-zero block
    nq = 34 * blocks
    xb, qb, yb = ctx.alloc(x.nbytes + 64), ctx.alloc(nq + 128), ctx.alloc(x.nbytes + 64)
    host = np.zeros(x.nbytes + 64, dtype=np.uint8)
    host[x_off:x_off + x.nbytes] = x.view(np.uint8)
    xb.write(host)
    for variant, name in ((0, "a"), (1, "b")):
        qb.write(np.full(nq + 128, 0xA5, dtype=np.uint8))
        vrt.q8_quantize(ctx, _span(xb, x_off, x.nbytes), x.size, variant, _span(qb, q_off, nq))
        ctx.sync()
        got = qb.read(np.uint8, nq + 128)
        assert np.array_equal(got[q_off:q_off + nq], oracle.quantize(x, name))
        assert np.all(got[:q_off] == 0xA5) and np.all(got[q_off + nq:] == 0xA5)
        vrt.q8_dequantize(ctx, _span(qb, q_off, nq), blocks, _span(yb, x_off, x.nbytes))
        ctx.sync()
        y = yb.read(np.uint8, x.nbytes + 64)[x_off:x_off + x.nbytes].view(np.float32)
        assert np.array_equal(y.view(np.uint32), oracle.dequant(oracle.quantize(x, name)).view(np.uint32))


@pytest.mark.parametrize("k,rows", ((640, 32768), (576, 32773), (640, 32767), (544, 40001), (608, 33000)))
def test_matvec_many_rows(ctx, k, rows):
    """Both sides of the rule that gives many rows of 17 to 20 blocks five blocks per lane; odd block counts put
    every other row two bytes off a dword."""
    w = synth.q8_matrix(5, "t", rows, k)
    x = synth.normal_f32(6, k, 1.0)
    wd, xd, yd = ctx.upload(w), ctx.upload(x), ctx.alloc(rows * 4)
    vrt.q8_matvec(ctx, wd, 0, xd, yd, k, rows, w_bytes=w.size)
    ctx.sync()
    ref = oracle.matvec_f64(w, x, rows)
    # limb and summation error, as bounded per row in the standalone kernels' tests, over this matrix's rows
    assert np.max(np.abs(yd.read(np.float32, rows) - ref)) <= 2e-6 * np.max(np.abs(ref))


@pytest.mark.parametrize("k", (32, 96, 512, 544, 2048, 2080, 8224, 16384))
def test_matvec_input_lengths(ctx, k):
    """Activations read by whole and partly filled passes of the limb build (128 values per wave, four waves, four
    passes in flight), from an address that is only 4-byte aligned, with NaNs on both sides of them."""
    rows = 67
    w = synth.q8_matrix(7, "t", rows, k)
    x = synth.normal_f32(8, k, 1.0)
    host = np.full(k + 160, np.nan, dtype=np.float32)
    host[1:1 + k] = x
    wd, xd, yd = ctx.upload(w), ctx.upload(host), ctx.alloc(rows * 4)
    vrt.q8_matvec(ctx, wd, 0, _span(xd, 4, x.nbytes), yd, k, rows, w_bytes=w.size)
    ctx.sync()
    ref = oracle.matvec_f64(w, x, rows)
    # limb and summation error, as bounded per row in the standalone kernels' tests, over this matrix's rows
    assert np.max(np.abs(yd.read(np.float32, rows) - ref)) <= 2e-6 * np.max(np.abs(ref))


@pytest.mark.parametrize("n", (1, 1023, 1025, 8191, 8192, 8193, 10240, 2097152, 2100001))
def test_argmax_lengths(ctx, n):
    """One workgroup and several, runs that end inside, at and past a pass; ties and NaNs across runs."""
    x = synth.normal_f32(n, n, 1.0)
    x[n // 3::97] = np.nan
    x[[n // 2, n - 1]] = 9.0
    xd, out = ctx.upload(x), ctx.alloc(8)
    vrt.argmax(ctx, xd, n, out)
    ctx.sync()
    got = out.read(np.uint32, 2)
    index, value = oracle.argmax(x)
    assert got[0] == index and got[1:].view(np.float32)[0] == np.float32(value)


@pytest.mark.parametrize("kv,tol", (("f16", 4e-4), ("bf16", 2e-3)))
@pytest.mark.parametrize("rows", (37, 700, 8300))
def test_prefill_matches_decode_16bit_cache(ctx, model, kv, tol, rows):
    """Both paths round keys and values to the cache's entries; one that lies near a tie may round the other way (the
    tolerances are an entry's rounding, 2^-11 and 2^-8, spread over the row)."""
    _compare(ctx, model, rows, tol, kv)


@pytest.mark.parametrize("base", (0, 1, 2, 3))
def test_weights_at_any_address(ctx, base):
    """Only the weights' offsets have to be multiples of four; the buffer itself may start anywhere (a view of a
    larger one). One kernel per load form: the FFN's gate/up rows, many rows of 20 blocks, a plain matrix."""
    k, ffn, out, many = 640, 96, 64, 32768
    x = synth.normal_f32(12, k, 1.0)
    parts = [synth.q8_matrix(13, n, r, c) for n, r, c in (("gate", ffn, k), ("up", ffn, k), ("down", out, ffn), ("big", many, k))]
    offs = np.concatenate([[0], np.cumsum([(p.size + 3) // 4 * 4 for p in parts])]).astype(int)
    host = np.zeros(offs[-1] + 64, dtype=np.uint8)
    for p, o in zip(parts, offs):
        host[base + o:base + o + p.size] = p
    wd, xd = ctx.upload(host), ctx.upload(x)
    w = _span(wd, base, int(offs[-1]) + 8)
    ws, y, yb = ctx.alloc(2 * ffn * 4), ctx.alloc(out * 4), ctx.alloc(many * 4)
    vrt.q8_ffn(ctx, w, *(int(o) for o in offs[:3]), k, ffn, out, xd, ws, y)
    vrt.q8_matvec(ctx, w, int(offs[3]), xd, yb, k, many)
    ctx.sync()
    up = oracle.matvec_f64(parts[1], x, ffn)
    gate = oracle.matvec_f64(parts[0], x, ffn)
    h = 0.5 * gate * (1.0 + np.tanh(0.7978845608028654 * (gate + 0.044715 * gate ** 3))) * up
    got = ws.read(np.float32, 2 * ffn)
    down = oracle.matvec_f64(parts[2], h.astype(np.float32), out)
    # limb and summation error, as in test_matvec_many_rows; h: that of its two factors and the GELU's own; the
    # product of h by the down matrix carries h's over
    for a, ref, tol in ((got[ffn:], up, 2e-6), (got[:ffn], h, 6e-6), (y.read(np.float32, out), down, 8e-6),
                        (yb.read(np.float32, many), oracle.matvec_f64(parts[3], x, many), 2e-6)):
        assert np.max(np.abs(a - ref)) <= tol * np.max(np.abs(ref))


def test_prefill_repeats_after_other_prompts(ctx, model, tmp_path):
    """A prompt's results do not depend, in any bit, on the prompts before it: the query tile that its length leaves
    partly filled holds another prompt's queries in the rows past the end. QK-norm weights of 2 spread the scores
    so far that those rows' maxima would move where the prompt's own do not."""
    path = os.path.join(str(tmp_path), "spread.gguf")
    hd = SHAPE["head_dim"]
    synth.edit_gguf(model, path, f32={f"blk.{l}.attn_{n}_norm.weight": np.full(hd, 2.0, np.float32) for l in range(2) for n in "qk"})
    ids = synth.uniform_ids(41, 300, 2, 1000)
    g = vrt.Gemma3(ctx, path)
    try:
        def run():
            (i, v), hid = g.prefill(ids, top_k=2, hidden=True)
            return hid, g.logits()
        runs = [run()]
        for seed in (42, 43, 44, 45):
            g.prefill(synth.uniform_ids(seed, 320, 2, 1000), top_k=0)
            runs.append(run())
        for hid, logits in runs[1:]:
            np.testing.assert_array_equal(hid, runs[0][0])
            np.testing.assert_array_equal(logits, runs[0][1])
    finally:
        g.close()


def test_executor_memory_follows_its_context(ctx, tmp_path):
    """An executor of 512 positions does not hold the attention partials of 8192 (268 MB at 4 heads of 256): its weights
    twice over (30 MB), the row buffers and K-split partials of 512 rows (45 MB) and 17 MB of partials, rounded up by
    the allocator."""
    hip = ctypes.CDLL("libamdhip64.so.7")   # the runtime that libvrt_hip.so is linked to

    def free_bytes():
        free, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return free.value
    path = os.path.join(str(tmp_path), "short.gguf")
    synth.write_gemma3_gguf(path, seed=23, **dict(SHAPE, context=512))
    vrt.Gemma3(ctx, path).close()   # what the first executor of a process allocates once
    free = free_bytes()
    g = vrt.Gemma3(ctx, path)
    try:
        took = free - free_bytes()
        print(f"[rowbatch] 512 positions: {took / 1e6:.0f} MB", flush=True)
        assert took < 150e6
        ids = synth.uniform_ids(47, 512, 2, 1000)
        g.prefill(ids, top_k=1)   # 64 pairs in up to 8 chunks
    finally:
        g.close()


# Batched steps against single-sequence decode. Shapes by what decides their kernels: K blocks of the LM head (20, and 24,
# 36: two groups of five per wave; 41: past k_gm_lm, the general GEMM and argmax, both of its tile widths), head
# dimensions without expanded weights (40, and 36, where a run of four straddles the RoPE halves). 26003 rows make
# 1626 tiles, the last of three rows: three or four in each of 512 chunks, six or seven in each of 256.
BATCH = dict(
    k20=dict(vocab=26003),
    k24=dict(d_model=768, vocab=1003),
    k36=dict(d_model=1152, vocab=26003),
    k41=dict(d_model=1312, head_dim=64, ffn=256, vocab=1003),
    k41w=dict(d_model=1312, head_dim=64, ffn=256, vocab=16384),
    hd40=dict(d_model=320, head_dim=40, ffn=640, vocab=1003),
    hd36=dict(d_model=288, n_heads=8, head_dim=36, ffn=576, vocab=1003),
)


@pytest.fixture(scope="module")
def batch_model(tmp_path_factory):
    d = str(tmp_path_factory.mktemp("batch"))

    def get(key, **kw):
        path = os.path.join(d, key + ".gguf")
        if not os.path.exists(path):
            synth.write_gemma3_gguf(path, seed=31, **dict(SHAPE, context=400, **BATCH.get(key, {})) | kw)
        return path
    return get


def _check_row(g, b, row, idx, val, token, pos, where):
    g.decode(token, pos, top_k=2)
    want, got = g.logits(), b.logits(row)
    assert _rel(got, want) <= TOL, where
    index, value = oracle.argmax(got)   # the row's own greedy token
    assert idx[row] == index and val[row] == np.float32(value), where


@pytest.mark.parametrize("key,n", [("k20", n) for n in (1, 8, 9, 16, 17, 32, 33, 64)] + [("k24", 7), ("k24", 16)] +
                         [("k36", n) for n in (9, 17, 33, 64)] +
                         [(k, n) for k in ("k41", "k41w", "hd40", "hd36") for n in (5, 64)])
def test_batch_rows_match_decode(ctx, batch_model, key, n):
    """Every row of a step of n sequences, a third of them two positions ahead, against the sequence decoded alone."""
    path = batch_model(key)
    vocab = BATCH[key]["vocab"]
    g = vrt.Gemma3(ctx, path)
    b = vrt.Gemma3Batch(g, n, 16)
    try:
        print(f"[rowbatch] {key}: {n} sequences", flush=True)
        ids = synth.uniform_ids(60 + n, 4 * n, 2, vocab).reshape(n, 4).astype(int)
        ahead = [i for i in range(n) if i % 3 == 0]
        for t in (0, 1):
            b.step(ahead, [ids[i][t] for i in ahead])
        order = list(range(n))[::-1]   # rows are not the sequences' numbers
        at = [2 if i in ahead else 0 for i in range(n)]
        for _ in range(2):
            idx, val = b.step(order, [ids[i][at[i]] for i in order])
            at = [a + 1 for a in at]
        for row, i in enumerate(order):
            g.reset()
            if at[i] > 1:
                g.forced(ids[i][:at[i] - 1].astype(np.uint32), 0)
            _check_row(g, b, row, idx, val, int(ids[i][at[i] - 1]), at[i] - 1, f"row {row}")
    finally:
        b.close()
        g.close()


# Six blocks (the last global), window 64.
LONG = dict(n_layers=6, window=64, ffn=256, vocab=1003)
BATCH.update(long64=dict(LONG, d_model=128, n_heads=2, head_dim=64), long36=dict(LONG, d_model=288, n_heads=8, head_dim=36),
             long256=dict(LONG, d_model=320, n_heads=1, head_dim=256))


@pytest.mark.parametrize("key", ("long64", "long36", "long256"))
def test_batch_passes_256_positions(ctx, batch_model, key):
    """Three sequences, one of them past 256 positions in the global block, where a step goes from the short
    attention to the chunked kernels and their merge: every row from position 250 to 262 of the longest, with
    rows of few positions in the same steps, against the sequences decoded alone; then the long one leaves
    and the others go back to the short kernel."""
    path = batch_model(key)
    g = vrt.Gemma3(ctx, path)
    b = vrt.Gemma3Batch(g, 3, 300)
    try:
        print(f"[rowbatch] {key}: past 256 positions", flush=True)
        n = (262, 40, 11)
        ids = [synth.uniform_ids(80 + i, 264, 2, 1003) for i in range(3)]
        results = {}   # (sequence, position) -> token, value, logits
        at = [0, 0, 0]

        def step(rows):
            idx, val = b.step(rows, [int(ids[i][at[i]]) for i in rows])
            for r, i in enumerate(rows):
                if i or at[i] >= 250:
                    results[i, at[i]] = idx[r], val[r], b.logits(r)
                at[i] += 1
        while at[0] < n[0]:   # the shorter ones join so that they end with the long one
            step([i for i in range(3) if at[0] >= n[0] - n[i] or i == 0])
        for _ in range(2):
            step([2, 1])
        for i in range(3):
            first = min(p for j, p in results if j == i)
            g.reset()
            if first:
                g.forced(ids[i][:first], 0)
            for p in range(first, at[i]):
                g.decode(int(ids[i][p]), p, top_k=2)
                want, (idx, val, got) = g.logits(), results[i, p]
                assert _rel(got, want) <= TOL, f"sequence {i} position {p}"
                assert (idx, val) == oracle.argmax(got), f"sequence {i} position {p}"
    finally:
        b.close()
        g.close()


@pytest.mark.parametrize("kv,tol", (("f32", 1e-5), ("f16", 4e-4), ("bf16", 2e-3)))
@pytest.mark.parametrize("rows", (8193, 8700))
def test_second_segment_with_a_global_block(ctx, batch_model, kv, tol, rows):
    """Prompts past the 8192 positions of one segment, of six blocks: the second segment's global block attends to all
    of the first through the cache (a history of 8192 keys, cut into chunks with the segment's own), its local ones
    to the window's start. Tolerances as above, the fp32 one for three times the blocks."""
    path = batch_model("segments", **dict(LONG, d_model=256, n_heads=2, head_dim=64, context=8800))
    _compare(ctx, path, rows, tol, kv)


def test_batch_table_not_on_16_bytes(ctx, batch_model, monkeypatch):
    """A tensor section that starts four bytes past a 16-byte unit: k_gm_lm's direct loads do not fit, so the LM head is
    the general GEMM and argmax, and the tokens are those of the aligned section."""
    path, n = batch_model("k20"), 5
    ids = synth.uniform_ids(90, 3 * n, 2, 26003).reshape(3, n)

    def run():
        g = vrt.Gemma3(ctx, path)
        b = vrt.Gemma3Batch(g, n, 16)
        try:
            out = [b.step(range(n), t) for t in ids]
            return g.arena.ptr, out, [b.logits(r) for r in range(n)]
        finally:
            b.close()
            g.close()
    at, want, logits = run()
    assert at % 16 == 0

    class Shifted(vrt.DeviceBuffer):
        def __init__(self, ctx, nbytes):
            super().__init__(ctx, nbytes + 64)
            self.ptr += 4

        def free(self):
            if getattr(self, "ptr", None):
                self.ptr -= 4
            super().free()
    monkeypatch.setattr(vrt, "DeviceBuffer", Shifted)
    at, got, logits4 = run()
    assert at % 16 == 4
    for (i, v), (j, w), in zip(got, want):
        np.testing.assert_array_equal(i, j)
        assert np.max(np.abs(v - w)) <= TOL * np.max(np.abs(w))
    for a, b in zip(logits4, logits):
        assert _rel(a, b) <= TOL
