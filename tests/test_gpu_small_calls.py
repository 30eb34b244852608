"""GPU parity of the kernels that a call's size chooses, at the sizes around
their limits, against the oracle: the arithmetic encoder's load groups, decode
attention by rows, few-row GEMMs, whole-stream decode, layer tail, 128 x 256
tiles and the wave counts of the unfused decoder step; and device memory that
jobs hand on."""
import ctypes as C
import queue
import threading

import numpy as np
import pytest

from conftest import MODEL_PATH

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def amd():
    import czip_amd
    if czip_amd.device_count() < 1:
        pytest.fail("no HIP device visible")
    return czip_amd


@pytest.fixture(scope="module")
def pair(amd, orc):
    return amd.Model(amd.ModelWeights(MODEL_PATH)), orc.Model.from_file(MODEL_PATH)


def free_device_memory():
    """Free bytes of the device, from the HIP runtime that the library links."""
    hip = C.CDLL("libamdhip64.so.7")
    free, total = C.c_size_t(), C.c_size_t()
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


@pytest.mark.parametrize("chunk", [1, 7, 8, 9, 16, 65])
def test_encoder_chunk_lengths(pair, chunk):
    """Chunk lengths around the encoder's groups of eight intervals, with a
    ragged last chunk; uniform ids, so that symbols of 20 to 30 bits (several
    words' worth of pending bits among them) are common."""
    gm, om = pair
    n = 67 * chunk + (chunk + 1) // 2
    toks = np.random.default_rng(chunk).integers(0, 1024, n).astype(np.uint32)
    assert gm.compress_chunks(toks, chunk) == om.compress_many(toks, chunk, threads=4)


def test_job_memory_reuse(pair):
    """Jobs of one context whose device memory comes back from earlier jobs of
    other sizes, two of them alive at once, and a decode after a compress:
    the bytes depend on nothing a block held before."""
    gm, om = pair
    rng = np.random.default_rng(5)
    sizes = [(3000, 512), (40, 64), (9001, 128), (40, 64), (3000, 512), (700, 1024)]
    ref = []
    for n, chunk in sizes:
        toks = rng.integers(0, 1024, n).astype(np.uint32)
        ref.append((toks, chunk, om.compress_many(toks, chunk, threads=4)))
    for toks, chunk, want in ref:
        assert gm.compress_chunks(toks, chunk) == want
        ntoks = [min(chunk, toks.size - i) for i in range(0, toks.size, chunk)]
        assert np.array_equal(gm.decompress_chunks(want, ntoks), toks)
    jobs = [gm.compress_plan(toks, chunk) for toks, chunk, _ in ref]
    for j in jobs[::2] + jobs[1::2]:
        j.run()
    for j, (_, _, want) in zip(jobs, ref):
        assert j.fetch() == want
        j.free()


def test_jobs_outlive_their_context(amd, pair):
    """A collector may finalize a model before its jobs: their memory goes with
    the context, and all that is left to do with them is to free them."""
    _, om = pair
    toks = np.random.default_rng(12).integers(0, 1024, 2000).astype(np.uint32)
    want = om.compress_many(toks, 64, threads=4)
    gm = amd.Model(amd.ModelWeights(MODEL_PATH))
    jobs = [gm.compress_plan(toks, 64), gm.decompress_plan(want, [64] * 31 + [16]), gm.compress_plan(toks, 64),
            gm.compress_plan(toks, 64)]
    for j in jobs[:3]:
        j.run()
    jobs[2].free()
    gm.close()
    for j in (jobs[0], jobs[1], jobs[3]):
        for call in (j.run, j.fetch):
            with pytest.raises(amd.CzipError) as e:
                call()
            assert e.value.code == -1
        j.free()
    # jobs freed by another thread while this one makes more
    gm = amd.Model(amd.ModelWeights(MODEL_PATH))
    made = queue.Queue()

    def free_all():
        while (j := made.get()) is not None:
            j.free()

    t = threading.Thread(target=free_all)
    t.start()
    for _ in range(300):
        made.put(gm.compress_plan(toks[:64], 64))
    made.put(None)
    t.join()
    assert gm.compress_chunks(toks, 64) == want
    gm.close()
    # a context after it, and a job freed out of order in it
    gm = amd.Model(amd.ModelWeights(MODEL_PATH))
    a, b, c = (gm.compress_plan(toks, 64) for _ in range(3))
    b.free()
    for j in (a, c):
        j.run()
        assert j.fetch() == want
        j.free()
    gm.close()


def test_job_memory_trim(amd, pair):
    """Freed jobs' memory goes back to the driver on demand, the live ones' stays."""
    _, om = pair
    gm = amd.Model(amd.ModelWeights(MODEL_PATH))
    toks = np.random.default_rng(8).integers(0, 1024, 300_000).astype(np.uint32)
    gm.compress_chunks(toks[:2000], 512)  # what a first launch takes for itself
    gm.trim()
    before = free_device_memory()
    gm.compress_chunks(toks, 512)
    live = gm.compress_plan(toks[:2000], 512)
    kept = before - free_device_memory()
    assert kept > 500e6  # 300 thousand rows of about 4 KB
    gm.trim()
    assert 0 <= before - free_device_memory() < 100e6  # the live job's
    live.run()
    assert live.fetch() == om.compress_many(toks[:2000], 512, threads=4)
    live.free()
    gm.trim()
    assert before - free_device_memory() < 16 << 20  # the runtime keeps a few pieces of 2 MB for small allocations
    assert gm.compress_chunks(toks[:2000], 512) == om.compress_many(toks[:2000], 512, threads=4)


@pytest.mark.parametrize("d_ff,env,want", [(1024, None, 0), (4160, None, 1), (1024, "0", 1)])
def test_split_k_workspace_only_where_used(amd, tmp_path, monkeypatch, d_ff, env, want):
    """A session's split-K workspace (64 KB a stream at d1024) is there where a
    launch can take the split-K row GEMM: K past 4096, or the few-row GEMMs off."""
    from czip_amd import synth
    path = synth.write_random_model(str(tmp_path / "w.czm"), d=1024, n_layers=1, n_heads=16, n_kv=1, d_ff=d_ff,
                                    vocab=1024, ctx=8, seed=860)
    if env is not None:
        monkeypatch.setenv("CZIP_SKINNY_ROWS", env)
    S = 4000
    gm = amd.Model(amd.ModelWeights(path, amd.KV_GQA))
    before = free_device_memory()
    gm.decode_begin(S, 4)
    used = before - free_device_memory()
    gm.decode_end()
    rest = S * (2 * 4 * 1024 + 7 * 1024 + d_ff + 2 * 64 * 64)  # tables and logits, rows, caches
    assert (used > rest + S * 32 * 1024) == bool(want), (used, rest)


def test_job_memory_threads(amd, pair):
    """A context per thread, both taking and returning device memory at the same time."""
    _, om = pair
    toks = np.random.default_rng(6).integers(0, 1024, 5000).astype(np.uint32)
    want = {c: om.compress_many(toks, c, threads=4) for c in (64, 200)}
    bad = []

    def work(c):
        try:
            gm = amd.Model(amd.ModelWeights(MODEL_PATH))
            for _ in range(6):
                if gm.compress_chunks(toks, c) != want[c]:
                    bad.append(c)
            gm.close()
        except Exception as e:  # reported below
            bad.append(e)

    ts = [threading.Thread(target=work, args=(c,)) for c in want]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad


# Decode steps of few rows take the one-row-per-wave attention kernel; one-layer
# models of 1024 tokens decode as a whole instead (CZIP_DECODE_FUSED=0: step by
# step).  The attention's edge cases through the row kernel, and through the
# kernel that packs streams or heads into a wave's rows (CZIP_ATTN_ROWS=0).
def test_decode_attention_row_edge_cases(amd, orc, tmp_path, monkeypatch):
    import test_gpu_parity as parity
    monkeypatch.setenv("CZIP_DECODE_FUSED", "0")
    parity.test_decompress_attention_edge_cases(amd, orc, tmp_path)


@pytest.mark.parametrize("sink", [False, True])
@pytest.mark.parametrize("kv,n_kv", [("rust", 1), ("gqa", 2)])
def test_decode_attention_row_general(amd, orc, tmp_path, sink, kv, n_kv):
    """Two layers whose scores pass 2^30 and wrap in their differences, an exp
    table whose first entry is not 65535, with and without a sink."""
    from test_gpu_parity import _write_model
    from czip_amd import synth
    t, meta = synth.random_model_tensors(d=256, n_layers=2, n_heads=4, n_kv=n_kv, d_ff=128, vocab=1024, ctx=256,
                                         seed=430 + n_kv, sink=sink)
    for l in range(2):
        t[f"layers.{l}.attn.score_mult"] = np.array([1 << 30, -(1 << 30), 1 << 27, -5], np.int32)
    t["lut.exp2"][0] = 65000
    path = _write_model(str(tmp_path / "g.czm"), t, meta)
    mode = amd.KV_GQA if kv == "gqa" else amd.KV_RUST_COMPAT
    gm, om = amd.Model(amd.ModelWeights(path, mode)), orc.Model.from_file(path, mode)
    gm.set_profiling(True)
    toks = synth.zipf_ids(3 * 150 - 41, 1024, seed=431)
    chunks = om.compress_many(toks, 150, threads=4)
    assert np.array_equal(gm.decompress_chunks(chunks, [150, 150, 109]), toks)
    assert gm.kernel_stats("dec_fused")[0] == 0 and gm.kernel_stats("attn_decode_rows")[0] == 2 * 150


@pytest.mark.parametrize("heads,most", [(8, 4), (16, 1), (10, 2)])
def test_decode_attention_rows_limit(amd, orc, tmp_path, monkeypatch, heads, most):
    """The most streams whose attention takes a row a wave: as many rows as the
    limit, three quarters of it for groups of more than 8 heads."""
    from czip_amd import synth
    path = synth.write_random_model(str(tmp_path / "l.czm"), d=64 * heads, n_layers=2, n_heads=heads, n_kv=1, d_ff=64,
                                    vocab=1024, ctx=70, seed=440 + heads)
    monkeypatch.setenv("CZIP_ATTN_ROWS", "32")
    gm, om = amd.Model(amd.ModelWeights(path, amd.KV_GQA)), orc.Model.from_file(path, amd.KV_GQA)
    gm.set_profiling(True)
    toks = synth.zipf_ids((most + 1) * 66, 1024, seed=441)
    chunks = om.compress_many(toks, 66, threads=4)
    for S in (most, most + 1):
        gm.reset_stats()
        assert np.array_equal(gm.decompress_chunks(chunks[:S], [66] * S), toks[:66 * S])
        assert gm.kernel_stats("attn_decode")[0] == 2 * 66
        assert gm.kernel_stats("attn_decode_rows")[0] == (2 * 66 if S == most else 0)


def test_decode_attention_tile_edge_cases(amd, orc, tmp_path, monkeypatch):
    import test_gpu_parity as parity
    monkeypatch.setenv("CZIP_ATTN_ROWS", "0")
    parity.test_decompress_attention_edge_cases(amd, orc, tmp_path)


def test_decode_attention_tile_wrap(amd, orc, tmp_path, monkeypatch):
    import test_gpu_parity as parity
    monkeypatch.setenv("CZIP_ATTN_ROWS", "0")
    parity.test_vacc_wrap(amd, orc, tmp_path)


@pytest.mark.parametrize("i", [0, 3, 7, 11, 16, 22, 28, 35])
def test_decode_attention_tile_random_shapes(orc, tmp_path, monkeypatch, i):
    import test_gpu_random_shapes as shapes
    monkeypatch.setenv("CZIP_ATTN_ROWS", "0")
    shapes.test_random_shape_roundtrip(orc, tmp_path, monkeypatch, i)


@pytest.mark.parametrize("n", [1, 3, 4, 5, 63, 64, 65, 128, 129])
def test_decode_attention_rows_key_counts(amd, pair, monkeypatch, n):
    """Key counts around the 4-key blocks and the 64-key tiles, and stream
    counts around a workgroup's four rows: step by step, and the whole-stream
    kernel's own rows."""
    _, om = pair
    toks = np.random.default_rng(100 + n).integers(0, 1024, 3 * n).astype(np.uint32)
    chunks = om.compress_many(toks, n, threads=4)
    for fused in (0, 4096):
        monkeypatch.setenv("CZIP_DECODE_FUSED", str(fused))
        gm = amd.Model(amd.ModelWeights(MODEL_PATH))
        gm.set_profiling(True)
        for s in (1, 2, 3):
            assert np.array_equal(gm.decompress_chunks(chunks[:s], [n] * s), toks[:s * n])
        assert gm.kernel_stats("dec_fused")[0] == (3 if fused else 0)
        assert gm.kernel_stats("attn_decode_rows")[0] == (0 if fused else 3 * n)


@pytest.mark.parametrize("heads,kv,d_ff", [(1, 1, 64), (5, 1, 1600), (6, 2, 128), (14, 7, 832), (16, 4, 3136)])
def test_few_row_gemms(amd, orc, tmp_path, heads, kv, d_ff):
    """The few-row GEMMs (and the row norms behind them) at row counts around
    their 16- and 64-row tiles and past their last one, for K of 1, 5, 6, 13,
    14, 16, 25 and 49 steps of 64 (all three wave counts, with and without a
    remainder)."""
    import test_gpu_parity as parity
    from czip_amd import synth
    path = synth.write_random_model(str(tmp_path / "m.czm"), d=64 * heads, n_layers=2, n_heads=heads, n_kv=kv,
                                    d_ff=d_ff, vocab=1088, ctx=600, seed=300 + heads)
    gm = amd.Model(amd.ModelWeights(path, amd.KV_GQA))
    om = orc.Model.from_file(path, amd.KV_GQA)
    gm.set_profiling(True)
    for lens in ([1], [16], [17], [63], [32, 32], [13, 5, 13, 13, 13], [129], [256], [257], [512], [513]):
        seen = gm.kernel_stats("few_row_gemm")[0]
        parity._check_logits(gm, om, max(lens), lens, 7 + len(lens), 1088)
        if max(lens) <= 512:  # QKV of the second layer, O, up and down of both, and the head up to 256 rows
            assert gm.kernel_stats("few_row_gemm")[0] - seen == (8 if len(lens) * max(lens) <= 256 else 7)


# The whole-stream decode kernel (one-layer models, V = 1024).  Up to 256
# streams it takes one stream a workgroup, then two, ... sixteen; the streams
# end at different steps, some before the first.
FUSED_SHAPES = [  # d, kv heads, d_ff, kv mode, sink, general attention
    (384, 1, 1024, "rust", False, False), (256, 2, 64, "gqa", True, False), (512, 4, 960, "gqa", False, False),
    (512, 2, 1024, "rust", True, True), (256, 1, 320, "rust", False, True), (384, 3, 448, "gqa", True, False)]


@pytest.mark.parametrize("i", range(len(FUSED_SHAPES)))
def test_fused_decode_shapes(amd, orc, tmp_path, monkeypatch, i):
    from test_gpu_parity import _write_model
    from czip_amd import synth
    d, n_kv, d_ff, kv, sink, general = FUSED_SHAPES[i]
    t, meta = synth.random_model_tensors(d=d, n_layers=1, n_heads=d // 64, n_kv=n_kv, d_ff=d_ff, vocab=1024, ctx=256,
                                         seed=400 + i, sink=sink)
    if general:  # scores past 2^30 and an exp table whose first entry is not 65535
        t["layers.0.attn.score_mult"] = np.resize(np.array([1 << 30, -(1 << 30), 1 << 27, -5], np.int32), d // 64)
        t["lut.exp2"][0] = 65000
    path = _write_model(str(tmp_path / "f.czm"), t, meta)
    mode = amd.KV_GQA if kv == "gqa" else amd.KV_RUST_COMPAT
    om = orc.Model.from_file(path, mode)
    rng = np.random.default_rng(410 + i)
    toks = synth.zipf_ids(5 * 200, 1024, seed=420 + i)
    chunks = om.compress_many(toks, 200, threads=8)
    gm = amd.Model(amd.ModelWeights(path, mode))
    gm.set_profiling(True)
    assert np.array_equal(gm.decompress_chunks(chunks, [200] * 5), toks)
    assert gm.kernel_stats("dec_fused")[0] == 1  # the kernel under test ran
    # many short streams of different lengths, some of them empty
    for S in (257, 700, 4000):
        lens = rng.integers(0, 6, S)
        part = [toks[r:r + n] for r, n in zip(rng.integers(0, 900, S), lens)]
        coded, seen = [], {}
        for c in part:
            k = c.tobytes()
            if k not in seen:
                seen[k] = om.compress_many(c, max(c.size, 1), threads=1)[0] if c.size else b""
            coded.append(seen[k])
        assert np.array_equal(gm.decompress_chunks(coded, lens), np.concatenate(part))


@pytest.mark.parametrize("T,most", [(1024, 2804), (800, 3173)])
def test_fused_decode_stream_limit(amd, pair, T, most):
    """The shipped model's streams decode as a whole up to the line where its
    row-wise attention falls behind, and step by step past it."""
    from czip_amd import synth
    gm = amd.Model(amd.ModelWeights(MODEL_PATH))
    gm.set_profiling(True)
    toks = synth.zipf_ids((most + 1) * T, 1024, seed=T)
    chunks = gm.compress_chunks(toks, T)
    for S in (most, most + 1):
        gm.reset_stats()
        assert np.array_equal(gm.decompress_chunks(chunks[:S], [T] * S), toks[:S * T])
        assert gm.kernel_stats("dec_fused")[0] == (1 if S == most else 0)


def test_fused_decode_truncated_bytes(amd, pair):
    """Streams cut short read zeros past their end, as the step kernels do."""
    gm, om = pair
    toks = np.random.default_rng(9).integers(0, 1024, 300).astype(np.uint32)
    chunks = om.compress_many(toks, 60, threads=2)
    for cut in (0, 1, 3, 7, 8, 9, 40):
        part = [c[:cut] for c in chunks]
        assert np.array_equal(gm.decompress_chunks(part, [60] * 5), om.decompress_many(part, [60] * 5))


@pytest.mark.parametrize("d,kv,d_ff,mode", [(256, 2, 64, "gqa"), (384, 1, 1024, "rust"), (512, 2, 2048, "gqa"), (512, 1, 704, "rust")])
def test_layer_tail(amd, orc, tmp_path, monkeypatch, d, kv, d_ff, mode):
    """A layer after its attention as one kernel: 16 rows a workgroup up to
    4096 rows, then 32, with partial last workgroups; prefill (logits) and
    decode steps (where it also projects the next layer's Q/K/V)."""
    from czip_amd import synth
    path = synth.write_random_model(str(tmp_path / "t.czm"), d=d, n_layers=2, n_heads=d // 64, n_kv=kv, d_ff=d_ff,
                                    vocab=1024, ctx=64, seed=500 + d_ff)
    m = amd.KV_GQA if mode == "gqa" else amd.KV_RUST_COMPAT
    monkeypatch.setenv("CZIP_SKINNY_ROWS", "0")  # also below the few-row GEMMs' limit
    monkeypatch.setenv("CZIP_TAIL_ROWS", "100000")
    gm = amd.Model(amd.ModelWeights(path, m))
    om = orc.Model.from_file(path, m)
    gm.set_profiling(True)
    rng = np.random.default_rng(d + d_ff)
    least = d * ((d + 128 * (kv if mode == "gqa" else 1)) + d + 3 * d_ff) // 2500  # fewest rows that take it
    for rows in (least + 1, 1537, 4096, 4097, 4131):
        toks = rng.integers(0, 1024, 6 * rows).astype(np.uint32)  # chunks of 6: one row a stream when decoded
        seen = gm.kernel_stats("layer_tail")[0]
        chunks = gm.compress_chunks(toks[:rows], 6)
        assert gm.kernel_stats("layer_tail")[0] > seen
        assert chunks == om.compress_many(toks[:rows], 6, threads=8)
        coded = gm.compress_chunks(toks, 6)
        some = sorted({0, 15, 16, rows // 2, rows - 1})
        assert [coded[i] for i in some] == om.compress_many(np.concatenate([toks[6 * i:6 * i + 6] for i in some]), 6, threads=8)
        seen = gm.kernel_stats("layer_tail")[0]
        assert np.array_equal(gm.decompress_chunks(coded, [6] * rows), toks)
        assert gm.kernel_stats("layer_tail")[0] > seen


@pytest.mark.parametrize("d,kv,d_ff,prefill,decode", [
    (512, 2, 2048, {8192: 1, 8193: 0, 12288: 0, 16400: 0}, {8192: 1, 8193: 0, 12287: 0, 12288: 1, 20480: 1, 20481: 0}),
    (512, 2, 1536, {8192: 1, 12287: 0, 12288: 1, 20481: 0}, {8193: 1, 20480: 1}),
    (384, 1, 3072, {4096: 1, 4097: 0, 6143: 0, 6144: 1, 8192: 1, 8193: 0}, {4096: 1, 4097: 0, 6144: 1, 8193: 0}),
    (256, 1, 512, {8193: 1, 20480: 1, 20481: 0}, {8193: 1, 20480: 1})])
def test_layer_tail_rounds(amd, tmp_path, monkeypatch, d, kv, d_ff, prefill, decode):
    """Row counts on both sides of the tail's rounds: the kernel expected there,
    and the bytes and intervals of the separate kernels."""
    from czip_amd import synth
    path = synth.write_random_model(str(tmp_path / "t.czm"), d=d, n_layers=2, n_heads=d // 64, n_kv=kv, d_ff=d_ff,
                                    vocab=1024, ctx=64, seed=900 + d_ff)
    gm = amd.Model(amd.ModelWeights(path, amd.KV_GQA))
    monkeypatch.setenv("CZIP_TAIL_ROWS", "0")
    other = amd.Model(amd.ModelWeights(path, amd.KV_GQA))
    gm.set_profiling(True)
    for rows, tail in prefill.items():
        toks = np.random.default_rng(rows).integers(0, 1024, rows).astype(np.uint32)
        gm.reset_stats()
        chunk = next(c for c in (32, 31, 29, 23, 19, 17, 13, 11, 7, 5, 3, 1) if rows % c == 0)  # whole chunks: rows rows
        assert gm.compress_chunks(toks, chunk) == other.compress_chunks(toks, chunk)
        assert gm.kernel_stats("layer_tail")[0] == 2 * tail
    for S, tail in decode.items():
        rng = np.random.default_rng(S)
        toks, values = rng.integers(0, 1024, (2, S)).astype(np.uint32), rng.integers(0, gm.target_total, (2, S)).astype(np.uint32)
        gm.reset_stats()
        out = []
        for m in (gm, other):
            m.decode_begin(S, 2)
            out.append([m.decode_step(toks[p], np.full(S, p, np.int32), values[p]) for p in range(2)])
            m.decode_end()
        assert np.array_equal(out[0], out[1])
        assert gm.kernel_stats("layer_tail")[0] == 4 * tail


def test_row_gemm_16_without_tail(amd, shipped, monkeypatch):
    """The 16-row row GEMM behind the tail (shapes whose weights outgrow an L2 take it)."""
    import test_gpu_parity as parity
    monkeypatch.setenv("CZIP_TAIL_ROWS", "0")
    gm = amd.Model(amd.ModelWeights(MODEL_PATH))
    parity.test_small_launch_row_gemm(gm, shipped, 4, 512)


# The kernels of more rows at launches that the few-row GEMMs, the layer tail
# and the whole-stream decode take by default: the shapes of the random-shape
# tests, and decode steps on both sides of the 16-row row GEMM's least rows
@pytest.mark.parametrize("i", [1, 5, 9, 13, 19, 24, 27, 33, 39, 44, 52, 61, 69, 74, 80, 88])
def test_random_shapes_many_row_kernels(orc, tmp_path, monkeypatch, i):
    import test_gpu_random_shapes as shapes
    monkeypatch.setenv("CZIP_SKINNY_ROWS", "0")
    monkeypatch.setenv("CZIP_TAIL_ROWS", "0")
    shapes.test_random_shape_roundtrip(orc, tmp_path, monkeypatch, i)


@pytest.mark.parametrize("n_chunks", [1600, 369, 368])
def test_decode_steps_many_row_kernels(amd, shipped, monkeypatch, n_chunks):
    import test_gpu_parity as parity
    monkeypatch.setenv("CZIP_SKINNY_ROWS", "0")
    monkeypatch.setenv("CZIP_TAIL_ROWS", "0")
    gm = amd.Model(amd.ModelWeights(MODEL_PATH))
    gm.set_profiling(True)
    parity.test_small_launch_row_gemm(gm, shipped, n_chunks, 64)
    for name in ("dec_fused", "layer_tail", "few_row_gemm"):
        assert gm.kernel_stats(name)[0] == 0


# projections of a layer that take the 128 x 256 tiles: QKV (not layer 0's,
# which comes from the table) and up of two layers, the head, and O and down
# where their own rule (d >= 768 with a row kernel) or the lack of a row
# kernel (11 and 13 heads) sends them there
@pytest.mark.parametrize("heads,kv,d_ff,vocab,per_pass", [
    (12, 4, 192, 1088, 8), (14, 2, 832, 2112, 8), (11, 1, 448, 1024, 8), (13, 13, 320, 1088, 8), (10, 5, 192, 1024, 4)])
def test_wide_gemms(amd, orc, tmp_path, monkeypatch, heads, kv, d_ff, vocab, per_pass):
    """The 128 x 256 tiles at row counts around their row blocks, for column
    counts with a partial last tile and numbers of K steps of 64 odd and even:
    10 to 14 for QKV, ReGLU and the head (11 and 13 among them), 3, 5, 7 and 13
    for the down projection, over ragged chunks; the norms behind them where
    the row count asks for them."""
    import test_gpu_parity as parity
    from czip_amd import synth
    path = synth.write_random_model(str(tmp_path / "w.czm"), d=64 * heads, n_layers=2, n_heads=heads, n_kv=kv,
                                    d_ff=d_ff, vocab=vocab, ctx=600, seed=600 + heads)
    monkeypatch.setenv("CZIP_SKINNY_ROWS", "0")
    monkeypatch.setenv("CZIP_TAIL_ROWS", "0")
    monkeypatch.setenv("CZIP_WIDE_ROWS", "1")
    gm = amd.Model(amd.ModelWeights(path, amd.KV_GQA))
    om = orc.Model.from_file(path, amd.KV_GQA)
    gm.set_profiling(True)
    for lens in ([1], [127], [64, 64], [129], [513], [200, 31, 200, 200]):
        seen = gm.kernel_stats("wide_gemm")[0]
        parity._check_logits(gm, om, max(lens), lens, 11 + len(lens), vocab)
        # (the row kernels' rule asks for twice the rows: one row is too few)
        n = per_pass if per_pass == 4 or heads in (11, 13) or len(lens) * max(lens) >= 2 else 4
        assert gm.kernel_stats("wide_gemm")[0] - seen == n


def test_wide_qkv_least_tiles(amd, tmp_path, monkeypatch):
    """A narrow QKV projection takes the 128 x 256 tiles from 256 of them on; the
    bytes are those of the other kernel."""
    from czip_amd import synth
    path = synth.write_random_model(str(tmp_path / "q.czm"), d=256, n_layers=2, n_heads=4, n_kv=2, d_ff=512, vocab=1024,
                                    ctx=64, seed=640)
    gm = amd.Model(amd.ModelWeights(path, amd.KV_GQA))
    monkeypatch.setenv("CZIP_WIDE_ROWS", str(1 << 30))
    other = amd.Model(amd.ModelWeights(path, amd.KV_GQA))
    gm.set_profiling(True)
    for rows, wide in ((8192, 0), (16352, 0), (16384, 1), (16416, 1)):
        toks = np.random.default_rng(rows).integers(0, 1024, rows).astype(np.uint32)
        gm.reset_stats()
        assert gm.compress_chunks(toks, 32) == other.compress_chunks(toks, 32)
        assert gm.kernel_stats("wide_gemm")[0] == wide


def test_general_requantization_leaves_the_wide_tiles(amd, orc, tmp_path, monkeypatch):
    """Projections off the fast requantization path (|mult| >= 2^26) keep the
    128 x 128 tiles, which are faster there; the head has none and does not."""
    import test_gpu_parity as parity
    from czip_amd import synth
    t, meta = synth.random_model_tensors(d=768, n_layers=2, n_heads=12, n_kv=4, d_ff=192, vocab=1088, ctx=600, seed=650)
    for l in range(2):
        for nm in ("attn.qkv", "attn.out", "ffn.up", "ffn.down"):
            t[f"layers.{l}.{nm}.mult"] = np.array(int(t[f"layers.{l}.{nm}.mult"]) << 17, np.int32)
            t[f"layers.{l}.{nm}.shift"] = np.array(int(t[f"layers.{l}.{nm}.shift"]) + 17, np.int8)
    path = parity._write_model(str(tmp_path / "g.czm"), t, meta)
    monkeypatch.setenv("CZIP_SKINNY_ROWS", "0")
    monkeypatch.setenv("CZIP_WIDE_ROWS", "1")
    gm, om = parity._model_pair(amd, orc, path, amd.KV_GQA)
    gm.set_profiling(True)
    parity._check_logits(gm, om, 200, [200, 31], 651, 1088)
    assert gm.kernel_stats("wide_gemm")[0] == 1


@pytest.mark.parametrize("vocab,env", [(1024, "CZIP_UNFUSED_HEAD"), (1088, None), (4096, None), (4160, None), (8192, None)])
def test_decode_step_wave_counts(amd, orc, tmp_path, monkeypatch, vocab, env):
    """The unfused head's decoder step with a row's logits over one, four and
    sixteen waves (up to 256 or 512 rows, then more), at the edges of their vocabulary
    ranges; streams that end at different steps and streams cut short."""
    from czip_amd import synth
    if env:
        monkeypatch.setenv(env, "1")
    path = synth.write_random_model(str(tmp_path / "c.czm"), d=128, n_layers=1, n_heads=2, n_kv=1, d_ff=64, vocab=vocab,
                                    ctx=64, seed=700 + vocab)
    gm = amd.Model(amd.ModelWeights(path, amd.KV_GQA))
    om = orc.Model.from_file(path, amd.KV_GQA)
    rng = np.random.default_rng(vocab)
    toks = rng.integers(0, vocab, 24 * 13).astype(np.uint32)
    coded = om.compress_many(toks, 13, threads=8)
    for S in (24, 256, 257, 512, 513):
        pick = rng.integers(0, 24, S)
        lens = rng.integers(0, 14, S).astype(np.int32)
        want = np.concatenate([toks[13 * c:13 * c + n] for c, n in zip(pick, lens)])
        assert np.array_equal(gm.decompress_chunks([coded[c] for c in pick], lens), want)
    cut = [c[:3 * i % (len(c) + 1)] for i, c in enumerate(coded)]
    assert np.array_equal(gm.decompress_chunks(cut, [13] * 24), om.decompress_many(cut, [13] * 24))


@pytest.mark.parametrize("heads,kv,d_ff,most", [(4, 2, 4160, 1024), (11, 1, 448, 1024), (12, 4, 448, 768)])
def test_few_row_gemms_row_limit(amd, orc, tmp_path, heads, kv, d_ff, most):
    """Row counts up to the few-row GEMMs' limit and just past it: 1024, and
    768 where a row GEMM of 640 columns or more takes over."""
    import test_gpu_parity as parity
    from czip_amd import synth
    path = synth.write_random_model(str(tmp_path / "l.czm"), d=64 * heads, n_layers=2, n_heads=heads, n_kv=kv,
                                    d_ff=d_ff, vocab=1088, ctx=600, seed=800 + heads)
    gm = amd.Model(amd.ModelWeights(path, amd.KV_GQA))
    om = orc.Model.from_file(path, amd.KV_GQA)
    gm.set_profiling(True)
    for lens in ([520], [384, 384], [385, 385], [512, 300], [513, 512]):
        seen = gm.kernel_stats("few_row_gemm")[0]
        parity._check_logits(gm, om, max(lens), lens, 17 + len(lens), 1088)
        assert (gm.kernel_stats("few_row_gemm")[0] > seen) == (len(lens) * max(lens) <= most)


@pytest.mark.parametrize("heads,layers,d_ff,most", [(10, 2, 1152, 768), (10, 24, 1152, 1024), (8, 2, 4160, 512)])
def test_few_row_gemms_decode_limit(amd, tmp_path, monkeypatch, heads, layers, d_ff, most):
    """Decode steps of a wide model take the few-row GEMMs up to 768 streams,
    up to 1024 with weights of more than 48 MB, and up to 512 with a
    feed-forward of more than 4096; the intervals are those of the other
    kernels."""
    from czip_amd import synth
    path = synth.write_random_model(str(tmp_path / "s.czm"), d=64 * heads, n_layers=layers, n_heads=heads, n_kv=2, d_ff=d_ff,
                                    vocab=1024, ctx=8, seed=850)
    gm = amd.Model(amd.ModelWeights(path, amd.KV_GQA))
    monkeypatch.setenv("CZIP_SKINNY_ROWS", "0")
    other = amd.Model(amd.ModelWeights(path, amd.KV_GQA))
    gm.set_profiling(True)
    other.set_profiling(True)
    for S in (512, 513, 768, 769, 1024, 1025):
        rng = np.random.default_rng(S)
        values = rng.integers(0, gm.target_total, (3, S)).astype(np.uint32)
        toks = rng.integers(0, 1024, (3, S)).astype(np.uint32)
        out = []
        seen = gm.kernel_stats("few_row_gemm")[0]
        for m in (gm, other):
            m.decode_begin(S, 3)
            out.append([m.decode_step(toks[p], np.full(S, p, np.int32), values[p]) for p in range(3)])
            m.decode_end()
        assert np.array_equal(out[0], out[1])
        assert (gm.kernel_stats("few_row_gemm")[0] > seen) == (S <= most)
    assert other.kernel_stats("few_row_gemm")[0] == 0
