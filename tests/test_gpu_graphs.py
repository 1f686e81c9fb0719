"""Recorded graphs of the attention ops (sd_graph_begin / sd_graph_end / sd_graph_run), after the reference's own uses of them:
crates/straydog-engine/tests/dspark_attention_gpu.rs:81-124 (a recorded op follows a device-resident position as it moves; what a
replay reads is what the buffers hold then) -- here for the DSpark block attention, a paged decode step (K/V append + attention) and
the whole Qwen decode stage.  Every replay is checked against the same work run eagerly, with eager work and waits between replays."""
import numpy as np
import pytest

from gpu_util import backend, close_enough, make_pool

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    with backend(4 << 30) as handle:
        yield handle


def _read(gpu, buffer, dtype, count):
    return gpu.read_buffer(buffer, 0, dtype, count)


def _bf16_pair(oracle, values):
    """(BF16 bit patterns, the FP32 values they stand for)."""
    bits = oracle.to_bf16(values)
    return bits, (bits.astype(np.uint32) << 16).view(np.float32).reshape(values.shape)


def test_graph_bookkeeping(gpu):
    from straydog_amd.backend import StraydogError
    assert not gpu.graph_run(12345), "no graph is stored under that key"
    with pytest.raises(StraydogError, match="no Straydog graph"):
        gpu.graph_end(1)
    gpu.graph_begin()
    with pytest.raises(StraydogError, match="already"):
        gpu.graph_begin()
    gpu.graph_end(1, keep=False)
    assert not gpu.graph_run(1), "a dropped graph is not stored"


def test_dspark_attention_recorded(gpu, oracle):
    from test_oracle_attention import _dspark_inputs
    from test_gpu_ops import _dspark_check
    q, ring, block, sinks = _dspark_inputs()
    qb, rb, bb, sb = (gpu.upload(a) for a in (q, ring, block, sinks))
    out = gpu.buffer(q.size * 4)
    anchor = gpu.upload(np.array([389], dtype=np.int32))
    gpu.graph_begin()
    gpu.dspark_attention(qb.base(), rb.base(), bb.base(), sb.base(), 64, 3, 389, anchor.base(), 128, out.base())
    gpu.graph_end(140)
    for at in (389, 200, 128, 389):
        gpu.write_buffer(anchor, 0, np.array([at], dtype=np.int32))
        assert gpu.graph_run(140)
        want = oracle.dspark_attention(q, ring, block, sinks, 64, 3, at, 128)
        _dspark_check(f"replayed at {at}", _read(gpu, out, np.float32, want.size), want)
    # the first capture, a key that changes later and the sink's mass are observable (dspark_attention_gpu.rs:101-124)
    gpu.write_buffer(qb, 0, np.zeros(q.size, np.float32))
    gpu.write_buffer(rb, 0, np.full(ring.size, 23.0, np.float32))
    keys = np.repeat(np.arange(1, 6, dtype=np.float32), 512)
    gpu.write_buffer(bb, 0, keys)
    gpu.write_buffer(sb, 0, np.zeros(64, np.float32))
    gpu.graph_begin()
    gpu.dspark_attention(qb.base(), rb.base(), bb.base(), sb.base(), 64, 5, 0, None, 0, out.base())
    gpu.graph_end(139)
    assert gpu.graph_run(139)
    _dspark_check("captured noncausal block", _read(gpu, out, np.float32, q.size), np.full(q.size, 2.5))
    keys[4 * 512:] = 11.0
    gpu.write_buffer(bb, 0, keys)
    assert gpu.graph_run(139)
    _dspark_check("future key changed", _read(gpu, out, np.float32, q.size), np.full(q.size, 3.5))
    for sink, expected in ((1000.0, 0.0), (-1000.0, 4.2)):
        gpu.write_buffer(sb, 0, np.full(64, sink, np.float32))
        assert gpu.graph_run(139)
        _dspark_check(f"sink={sink}", _read(gpu, out, np.float32, q.size), np.full(q.size, expected))
    for b in (qb, rb, bb, sb, out, anchor):
        gpu.release(b)


def test_paged_decode_step_recorded(gpu, oracle):
    # one decode step of a ragged batch -- append the new K/V rows, attend -- recorded once and replayed as the positions advance
    rng = np.random.default_rng(5)
    seqs, heads, kv_heads, dim, page_tokens, row_bytes = 3, 16, 2, 128, 64, 136
    lengths = [700, 65, 1000]
    capacity = [n + 8 for n in lengths]
    pool, buffer, host, table, table_buffer = make_pool(gpu, oracle, rng, capacity, kv_heads, dim, page_tokens, row_bytes)
    max_context = max(capacity)
    positions = gpu.upload(np.array(lengths, dtype=np.int32))
    kb, vb = gpu.buffer(seqs * kv_heads * dim * 4), gpu.buffer(seqs * kv_heads * dim * 4)
    qb, out = gpu.buffer(seqs * heads * dim * 4), gpu.buffer(seqs * heads * dim * 4)
    scratch = gpu.buffer(gpu.paged_attention_scratch(seqs, 1, heads, dim, max_context))

    def step():
        gpu.kv_write(pool, table_buffer.base(), table.shape[1], positions.base(), kb.base(), vb.base(), False, seqs, 1)
        gpu.paged_attention(pool, table_buffer.base(), table.shape[1], positions.base(), max_context, qb.base(), False, seqs, 1, heads, 0.088, out.base(),
                            False, scratch)
    step()                                  # once eagerly: whatever a first call sets up is set up outside the recording
    gpu.graph_begin()
    step()
    gpu.graph_end(7)
    for turn in range(4):
        at = np.array([n + turn for n in lengths], dtype=np.int32)
        k = rng.standard_normal((seqs, 1, kv_heads, dim)).astype(np.float32)
        v = rng.standard_normal((seqs, 1, kv_heads, dim)).astype(np.float32)
        q = rng.standard_normal((seqs, 1, heads, dim)).astype(np.float32)
        for b, a in ((positions, at), (kb, k), (vb, v), (qb, q)):
            gpu.write_buffer(b, 0, a)
        assert gpu.graph_run(7)
        got = _read(gpu, out, np.float32, q.size).reshape(q.shape)
        oracle.kv_write(host, row_bytes, page_tokens, kv_heads, dim, table, at, k, v)
        want = oracle.paged_attention(host, row_bytes, page_tokens, kv_heads, dim, table, at, q, 0.088)
        close_enough(got, want, f"replay {turn}")
        assert np.array_equal(_read(gpu, buffer, np.uint8, host.size), host), "the appended rows"
    for b in (buffer, table_buffer, positions, kb, vb, qb, out, scratch):
        gpu.release(b)


def test_qwen_decode_stage_recorded(gpu, oracle):
    # sdx_qsa_decode_attend recorded once; replays at advancing device-resident positions give the bits of eager calls on a twin state
    rng = np.random.default_rng(6)
    heads, kv_heads, context, first, row_bytes = 24, 2, 4096, 2300, 272
    pool_blocks, stride = context // 4 + 1, 24 * 512 + 2 * 512 + 640
    blocks = np.zeros((128, pool_blocks), dtype=np.float32)
    blocks[:, :first // 4] = rng.standard_normal((128, first // 4)).astype(np.float32)
    history = rng.standard_normal((16, 128)).astype(np.float32)
    norms = [(0.4 + 1.2 * rng.random(n)).astype(np.float32) for n in (256, 256, 128, 128)]
    cached = np.zeros(context * 4 * row_bytes, dtype=np.uint8)
    oracle.kv_write(cached, row_bytes, context, kv_heads, 256, np.zeros((1, 1), np.int32), np.zeros(1, np.int32),
                    rng.standard_normal((1, first, kv_heads, 256)).astype(np.float32), rng.standard_normal((1, first, kv_heads, 256)).astype(np.float32))

    def twin():
        kv, buffer = gpu.kv_pool(1, context, kv_heads, 256, row_bytes)
        gpu.write_buffer(buffer, 0, cached)
        s = dict(kv=kv, buffer=buffer, projections=gpu.buffer(stride * 4), blocks=gpu.upload(blocks), history=gpu.upload(history),
                 norms=[gpu.upload(n) for n in norms], position=gpu.upload(np.array([first], dtype=np.uint32)), attended=gpu.buffer(heads * 256 * 4),
                 scratch=gpu.buffer(gpu.qsa_decode_attend_scratch(1, heads, kv_heads, context)))
        s["state"] = gpu.qsa_state(kv, None, context, s["blocks"].base(), s["history"].base(), *[n.base() for n in s["norms"]], heads)
        return s

    def call(s):
        gpu.qsa_decode_attend(s["state"], s["projections"].base(), stride, 1, s["position"].base(), s["position"].base(), s["scratch"], s["attended"].base())
    recorded, eager = twin(), twin()
    warm = twin()
    call(warm)                               # a first call outside the recording
    gpu.graph_begin()
    call(recorded)
    gpu.graph_end(9)
    for turn in range(6):                    # positions 2300 .. 2305: a block is completed at 2303
        row = (rng.standard_normal(stride) * 2).astype(np.float32)
        at = np.array([first + turn], dtype=np.uint32)
        for s in (recorded, eager):
            gpu.write_buffer(s["projections"], 0, row)
            gpu.write_buffer(s["position"], 0, at)
        assert gpu.graph_run(9)
        call(eager)
        for what, count, dtype in (("attended", heads * 256, np.float32), ("blocks", blocks.size, np.float32), ("history", history.size, np.float32),
                                   ("buffer", cached.size, np.uint8)):
            a, b = _read(gpu, recorded[what], dtype, count), _read(gpu, eager[what], dtype, count)
            assert np.array_equal(a.view(np.uint8), b.view(np.uint8)), f"replay {turn}: {what}"
        assert np.abs(_read(gpu, recorded["attended"], np.float32, heads * 256)).max() > 0


def test_prompt_chunk_stage_recorded(gpu, oracle):
    # sdx_qsa_prefill_attend recorded once at a position past 32768 (the selection by intervals); replays on new projections give
    # the bits of eager calls on a twin state
    rng = np.random.default_rng(16)
    heads, kv_heads, context, first, row_bytes, steps = 24, 2, 36864, 34000, 272, 24
    pool_blocks, stride = context // 4 + 1, 24 * 512 + 2 * 512 + 640
    blocks = np.zeros((128, pool_blocks), dtype=np.float32)
    blocks[:, :first // 4] = rng.standard_normal((128, first // 4)).astype(np.float32)
    history = rng.standard_normal((16, 128)).astype(np.float32)
    norms = [(0.4 + 1.2 * rng.random(n)).astype(np.float32) for n in (256, 256, 128, 128)]
    cached = rng.integers(0, 256, context * 4 * row_bytes, dtype=np.uint8)
    cached.reshape(-1, row_bytes)[:, 256:] = np.tile(np.frombuffer(np.float16(0.01).tobytes(), np.uint8), 8)

    def twin():
        kv, buffer = gpu.kv_pool(1, context, kv_heads, 256, row_bytes)
        gpu.write_buffer(buffer, 0, cached)
        s = dict(kv=kv, buffer=buffer, projections=gpu.buffer(steps * stride * 4), blocks=gpu.upload(blocks), history=gpu.upload(history),
                 norms=[gpu.upload(n) for n in norms], attended=gpu.buffer(steps * heads * 256 * 4),
                 scratch=gpu.buffer(gpu.qsa_prefill_attend_scratch(steps, heads, kv_heads, context)))
        s["state"] = gpu.qsa_state(kv, None, context, s["blocks"].base(), s["history"].base(), *[n.base() for n in s["norms"]], heads)
        return s

    def call(s):
        gpu.qsa_prefill_attend(s["state"], s["projections"].base(), stride, steps, first, s["scratch"], s["attended"].base())
    recorded, eager, warm = twin(), twin(), twin()
    gpu.write_buffer(warm["projections"], 0, rng.standard_normal(steps * stride).astype(np.float32))
    call(warm)                               # a first call outside the recording
    gpu.graph_begin()
    call(recorded)
    gpu.graph_end(19)
    for turn in range(3):
        rows = (rng.standard_normal(steps * stride) * 2).astype(np.float32)
        for s in (recorded, eager):
            gpu.write_buffer(s["projections"], 0, rows)
        assert gpu.graph_run(19)
        call(eager)
        for what, count, dtype in (("attended", steps * heads * 256, np.float32), ("blocks", blocks.size, np.float32), ("history", history.size, np.float32),
                                   ("buffer", cached.size, np.uint8)):
            a, b = _read(gpu, recorded[what], dtype, count), _read(gpu, eager[what], dtype, count)
            assert np.array_equal(a.view(np.uint8), b.view(np.uint8)), f"replay {turn}: {what}"
        assert np.abs(_read(gpu, recorded["attended"], np.float32, steps * heads * 256)).max() > 0


def test_prompt_chunk_call_recorded(gpu, oracle):
    # sdx_prefill_chunk -- a chunk's K/V append, its tiles and its attention -- recorded once and replayed chunk after chunk of a
    # prompt as the device-resident positions advance: every replay's cache bytes and outputs against the oracle
    rng = np.random.default_rng(12)
    seqs, heads, kv_heads, dim, page_tokens, row_bytes, span, chunks = 2, 16, 2, 128, 64, 136, 96, 4
    begins = [0, 40]                        # the second sequence's prompt starts behind 40 cached tokens
    capacity = [b + chunks * span for b in begins]
    pool, buffer, host, table, table_buffer = make_pool(gpu, oracle, rng, capacity, kv_heads, dim, page_tokens, row_bytes)
    max_context = max(capacity)
    positions = gpu.upload(np.array(begins, dtype=np.int32))
    kb, vb = gpu.buffer(seqs * span * kv_heads * dim * 2), gpu.buffer(seqs * span * kv_heads * dim * 2)
    qb, out = gpu.buffer(seqs * span * heads * dim * 2), gpu.buffer(seqs * span * heads * dim * 4)
    tiles = gpu.buffer(gpu.prefill_tiles_bytes(seqs, kv_heads, dim, max_context))
    valid = gpu.upload(np.zeros(seqs, dtype=np.int32))      # what the tiles hold: nothing before the first chunk, then the positions

    def call():
        gpu.prefill_chunk(pool, table_buffer.base(), table.shape[1], positions.base(), max_context, kb.base(), vb.base(), True, qb.base(), True,
                          seqs, span, heads, 0.088, out.base(), False, tiles, valid.base())
    gpu.graph_begin()
    call()
    gpu.graph_end(11)
    for turn in range(chunks):
        at = np.array([b + turn * span for b in begins], dtype=np.int32)
        k = rng.standard_normal((seqs, span, kv_heads, dim)).astype(np.float16)
        v = rng.standard_normal((seqs, span, kv_heads, dim)).astype(np.float16)
        q = rng.standard_normal((seqs, span, heads, dim)).astype(np.float16)
        for b, a in ((positions, at), (kb, k), (vb, v), (qb, q)):
            gpu.write_buffer(b, 0, a)
        gpu.write_buffer(valid, 0, at if turn else np.zeros(seqs, dtype=np.int32))
        assert gpu.graph_run(11)
        got = _read(gpu, out, np.float32, q.size).reshape(q.shape)
        oracle.kv_write(host, row_bytes, page_tokens, kv_heads, dim, table, at, k.astype(np.float32), v.astype(np.float32))
        want = oracle.paged_attention(host, row_bytes, page_tokens, kv_heads, dim, table, at, q.astype(np.float32), 0.088)
        close_enough(got, want, f"replay {turn}")
        assert np.array_equal(_read(gpu, buffer, np.uint8, host.size), host), "the appended rows"
    for b in (buffer, table_buffer, positions, kb, vb, qb, out, tiles, valid):
        gpu.release(b)


def test_graphs_are_dropped_when_the_workspace_moves(gpu, oracle):
    # ops that use the handle's workspace bake its address into a recorded graph; when a later, larger call makes the workspace
    # grow (and move), the kept graphs are dropped: sd_graph_run answers "none stored" and the caller records again, instead of
    # replaying on freed memory.  Growth while recording is refused.
    from straydog_amd.backend import StraydogError
    rng = np.random.default_rng(8)

    def latent_case(batch, groups, k, heads=64):
        q = rng.standard_normal((batch, heads, 576)).astype(np.float32)
        latents = rng.standard_normal((batch, groups, 576)).astype(np.float32)
        selected = np.stack([np.sort(rng.choice(groups, size=k, replace=False)) for _ in range(batch)]).astype(np.int32)
        bf = lambda a: (a.view(np.uint32) >> 16).astype(np.uint16)     # truncation is fine here: both sides see the same bits
        qb, lb, sb = gpu.upload(bf(q)), gpu.upload(bf(latents)), gpu.upload(selected)
        out = gpu.buffer(batch * heads * 512 * 4)
        def run():
            gpu.latent_attention(qb.base(), lb.base(), sb.base(), batch, groups, k, heads, 576, 512, 1.0 / 24.0, out.base())
        return run, out, (qb, lb, sb, out)

    small, small_out, small_buffers = latent_case(1, 512, 128)
    small()                                              # sizes the workspace for this shape
    eager = _read(gpu, small_out, np.float32, 64 * 512).copy()
    gpu.graph_begin()
    small()
    gpu.graph_end(21)
    gpu.write_buffer(small_out, 0, np.zeros(64 * 512, np.float32))
    assert gpu.graph_run(21)
    assert np.array_equal(_read(gpu, small_out, np.float32, 64 * 512), eager)
    large, large_out, large_buffers = latent_case(4, 4096, 2048)
    gpu.graph_begin()
    with pytest.raises(StraydogError, match="cannot grow while a graph is recorded"):
        large()
    gpu.graph_end(22, keep=False)
    assert gpu.graph_run(21), "a refused growth leaves the kept graphs alone"
    large()                                              # eager: the workspace grows and moves
    assert not gpu.graph_run(21), "the graph that held the old workspace address is gone"
    gpu.graph_begin()
    small()
    gpu.graph_end(21)
    gpu.write_buffer(small_out, 0, np.zeros(64 * 512, np.float32))
    assert gpu.graph_run(21)
    assert np.array_equal(_read(gpu, small_out, np.float32, 64 * 512), eager)
    for b in small_buffers + large_buffers:
        gpu.release(b)


def test_batched_sparse_step_recorded(gpu, oracle):
    # the batched sparse path -- matrix-core indexer with its histograms, top-k, gather attention over the selection -- recorded
    # once and replayed with other queries and other visible lengths: the histograms one replay leaves must be what the next one
    # expects, and every replay picks the indices and gives the outputs of the same work run eagerly
    rng = np.random.default_rng(41)
    batch, groups, iheads, idim, k, heads, kdim, vdim = 4, 9000, 64, 128, 512, 32, 576, 512
    key_bits, key_vals = _bf16_pair(oracle, rng.standard_normal((batch, groups, idim)).astype(np.float32))
    lat_bits, _ = _bf16_pair(oracle, rng.standard_normal((batch, groups, kdim)).astype(np.float32))
    kb, lb = gpu.upload(key_bits), gpu.upload(lat_bits)
    qb, wb, vb = gpu.buffer(batch * iheads * idim * 2), gpu.buffer(batch * iheads * 4), gpu.buffer(batch * 4)
    ab, indices, out = gpu.buffer(batch * heads * kdim * 2), gpu.buffer(batch * k * 4), gpu.buffer(batch * heads * vdim * 4)
    scale = float(1.0 / np.sqrt(kdim))

    def load(turn):
        q_bits, q_vals = _bf16_pair(oracle, rng.standard_normal((batch, iheads, idim)).astype(np.float32))
        a_bits, a_vals = _bf16_pair(oracle, rng.standard_normal((batch, heads, kdim)).astype(np.float32))
        weights = rng.random((batch, iheads)).astype(np.float32)
        visible = np.array([groups, groups - 1000 * turn, 300 + turn, max(1, groups // (turn + 1))], dtype=np.int32)   # (row 2: fewer than k)
        for b, a in ((qb, q_bits), (wb, weights), (vb, visible), (ab, a_bits)):
            gpu.write_buffer(b, 0, a)
        return q_vals, a_vals, weights, visible

    def step():
        gpu.index_top_k(qb.base(), kb.base(), wb.base(), vb.base(), batch, groups, iheads, idim, 0.5, None, k, indices.base())
        gpu.latent_attention(ab.base(), lb.base(), indices.base(), batch, groups, k, heads, kdim, vdim, scale, out.base())
    load(0)
    step()                                  # once eagerly: whatever a first call sets up is set up outside the recording
    gpu.graph_begin()
    step()
    gpu.graph_end(11)
    for turn in range(4):
        q_vals, a_vals, weights, visible = load(turn)
        assert gpu.graph_run(11)
        got_indices = _read(gpu, indices, np.int32, batch * k).reshape(batch, k)
        got = _read(gpu, out, np.float32, batch * heads * vdim).reshape(batch, heads, vdim)
        for b in range(batch):
            scores = oracle.index_scores(q_vals[b:b + 1], key_vals[b], weights[b:b + 1], visible[b:b + 1], 0.5)
            assert np.array_equal(got_indices[b], oracle.top_k(scores, k)[0]), f"replay {turn}, sequence {b}"
            want = oracle.latent_attention(a_vals[b:b + 1], None, None, 0, lat_bits[b], got_indices[b:b + 1], None, vdim, scale)
            close_enough(got[b], want[0], f"replay {turn}, sequence {b}")
        if turn == 1:
            step()                          # eager work between replays, through the same histograms and workspace
            gpu.synchronize()
    for b in (kb, lb, qb, wb, vb, ab, indices, out):
        gpu.release(b)


class _Dense:
    """sd_op_attention of rows whose keys are cut into more runs than the caller's scratch holds: it takes an optional workspace."""

    def __init__(self, gpu, oracle, rows=1, context=4200, heads=16, kv_heads=2, dim=256):
        rng = np.random.default_rng(context)
        self.gpu, self.shape = gpu, (context, rows, heads, kv_heads, dim)
        q, keys, values = (rng.standard_normal(n).astype(np.float32) for n in ((rows, heads, dim), (context, kv_heads, dim), (context, kv_heads, dim)))
        positions = np.arange(context - rows, context, dtype=np.int32)
        self.buffers = [gpu.upload(x) for x in (q, keys, values, positions)]
        pairs = rows * heads
        self.scratch, self.out = gpu.buffer(pairs * min(64, max(1, 256 // pairs)) * (dim + 2) * 4), gpu.buffer(q.size * 4)
        if oracle:
            self.want, self.bound = oracle.op_attention_f64(q, keys, values, positions, float(np.float32(dim ** -0.5)), None)

    def queue(self):
        context, rows, heads, kv_heads, dim = self.shape
        q, keys, values, positions = (b.base() for b in self.buffers)
        self.gpu.attention(q, keys, values, context, positions, rows, heads, kv_heads, dim, float(dim ** -0.5), None, self.scratch, self.out.base())

    def right(self, how):
        self.gpu.write_buffer(self.out, 0, np.zeros(self.want.size, np.float32))
        ran = how()
        got = _read(self.gpu, self.out, np.float32, self.want.size).reshape(self.want.shape)
        assert np.abs((got - self.want) / self.bound).max() <= 1.0
        return ran


def test_optional_workspaces_are_given_back_where_that_helps(oracle):
    # an allocation that fits once the ops' optional workspaces are gone takes them, and the graphs that hold them; one that would not fit
    # even then is refused and leaves both as they are
    from straydog_amd.backend import StraydogError
    budget = 64 << 20
    with backend(budget) as gpu:
        work = _Dense(gpu, oracle)
        gpu.graph_begin()
        gpu.graph_end(7, keep=False)           # (what a first recording reserves)
        used, before = gpu.memory()[0], gpu.device_state()[0]
        work.right(work.queue)
        assert before - gpu.device_state()[0] >= 2 << 20, "the op has taken a workspace"
        assert gpu.memory() == (used, budget), "what an allocation can have is not less for it"
        gpu.graph_begin()
        work.queue()
        gpu.graph_end(7)
        for size in (budget, budget << 10, budget - (8 << 20)):
            with pytest.raises(StraydogError, match="budget exceeded"):
                gpu.buffer(size)
            assert work.right(lambda: gpu.graph_run(7)), "a refused allocation drops no graph"
        rest = gpu.buffer(budget - used - 64)
        assert not gpu.graph_run(7), "the graph that held the workspace is gone with it"
        work.right(work.queue)                 # without room it does with the caller's scratch
        gpu.graph_begin()
        work.queue()
        gpu.graph_end(7)
        gpu.release(rest)
        for _ in range(2):
            work.right(work.queue)             # (with a workspace again)
            assert work.right(lambda: gpu.graph_run(7))


@pytest.mark.parametrize("recorded", [False, True])
def test_optional_workspaces_grow_into_the_room_there_is(oracle, recorded):
    # partial results of 25 and of 32 MB: the second workspace fits the budget, twice the first does not; where a graph was recorded
    # over the first it stays, and the graph is right
    with backend(4 << 30) as gpu:
        for rows in (44, 60):
            _Dense(gpu, None, rows, 1120)
        used = gpu.memory()[0]
    with backend(used + (2 << 20) + ((72 if recorded else 44) << 20)) as gpu:
        first, second = (_Dense(gpu, oracle, rows, 1120) for rows in (44, 60))
        first.right(first.queue)
        free = gpu.device_state()[0]
        if recorded:
            gpu.graph_begin()
            first.queue()
            gpu.graph_end(1)
        second.right(second.queue)
        assert free - gpu.device_state()[0] >= (30 if recorded else 2) << 20, "the second call has a workspace of its size"
        for _ in range(2):
            first.right(first.queue)
            second.right(second.queue)
            if recorded:
                assert first.right(lambda: gpu.graph_run(1))


def test_optional_workspaces_under_allocations_of_another_thread(oracle):
    # one thread queues an op that takes an optional workspace while another allocates what only fits without it: the op's kernels keep
    # the workspace they were given
    import threading
    budget = 64 << 20
    with backend(budget) as gpu:
        work = _Dense(gpu, oracle)
        rest, done, failed = budget - gpu.memory()[0] - 64, threading.Event(), []

        def allocate():
            try:
                while not done.is_set():
                    gpu.release(gpu.buffer(rest))
            except Exception as error:
                failed.append(error)
        other = threading.Thread(target=allocate)
        other.start()
        try:
            for _ in range(50):
                work.right(work.queue)
        finally:
            done.set()
            other.join()
        assert not failed
