"""The work that users of the attention library have it do, as cases to be timed.

A case names a path (a sequence of public entry points as a model's attention layer calls them) and its sizes.  The paths:

  decode      a batch of sequences in the paged K/V cache: each appends the rows of its newest tokens (one, or a speculative span
              to verify) and attends everything before and with them           kv_write, paged_attention
  prompt      prompts read in chunks: the chunk's rows appended and attended   prefill_chunk, or kv_write + paged_attention
  stage       the whole attention stage of a model with a block indexer        qsa_decode_attend / qsa_prefill_attend
  topk        a batch of decode rows: indexer over BF16 keys, top-k, gather attention over BF16 latents
                                                                               index_top_k, latent_attention
  compressed  rows over a window ring and the best compressed rows of one sequence
                                                                               index_select, sparse_attention
  dense       rows over FP32 caches, gated                                     attention

Inputs are made on the GPU from the seed.  The library works on allocations of its own; torch sees them as views.
"""
import numpy as np
import torch

from straydog_amd.abi import KvPool
from straydog_amd.backend import Backend, tagged_bf16

_handle = None


def _gpu():
    """The program's one device handle."""
    global _handle
    if _handle is None:
        _handle = Backend(0, 256 << 30)
    return _handle


class _Memory:
    """A buffer of the library as torch takes it.  Every torch view of it holds on to this object; the buffer is given back with the
    last of them."""

    def __init__(self, gpu, size):
        self.gpu, self.buffer = gpu, gpu.buffer(max(size, 16))

    def view(self, count, dtype):
        if dtype is torch.bfloat16:      # (no array interface names it)
            return self.view(count, torch.float16).view(torch.bfloat16)
        self.__cuda_array_interface__ = {"shape": (count,), "typestr": _KINDS[dtype], "data": (self.buffer.base(), False), "version": 2}
        return torch.as_tensor(self, device="cuda")

    def __del__(self):
        if hasattr(self, "buffer"):
            try:
                self.gpu.release(self.buffer)
            except Exception:            # the interpreter is going down
                pass


_KINDS = {torch.uint8: "|u1", torch.int32: "<i4", torch.float16: "<f2", torch.float32: "<f4"}


class _State:
    """What a program holds for one case: buffers by name, each with a torch view."""

    def __init__(self, case, seed):
        self.case, self.gpu, self.memory, self.buffers, self.views = dict(case), _gpu(), {}, {}, {}
        self.random = torch.Generator(device="cuda")
        self.random.manual_seed(seed)
        self.order = np.random.default_rng(seed)

    def empty(self, name, count, dtype):
        self.memory[name] = _Memory(self.gpu, count * torch.empty(0, dtype=dtype).element_size())
        self.buffers[name] = self.memory[name].buffer
        self.views[name] = self.memory[name].view(count, dtype)
        return self.views[name]

    def normal(self, name, count, dtype):
        self.empty(name, count, dtype).normal_(generator=self.random)

    def uniform(self, name, count, low, high):
        self.empty(name, count, torch.float32).uniform_(low, high, generator=self.random)

    def put(self, name, values):
        values = np.ascontiguousarray(values)
        kind = {"int32": torch.int32, "uint32": torch.int32, "float32": torch.float32}[str(values.dtype)]
        self.empty(name, values.size, kind)
        self.gpu.write_buffer(self.buffers[name], 0, values)

    def drop(self, name):
        del self.views[name], self.buffers[name], self.memory[name]

    def at(self, name, offset=0):
        return self.buffers[name].at(offset)

    def ready(self):
        torch.cuda.synchronize()         # (views are written on torch's stream, the library works on its own)


# ---- the cases -----------------------------------------------------------------------------------------------------

def listed():
    return [
        # one user's conversation, token by token: the smallest call, bound by launches and latency
        {"name": "decode_one", "path": "decode", "seqs": 1, "low": 4096, "high": 4096, "span": 1, "heads": 16, "kv_heads": 2, "dim": 128, "q8": True,
         "page_tokens": 256, "io16": False},
        # a serving batch of mixed lengths
        {"name": "decode_ragged_32", "path": "decode", "seqs": 32, "low": 1024, "high": 32768, "span": 1, "heads": 32, "kv_heads": 4, "dim": 128, "q8": True,
         "page_tokens": 256, "io16": True},
        # a small batch of a model with 256 columns a head, its cache kept in FP16
        {"name": "decode_256_f16", "path": "decode", "seqs": 8, "low": 777, "high": 16384, "span": 1, "heads": 24, "kv_heads": 2, "dim": 256, "q8": False,
         "page_tokens": 128, "io16": True},
        # speculative decoding at long context: the accepted token and four drafts verified in one pass
        {"name": "verify_5", "path": "decode", "seqs": 16, "low": 65541, "high": 65541, "span": 5, "heads": 32, "kv_heads": 4, "dim": 128, "q8": True,
         "page_tokens": 256, "io16": True},
        # one long prompt, read chunk by chunk
        {"name": "prompt_8192", "path": "prompt", "seqs": 1, "tokens": 8192, "chunk": 2048, "heads": 32, "kv_heads": 4, "dim": 128, "q8": True,
         "page_tokens": 256, "fused": True},
        # two short prompts of odd length at once, 256 columns a head
        {"name": "prompt_2x1531_256", "path": "prompt", "seqs": 2, "tokens": 1531, "chunk": 1531, "heads": 24, "kv_heads": 2, "dim": 256, "q8": True,
         "page_tokens": 256, "fused": False},
        # the indexed model: a decode token at very long context
        {"name": "stage_decode_242k", "path": "stage", "rows": 1, "chunks": 1, "base": 242000, "heads": 24, "kv_heads": 2, "q8": True},
        # ... and two chunks of its prompt further on
        {"name": "stage_prompt_98k", "path": "stage", "rows": 1024, "chunks": 2, "base": 98304, "heads": 24, "kv_heads": 2, "q8": True},
        # indexed decode over latents for a serving batch
        {"name": "topk_batch_8", "path": "topk", "batch": 8, "context": 131072, "index_heads": 64, "k": 2048, "heads": 64},
        # the compressed model: a decode token
        {"name": "compressed_decode", "path": "compressed", "rows": 1, "position": 65000, "index_heads": 64, "heads": 64, "k": 512, "bf16": True},
        # ... and a chunk of its prompt
        {"name": "compressed_prompt", "path": "compressed", "rows": 256, "position": 32768, "index_heads": 64, "heads": 64, "k": 512, "bf16": True},
        # a chunk of rows of a dense gated layer over its FP32 caches
        {"name": "dense_128_rows", "path": "dense", "rows": 128, "position": 4096, "heads": 16, "kv_heads": 2, "dim": 256},
    ]


def _size(rng, low, high):
    """A whole number of [low, high], spread over its logarithm."""
    return int(round(low * (high / low) ** rng.random()))


def draw(rng):
    path = rng.choice(["decode", "decode", "decode", "prompt", "prompt", "stage", "stage", "topk", "compressed", "compressed", "dense"])
    if path == "decode":
        dim = rng.choice([128, 128, 256])
        heads, kv_heads = rng.choice([(16, 2), (32, 4), (32, 8)]) if dim == 128 else rng.choice([(24, 2), (16, 2)])
        seqs, high, q8 = _size(rng, 1, 64), _size(rng, 200, 65536), rng.random() < 0.7
        row = dim + dim // 16 if q8 else 2 * dim
        high = max(64, min(high, int(1.1e9 / (seqs * kv_heads * 2 * row))))
        span = rng.choice([1, 1, 1, 2, 3, 4, 5, 8])
        return {"path": path, "seqs": seqs, "low": max(span, high // rng.choice([1, 2, 8, 32])), "high": high, "span": span, "heads": heads,
                "kv_heads": kv_heads, "dim": dim, "q8": q8, "page_tokens": rng.choice([64, 256, 256]), "io16": rng.random() < 0.8}
    if path == "prompt":
        dim = rng.choice([128, 128, 256])
        heads, kv_heads = rng.choice([(16, 2), (32, 4)]) if dim == 128 else (24, 2)
        seqs, tokens = rng.choice([1, 1, 2, 3, 5]), _size(rng, 100, 8192 if dim == 128 else 4096)
        tokens = min(tokens, int(((5.4e11 if dim == 128 else 1.2e11) / (2 * heads * dim * seqs)) ** 0.5))
        return {"path": path, "seqs": seqs, "tokens": tokens, "chunk": rng.choice([tokens, tokens, min(tokens, 2048), min(tokens, 512)]), "heads": heads,
                "kv_heads": kv_heads, "dim": dim, "q8": rng.random() < 0.8, "page_tokens": 256, "fused": dim == 128 and rng.random() < 0.7}
    if path == "stage":
        if rng.random() < 0.5:
            rows, chunks = rng.choice([1, 1, 2, 3, 4, 5, 8]), 1
        else:
            rows, chunks = _size(rng, 32, 1024), rng.choice([1, 2])
        return {"path": path, "rows": rows, "chunks": chunks, "base": 4 * _size(rng, 300, 24000 if rows > 8 else 60000), "heads": 24, "kv_heads": 2,
                "q8": rng.random() < 0.7}
    if path == "topk":
        return {"path": path, "batch": _size(rng, 1, 8), "context": _size(rng, 4096, 131072), "index_heads": rng.choice([32, 64]), "k": rng.choice([512, 1024, 2048]),
                "heads": rng.choice([16, 32, 64])}
    if path == "compressed":
        rows = rng.choice([1, 1, 2, 4, _size(rng, 8, 256), _size(rng, 8, 256)])
        return {"path": path, "rows": rows, "position": _size(rng, 500, 65000 if rows < 8 else 32768), "index_heads": rng.choice([32, 64]),
                "heads": rng.choice([32, 64]), "k": 512, "bf16": rng.random() < 0.8}
    dim = rng.choice([128, 256, 256])
    return {"path": path, "rows": rng.choice([1, 2, _size(rng, 3, 128), _size(rng, 16, 128)]), "position": _size(rng, 50, 4096), "heads": 16,
            "kv_heads": rng.choice([2, 4]), "dim": dim}


def _lengths(case):
    """Cached tokens of each sequence of a decode case, its span included: a fixed spread over [low, high] (the seed shuffles which
    sequence has which, so that every seed is the same amount of work)."""
    n, low, high = case["seqs"], max(case["low"], case["span"]), case["high"]
    return [high] if n == 1 else [low + (high - low) * i // (n - 1) for i in range(n)]


# ---- what a program has in hand ----------------------------------------------------------------------------------------

def _row_bytes(case, dim):
    return dim + dim // 16 if case["q8"] else 2 * dim


def _paged(s, lengths):
    """A pool whose pages are dealt to the sequences in a shuffled order, filled by the library's own writer from N(0, 1) rows."""
    c, g, page = s.case, s.gpu, s.case["page_tokens"]
    row = _row_bytes(c, c["dim"])
    pages = [(n + page - 1) // page for n in lengths]
    s.stride = max(pages)
    table, order, at = np.zeros((len(lengths), s.stride), np.int32), s.order.permutation(sum(pages)).astype(np.int32), 0
    for i, n in enumerate(pages):
        table[i, :n] = order[at:at + n]
        at += n
    s.put("table", table)
    s.empty("pages", sum(pages) * 2 * c["kv_heads"] * page * row, torch.uint8)
    s.pool = KvPool(s.at("pages"), sum(pages), page, c["kv_heads"], c["dim"], row)


def _fill(s, sequence, tokens):
    """Rows 0 .. tokens - 1 of a sequence, written before the pass that is measured."""
    c, g, step = s.case, s.gpu, 16384
    width = c["kv_heads"] * c["dim"]
    s.empty("fill", 2 * step * width, torch.float16)
    for first in range(0, tokens, step):
        s.views["fill"].normal_(generator=s.random)
        s.put("fill_at", np.array([first], np.int32))
        s.ready()
        g.kv_write(s.pool, s.at("table", sequence * s.stride * 4), s.stride, s.at("fill_at"), s.at("fill"), s.at("fill", step * width * 2), True, 1,
                   min(step, tokens - first))
        s.ready()
        s.drop("fill_at")
    s.drop("fill")


def _prepare_decode(s):
    c = s.case
    lengths = s.order.permutation(_lengths(c))
    _paged(s, [int(n) for n in lengths])
    for i, n in enumerate(lengths):
        _fill(s, i, int(n) - c["span"])
    s.put("positions", (lengths - c["span"]).astype(np.int32))
    kind = torch.float16 if c["io16"] else torch.float32
    rows = c["seqs"] * c["span"]
    s.normal("k", rows * c["kv_heads"] * c["dim"], kind)
    s.normal("v", rows * c["kv_heads"] * c["dim"], kind)
    s.normal("q", rows * c["heads"] * c["dim"], kind)
    s.empty("out", rows * c["heads"] * c["dim"], kind)
    s.context, s.scale = int(lengths.max()), c["dim"] ** -0.5
    s.empty("scratch", s.gpu.paged_attention_scratch(c["seqs"], c["span"], c["heads"], c["dim"], s.context), torch.uint8)


def _run_decode(s):
    c, g = s.case, s.gpu
    g.kv_write(s.pool, s.at("table"), s.stride, s.at("positions"), s.at("k"), s.at("v"), c["io16"], c["seqs"], c["span"])
    g.paged_attention(s.pool, s.at("table"), s.stride, s.at("positions"), s.context, s.at("q"), c["io16"], c["seqs"], c["span"], c["heads"], s.scale, s.at("out"),
                      c["io16"], s.buffers["scratch"])
    return {"out": s.views["out"], "pages": s.views["pages"]}


def _prepare_prompt(s):
    c = s.case
    _paged(s, [c["tokens"]] * c["seqs"])
    s.chunks = [(first, min(c["chunk"], c["tokens"] - first)) for first in range(0, c["tokens"], c["chunk"])]
    rows = c["seqs"] * c["tokens"]
    # (a chunk's rows lie together, sequence by sequence)
    s.put("starts", np.array([[first] * c["seqs"] for first, _ in s.chunks], np.int32))
    s.normal("k", rows * c["kv_heads"] * c["dim"], torch.float16)
    s.normal("v", rows * c["kv_heads"] * c["dim"], torch.float16)
    s.normal("q", rows * c["heads"] * c["dim"], torch.float16)
    s.empty("out", rows * c["heads"] * c["dim"], torch.float16)
    s.scale = c["dim"] ** -0.5
    if c["fused"]:
        s.empty("tiles", s.gpu.prefill_tiles_bytes(c["seqs"], c["kv_heads"], c["dim"], c["tokens"]), torch.uint8)
    else:
        s.empty("scratch", s.gpu.paged_attention_scratch(c["seqs"], max(n for _, n in s.chunks), c["heads"], c["dim"], c["tokens"]), torch.uint8)


def _run_prompt(s):
    c, g = s.case, s.gpu
    for i, (first, n) in enumerate(s.chunks):
        kv, q, start = first * c["seqs"] * c["kv_heads"] * c["dim"] * 2, first * c["seqs"] * c["heads"] * c["dim"] * 2, s.at("starts", 4 * i * c["seqs"])
        if c["fused"]:
            g.prefill_chunk(s.pool, s.at("table"), s.stride, start, c["tokens"], s.at("k", kv), s.at("v", kv), True, s.at("q", q), True, c["seqs"], n, c["heads"],
                            s.scale, s.at("out", q), True, s.buffers["tiles"], start)
        else:
            g.kv_write(s.pool, s.at("table"), s.stride, start, s.at("k", kv), s.at("v", kv), True, c["seqs"], n)
            g.paged_attention(s.pool, s.at("table"), s.stride, start, first + n, s.at("q", q), True, c["seqs"], n, c["heads"], s.scale, s.at("out", q), True,
                              s.buffers["scratch"])
    return {"out": s.views["out"], "pages": s.views["pages"]}


def _stage_context(case):
    return (case["base"] + case["rows"] * case["chunks"] + 255) // 256 * 256


def _prepare_stage(s):
    c, context = s.case, _stage_context(s.case)
    c.update(dim=256, page_tokens=context)
    rows, pool = c["rows"] * c["chunks"], context // 4 + 1
    _paged(s, [context])
    _fill(s, 0, c["base"])
    s.row = c["heads"] * 512 + c["kv_heads"] * 512 + 640
    # the layer's projections; neighbouring tokens ask for much the same, so their index queries differ little
    s.normal("projected", rows * s.row, torch.float32)
    at, alike = s.row - 640, 16
    index = s.views["projected"].view(rows, s.row)[:, at:at + 512]
    shared = torch.randn((rows + alike - 1) // alike, 512, device="cuda", generator=s.random)
    index.mul_(0.05).add_(shared.repeat_interleave(alike, 0)[:rows])
    s.empty("projections", rows * s.row, torch.float32)
    s.normal("blocks", 128 * pool, torch.float32)
    s.normal("history", 16 * 128, torch.float32)
    for name, n in (("q_norm", 256), ("k_norm", 256), ("index_q_norm", 128), ("index_k_norm", 128)):
        s.uniform(name, n, 0.5, 1.5)
    s.put("positions", np.arange(c["base"], c["base"] + rows, dtype=np.uint32))
    s.empty("attended", rows * c["heads"] * 256, torch.float32)
    s.state = s.gpu.qsa_state(s.pool, None, context, *[s.at(n) for n in ("blocks", "history", "q_norm", "k_norm", "index_q_norm", "index_k_norm")], c["heads"])
    size = s.gpu.qsa_decode_attend_scratch if c["rows"] <= 8 else s.gpu.qsa_prefill_attend_scratch
    s.empty("scratch", size(c["rows"], c["heads"], c["kv_heads"], context), torch.uint8)


def _run_stage(s):
    c, g = s.case, s.gpu
    # the projections arrive (the stage turns its index queries in place)
    g.copy(s.at("projections"), s.at("projected"), s.buffers["projections"].size)
    valid = [0]
    for i in range(c["chunks"]):
        first = i * c["rows"]
        rows, out = s.at("projections", first * s.row * 4), s.at("attended", first * c["heads"] * 256 * 4)
        if c["rows"] <= 8:
            g.qsa_decode_attend(s.state, rows, s.row, c["rows"], s.at("positions", 4 * first), s.at("positions", 4 * first), s.buffers["scratch"], out)
        else:
            g.qsa_prefill_attend(s.state, rows, s.row, c["rows"], c["base"] + first, s.buffers["scratch"], out, valid)
    return {name: s.views[name] for name in ("attended", "pages", "blocks", "history")}


def _prepare_topk(s):
    c = s.case
    c.update(dim=128, kdim=576, vdim=512)
    s.normal("q_index", c["batch"] * c["index_heads"] * c["dim"], torch.bfloat16)
    s.normal("keys", c["batch"] * c["context"] * c["dim"], torch.bfloat16)
    s.uniform("weights", c["batch"] * c["index_heads"], 0.0, 1.0)
    s.put("visible", np.full(c["batch"], c["context"], np.int32))
    s.empty("indices", c["batch"] * c["k"], torch.int32)
    s.normal("q", c["batch"] * c["heads"] * c["kdim"], torch.bfloat16)
    s.normal("latents", c["batch"] * c["context"] * c["kdim"], torch.bfloat16)
    s.empty("out", c["batch"] * c["heads"] * c["vdim"], torch.float32)


def _run_topk(s):
    c, g = s.case, s.gpu
    g.index_top_k(s.at("q_index"), s.at("keys"), s.at("weights"), s.at("visible"), c["batch"], c["context"], c["index_heads"], c["dim"], 1.0, None, c["k"],
                  s.at("indices"))
    g.latent_attention(s.at("q"), s.at("latents"), s.at("indices"), c["batch"], c["context"], c["k"], c["heads"], c["kdim"], c["vdim"], c["kdim"] ** -0.5, s.at("out"))
    return {"indices": s.views["indices"], "out": s.views["out"]}


_WINDOW, _RATIO, _ROPE = 128, 4, 64


def _prepare_compressed(s):
    c = s.case
    c.update(dim=512, index_dim=128)
    rows = c["rows"]
    positions = np.arange(c["position"], c["position"] + rows, dtype=np.int32)
    s.groups = int(positions[-1] + 1) // _RATIO
    kind = torch.bfloat16 if c["bf16"] else torch.float32
    s.put("positions", positions)
    s.put("visible", (positions + 1) // _RATIO)
    s.put("frequencies", (np.float32(1.6e5) ** (-(2.0 * np.arange(_ROPE // 2, dtype=np.float32)) / np.float32(_ROPE))).astype(np.float32))
    s.normal("index_q", rows * c["index_heads"] * c["index_dim"], torch.float32)
    s.normal("index_keys", s.groups * c["index_dim"], kind)
    s.uniform("weights", rows * c["index_heads"], 0.0, 1.0)
    s.empty("scores", rows * s.groups, torch.float32)
    s.empty("selected", rows * c["k"], torch.int32)
    s.ring = _WINDOW if rows == 1 else (_WINDOW + rows + 127) // 128 * 128
    s.normal("q", rows * c["heads"] * c["dim"], torch.float32)
    s.normal("raw", s.ring * c["dim"], torch.float32)
    s.normal("rows", s.groups * c["dim"], kind)
    s.normal("sinks", c["heads"], torch.float32)
    s.empty("out", rows * c["heads"] * c["dim"], torch.float32)


def _run_compressed(s):
    c, g = s.case, s.gpu
    tag = tagged_bf16 if c["bf16"] else lambda pointer: pointer
    g.index_select(s.at("index_q"), tag(s.at("index_keys")), s.at("weights"), s.at("visible"), c["rows"], s.groups, c["index_heads"], c["index_dim"],
                   (c["index_dim"] * c["index_heads"]) ** -0.5, (_ROPE, s.at("positions"), s.at("frequencies")), s.at("scores"), c["k"], s.at("selected"))
    g.sparse_attention(s.at("q"), s.at("raw"), s.ring, s.at("positions"), _WINDOW, tag(s.at("rows")), s.groups, s.at("selected"), c["k"], s.at("sinks"), c["rows"],
                       c["heads"], c["dim"], c["dim"] ** -0.5, _ROPE, s.at("frequencies"), None, s.at("out"))
    return {"scores": s.views["scores"], "selected": s.views["selected"], "out": s.views["out"]}


def _prepare_dense(s):
    c = s.case
    s.context = c["position"] + c["rows"]
    s.put("positions", np.arange(c["position"], s.context, dtype=np.int32))
    s.normal("q", c["rows"] * c["heads"] * c["dim"], torch.float32)
    s.normal("gate", c["rows"] * c["heads"] * c["dim"], torch.float32)
    s.normal("keys", s.context * c["kv_heads"] * c["dim"], torch.float32)
    s.normal("values", s.context * c["kv_heads"] * c["dim"], torch.float32)
    pairs = c["rows"] * c["heads"]
    s.empty("scratch", pairs * min(64, max(1, 256 // pairs)) * (c["dim"] + 2) * 4, torch.uint8)
    s.empty("out", c["rows"] * c["heads"] * c["dim"], torch.float32)


def _run_dense(s):
    c = s.case
    s.gpu.attention(s.at("q"), s.at("keys"), s.at("values"), s.context, s.at("positions"), c["rows"], c["heads"], c["kv_heads"], c["dim"], c["dim"] ** -0.5,
                    s.at("gate"), s.buffers["scratch"], s.at("out"))
    return s.views["out"]


_PATHS = {"decode": (_prepare_decode, _run_decode), "prompt": (_prepare_prompt, _run_prompt), "stage": (_prepare_stage, _run_stage),
          "topk": (_prepare_topk, _run_topk), "compressed": (_prepare_compressed, _run_compressed), "dense": (_prepare_dense, _run_dense)}


def prepare(case, seed):
    state = _State(case, seed)
    _PATHS[case["path"]][0](state)
    state.ready()
    return state


def run(state):
    return _PATHS[state.case["path"]][1](state)


# ---- what a pass cannot do without ---------------------------------------------------------------------------------------

def work(case):
    c, path = case, case["path"]
    if path == "decode":
        lengths, rows, size = _lengths(c), c["seqs"] * c["span"], 2 if c["io16"] else 4
        cache = sum(lengths) * c["kv_heads"] * 2 * _row_bytes(c, c["dim"])
        io = rows * c["dim"] * size * (2 * c["heads"] + 2 * c["kv_heads"])
        return {"bytes": cache + io, "flops": 4 * c["heads"] * c["dim"] * c["span"] * sum(lengths)}
    if path == "prompt":
        tokens = c["seqs"] * c["tokens"]
        return {"bytes": tokens * c["dim"] * 4 * (c["heads"] + c["kv_heads"]) + tokens * c["kv_heads"] * 2 * _row_bytes(c, c["dim"]),
                "flops": 4 * c["heads"] * c["dim"] * c["seqs"] * (c["tokens"] * (c["tokens"] + 1) // 2)}
    if path == "stage":
        rows, end = c["rows"] * c["chunks"], c["base"] + c["rows"] * c["chunks"]
        seen = min(2052, end)
        row = c["heads"] * 512 + c["kv_heads"] * 512 + 640
        cache = min(rows * seen, end) * c["kv_heads"] * 2 * _row_bytes(c, 256)
        return {"bytes": end // 4 * 512 + cache + rows * (row + c["heads"] * 256) * 4, "flops": rows * (end // 4 * 1024 + seen * c["heads"] * 1024)}
    if path == "topk":
        gathered = c["batch"] * c["k"] * 576 * 2
        return {"bytes": c["batch"] * c["context"] * 256 + gathered + c["batch"] * (c["index_heads"] * 260 + c["k"] * 4 + c["heads"] * (576 * 2 + 512 * 4)),
                "flops": c["batch"] * (c["context"] * c["index_heads"] * 256 + c["k"] * c["heads"] * 2 * (576 + 512))}
    if path == "compressed":
        rows, groups, value = c["rows"], (c["position"] + c["rows"]) // _RATIO, 2 if c["bf16"] else 4
        cache = groups * 128 * value + min(rows * c["k"], groups) * 512 * value + min(c["position"], _WINDOW + rows) * 2048
        return {"bytes": cache + rows * (groups * 4 + c["index_heads"] * 516 + c["k"] * 4 + c["heads"] * 4096),
                "flops": rows * (groups * c["index_heads"] * 256 + (_WINDOW + c["k"]) * c["heads"] * 2048)}
    context = c["position"] + c["rows"]
    return {"bytes": context * c["kv_heads"] * c["dim"] * 8 + c["rows"] * c["heads"] * c["dim"] * 12,
            "flops": 4 * c["rows"] * c["heads"] * c["dim"] * (c["position"] + c["rows"] // 2)}


def tolerance(case):
    # Four times what the paths were measured to differ from themselves in 64 bits on the same stored rows.  FP16 operands and weights
    # (and FP16 outputs): 2.5e-4 to 5e-4; over selected rows of a long context, where few rows carry the weight, up to 1e-3.  FP32: up to
    # 1.5e-6.  Whole numbers (selected rows, cache bytes) are the same.
    return {"rel": {"decode": 2e-3, "prompt": 2e-3, "stage": 4e-3}.get(case["path"], 1e-5)}
