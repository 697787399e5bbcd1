"""The work that a serving program has this framework do, as measurable cases.

Each case is one pass through the public entry points: a whole small decode
step, the decode attention of a step's layers at several head shapes and batch
forms, prompt attention, the all-layer KV append, the de-page of sequences and
a swap round trip.  Geometries are the ones the framework's workloads and tests
name; a pool holds a few of a model's layers, so that a case fits beside two
more of its kind.

``listed`` names the cases, ``draw`` makes more of the same ranges, ``prepare``
makes what a program has in hand before the call, ``run`` is the pass,
``work`` the bytes and operations it cannot do without, ``tolerance`` and
``exact`` what its outputs are compared with.
"""
import math

import numpy as np
import torch

from aegaeon_amd import attention as A
from aegaeon_amd import ops
from aegaeon_amd.inputs import prepare_model_inputs

BLOCK = 16  # tokens per KV block
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def _case(name, kind, dtype, hq, hkv, dim, layers, seqs, mean, sigma, lo, hi, lens_seed=0, **more):
    """``seqs`` sequences (prompts) whose lengths are lognormal with arithmetic
    mean ``mean`` and ``sigma``, clipped to [lo, hi]; sigma 0: all ``mean``."""
    return dict(name=name, kind=kind, dtype=dtype, hq=hq, hkv=hkv, dim=dim, layers=layers,
                seqs=seqs, mean=mean, sigma=sigma, lo=lo, hi=hi, lens_seed=lens_seed, **more)


def listed():
    return [
        # The smallest whole decode step: request lists to device inputs, the
        # KV write and the attention of one layer (8 short sequences): latency.
        _case("step_tiny", "step", "fp16", 2, 2, 64, 1, 8, 60, 0.8, 1, 128),
        # Decode attention of a loaded engine: Qwen2.5-7B heads, 128 sequences
        # of very different lengths, one plan for the step's layers.
        _case("decode_qwen_128", "decode", "bf16", 28, 4, 128, 4, 128, 1500, 1.0, 16, 8192,
              append=False),
        # A smaller batch (Yi-1.5-9B heads) whose KV write is fused into the call.
        _case("decode_append_yi_64", "decode", "bf16", 32, 4, 128, 4, 64, 1000, 1.0, 16, 4096,
              append=True),
        # Multi-head attention without grouping (Llama-2-13B): the most KV bytes
        # per token, sequences of one length.
        _case("decode_llama_32", "decode", "fp16", 40, 40, 128, 1, 32, 2048, 0.0, 1, 4096,
              append=False),
        # One very long context (a document being discussed): one sequence over
        # the whole chip.
        _case("decode_long_context", "decode", "bf16", 28, 4, 128, 2, 1, 131001, 0.0, 1, 131072,
              append=False),
        # One kv head per GPU: Qwen2.5-7B cut over four GPUs by kv head, or a
        # multi-query model.
        _case("decode_one_kv_head", "decode", "bf16", 7, 1, 128, 4, 256, 1000, 1.0, 16, 4096,
              append=True),
        # Prompt run of four long prompts, causal, q/k/v views of the fused
        # projection's output.
        _case("prefill_qwen_4x2048", "prefill", "bf16", 28, 4, 128, 1, 4, 2048, 0.0, 1, 2048,
              causal=True),
        # One long document.
        _case("prefill_qwen_1x8192", "prefill", "bf16", 28, 4, 128, 1, 1, 8192, 0.0, 1, 8192,
              causal=True),
        # Many chat-sized prompts of different lengths in one batch.
        _case("prefill_short_48", "prefill", "fp16", 32, 4, 128, 1, 48, 220, 0.8, 16, 1024,
              causal=True),
        # The KV write of a decode step for every layer at once (Qwen2.5-7B, 256
        # sequences x 28 layers).
        _case("append_qwen_256", "append", "bf16", 28, 4, 128, 28, 256, 40, 0.5, 1, 96),
        # De-page of a batch's sequences into contiguous K and V, one layer.
        _case("gather_qwen_256", "gather", "bf16", 28, 4, 128, 1, 256, 600, 1.0, 16, 4096),
        # Model switch: a request set's blocks out to pinned host memory and back
        # into other blocks of the pool (all 28 layers of a Qwen2.5-7B block).
        _case("swap_qwen_256", "swap", "bf16", 28, 4, 128, 28, 16, 256, 0.0, 16, 256),
    ]


# (query heads, kv heads, head dim) of the framework's models and tests
_SHAPES = [(28, 4, 128), (32, 4, 128), (40, 40, 128), (8, 8, 128), (16, 1, 64), (7, 1, 128),
           (14, 2, 128), (12, 6, 128), (2, 2, 64), (6, 2, 256)]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed ones' ranges."""
    kind = rng.choice(["step", "decode", "decode", "decode", "prefill", "prefill", "append",
                       "gather", "swap"])
    dtype = rng.choice(["bf16", "fp16"])
    hq, hkv, dim = rng.choice(_SHAPES)
    seed = rng.randrange(1 << 20)
    row = 4 * hkv * dim  # K and V bytes of a token in a layer
    if kind == "step":
        layers, seqs, hi = rng.randint(1, 4), _log_int(rng, 1, 256), 512
        mean = _log_int(rng, 4, 200)
        return _draw(kind, dtype, hq, hkv, dim, layers, seqs, mean, 0.8, 1, hi, seed)
    if kind == "decode":
        layers = rng.randint(1, 4)
        budget = (1 << 30) // (row * layers)  # tokens
        seqs = _log_int(rng, 1, 512)
        mean = _log_int(rng, 24, max(32, min(65536, budget // seqs)))
        sigma = rng.choice([0.0, 0.5, 1.0])
        return _draw(kind, dtype, hq, hkv, dim, layers, seqs, mean, sigma, 1,
                     max(32, min(131072, 6 * mean)), seed, append=rng.random() < 0.5)
    if kind == "prefill":
        if dim == 256:
            hq, hkv, dim = 28, 4, 128
        seqs = _log_int(rng, 1, 64)
        causal = rng.random() < 0.8
        # at most the one-document case's operations
        top = int(math.sqrt(2.2e11 / (4 * hq * dim * seqs))) if causal else \
            int(math.sqrt(1.1e11 / (4 * hq * dim * seqs)))
        mean = _log_int(rng, 16, max(32, min(8192, top)))
        sigma = rng.choice([0.0, 0.4, 0.8])
        return _draw(kind, dtype, hq, hkv, dim, 1, seqs, mean, sigma, 1,
                     max(32, min(8192, 3 * mean)), seed, causal=causal)
    if kind == "append":
        layers, seqs = rng.choice([1, 8, 28, 40]), _log_int(rng, 1, 512)
        while seqs * layers * row > 60 << 20:
            seqs = (seqs + 1) // 2
        return _draw(kind, dtype, hq, hkv, dim, layers, seqs, rng.randint(8, 48), 0.5, 1, 96, seed)
    if kind == "gather":
        layers, seqs = rng.randint(1, 3), _log_int(rng, 1, 512)
        budget = (300 << 20) // (row * layers)
        mean = _log_int(rng, 16, max(32, min(8192, budget // seqs)))
        return _draw(kind, dtype, hq, hkv, dim, layers, seqs, mean, rng.choice([0.0, 0.8]), 1,
                     max(32, 4 * mean), seed)
    layers, seqs = rng.choice([4, 28]), _log_int(rng, 1, 16)
    budget = (200 << 20) // (row * layers)
    mean = _log_int(rng, 16, max(24, min(2048, budget // seqs)))
    return _draw("swap", dtype, hq, hkv, dim, layers, seqs, mean, 0.4, 1, 2 * mean, seed)


def _draw(kind, *args, **more):
    c = _case("", kind, *args, **more)
    del c["name"]
    return c


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _lengths(case):
    """The case's lengths (the same for every seed; prepare orders them by it)."""
    n, mean, sigma = case["seqs"], case["mean"], case["sigma"]
    if sigma == 0:
        return np.full(n, max(case["lo"], min(case["hi"], mean)), dtype=np.int64)
    rng = np.random.default_rng(case["lens_seed"])
    x = rng.lognormal(math.log(mean) - sigma * sigma / 2, sigma, size=n)
    return np.clip(np.rint(x), case["lo"], case["hi"]).astype(np.int64)


class State:
    """What the program holds: tensors and lists by name."""

    def __init__(self, **kw):
        self.__dict__.update(kw)


def _normal(gen, shape, dtype):
    return torch.empty(shape, dtype=dtype, device="cuda").normal_(generator=gen)


def _tables(rng, need, pool):
    ids = rng.permutation(pool)
    out, o = [], 0
    for n in need:
        out.append(ids[o:o + n].astype(np.int32).tolist())
        o += n
    return out, ids[o:]


def _pool_blocks(need):
    return int(sum(need) * 5 // 4) + 16


def _padded(tables):
    w = max(len(t) for t in tables)
    out = np.zeros((len(tables), w), dtype=np.int32)
    for i, t in enumerate(tables):
        out[i, :len(t)] = t
    return torch.from_numpy(out).cuda()


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dt = DTYPES[case["dtype"]]
    hq, hkv, dim, layers = case["hq"], case["hkv"], case["dim"], case["layers"]
    kind = case["kind"]
    lens = rng.permutation(_lengths(case))
    n = len(lens)
    scale = 1.0 / math.sqrt(dim)
    if kind == "prefill":
        cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
        qkv = _normal(gen, (int(cu[-1]), (hq + 2 * hkv) * dim), dt)
        q, k, v = qkv.split([hq * dim, hkv * dim, hkv * dim], dim=1)
        return State(kind=kind, q=q.unflatten(1, (hq, dim)), k=k.unflatten(1, (hkv, dim)),
                     v=v.unflatten(1, (hkv, dim)), cu=torch.from_numpy(cu).cuda(),
                     longest=int(lens.max()), lens=lens, scale=scale, causal=case["causal"])
    # the sequences' last token is the step's new one
    need = [-(-int(x) // BLOCK) for x in lens]
    pool = _pool_blocks(need)
    tables, spare = _tables(rng, need, pool if kind != "swap" else 2 * pool)
    if kind == "swap":
        cache = _normal(gen, (2 * pool, layers, 2, BLOCK, hkv, dim), dt)
        ids = [b for t in tables for b in t]
        host = torch.empty((len(ids), layers, 2, BLOCK, hkv, dim), dtype=dt, pin_memory=True)
        return State(kind=kind, cache=cache, host=host, gpu_ids=ids,
                     cpu_ids=list(range(len(ids))), back_ids=spare[:len(ids)].tolist())
    cache = _normal(gen, (pool, layers, 2, BLOCK, hkv, dim), dt)
    seq = torch.from_numpy(lens.astype(np.int32)).cuda()
    st = State(kind=kind, cache=cache, lens=lens, tables=tables, seq_lens=seq,
               longest=int(lens.max()), scale=scale)
    if kind == "gather":
        st.block_tables = _padded(tables)
        st.total = int(lens.sum())
        st.cu = torch.zeros(n + 1, dtype=torch.int32, device="cuda")
        torch.cumsum(seq, 0, dtype=torch.int32, out=st.cu[1:])
        return st
    st.k = _normal(gen, (layers, n, hkv, dim), dt)
    st.v = _normal(gen, (layers, n, hkv, dim), dt)
    if kind == "append":
        last = lens - 1
        slots = [t[p // BLOCK] * BLOCK + p % BLOCK for t, p in zip(tables, last)]
        st.slots = torch.tensor(slots, dtype=torch.int64, device="cuda")
        return st
    st.q = _normal(gen, (layers, n, hq, dim), dt)
    if kind == "step":
        st.requests = [(i, [int(rng.integers(0, 32000))], int(x), int(x) - 1)
                       for i, x in enumerate(lens)]
        # a first token has no context: such a request decodes its second one
        st.requests = [r if r[3] > 0 else (r[0], r[1], 2, 1) for r in st.requests]
        st.lens = np.maximum(lens, 2)
        return st
    st.block_tables = _padded(tables)
    st.append = case["append"]
    return st


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(st):
    if st.kind == "step":
        tokens, positions, md = prepare_model_inputs(st.requests, st.tables, st.cache.device)
        outs = []
        for l in range(st.cache.size(1)):
            kc, vc = st.cache[:, l, 0], st.cache[:, l, 1]
            A.reshape_and_cache_flash(st.k[l], st.v[l], kc, vc, md["slot_mapping"])
            outs.append(A.flash_attn_with_kvcache(
                st.q[l].unsqueeze(1), kc, vc, cache_seqlens=md["seq_lens_tensor"],
                block_table=md["block_tables"], softmax_scale=st.scale,
                max_seqlen=md["max_decode_seq_len"]))
        return {"out": outs, "cache": st.cache, "tokens": tokens, "positions": positions,
                "slots": md["slot_mapping"]}
    if st.kind == "decode":
        plan = A.DecodePlan(st.block_tables, st.seq_lens, st.longest, st.cache.size(4))
        outs = []
        for l in range(st.cache.size(1)):
            outs.append(A.paged_decode_attention(
                st.q[l], st.cache[:, l, 0], st.cache[:, l, 1], None, None, st.scale, st.longest,
                plan=plan, key=st.k[l] if st.append else None,
                value=st.v[l] if st.append else None))
        return {"out": outs, "cache": st.cache} if st.append else {"out": outs}
    if st.kind == "prefill":
        return {"out": A.flash_attn_varlen_func(st.q, st.k, st.v, st.cu, st.cu, st.longest,
                                                st.longest, softmax_scale=st.scale,
                                                causal=st.causal)}
    if st.kind == "append":
        A.append_kv(st.k, st.v, st.cache, st.slots)
        return {"cache": st.cache}
    if st.kind == "gather":
        k, v = A.gather_tokens(st.cache, st.block_tables, st.seq_lens, st.total, st.longest,
                               cu_seqlens=st.cu)
        return {"k": k, "v": v}
    ops.swap(st.gpu_ids, st.cpu_ids, False, st.cache, st.host)
    ops.swap(st.cpu_ids, st.back_ids, True, st.cache, st.host)
    return {"host": st.host, "cache": st.cache}


# ---------------------------------------------------------------------------
# what a pass cannot do without, and what its outputs are compared with
# ---------------------------------------------------------------------------
def work(case):
    hq, hkv, dim, layers = case["hq"], case["hkv"], case["dim"], case["layers"]
    lens = _lengths(case)
    if case["kind"] == "step":
        lens = np.maximum(lens, 2)
    n, total = len(lens), int(lens.sum())
    row = 2 * hkv * dim * 2  # K and V of a token
    blocks = int(sum(-(-int(x) // BLOCK) for x in lens))
    if case["kind"] == "prefill":
        pairs = int(sum(int(x) * (int(x) + 1) // 2 if case["causal"] else int(x) ** 2
                        for x in lens))
        return {"bytes": total * (2 * hq * dim * 2 + row) + 4 * (n + 1),
                "flops": 4 * hq * dim * pairs}
    if case["kind"] == "swap":  # the pool's blocks read once, other ones written once
        return {"bytes": 2 * blocks * layers * BLOCK * row, "flops": 0}
    if case["kind"] == "append":
        return {"bytes": 2 * n * layers * row + 8 * n, "flops": 0}
    if case["kind"] == "gather":
        return {"bytes": 2 * total * layers * row + 4 * blocks + 8 * n, "flops": 0}
    per_layer = total * row + 2 * n * hq * dim * 2
    if case["kind"] == "step" or case["append"]:
        per_layer += n * row  # the cache rows written (the new rows count as read above)
    return {"bytes": layers * per_layer + 4 * blocks + 4 * n,
            "flops": 4 * layers * hq * dim * total}


def tolerance(case):
    """Byte moves are exact.  Attention accumulates in 32 bits and rounds its
    output to 16: the relative error against 64 bits is that rounding's
    (measured: bf16 1.7e-3, fp16 2.1e-4) in decode, and with P rounded to 16
    bits as well in the prompt run (bf16 2.1e-3, fp16 2.4e-4); four times that."""
    if case["kind"] in ("append", "gather", "swap"):
        return "exact"
    if case["kind"] == "prefill":
        return {"rel": 8.5e-3} if case["dtype"] == "bf16" else {"rel": 1e-3}
    return {"rel": 7e-3} if case["dtype"] == "bf16" else {"rel": 9e-4}


def _softmax_pv(q, k, v, scale, mask=None):
    """[Hkv, m, D] x [Hkv, n, D] -> [Hkv, m, D], all in 64 bits."""
    s = torch.matmul(q, k.transpose(1, 2).contiguous()) * scale
    if mask is not None:
        s.masked_fill_(mask, -math.inf)
    return torch.matmul(torch.softmax(s, -1), v)


def exact(case, seed):
    if case["kind"] in ("append", "gather", "swap"):
        return None  # copies of 16-bit values
    st = prepare(case, seed)
    hq, hkv, dim, layers = case["hq"], case["hkv"], case["dim"], case["layers"]
    group = hq // hkv
    if case["kind"] == "prefill":
        out = torch.zeros(st.q.shape, dtype=torch.float64, device="cuda")
        t0 = 0
        for x in st.lens:
            x = int(x)
            pos = torch.arange(x, device="cuda")
            mask = pos[None, :] > pos[:, None] if st.causal else None
            for h in range(hq):
                kh, vh = st.k[t0:t0 + x, h // group], st.v[t0:t0 + x, h // group]
                out[t0:t0 + x, h] = _softmax_pv(st.q[t0:t0 + x, h].double()[None],
                                                kh.double()[None], vh.double()[None], st.scale,
                                                mask)[0]
            t0 += x
        return {"out": out}
    outs = []
    appends = case["kind"] == "step" or case["append"]
    for l in range(layers):
        out = torch.zeros((len(st.lens), hq, dim), dtype=torch.float64, device="cuda")
        for b, x in enumerate(st.lens):
            x = int(x)
            ids = torch.tensor(st.tables[b], dtype=torch.int64, device="cuda")
            kv = st.cache[:, l].index_select(0, ids).double()  # [blocks, 2, 16, Hkv, D]
            k = kv[:, 0].reshape(-1, hkv, dim)[:x].transpose(0, 1).contiguous()
            v = kv[:, 1].reshape(-1, hkv, dim)[:x].transpose(0, 1).contiguous()
            if appends:
                k[:, x - 1] = st.k[l, b].double()
                v[:, x - 1] = st.v[l, b].double()
            out[b] = _softmax_pv(st.q[l, b].double().view(hkv, group, dim), k, v,
                                 st.scale).view(hq, dim)
        outs.append(out.unsqueeze(1) if case["kind"] == "step" else out)
    if case["kind"] == "step":
        return {"out": outs, "cache": None, "tokens": None, "positions": None, "slots": None}
    return {"out": outs, "cache": None} if appends else {"out": outs}
