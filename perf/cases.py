"""Performance cases of the reshard engine: what a user's program has it do.

A case is one destination rank's share of a plan change (tensor-parallel
degree, pipeline stages) of a GPT, Llama or Qwen2 model's training state,
through one of the public entry points (``entry``):

* ``send``      ``TransferOp.get_send_tensor`` of every piece that is cut from
                a coarser shard (the sending side's loop);
* ``migrate``   ``schedule_and_execute_param_transfer``: the whole drop-in call,
                schedule included, as a job that migrates once makes it;
* ``call``      ``execute_param_transfer`` of a schedule, fresh destinations;
* ``adopt``     the same with ``arena=True``: the state of a whole model in one
                allocation, which the model then adopts;
* ``resume``    ``execute_param_transfer`` with the sources in host memory, as a
                checkpoint leaves them, and the result on the GPU;
* ``reshard``   a kept ``ReshardPlan``: one direct gather into kept destinations;
* ``refresh``   the same into fresh destinations at every call;
* ``exchange``  a kept plan's pack into per-peer buffers, then the unpack;
* ``noalloc``   ``sr_gather_noalloc``, for programs that may not allocate.

State fields (``fields``): ``f32x3`` = f32 param, exp_avg, exp_avg_sq; ``mixed``
= bf16 param with f32 master and moments; ``recast`` = f32 master and moments,
the bf16 param rounded from master on the way.

Every output is a copy of input bytes or one defined rounding of an f32
value, so all results are compared exactly.
"""
import torch

from suika_amd import execute_param_transfer, schedule_and_execute_param_transfer, schedule_param_transfer
from suika_amd.inventory import ModelSpec, Parallel, build_layout
from suika_amd.plan import ReshardPlan

ALIGN = 256          # bytes between the kept destinations' starting points
MAX_OUTPUTS = 64     # more tensors than this come back as one flat tensor per field

# field -> dtype of the source state
FIELDS = {
    "f32x3": {"param": torch.float32, "exp_avg": torch.float32, "exp_avg_sq": torch.float32},
    "mixed": {"param": torch.bfloat16, "master": torch.float32, "exp_avg": torch.float32,
              "exp_avg_sq": torch.float32},
    "recast": {"master": torch.float32, "exp_avg": torch.float32, "exp_avg_sq": torch.float32},
}
STD = {"param": 0.02, "master": 0.02, "exp_avg": 1e-3, "exp_avg_sq": 1e-6}


def _case(name, entry, family, fields, src, dst, at=(0, 0), layers=1, hidden=768, heads=12, kv_heads=0, head_dim=0,
          ffn=3072, vocab=50304, fused_qkv=False, vocab_parallel=False, positions=0, embeddings=True):
    """``src`` / ``dst``: (tensor-parallel, pipeline) degrees; ``at``: the
    destination's (stage, tensor-parallel rank)."""
    c = {"entry": entry, "family": family, "fields": fields, "src_tp": src[0], "src_pp": src[1], "dst_tp": dst[0],
         "dst_pp": dst[1], "at_pp": at[0], "at_tp": at[1], "layers": layers, "hidden": hidden, "heads": heads,
         "kv_heads": kv_heads, "head_dim": head_dim, "ffn": ffn, "vocab": vocab, "fused_qkv": fused_qkv,
         "vocab_parallel": vocab_parallel, "positions": positions, "embeddings": embeddings}
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # The sending side of a migration step: the pieces of one GPT-125M block, tensor by tensor.
        _case("send_gpt125m_block", "send", "gpt", "f32x3", (1, 1), (2, 1), embeddings=False),
        # The smallest whole migration: the test model's shapes, where launches and host work are all there is.
        _case("migrate_gpt_test", "migrate", "gpt", "f32x3", (1, 1), (2, 1), at=(0, 1), hidden=16, heads=4, ffn=64,
              vocab=128),
        # One pipeline stage's share through the drop-in call: GPT-125M's embedding, head and a block, TP2 -> TP4.
        _case("call_gpt125m_stage", "call", "gpt", "f32x3", (2, 1), (4, 1)),
        # The whole GPT-125M share, adopted by the model from one allocation.
        _case("adopt_gpt125m", "adopt", "gpt", "f32x3", (2, 1), (4, 1), layers=12),
        # Blocks merged TP4 -> TP2 by a kept plan into fresh tensors each time: a few MB, launch bound.
        _case("refresh_gpt125m_block", "refresh", "gpt", "f32x3", (4, 1), (2, 1), at=(0, 1), embeddings=False),
        # A serving loop that may not allocate: GPT-125M TP2 -> TP4.
        _case("noalloc_gpt125m", "noalloc", "gpt", "f32x3", (2, 1), (4, 1), at=(0, 1), layers=12),
        # The headline plan change, TP4 PP2 -> TP2 PP2 at Llama2-7B's width, pack and unpack (8 of its 32 layers).
        _case("exchange_llama7b", "exchange", "llama", "mixed", (4, 2), (2, 2), layers=8, hidden=4096, heads=32,
              ffn=11008, vocab=32000, vocab_parallel=True),
        # Head-granular fused QKV at Llama2-13B's width, TP8 -> TP4 PP2, second stage (8 of 40 layers).
        _case("reshard_llama13b_qkv", "reshard", "llama", "mixed", (8, 1), (4, 2), at=(1, 2), layers=8, hidden=5120,
              heads=40, ffn=13824, vocab=32000, fused_qkv=True, vocab_parallel=True),
        # f32 state split TP2 -> TP4 with the bf16 parameter rounded on the way, Qwen2-7B's width (4 of 28 layers).
        _case("reshard_qwen7b_recast", "reshard", "qwen", "recast", (2, 1), (4, 1), at=(0, 3), layers=4, hidden=3584,
              heads=28, kv_heads=4, head_dim=128, ffn=18944, vocab=152064, vocab_parallel=True),
        # A feed-forward width that is no multiple of 16 bytes per rank (the Qwen2 test model's), merged TP2 -> TP1.
        _case("exchange_ragged_merge", "exchange", "qwen", "mixed", (2, 1), (1, 1), layers=24, hidden=1024, heads=4,
              kv_heads=2, head_dim=256, ffn=2028, vocab=1024),
        # An 8/3 feed-forward width left unrounded (2730 of 1024): odd columns per rank, split with the rounding.
        _case("reshard_ragged_split", "reshard", "llama", "recast", (1, 1), (2, 1), at=(0, 1), layers=12, hidden=1024,
              heads=8, ffn=2730, vocab=32002),
        # Resuming from a checkpoint in host memory: GPT-125M's embedding, head and a block to the GPU.
        _case("resume_gpt125m_stage", "resume", "gpt", "f32x3", (2, 1), (4, 1), at=(0, 1)),
    ]


# ------------------------------------------------------------------ shapes

def _spec(c):
    return ModelSpec(c["family"], n_layer=c["layers"], hidden=c["hidden"], n_head=c["heads"], ffn=c["ffn"],
                     vocab=c["vocab"], n_kv_head=c["kv_heads"] or None, head_dim=c["head_dim"] or None,
                     fused_qkv=c["fused_qkv"], vocab_parallel=c["vocab_parallel"], positions=c["positions"],
                     embeddings=c["embeddings"])


def _plans(c):
    return Parallel(c["src_tp"], c["src_pp"]), Parallel(c["dst_tp"], c["dst_pp"])


def _layouts(c):
    """Source and target layouts, the destination rank and its names."""
    m, (src, dst) = _spec(c), _plans(c)
    dtypes = FIELDS[c["fields"]]
    spl = build_layout(m, src, dtypes.get("param", torch.float32))
    tpl = build_layout(m, dst, torch.float32 if c["fields"] == "f32x3" else torch.bfloat16)
    return spl, tpl, dst.rank(c["at_pp"], c["at_tp"])


def _outputs_of(c):
    """Destination fields and their dtypes, in result order."""
    out = dict(FIELDS[c["fields"]])
    if c["fields"] == "recast":
        out = {"param": torch.bfloat16, **out}
    return out


def _flat(c, names):
    return len(names) * len(_outputs_of(c)) > MAX_OUTPUTS


def _numel(shape):
    n = 1
    for s in shape:
        n *= int(s)
    return n


def work(c):
    """Bytes read once and written once; nothing is computed but roundings."""
    _, tpl, rank = _layouts(c)
    names = tpl.layout[rank]
    if c["entry"] == "send":
        cut = sum(_numel(m.actual_shape()) for n, m in names.items() if _kind(c, n) != "repl")
        return {"bytes": 2 * 4 * cut, "flops": 0}
    read = sum(d.itemsize for d in FIELDS[c["fields"]].values())
    wrote = sum(d.itemsize for d in _outputs_of(c).values())
    elems = 0     # read from sources: a padded vocabulary's empty rows are not
    total = 0
    for n, m in names.items():
        shape = [int(s) for s in m.actual_shape()]
        total += _numel(shape)
        if _kind(c, n) == "vocab":
            lo, hi = m.valid_rows()
            shape[0] = hi - lo
        elems += _numel(shape)
    if c["entry"] == "exchange":   # pack writes and unpack reads the buffers
        return {"bytes": 3 * elems * read + total * wrote, "flops": 0}
    return {"bytes": elems * read + total * wrote, "flops": 0}


def tolerance(c):
    return "exact"


# ------------------------------------------------------------------ state

def _sources(c, seed, device="cuda"):
    """{rank: {name: {field: shard}}} of the source ranks that the share
    reads, drawn on the device, and the schedule."""
    spl, tpl, rank = _layouts(c)
    schedule = schedule_param_transfer(spl, tpl, minimum_est_peers=2)
    reads = sorted({(op.src_rank, op.param_name) for op in schedule if op.dst_rank == rank})
    gen = torch.Generator(device=device)
    gen.manual_seed(int(seed))
    out = {}
    for r, name in reads:
        shape = tuple(int(s) for s in spl.layout[r][name].actual_shape())
        entry = {}
        for f, dt in FIELDS[c["fields"]].items():
            if f == "param" and c["fields"] == "mixed":
                continue
            t = torch.randn(shape, generator=gen, device=device).mul_(STD[f])
            entry[f] = t.abs_() if f == "exp_avg_sq" else t
        if c["fields"] == "mixed":
            entry["param"] = entry["master"].to(torch.bfloat16)
        out.setdefault(r, {})[name] = {f: entry[f] for f in FIELDS[c["fields"]]}
    return out, schedule, spl, tpl, rank


def _kept_destinations(c, metas):
    """One zeroed buffer per field and every destination tensor as a view of
    it, each at an aligned place; the flat buffers are the outputs."""
    flats, dst = {}, {n: {} for n in metas}
    for f, dt in _outputs_of(c).items():
        at, end = {}, 0
        for n, m in metas.items():
            at[n] = end
            size = _numel(m.actual_shape()) * dt.itemsize
            end += -(-size // ALIGN) * ALIGN
        flats[f] = torch.zeros(end // dt.itemsize, dtype=dt, device="cuda")
        for n, m in metas.items():
            shape = tuple(int(s) for s in m.actual_shape())
            a = at[n] // dt.itemsize
            dst[n][f] = flats[f][a:a + _numel(shape)].view(shape)
    return flats, dst


def prepare(c, seed):
    src, schedule, spl, tpl, rank = _sources(c, seed)
    metas = tpl.layout[rank]
    recast = {"param": "master"} if c["fields"] == "recast" else {}
    s = {"case": c, "src": src, "rank": rank, "names": list(metas), "recast": recast,
         "fields": [(f, "normal") for f in FIELDS[c["fields"]]], "device": torch.device("cuda", 0)}
    entry = c["entry"]
    if entry == "migrate":
        s.update(spl=spl, tpl=tpl, context={"expected_sub_fields": s["fields"]})
    elif entry in ("call", "adopt"):
        s["schedule"] = schedule
    elif entry == "resume":
        s["schedule"] = schedule
        s["src"] = {r: {n: {f: t.cpu() for f, t in e.items()} for n, e in ents.items()} for r, ents in src.items()}
    elif entry == "send":
        s["ops"] = [op for op in schedule if op.dst_rank == rank and _kind(c, op.param_name) != "repl"]
    else:
        ops = [op for op in schedule if op.dst_rank == rank]
        plan, src_ptrs = ReshardPlan.from_sources(ops, lambda r: src[r], list(FIELDS[c["fields"]]), s["device"],
                                                  recast=recast)
        s.update(plan=plan, src_ptrs=src_ptrs)
        if entry != "refresh":
            s["flats"], dst = _kept_destinations(c, metas)
            s["dst"] = dst
            s["dst_ptrs"] = plan.dst_pointers(dst)
        if entry == "exchange":
            s["bufs"] = plan.alloc_buffers(s["device"])
            s["buf_ptrs"] = plan.buf_pointers(s["bufs"])
    torch.cuda.synchronize()
    return s


def _result(s, state):
    """A returned state dict: its tensors, or where they are many the spans
    of the one allocation that they lie in (sizes without gaps)."""
    names = s["names"]
    if not _flat(s["case"], names):
        return state
    out = {}
    for f in _outputs_of(s["case"]):
        first, last = state[names[0]][f], state[names[-1]][f]
        n = last.storage_offset() + last.numel() - first.storage_offset()
        out[f] = first.as_strided((n,), (1,))
    return out


def run(s):
    entry = s["case"]["entry"]
    if entry == "reshard":
        s["plan"].gather_ptrs(s["src_ptrs"], s["dst_ptrs"])
        return s["flats"]
    if entry == "exchange":
        s["plan"].pack_ptrs(s["src_ptrs"], s["buf_ptrs"])
        s["plan"].unpack_ptrs(s["buf_ptrs"], s["dst_ptrs"])
        return s["flats"]
    if entry == "noalloc":
        s["plan"].gather_noalloc_ptrs(s["src_ptrs"], s["dst_ptrs"])
        return s["flats"]
    if entry == "refresh":
        dst, dst_ptrs = s["plan"].alloc_dst_ptrs(s["device"])
        s["plan"].gather_ptrs(s["src_ptrs"], dst_ptrs)
        return dst
    if entry == "send":
        return {op.param_name: op.get_send_tensor(s["src"][op.src_rank][op.param_name]["param"]) for op in s["ops"]}
    if entry == "migrate":
        return schedule_and_execute_param_transfer(s["spl"], s["tpl"], {}, s["context"], s["device"], None, None,
                                                   False, rank=s["rank"], recast=s["recast"],
                                                   fake_source_state_dicts=s["src"])
    state = execute_param_transfer(s["schedule"], {}, s["device"], s["fields"], rank=s["rank"], recast=s["recast"],
                                   fake_source_state_dicts=s["src"], arena=entry == "adopt")
    return _result(s, state)


# ------------------------------------------------------------------ the same by plain torch

def _kind(c, name):
    """How a tensor is split over the tensor-parallel ranks."""
    if name.endswith(("c_proj.linear.weight", "o_proj.weight", "down_proj.weight")):
        return "row"
    if name == "wte.weight":
        return "vocab" if c["vocab_parallel"] else "repl"
    if "qkv_proj" in name:
        return "qkv"
    if "ln_" in name or "norm" in name or name.endswith("c_proj.linear.bias") or name == "wpe.weight":
        return "repl"
    return "col"


def _projections(c, t, parts):
    """A fused QKV shard of 1/parts of the heads: its Q, K and V rows."""
    hd = c["head_dim"] or c["hidden"] // c["heads"]
    q, kv = c["heads"] * hd // parts, (c["kv_heads"] or c["heads"]) * hd // parts
    return t.split([q, kv, kv], 0)


def _expected(c, name, shards):
    """One destination tensor from {source tensor-parallel rank: shard}."""
    kind, a, b, i = _kind(c, name), c["src_tp"], c["dst_tp"], c["at_tp"]
    if kind == "repl":
        return next(iter(shards.values()))
    if kind == "vocab":
        v, per = c["vocab"], -(-c["vocab"] // (128 * b)) * 128
        held = -(-v // (128 * a)) * 128
        out = next(iter(shards.values())).new_zeros(per, c["hidden"])
        for k, t in shards.items():
            lo, hi = max(k * held, i * per), min(k * held + held, i * per + per, v)
            if lo < hi:
                out[lo - i * per:hi - i * per] = t[lo - k * held:hi - k * held]
        return out
    dim = -1 if kind == "row" else 0
    if b >= a:
        n = b // a
        t = shards[i // n]
        if kind == "qkv":
            return torch.cat([p.chunk(n, 0)[i % n] for p in _projections(c, t, a)], 0)
        return t.chunk(n, dim)[i % n].contiguous()
    n = a // b
    parts = [shards[i * n + k] for k in range(n)]
    if kind == "qkv":
        return torch.cat([torch.cat(p, 0) for p in zip(*(_projections(c, t, a) for t in parts))], 0)
    return torch.cat(parts, dim)


def exact(c, seed):
    src, _, _, tpl, rank = _sources(c, seed)
    names = list(tpl.layout[rank])
    state = {}
    for n in names:
        state[n] = {}
        shards = {f: {r % c["src_tp"]: e[n][f] for r, e in src.items() if n in e} for f in FIELDS[c["fields"]]}
        if c["entry"] == "send" and _kind(c, n) == "repl":
            continue
        for f in _outputs_of(c):
            held = "master" if f == "param" and c["fields"] == "recast" else f
            state[n][f] = _expected(c, n, shards[held])   # a rounded field: the value before the rounding
    if c["entry"] == "send":
        return {n: e["param"] for n, e in state.items() if e}
    kept = c["entry"] in ("reshard", "exchange", "noalloc")
    if not kept and not _flat(c, names):
        return state
    out = {}
    for f, dt in _outputs_of(c).items():
        parts = []
        for k, n in enumerate(names):
            t = state[n][f].reshape(-1)
            parts.append(t)
            if kept:   # the kept destinations' places
                parts.append(t.new_zeros(-t.numel() % (ALIGN // dt.itemsize)))
        out[f] = torch.cat(parts)
    return out


# ------------------------------------------------------------------ more of the same

def _log_uniform(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    while True:
        entry = rng.choice(["send", "migrate", "call", "adopt", "resume", "reshard", "reshard", "refresh", "exchange",
                            "exchange", "noalloc"])
        a, b = rng.choice([(1, 2), (2, 1), (2, 4), (4, 2), (8, 4), (4, 8), (1, 4), (8, 1)])
        if entry == "send" and a >= b:   # a shard as fine as the piece is sent as it is
            continue
        t = max(a, b)
        family = rng.choice(["gpt", "llama", "qwen"])
        hd = rng.choice([4, 25, 32, 64, 80, 96, 100, 127, 128])
        most = 4096 if entry in ("reshard", "exchange") else 2048
        heads = t * max(1, _log_uniform(rng, 16, most) // (t * hd))
        kv = rng.choice([0, t]) if family != "gpt" else 0
        hidden = heads * hd
        ffn = t * max(1, int(hidden * rng.choice([2.5, 8 / 3, 4]) / t) + rng.choice([0, 0, 1, 3]))
        fields = "f32x3" if entry == "send" else rng.choice(["f32x3", "mixed", "recast"])
        # a padded vocabulary keeps rows on every rank
        vocab = t * (128 * t + _log_uniform(rng, 16, 4096))
        layers = 1 if entry in ("send", "migrate", "call", "adopt", "resume", "refresh") else _log_uniform(rng, 1, 16)
        pp = rng.choice([1, 1, 2]) if layers > 1 else 1
        embeddings = entry != "send" and rng.random() < 0.7
        c = _case(None, entry, family, fields, (a, 1), (b, pp), at=(rng.randrange(pp), rng.randrange(b)),
                  layers=layers, hidden=hidden, heads=heads, kv_heads=kv, head_dim=hd, ffn=ffn, vocab=vocab,
                  fused_qkv=family != "gpt" and rng.random() < 0.5, vocab_parallel=rng.random() < 0.5,
                  positions=128 if family == "gpt" and rng.random() < 0.3 else 0, embeddings=embeddings)
        _, tpl, rank = _layouts(c)
        if entry in ("migrate", "call", "adopt", "resume", "refresh") and _flat(c, tpl.layout[rank]):
            continue
        # bytes of the pass, and of the source shards that it reads parts of
        moved = work(c)["bytes"]
        if moved * max(1, b // a) <= ((1 << 30) if entry == "resume" else (8 << 30)):
            return c
