"""What this framework is timed on: the work of a speculative-decoding verify loop, through the package's public
entry points, from one small recurrence to a stack of layers at a 32K context.

A case is a dict of plain values; ``op`` says which part of the loop it is:

  replay    DFlashKernels.tape_replay_kernel: one recurrent cache rolled back to the accepted prefix
  forward   DFlashKernels.gated_delta_kernel_with_tape: one GatedDelta layer's recurrence (a draft block, or a
            longer stretch of a prompt)
  layer     DFlashKernels.gdn_layer: the layer's body between its projections in one call
  attn      DFlashKernels.batched_sdpa_2pass / _append / _paged: the block's attention over the cached keys
  cycle     one eager verify cycle of a host program: arm the caches, run the recurrences, record the tapes, take
            the greedy tokens, count the accepted ones, roll every cache back
  step      HybridVerifyStack: whole verify steps, captured once in a HIP graph and replayed (or enqueued eagerly)
"""

import torch

from swiftlm_amd import DFlashKernels, DFlashRuntime, HybridGDNEngine, KVCacheSimple, RecurrentRollbackCache
from swiftlm_amd.verify_step import HybridVerifyStack, StackConfig

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
BYTES = {"bf16": 2, "f16": 2, "f32": 4}
BLOCK = 16          # tokens of a verify block
CONV = 4            # taps of the layers' short convolution


def _forward(**kw):
    return dict(dict(op="forward", B=1, T=16, Hk=16, Hv=32, Dk=128, Dv=128, dtype="bf16", state="f32", channel_gate=False,
                     masked=False), **kw)


def _attn(**kw):
    return dict(dict(op="attn", B=1, Hq=16, Hk=2, D=256, N=4112, dtype="bf16", ragged=False, masked=False, kind="plain",
                     page=0, lse=True, own_workspace=True), **kw)


def _step(**kw):
    return dict(dict(op="step", layers=16, context=32768, steps=4, page=0, graph=True), **kw)


def listed():
    return [
        # the smallest call: a rejected block of eight tokens rolled back in one small layer
        dict(name="replay_small", op="replay", B=1, T=8, Hk=4, Hv=8, Dk=64, Dv=64, dtype="f32", state="f32",
             channel_gate=False, masked=False),
        # one linear-attention layer of a large hybrid model scoring a 16-token draft
        _forward(name="forward_block"),
        # four sequences whose drafts have different lengths (step mask), one decay per channel, state kept in bf16
        _forward(name="forward_channel_gate", B=4, T=13, Hk=8, Hv=16, state="bf16", channel_gate=True, masked=True),
        # a stretch of prompt run through the recurrence, its length no multiple of anything
        _forward(name="forward_prompt", T=1003),
        # the whole layer body of two sequences between the input and the output projection
        dict(name="layer_block", op="layer", B=2, T=16, Hk=16, Hv=32, Dk=128, Dv=128, dtype="bf16", carry=True, gate="silu"),
        # attention early in a conversation, called the simplest way (no workspace kept, no logsumexp)
        _attn(name="attn_short", Hq=32, Hk=8, D=128, N=512, lse=False, own_workspace=False),
        # attention over a context of four thousand tokens
        _attn(name="attn_4k"),
        # attention over a very long context
        _attn(name="attn_100k", N=102416),
        # four sequences of unequal length, 8K to 64K, in one call
        _attn(name="attn_ragged_batch", B=4, N=65552, ragged=True),
        # eight sequences over paged f16 caches, the block's rows appended by the same call
        _attn(name="attn_paged_append", B=8, Hq=32, Hk=8, D=128, N=3000, dtype="f16", ragged=True, kind="paged_append", page=64),
        # an eager host program: six recurrent and two attention caches, 151936-token vocabulary
        dict(name="cycle_eager", op="cycle", layers=6, attn=2, Hk=16, Hv=32, Dk=128, Dv=128, dtype="bf16", vocab=151936),
        # a hybrid stack, three recurrent layers to one of attention, four steps at a 32K context in one graph
        _step(name="step_32k"),
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    op = rng.choice(["replay", "forward", "forward", "forward_long", "layer", "attn", "attn", "attn", "cycle", "step", "step"])
    Hk = rng.choice([2, 4, 8, 16])
    heads = dict(Hk=Hk, Hv=Hk * rng.choice([1, 2, 2]), Dk=rng.choice([64, 128, 128, 256]), Dv=rng.choice([64, 128, 128]))
    if op in ("replay", "forward"):
        dtype = rng.choice(["bf16", "bf16", "f16", "f32"])
        return dict(op=op, B=rng.choice([1, 1, 2, 4]), T=rng.randint(1, BLOCK), dtype=dtype, state=rng.choice(["f32", "f32", dtype]),
                    channel_gate=rng.random() < 0.3, masked=rng.random() < 0.3, **heads)
    if op == "forward_long":
        return dict(op="forward", B=rng.choice([1, 1, 2]), T=_log(rng, 17, 1024), dtype="bf16", state="f32",
                    channel_gate=rng.random() < 0.25, masked=False, **heads)
    if op == "layer":
        return dict(op="layer", B=rng.choice([1, 1, 2, 4]), T=rng.randint(1, BLOCK), dtype=rng.choice(["bf16", "bf16", "f16"]),
                    carry=rng.random() < 0.8, gate=rng.choice(["silu", "sigmoid"]), **heads)
    if op == "attn":
        D = rng.choice([128, 256])
        Hk = rng.choice([1, 2, 4, 8])
        B = rng.choice([1, 1, 1, 2, 4, 8])
        kind = rng.choice(["plain", "plain", "append", "paged", "paged_append"])
        masked = kind == "plain" and rng.random() < 0.25
        most = min(102416, 400_000_000 // (B * Hk * D * 4))
        N = _log(rng, 24, min(most, 16384) if masked else most)
        return dict(op="attn", B=B, Hq=Hk * rng.choice([1, 4, 6, 8]), Hk=Hk, D=D, N=N, dtype=rng.choice(["bf16", "bf16", "f16"]),
                    ragged=B > 1 and rng.random() < 0.6, masked=masked, kind=kind,
                    page=rng.choice([32, 64, 256]) if kind.startswith("paged") else 0, lse=rng.random() < 0.5,
                    own_workspace=rng.random() < 0.5)
    if op == "cycle":
        return dict(op="cycle", layers=rng.randint(1, 12), attn=rng.randint(0, 4), dtype=rng.choice(["bf16", "bf16", "f16"]),
                    vocab=_log(rng, 32000, 152000), **heads)
    return dict(op="step", layers=4 * rng.randint(1, 4), context=_log(rng, 300, 32768), steps=rng.choice([2, 4]),
                page=rng.choice([0, 0, 0, 64]), graph=rng.random() < 0.7)


# ---- inputs ------------------------------------------------------------------------------------------------------

def _source(seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    return lambda *shape: torch.randn(*shape, generator=gen, device="cuda")


def _unit(x):
    return torch.nn.functional.normalize(x, dim=-1)


def _recurrence(c, randn, T):
    """What a model's projections hand to the recurrence: normalised q and k, decays below one, betas in (0, 1)."""
    dt, B, Hk, Hv, Dk, Dv = DTYPES[c["dtype"]], c.get("B", 1), c["Hk"], c["Hv"], c["Dk"], c["Dv"]
    gate = (B, T, Hv, Dk) if c.get("channel_gate") else (B, T, Hv)
    return dict(q=_unit(randn(B, T, Hk, Dk)).to(dt), k=_unit(randn(B, T, Hk, Dk)).to(dt), v=randn(B, T, Hv, Dv).to(dt),
                g=torch.exp(-torch.nn.functional.softplus(randn(*gate))).to(dt), beta=torch.sigmoid(randn(B, T, Hv)).to(dt),
                state=(0.1 * randn(B, Hv, Dv, Dk)).to(DTYPES[c.get("state", "f32")]))


def _step_mask(c, randn):
    if not c["masked"]:
        return None
    # drafts of different lengths padded to T: a prefix of each sequence's steps runs
    lens = (randn(c["B"]).abs() * c["T"] / 2).long().clamp(max=c["T"] - 1) + 1
    return (torch.arange(c["T"], device="cuda")[None] < lens[:, None]).to(torch.uint8)


def _commit_counts(seed, n):
    """Committed tokens per block: geometric with p = 1/4, clipped to the block."""
    u = torch.rand(n, generator=torch.Generator().manual_seed(seed), dtype=torch.float64)
    return (torch.log1p(-u) / torch.log(torch.tensor(0.75, dtype=torch.float64))).floor().long().clamp(max=BLOCK - 1) + 1


def _token_ids(seed, commits, vocab):
    """[step, ids | posterior, BLOCK]: the posterior agrees with the draft up to the committed prefix."""
    gen = torch.Generator().manual_seed(seed)
    ids = torch.randint(0, vocab - 2, (len(commits), BLOCK), generator=gen, dtype=torch.int32)
    post = torch.cat([ids[:, 1:], torch.full((len(commits), 1), 7, dtype=torch.int32)], dim=1)
    for s, n in enumerate(commits.tolist()):
        if n < BLOCK:
            post[s, n - 1] = ids[s, n] + 1
    return torch.stack([ids, post], dim=1)


def prepare(case, seed):
    c, randn = case, _source(seed)
    if c["op"] in ("replay", "forward"):
        s = _recurrence(c, randn, c["T"])
        s["mask"] = _step_mask(c, randn)
        if c["op"] == "replay":
            s["tape"] = randn(c["B"], c["T"], c["Hv"], c["Dv"])
    elif c["op"] == "layer":
        dt, B, T, Hv = DTYPES[c["dtype"]], c["B"], c["T"], c["Hv"]
        C = 2 * c["Hk"] * c["Dk"] + Hv * c["Dv"]
        s = dict(mixed_qkv=randn(B, T, C).to(dt), conv_state=randn(B, CONV - 1, C).to(dt) if c["carry"] else None,
                 conv_weight=(0.5 * randn(C, CONV)).to(dt), a_logits=randn(B, T, Hv).to(dt), b_logits=randn(B, T, Hv).to(dt),
                 a_log=0.5 * randn(Hv), dt_bias=randn(Hv), state=0.1 * randn(B, Hv, c["Dv"], c["Dk"]),
                 Hk=c["Hk"], Hv=Hv, Dk=c["Dk"], Dv=c["Dv"], q_scale=1.0 / c["Dk"], k_scale=c["Dk"] ** -0.5,
                 gate=randn(B, T, Hv, c["Dv"]).to(dt), norm_weight=(1 + 0.1 * randn(c["Dv"])).to(dt), gate_kind=c["gate"])
    elif c["op"] == "attn":
        s = _prepare_attention(c, randn, seed)
    elif c["op"] == "cycle":
        s = _prepare_cycle(c, randn, seed)
    else:
        s = _prepare_step(c, seed)
    s["case"] = c
    return s


def _prepare_attention(c, randn, seed):
    dt, B, Hq, Hk, D, N = DTYPES[c["dtype"]], c["B"], c["Hq"], c["Hk"], c["D"], c["N"]
    append = c["kind"].endswith("append")
    s = dict(q=randn(B, Hq, BLOCK, D).to(dt), scale=D ** -0.5, lengths=None, mask=None, k_new=None, v_new=None)
    if append:
        s["k_new"], s["v_new"] = randn(B, Hk, BLOCK, D).to(dt), randn(B, Hk, BLOCK, D).to(dt)
    if c["ragged"] or append:
        # key counts from an eighth of the bound up, the longest at the bound; an append counts the rows cached before it
        gen = torch.Generator().manual_seed(seed)
        lens = N - ((N - BLOCK) * 7 // 8 * torch.rand(B, generator=gen, dtype=torch.float64)).long() if c["ragged"] else torch.full((B,), N)
        lens[0] = N
        s["lengths"] = (lens - (BLOCK if append else 0)).to(torch.int32).cuda()
    if c["masked"]:
        drop = randn(B, 1, 1, N) > 1.5                      # keys that an application hides, on top of a small bias
        drop[..., 0] = False
        s["mask"] = (0.1 * randn(B, Hq, BLOCK, N)).masked_fill(drop, float("-inf")).to(dt)
    if c["page"]:
        P = c["page"]
        pages = -(-N // P)
        order = torch.randperm(B * pages, generator=torch.Generator().manual_seed(seed))
        s["page_table"] = order.view(B, pages).to(torch.int32).cuda()
        shape = (B * pages, Hk, P, D)
    else:
        shape = (B, Hk, N, D)
    s["k"], s["v"] = randn(*shape).to(dt), randn(*shape).to(dt)
    s["workspace"] = None
    if c["own_workspace"]:
        s["workspace"] = torch.empty(DFlashKernels.sdpa_workspace_bytes(B, Hq, Hk, BLOCK, N, D), dtype=torch.uint8, device="cuda")
    return s


def _prepare_cycle(c, randn, seed):
    dt, V = DTYPES[c["dtype"]], c["vocab"]
    C = 2 * c["Hk"] * c["Dk"] + c["Hv"] * c["Dv"]
    layers, caches = [], []
    for _ in range(c["layers"]):
        layer = _recurrence(c, randn, BLOCK)
        layer["qkv"] = randn(1, BLOCK, C).to(dt)
        cache = RecurrentRollbackCache()
        cache[0], cache[1] = randn(1, CONV - 1, C).to(dt), layer.pop("state")
        layers.append(layer)
        caches.append(cache)
    ids, post = _token_ids(seed, _commit_counts(seed, 1), V)[0]
    logits = randn(BLOCK, V)
    logits[torch.arange(BLOCK), post.long()] = 12.0
    suppress = DFlashRuntime.build_suppress_token_mask(V, [V - 1, V - 2])
    return dict(layers=layers, caches=caches, kv=[KVCacheSimple() for _ in range(c["attn"])], logits=logits.to(dt), suppress=suppress,
                ids=ids.cuda(), engine=HybridGDNEngine())


def _prepare_step(c, seed):
    stack = HybridVerifyStack(StackConfig(n_layers=c["layers"], context=c["context"], max_steps=c["steps"], page_size=c["page"]),
                              seed=seed, n_slots=c["steps"])
    s = dict(stack=stack, tokens=_token_ids(seed, _commit_counts(seed, c["steps"]), 1000).cuda(), offset=stack.offset.clone(), graph=None)
    if c["graph"]:
        for i in range(2):                                  # code objects are loaded before the capture
            stack.enqueue_step(slot=i)
        torch.cuda.synchronize()
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        s["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["graph"], stream=side):
            for i in range(c["steps"]):
                stack.enqueue_step(slot=i)
        torch.cuda.current_stream().wait_stream(side)
    return s


# ---- one pass ----------------------------------------------------------------------------------------------------

def run(s):
    c = s["case"]
    if c["op"] == "replay":
        return DFlashKernels.tape_replay_kernel(s["tape"], s["k"], s["g"], s["state"], s["mask"])
    if c["op"] == "forward":
        return DFlashKernels.gated_delta_kernel_with_tape(s["q"], s["k"], s["v"], s["g"], s["beta"], s["state"], s["mask"])
    if c["op"] == "layer":
        return DFlashKernels.gdn_layer(**{k: v for k, v in s.items() if k != "case"})
    if c["op"] == "attn":
        return _run_attention(c, s)
    if c["op"] == "cycle":
        return _run_cycle(s)
    return _run_step(c, s)


def _run_attention(c, s):
    opts = dict(return_lse=c["lse"], workspace=s["workspace"])
    if c["kind"] == "plain":
        return DFlashKernels.batched_sdpa_2pass(s["q"], s["k"], s["v"], s["scale"], s["mask"], kv_len=s["lengths"], **opts)
    if c["kind"] == "append":
        out = DFlashKernels.batched_sdpa_2pass_append(s["q"], s["k"], s["v"], s["k_new"], s["v_new"], s["scale"], c["N"],
                                                      cache_len=s["lengths"], **opts)
    else:
        out = DFlashKernels.batched_sdpa_2pass_paged(s["q"], s["k"], s["v"], s["page_table"], s["scale"], c["N"], k_new=s["k_new"],
                                                     v_new=s["v_new"], lengths=s["lengths"], **opts)
        if c["kind"] == "paged":
            return out
    return out, s["k"], s["v"]


def _run_cycle(s):
    start, engine, caches = 1000, s["engine"], s["caches"]
    every = caches + s["kv"]
    engine.arm_rollback(every, start)
    kept = []
    for layer, cache in zip(s["layers"], caches):
        y, state, tape = DFlashKernels.gated_delta_kernel_with_tape(layer["q"], layer["k"], layer["v"], layer["g"], layer["beta"], cache[1])
        cache[1], cache[0] = state, layer["qkv"][:, 1 - CONV:].clone()
        cache.record_tape(tape, layer["k"], layer["g"], layer["qkv"])
        kept.append(y)
    for kv in s["kv"]:
        kv.offset = start + BLOCK
    accept, posterior = DFlashRuntime.greedy_accept_commit(s["logits"], s["suppress"], s["ids"], start)
    engine.rollback(every, accept.start, accept.acceptance_len, BLOCK - 1)
    return dict(y=kept, state=[x[1] for x in caches], conv=[x[0] for x in caches], posterior=posterior,
                accept=[accept.acceptance_len, accept.commit_count, accept.staged_first_next, accept.start],
                offsets=[x.offset for x in s["kv"]])


def _run_step(c, s):
    stack = s["stack"]
    # the drafter's tokens and the cache length of the blocks at hand
    stack.accept_inputs.copy_(s["tokens"], non_blocking=True)
    stack.offset.copy_(s["offset"], non_blocking=True)
    if s["graph"] is not None:
        s["graph"].replay()
    else:
        for i in range(c["steps"]):
            stack.enqueue_step(slot=i)
    return dict(gdn=[(x["state"][stack.phase], x["y"], x["tape"]) for x in stack.gdn], attn=[(x["out"], x["lse"]) for x in stack.attn],
                cache=[(x["k_pool"], x["v_pool"]) if c["page"] else (x["k_cache"], x["v_cache"]) for x in stack.attn],
                accept=stack.accept, offset=stack.offset)


# ---- what a pass cannot do without ---------------------------------------------------------------------------------

def _recurrence_work(c, B, T, forward):
    Hk, Hv, Dk, Dv, e = c["Hk"], c["Hv"], c["Dk"], c["Dv"], BYTES[c["dtype"]]
    gate = Hv * (Dk if c.get("channel_gate") else 1) * e
    per_step = Hk * Dk * e + gate + 4 * Hv * Dv                         # k, g, tape
    if forward:
        per_step += Hk * Dk * e + 2 * Hv * Dv * e + Hv * e              # q, v, y, beta
    state = 2 * B * Hv * Dv * Dk * BYTES[c.get("state", "f32")]
    return state + B * T * per_step, (7 if forward else 3) * B * T * Hv * Dv * Dk


def _attention_work(B, Hq, Hk, D, keys, e, lse, append):
    """keys: key count summed over the batch."""
    nbytes = 2 * B * Hq * BLOCK * D * e + 2 * Hk * keys * D * e + (4 * B * Hq * BLOCK if lse else 0)
    return nbytes + (2 * B * Hk * BLOCK * D * e if append else 0), 4 * Hq * BLOCK * keys * D


def work(case):
    c = case
    if c["op"] in ("replay", "forward"):
        b, f = _recurrence_work(c, c["B"], c["T"], c["op"] == "forward")
    elif c["op"] == "layer":
        e, B, T = BYTES[c["dtype"]], c["B"], c["T"]
        C = 2 * c["Hk"] * c["Dk"] + c["Hv"] * c["Dv"]
        rows = c["Hv"] * c["Dv"]
        b = (2 * 4 * B * rows * c["Dk"] + e * (B * T * C + (2 if c["carry"] else 1) * B * (CONV - 1) * C + C * CONV)
             + e * B * T * (3 * c["Hv"] + c["Hk"] * c["Dk"]) + B * T * rows * (3 * e + 4))
        f = 7 * B * T * rows * c["Dk"] + 2 * CONV * B * T * C
    elif c["op"] == "attn":
        keys = c["B"] * c["N"]
        if c["ragged"]:
            keys = c["N"] + int((c["B"] - 1) * (c["N"] - (c["N"] - BLOCK) * 7 / 16))       # the mean of the drawn lengths
        b, f = _attention_work(c["B"], c["Hq"], c["Hk"], c["D"], keys, 2, c["lse"], c["kind"].endswith("append"))
        if c["masked"]:
            b += 2 * c["Hq"] * BLOCK * keys
    elif c["op"] == "cycle":
        fb, ff = _recurrence_work(c, 1, BLOCK, True)
        rb, rf = _recurrence_work(c, 1, 4, False)
        C = 2 * c["Hk"] * c["Dk"] + c["Hv"] * c["Dv"]
        e = BYTES[c["dtype"]]
        b = c["layers"] * (fb + rb + 2 * e * (CONV - 1) * C) + BLOCK * c["vocab"] * e + c["vocab"]
        f = c["layers"] * (ff + rf)
    else:
        k = StackConfig(n_layers=c["layers"])
        r = dict(Hk=k.Hk, Hv=k.Hv, Dk=k.Dk, Dv=k.Dv, dtype="bf16")
        fb, ff = _recurrence_work(r, 1, BLOCK, True)
        rb, rf = _recurrence_work(r, 1, 4, False)
        ab, af = _attention_work(1, k.Hq, k.Hkv, k.D, c["context"] + 2 * c["steps"] + BLOCK, 2, True, True)
        n_attn = c["layers"] // k.attn_every
        n_gdn = c["layers"] - n_attn
        b = c["steps"] * (n_gdn * (fb + rb) + n_attn * ab)
        f = c["steps"] * (n_gdn * (ff + rf) + n_attn * af)
    return {"bytes": b, "flops": f}


def tolerance(case):
    """32-bit sums differ in their order only; 16-bit outputs by their rounding (attention also rounds its weights
    and partial rows); a 16-bit state is rounded after every step."""
    c = case
    if c["op"] == "attn":
        return {"rel": 1e-2 if c["dtype"] == "bf16" else 2e-3}
    if c["op"] == "step":
        return {"rel": 1e-2}
    if c.get("state", "f32") != "f32":
        return {"rel": 1e-2 if c["dtype"] == "bf16" else 2e-3}
    if c["op"] == "replay":
        return {"rel": 1e-5}
    return {"rel": {"bf16": 5e-3, "f16": 1e-3, "f32": 2e-5}[c["dtype"]]}
