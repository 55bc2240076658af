"""Performance cases of the RecoverSSM path: what a serving program has it do.

A case is one decode step of a stack of Gated DeltaNet layers, or the part of
it that one entry point covers, on inputs with the distributions of the
benchmark's workloads:

* flow ``step``: the verify of every layer (``gdn_recoverssm_verify``), then
  the commit of the accepted prefixes over all of them, conv states included,
  through one commit context or (``commit: grouped``) the coordinator with the
  layers in four cache groups;
* flow ``gated``: the verify with the gating and the q/k L2 norm fused in
  (``gdn_recoverssm_verify_gated``) of every layer;
* flow ``deferred``: the verify of every layer that applies the previous
  step's pending commit (``gdn_recoverssm_verify_deferred``), then the plan and
  conv compaction of this step (``commit_deferred``).

With ``graph`` the verifies of a step are captured in a HIP graph, as a serving
engine runs its decode step; the commit runs after sampling and is called
eagerly. Sizes are those of the benchmark workloads (48 layers of Hk=16, Hv=32,
Dk=Dv=128, Q=4), of one tensor-parallel rank of eight (Hk=2, Hv=4), of the
record geometry Hk=4, Hv=12, and of the tests' other head dims.
"""

import math
import os
import sys
from types import SimpleNamespace

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gdn-recoverssm-ascend_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

_DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
_BLOCK = 64            # tokens per cache block in align mode
_MAX_POSITION = 8192   # positions are uniform in [0, 8192)
_CROSSING = 0.25       # share of the rows whose window crosses a block boundary
_CONV_HISTORY = 3      # conv kernel 4
_GROUPS = 4            # cache groups of a grouped commit


def _case(name=None, **kw):
    c = dict(flow="step", layers=1, rows=64, H=16, HV=32, K=128, V=128, Q=4, state="f32", act="bf16", align=True,
             accept="uniform", ragged=False, padded=0, commit="single", graph=True)
    unknown = set(kw) - set(c)
    assert not unknown, unknown
    c.update(kw)
    return dict(c, name=name) if name else c


def listed():
    return [
        # One layer of a toy model called eagerly: the latency of the two host
        # calls and of kernels with 16 (row, head) tiles.
        _case("plumbing_b4", rows=4, H=2, HV=4, K=64, V=64, align=False, graph=False),
        # A single user: 48 layers with one row each.
        _case("single_user_l48", layers=48, rows=1, accept="live"),
        # One tensor-parallel rank of eight with a few requests, windows of
        # unequal length.
        _case("tp8_rank_b6_l48", layers=48, rows=6, H=2, HV=4, ragged=True),
        # A small serving batch.
        _case("small_batch_b16_l24", layers=24, rows=16, align=False),
        # A medium batch committed by the coordinator over four cache groups.
        _case("grouped_b64_l12", layers=12, rows=64, commit="grouped", padded=1),
        # The headline step: one layer, B=256, prefix-cache align mode.
        _case("align_b256", rows=256, padded=6),
        # Plain decode through the same kernels: Q=1, every token accepted.
        _case("decode_q1_b256", rows=256, Q=1, align=False, accept="all"),
        # The longest window with skewed acceptance.
        _case("skewed_q8_b256", rows=256, Q=8, align=False, accept="geometric"),
        # The fused producers (gating, q/k L2 norm) on a ragged batch.
        _case("gated_b37_l16", flow="gated", layers=16, rows=37, ragged=True),
        # The decode loop's layers with the deferred commit.
        _case("deferred_b128_l8", flow="deferred", layers=8, rows=128, padded=2),
        # Head dims off the 128 x 128 tile, FP16 activations and pages, an odd
        # ragged batch with a grouped-query ratio of three.
        _case("ragged_f16_b29_l12", layers=12, rows=29, H=4, HV=12, K=96, V=192, state="f16", act="f16", ragged=True,
              padded=1),
        # BF16 checkpoint pages.
        _case("bf16_pages_b96_l8", layers=8, rows=96, state="bf16", align=False),
    ]


def _row_elements(c):
    return c["HV"] * c["V"] * c["K"]


_LARGEST = 8 * 128 * 32 * 128 * 128  # state elements of the largest listed case


def draw(rng):
    """One more case of the same ranges."""
    H, HV = rng.choice([(2, 4), (4, 8), (4, 12), (8, 16), (16, 32), (16, 32)])
    K, V = rng.choice([(128, 128)] * 5 + [(64, 64), (128, 96), (64, 192), (256, 128)])
    rows = max(1, min(256, int(round(math.exp(rng.uniform(0.0, math.log(256.0)))))))
    flow = rng.choice(["step"] * 5 + ["gated", "gated", "deferred", "deferred", "deferred"])
    state = rng.choice(["f32"] * 7 + ["bf16", "bf16", "f16"])
    most = max(1, min(48, _LARGEST // (rows * HV * V * K)))
    layers = min(most, rng.choice([8, 12, 24, 48]))
    return _case(
        flow=flow, layers=layers, rows=rows, H=H, HV=HV, K=K, V=V,
        Q=rng.choice([4, 4, 4, 4, 1, 2, 3, 5, 6, 8]), state=state, act="f16" if state == "f16" else "bf16",
        align=rng.random() < 0.6, accept=rng.choice(["uniform", "uniform", "geometric", "live", "all"]),
        ragged=rng.random() < 0.35, padded=rng.choice([0, 0, 1, 2]) if rows > 4 else 0,
        commit="grouped" if flow == "step" and layers % _GROUPS == 0 and rng.random() < 0.4 else "single",
        graph=layers > 1)


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------


def _accepted(c, gen):
    """Accepted lengths with the same counts for every seed, in a random order."""
    B, Q = c["rows"], c["Q"]
    place = torch.randperm(B, generator=gen)
    if c["accept"] == "all":
        return torch.full((B,), Q, dtype=torch.int64)
    if c["accept"] == "live":
        return 1 + (place + (Q - 1) // 2) % Q
    if c["accept"] == "geometric":
        u = (place.double() + 0.5) / B
        return torch.floor(torch.log(u) / math.log(0.7)).clamp(max=Q).long()
    return (place + (Q + 1) // 2) % (Q + 1)


def _next_pages(c, qlens, accepted, C, table, src, valid):
    """The commit's plan (count, final page, boundary page and length)."""
    n = torch.where(valid, torch.minimum(accepted, qlens), torch.zeros_like(qlens))
    zero = torch.zeros_like(n)
    if not c["align"]:
        return n, torch.where(n > 0, src, zero), zero, zero
    rows = torch.arange(c["rows"])
    final = table[rows, (C + n - 1).clamp(min=0) // _BLOCK]
    boundary = (C // _BLOCK + 1) * _BLOCK
    crosses = (n > 0) & (C + n >= boundary)
    page = table[rows, boundary // _BLOCK - 1]
    return (n, torch.where(n > 0, final, zero), torch.where(crosses, page, zero),
            torch.where(crosses, boundary - C, zero))


def _meta(c, seed):
    """The scheduler's view of the batch, on the host: page tables, positions,
    windows, accepted lengths, and the plan that follows from them; one entry
    per step (the deferred flow has the pending step and the current one)."""
    gen = torch.Generator().manual_seed(int(seed))
    B, Q, steps = c["rows"], c["Q"], 2 if c["flow"] == "deferred" else 1
    qlens = torch.full((B,), Q, dtype=torch.int64)
    if c["ragged"]:
        qlens = 1 + torch.randperm(B, generator=gen) % Q
    accepted = [_accepted(c, gen) for _ in range(steps)]
    C = torch.randint(0, _MAX_POSITION, (B,), generator=gen)
    per_row = 1 + steps if c["align"] else 2
    table = None
    if c["align"]:
        n = torch.minimum(accepted[0], qlens)
        place = torch.randperm(B, generator=gen)
        ahead = 1 + (torch.rand(B, generator=gen) * n).long().clamp(max=Q)
        moved = (n > 0) & (place < max(1, round(_CROSSING * B / max(float((n > 0).float().mean()), 0.1))))
        moved &= place < B
        C = torch.where(moved, (C // _BLOCK).clamp(min=1) * _BLOCK - torch.minimum(ahead, n.clamp(min=1)), C)
        first = (C - 1).clamp(min=0) // _BLOCK
        table = torch.zeros(B, _MAX_POSITION // _BLOCK + 2 + steps, dtype=torch.int64)
        for j in range(per_row):
            table[torch.arange(B), first + j] = 1 + per_row * torch.arange(B) + j
        src = table[torch.arange(B), first]
    else:
        src = 1 + torch.randperm(per_row * B, generator=gen)[:B]
    pages = 1 + per_row * B
    pad = torch.randperm(B, generator=gen)[:c["padded"]]
    src[pad] = -1
    qsl = torch.zeros(B + 1, dtype=torch.int64)
    qsl[1:] = torch.cumsum(qlens, 0)
    out = []
    for i in range(steps):
        valid = src > 0
        n, final, boundary, blen = _next_pages(c, qlens, accepted[i], C, table, src, valid)
        out.append(SimpleNamespace(qlens=qlens, qsl=qsl, accepted=accepted[i], C=C, table=table, src=src, valid=valid,
                                   n=n, final=final, boundary=boundary, blen=blen, pages=pages))
        src, C = torch.where(n > 0, final, src), C + n
    return out


def _unit(x):
    return x * torch.rsqrt((x * x).sum(-1, keepdim=True) + 1e-6)


def _tensors(c, seed, tokens, pages):
    """Activations of every step and layer, pages and conv states, on the GPU."""
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(int(seed) + 1)
    act, L, H, HV, K, V = _DTYPES[c["act"]], c["layers"], c["H"], c["HV"], c["K"], c["V"]

    def randn(*shape):
        return torch.randn(*shape, generator=gen, device=dev)

    steps = []
    for _ in range(2 if c["flow"] == "deferred" else 1):
        x = SimpleNamespace(q=randn(L, 1, tokens, H, K), k=randn(L, 1, tokens, H, K))
        if c["flow"] == "gated":
            x.q, x.k = x.q.to(act), x.k.to(act)
            x.g, x.beta = randn(L, tokens, HV).to(act), randn(L, tokens, HV).to(act)
            x.A_log = torch.log(0.05 + 4.0 * torch.rand(L, HV, generator=gen, device=dev))
            x.dt_bias = randn(L, HV)
        else:
            x.q, x.k = _unit(x.q).to(act), _unit(x.k).to(act)
            x.g = -torch.nn.functional.softplus(randn(L, tokens, HV))
            x.beta = torch.sigmoid(randn(L, tokens, HV))
        x.v = randn(L, 1, tokens, HV, V).to(act)
        steps.append(x)
    state = torch.empty(L, pages, HV, V, K, dtype=_DTYPES[c["state"]], device=dev)
    conv = torch.empty(L, pages, 2 * H * K + HV * V, _CONV_HISTORY + c["Q"] - 1, dtype=act, device=dev)
    for layer in range(L):
        state[layer] = randn(pages, HV, V, K) * 0.1
        conv[layer] = randn(*conv.shape[1:])
    return steps, state, conv


# ---------------------------------------------------------------------------
# The path
# ---------------------------------------------------------------------------


def _records(c, key_dtype):
    """One record set per layer (views of three stacked planes) and the planes."""
    from gdn_recoverssm_ascend import ReplayRecordBuffers

    L, B, H, HV, K, V, Q = (c[x] for x in ("layers", "rows", "H", "HV", "K", "V", "Q"))
    dev = torch.device("cuda")
    planes = (torch.zeros(L, B, HV, Q, V, device=dev), torch.zeros(L, B, H, Q, K, dtype=key_dtype, device=dev),
              torch.zeros(L, B, HV, Q, device=dev))
    return [ReplayRecordBuffers(*(p[i] for p in planes)) for i in range(L)], planes


def _commit_inputs(m, align):
    """One step's commit metadata on the GPU, as the engine holds it."""
    dev = torch.device("cuda")

    def i32(t):
        return t.to(torch.int32).to(dev)

    s = SimpleNamespace(accepted=i32(m.accepted), qsl=i32(m.qsl), src=i32(m.src), align={})
    if align:
        s.align = dict(block_table=i32(m.table), num_computed_tokens=i32(m.C), mamba_block_size=_BLOCK)
    return s


def _verify_calls(c, x, meta, state, records, outs, pending=None):
    """One function that runs the verify of every layer, in layer order."""
    import gdn_recoverssm_ascend as G

    def call():
        for i in range(c["layers"]):
            kw = dict(checkpoint_state=state[i], replay_cache=records[i], query_start_loc=meta.qsl,
                      state_indices=meta.src, spec_query_len=c["Q"], out=outs[i])
            if c["flow"] == "gated":
                G.gdn_recoverssm_verify_gated(x.g[i], x.beta[i], x.q[i], x.k[i], x.v[i], A_log=x.A_log[i],
                                              dt_bias=x.dt_bias[i], **kw)
            elif pending is not None:
                G.gdn_recoverssm_verify_deferred(x.g[i], x.beta[i], x.q[i], x.k[i], x.v[i], pending=pending[i], **kw)
            else:
                G.gdn_recoverssm_verify(x.g[i], x.beta[i], x.q[i], x.k[i], x.v[i], **kw)

    return call


def _captured(call):
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        call()
    return graph.replay


def _group_metadata(c, contexts, meta, m):
    payload = SimpleNamespace(
        state_indices=meta.src, query_start_loc=meta.qsl,
        request_indices=torch.arange(c["rows"], device="cuda"), block_table=meta.align.get("block_table"),
        num_computed_tokens=meta.align.get("num_computed_tokens"), block_size=meta.align.get("mamba_block_size"),
        request_rows=tuple(range(c["rows"])), query_lens=tuple(m.qlens.tolist()))
    return [SimpleNamespace(recoverssm_commit=payload, recoverssm_builder=SimpleNamespace(), recoverssm_context=x)
            for x in contexts]


def prepare(case, seed):
    """The engine's state before the step: activations, pages, records, commit
    contexts and the captured verifies."""
    import gdn_recoverssm_ascend as G

    c = dict(case)
    metas = _meta(c, seed)
    tokens, pages = int(metas[0].qsl[-1]), metas[0].pages
    steps, state, conv = _tensors(c, seed, tokens, pages)
    L, B, Q = c["layers"], c["rows"], c["Q"]
    key_dtype = torch.float32 if c["flow"] == "gated" else _DTYPES[c["act"]]
    outs = torch.zeros_like(steps[0].v)
    records, planes = _records(c, key_dtype)

    def context(recs, part=slice(None)):
        return G.GDNRecoverSSMCommitContext.from_tensors(list(conv[part]), list(state[part]), recs[part],
                                                         spec_query_len=Q, max_num_reqs=B)

    meta = _commit_inputs(metas[-1], c["align"])
    s = dict(case=c, meta=meta, outs=outs, planes=planes, state=state, conv=conv, keep=(steps, records))
    if c["flow"] == "deferred":
        # The step before: its verify, and its commit left pending.
        before = _commit_inputs(metas[0], c["align"])
        first, _ = _records(c, key_dtype)
        _verify_calls(c, steps[0], before, state, first, outs)()
        ctx = context(first)
        pending = ctx.commit_deferred(before.accepted, before.src, before.qsl, **before.align)
        s["keep"] += (ctx, before, pending)
        # A verify of one row in a pool of its own, so that the capture below
        # finds the kernels loaded.
        one = torch.zeros(2, *state.shape[2:], dtype=state.dtype, device="cuda")
        zero = [t[0].contiguous() for t in (steps[0].q, steps[0].k, steps[0].v)]
        G.gdn_recoverssm_verify_deferred(
            steps[0].g[0][:1], steps[0].beta[0][:1], *(t[:, :1] for t in zero), checkpoint_state=one,
            replay_cache=records[0], pending=pending[0], query_start_loc=torch.arange(2, device="cuda"),
            state_indices=torch.zeros(1, dtype=torch.int64, device="cuda"), spec_query_len=Q, out=outs[0][:, :1])
        call = _verify_calls(c, steps[1], meta, state, records, outs, pending)
        s["context"] = context(records)
    else:
        call = _verify_calls(c, steps[0], meta, state, records, outs)
        call()  # reads the pages only: loads the kernels before a capture
        if c["flow"] == "step" and c["commit"] == "grouped":
            per = L // _GROUPS
            contexts = [context(records, slice(g * per, (g + 1) * per)) for g in range(_GROUPS)]
            s["coordinator"] = G.GroupedCommitCoordinator()
            s["metadata"] = _group_metadata(c, contexts, meta, metas[-1])
            s["mapping"] = torch.arange(B, dtype=torch.int32, device="cuda")
            s["columns"] = torch.full((B,), -1, dtype=torch.int32, device="cuda")
            s["acceptance"] = torch.zeros(B, dtype=torch.int32, device="cuda")
        elif c["flow"] == "step":
            s["context"] = context(records)
    s["verify"] = _captured(call) if c["graph"] else call
    return s


def run(s):
    """One step: the verifies, then the commit."""
    c, m = s["case"], s["meta"]
    out = {"out": s["outs"], "correction": s["planes"][0], "key": s["planes"][1], "decay": s["planes"][2]}
    s["verify"]()
    if c["flow"] == "gated":
        return out
    if "coordinator" in s:
        s["coordinator"].commit(s["metadata"], m.accepted, s["mapping"], s["columns"], s["acceptance"])
        out["columns"] = s["columns"]
    elif c["flow"] == "deferred":
        s["context"].commit_deferred(m.accepted, m.src, m.qsl, **m.align)
    else:
        s["context"].commit(m.accepted, m.src, m.qsl, **m.align)
    if "context" in s:
        out["lengths"], out["final"] = s["context"].commit_lens, s["context"].final_state_indices
    out["state"], out["conv"] = s["state"], s["conv"]
    return out


# ---------------------------------------------------------------------------
# Work, tolerance and the same step in 64 bits
# ---------------------------------------------------------------------------


def work(case):
    """State pages read once by the verify; the commit reads the committed
    ones again and writes them (the deferred flow reads each page once), with
    the activations, outputs, records and conv histories beside them."""
    c = dict(case)
    L, H, HV, K, V, Q = (c[x] for x in ("layers", "H", "HV", "K", "V", "Q"))
    m = _meta(c, 0)
    page = _row_elements(c) * (4 if c["state"] == "f32" else 2)
    key = H * K * (4 if c["flow"] == "gated" else 2)
    gate = HV * (4 if c["flow"] == "gated" else 8)
    now = m[-1]
    rows, tokens = int(now.valid.sum()), int(now.qlens[now.valid].sum())
    nbytes = rows * page + tokens * ((2 * H * K + 2 * HV * V) * 2 + gate + HV * V * 4 + key + HV * 4)
    flops = tokens * HV * V * K * 4 + tokens * HV * V * Q * 4

    def conv(x):
        return (int((x.n > 0).sum()) + int((x.blen > 0).sum())) * (2 * H * K + HV * V) * _CONV_HISTORY * 2 * 2

    def records(x):
        return int(x.n.sum()) * (HV * V * 4 + key + HV * 4)

    def snapshots(x):
        return int(((x.blen > 0) & (x.boundary != x.final)).sum())

    if c["flow"] == "step":
        active = int((now.n > 0).sum())
        nbytes += (2 * active + snapshots(now)) * page + records(now) + conv(now)
        flops += int(now.n.sum()) * HV * V * K * 3
    elif c["flow"] == "deferred":
        past = m[0]
        nbytes += (int((past.n > 0).sum()) + snapshots(past)) * page + records(past) + conv(now)
        flops += int(past.n.sum()) * HV * V * K * 3
    return {"bytes": L * nbytes, "flops": L * flops}


def tolerance(case):
    """Whole numbers are the same; the 16-bit outputs (and pages) of another
    correct implementation differ where its FP32 value rounds the other way.
    Measured against the 64-bit step rounded to the outputs' own types over the
    listed cases and drawn ones: at most 4e-5 of the norm, one BF16 spacing
    (7.8e-3) in a value; four times that."""
    return {"rel": 2e-4, "max": 3.2e-2}


def _windows(t, m):
    """[L, T, ...] -> [L, B, Q, ...] in 64 bits, zero past a row's window."""
    Q = int(m.qlens.max())
    at = (m.qsl[:-1, None] + torch.arange(Q)[None]).clamp(max=int(m.qsl[-1]) - 1)
    return t[:, at.to(t.device)].double()


def _exact_verify(c, x, m, pages):
    """The token-by-token gated delta rule from `pages` (64-bit [L, B, HV, V, K])."""
    dev = pages.device
    L, H, HV, Q = c["layers"], c["H"], c["HV"], int(m.qlens.max())
    q, k, v = (_windows(t[:, 0], m) for t in (x.q, x.k, x.v))
    g, beta = _windows(x.g, m), _windows(x.beta, m)
    if c["flow"] == "gated":
        q, k = _unit(q), _unit(k)
        raw = g + x.dt_bias.double()[:, None, None]
        g = -torch.exp(x.A_log.double())[:, None, None] * torch.nn.functional.softplus(raw)
        beta = torch.sigmoid(beta)
    live = (m.valid[:, None] & (torch.arange(Q)[None] < m.qlens[:, None])).to(dev)
    heads = torch.arange(HV, device=dev) // (HV // H)
    S = pages.clone()
    o, corr = torch.zeros_like(v), torch.zeros_like(v)
    decay = torch.exp(g)
    for t in range(Q):
        on = live[:, t][None, :, None]
        kt, qt = k[:, :, t][:, :, heads], q[:, :, t][:, :, heads] * c["K"] ** -0.5
        d = torch.where(on, decay[:, :, t], torch.ones_like(decay[:, :, t]))
        S.mul_(d[..., None, None])
        ct = (v[:, :, t] - (S * kt[..., None, :]).sum(-1)) * beta[:, :, t][..., None]
        ct = torch.where(on[..., None], ct, torch.zeros_like(ct))
        S.add_(ct[..., None] * kt[..., None, :])
        o[:, :, t] = (S * qt[..., None, :]).sum(-1) * on[..., None]
        corr[:, :, t] = ct
    return o, corr, k, decay, live, heads


def _exact_fold(c, m, pages, corr, k, decay, heads):
    """The accepted prefix replayed; returns the final pages and the snapshots."""
    dev = pages.device
    S, snap = pages.clone(), pages.clone()
    n, blen = m.n.to(dev), m.blen.to(dev)
    for t in range(corr.shape[2]):
        on = (t < n)[None, :, None, None, None]
        new = S * decay[:, :, t][..., None, None] + corr[:, :, t][..., None] * k[:, :, t][:, :, heads][..., None, :]
        S = torch.where(on, new, S)
        snap = torch.where((t + 1 == blen)[None, :, None, None, None], S, snap)
    return S, snap


def _scatter(pool, m, final, snap):
    """Boundary snapshots, then final pages, into the pool."""
    b = ((m.blen > 0) & (m.boundary != m.final)).nonzero().flatten()
    a = (m.n > 0).nonzero().flatten()
    dev = pool.device
    pool[:, m.boundary[b].to(dev)] = snap[:, b.to(dev)].to(pool.dtype)
    pool[:, m.final[a].to(dev)] = final[:, a.to(dev)].to(pool.dtype)


def _exact_conv(m, conv):
    h = _CONV_HISTORY
    rows = (m.n > 0).nonzero().flatten()
    moves = []
    for r in rows.tolist():
        window = conv[:, int(m.src[r])]
        n, b = int(m.n[r]), int(m.blen[r])
        if b > 0:
            moves.append((int(m.boundary[r]), window[..., b - 1:b - 1 + h].clone()))
        moves.append((int(m.final[r]), window[..., n - 1:n - 1 + h].clone()))
    for page, part in moves:
        conv[:, page, :, :h] = part


def exact(case, seed):
    """What `run` returns for these inputs, in 64 bits, by the plain recurrence."""
    c = dict(case)
    metas = _meta(c, seed)
    steps, state, conv = _tensors(c, seed, int(metas[0].qsl[-1]), metas[0].pages)
    dev = state.device
    pool = state.double()
    del state
    for i, (x, m) in enumerate(zip(steps, metas)):
        src = m.src.clamp(min=0).to(dev)
        pages = pool[:, src]
        o, corr, k, decay, live, heads = _exact_verify(c, x, m, pages)
        last = i + 1 == len(steps)
        if c["flow"] == "step" or not last:
            final, snap = _exact_fold(c, m, pages, corr, k, decay, heads)
            _scatter(pool, m, final, snap)
            if c["state"] != "f32" and not last:
                pool = pool.to(_DTYPES[c["state"]]).double()  # the pages this step's verify reads are stored ones
            del final, snap
        del pages
        if c["flow"] != "gated":
            _exact_conv(m, conv)
    L, B, Q = c["layers"], c["rows"], c["Q"]
    T = int(m.qsl[-1])
    flat = torch.zeros(L, 1, T, *o.shape[3:], dtype=torch.float64, device=dev)
    in_window = torch.arange(o.shape[2])[None] < m.qlens[:, None]
    flat[:, 0] = o[:, in_window.to(dev)]

    def record(t, per_token):
        out = torch.zeros(L, B, t.shape[3], Q, *t.shape[4:], dtype=torch.float64, device=dev)
        on = live.view(1, B, 1, -1, *([1] * (t.dim() - 4)))
        out[:, :, :, :t.shape[2]] = torch.where(on, t.transpose(2, 3), torch.zeros((), dtype=t.dtype, device=dev))
        return out

    out = {"out": flat, "correction": record(corr, True), "key": record(k, False), "decay": record(decay, True)}
    if c["flow"] == "gated":
        return out
    if c["flow"] == "step" and c["commit"] == "grouped":
        out["columns"] = None
    else:
        out["lengths"] = out["final"] = None
    out["state"], out["conv"] = pool, conv.double()
    return out
