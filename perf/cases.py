"""Performance cases: the calls a serving loop makes into this framework.

Every case is one entry point (or one prepared call) on inputs made from a seed, over the
sizes of the repository's own configurations (strim_amd/workloads.py, bench.py and the
tests): vocabularies of 8 k to 262 k, 1 to 64 rows, 1 to 8 drafts. `listed()` gives the
named ones, `draw()` others of the same ranges. See each case's comment for what it
stands for.
"""
import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "strim-engine_amd"))

from strim_amd import _native as N  # noqa: E402
from strim_amd import ops, workloads  # noqa: E402
from strim_amd.grammar import DeviceGrammar  # noqa: E402

DEV = "cuda:0"

# the options of one sampling call, all plain values
SAMPLE = dict(op="sample", B=8, V=151_936, dtype="bf16", dist="zipf", T=0.8, top_k=0,
              top_p=1.0, min_p=0.0, mixed=False, rep=1.0, pres=0.0, freq=0.0, H=0, mask="none",
              noise="icdf", sampler_flags=False)
VERIFY = dict(op="verify", B=4, k=3, V=151_936, Vd=0, dtype="bf16", T=0.7, top_k=0, top_p=1.0,
              noise="gumbel")
HEAD = dict(op="head", B=8, K=5120, V=151_936)
DRAFT = dict(op="draft", B=4, Vd=32_768, dtype="bf16")
GRAMMAR = dict(op="grammar", B=8, V=151_936)


def listed():
    return [
        # one chat stream, float32 logits, repetition penalty, top-k 20 + top-p 0.95: the
        # smallest call, where the launches and their latency are all there is
        dict(SAMPLE, name="sample_b1_f32", B=1, dtype="f32", dist="spikes", T=0.7, top_k=20,
             top_p=0.95, rep=1.05, H=256),
        # the ordinary constrained decode step: 8 requests with penalties over a 4,096-token
        # history, grammar masks of every density, top-p
        dict(SAMPLE, name="sample_b8_chain", T=0.8, top_p=0.9, pres=0.5, freq=0.3, H=4096,
             mask="grammar"),
        # a loaded server: 64 requests, 2,048-token histories, 5 % masks, every filter on
        dict(SAMPLE, name="sample_b64", B=64, dist="normal", T=0.8, top_k=40, top_p=0.95,
             min_p=0.02, pres=0.5, freq=0.3, H=2048, mask="sparse", noise="philox"),
        # creative sampling: flat distributions at T 1 whose top-p nucleus holds tens of
        # thousands of tokens
        dict(SAMPLE, name="sample_b8_wide", dist="flat", T=1.0, top_p=0.95),
        # a chat request that sets temperature and top_p alone, through the non-speculative
        # sampler's rules (ties kept, rank-indexed Gumbel noise), one stream at the vocabulary
        # that the real draft table belongs to
        dict(SAMPLE, name="sampler_v248k", B=1, V=248_320, T=0.8, top_p=0.95, noise="gumbel",
             sampler_flags=True),
        # a speculative round with argmax drafts, no filter
        dict(VERIFY, name="verify_onehot"),
        # a speculative round with drafts sampled from a truncated draft vocabulary
        dict(VERIFY, name="verify_draft", Vd=32_768),
        # the same with the filters of ordinary chat settings
        dict(VERIFY, name="verify_draft_filtered", Vd=32_768, top_k=20, top_p=0.95),
        # the producer of the logits for a batch of 8: memory traffic of the lm_head
        dict(HEAD, name="head_b8"),
        # the same at the largest batch
        dict(HEAD, name="head_b64", B=64),
        # one draft step's argmax over the truncated vocabulary
        dict(DRAFT, name="draft_argmax"),
        # masks of 8 requests in states of a JSON-object grammar met for the first time
        dict(GRAMMAR, name="grammar_masks"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["sample"] * 5 + ["verify"] * 3 + ["head"] * 2 + ["draft", "grammar"])
    V = _log_int(rng, 8_192, 262_144)
    dtype = rng.choice(["bf16", "bf16", "f32"])
    if op == "sample":
        c = dict(SAMPLE, B=min(_log_int(rng, 1, 64), 64 * 151_936 // V), V=V, dtype=dtype,
                 dist=rng.choice(["zipf", "normal", "flat", "spikes"]),
                 T=round(rng.uniform(0.5, 1.1), 2), mixed=rng.random() < 0.2,
                 mask=rng.choice(["none", "none", "grammar", "sparse"]),
                 noise=rng.choice(["icdf", "philox", "gumbel"]))
        kind = rng.choice(["top_p", "top_k", "both", "all", "none", "greedy"])
        if kind in ("top_p", "both", "all"):
            c["top_p"] = round(rng.uniform(0.8, 0.99), 3)
        if kind in ("top_k", "both", "all"):
            c["top_k"] = _log_int(rng, 10, 200)
        if kind == "all":
            c["min_p"] = round(rng.uniform(0.01, 0.1), 3)
        if kind == "greedy":
            c["T"] = 0.0
        if rng.random() < 0.5:
            c.update(H=_log_int(rng, 64, 4096), rep=rng.choice([1.0, 1.05]), pres=0.5,
                     freq=rng.choice([0.0, 0.3]))
        c["sampler_flags"] = c["noise"] == "gumbel" and rng.random() < 0.3
        return c
    if op == "verify":
        c = dict(VERIFY, B=_log_int(rng, 1, 8), k=rng.randint(1, 5), V=V, dtype=dtype,
                 T=round(rng.uniform(0.5, 1.0), 2), noise=rng.choice(["gumbel", "icdf"]))
        if rng.random() < 0.6:
            c["Vd"] = min(V, _log_int(rng, 4_096, 32_768))
        if rng.random() < 0.5:
            c.update(top_k=_log_int(rng, 10, 100), top_p=round(rng.uniform(0.8, 0.99), 3))
        return c
    if op == "head":
        return dict(HEAD, B=_log_int(rng, 1, 64), K=256 * rng.randint(4, 20),
                    V=min(V, 151_936))
    if op == "draft":
        return dict(DRAFT, B=_log_int(rng, 1, 16), Vd=_log_int(rng, 4_096, 65_536), dtype=dtype)
    return dict(GRAMMAR, B=_log_int(rng, 1, 16), V=max(V, 32_768))


# ---- inputs -----------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 7919 + 17)
    return g


def _dt(case):
    return torch.bfloat16 if case["dtype"] == "bf16" else torch.float32


def _logits(g, rng, rows, V, dist):
    """Rows of logits, float32: "zipf" N(0, 2.5^2) on a Zipf(1.1) rank bias, "normal"
    N(0, 2^2) with one dominant token in 30 % of the rows, "flat" N(0, 1), "spikes" N(0, 3^2)
    with five tokens at +15."""
    x = torch.randn(rows, V, device=DEV, generator=g)
    if dist == "zipf":
        bias = -1.1 * torch.log(torch.arange(V, device=DEV, dtype=torch.float32) + 1.0)
        return 2.5 * x + bias[torch.randperm(V, device=DEV, generator=g)]
    if dist == "normal":
        x = 2.0 * x
        for r in np.nonzero(rng.random(rows) < 0.3)[0].tolist():
            x[r, int(rng.integers(V))] = 20.0
        return x
    if dist == "spikes":
        x = 3.0 * x
        x[:, torch.randint(0, V, (5,), device=DEV, generator=g)] = 15.0
        return x
    return x


def _params(case, rng, rows):
    p = N.params_array(rows, temperature=case["T"], top_k=case["top_k"], top_p=case["top_p"],
                       min_p=case.get("min_p", 0.0), repetition_penalty=case.get("rep", 1.0),
                       presence_penalty=case.get("pres", 0.0),
                       frequency_penalty=case.get("freq", 0.0),
                       seed=rng.integers(0, 2**63, size=rows, dtype=np.uint64),
                       position=int(rng.integers(1, 4096)))
    if case.get("sampler_flags"):
        p["flags"] = N.FLAG_SAMPLER_COMPAT
    if case.get("mixed"):  # requests of one batch with settings of their own
        p["temperature"] = np.array([0.6, 0.8, 1.0], np.float32)[np.arange(rows) % 3]
        p["top_k"] = np.array([0, 20, 50], np.int32)[(np.arange(rows) // 3) % 3]
        p["top_p"] = rng.uniform(0.8, 1.0, size=rows).astype(np.float32)
        p["min_p"] = 0.05
    return p


def _masks(g, rng, x, kind):
    """Packed allow-masks: "sparse" 5 % at random; "grammar" densities 0.01 / 1 / 10 / 30 %
    by row, in clusters of 64 and scattered in turn, every seventh row one token, every
    eighth without its 200 likeliest tokens."""
    if kind == "none":
        return None
    B, V = x.shape
    u = torch.rand(B, V, device=DEV, generator=g)
    if kind == "sparse":
        return ops.pack_mask(u < 0.05).contiguous()
    dens = torch.tensor([1e-4, 0.01, 0.1, 0.3], device=DEV)[torch.arange(B, device=DEV) % 4]
    runs = u[:, : (V + 63) // 64].repeat_interleave(64, dim=1)[:, :V]
    clustered = ((torch.arange(B, device=DEV) // 4) % 2 == 0)[:, None]
    allowed = torch.where(clustered, runs, u) < dens[:, None]
    for r in range(B):
        if r % 8 == 6:
            allowed[r] = False
        elif r % 8 == 7:
            allowed[r, torch.topk(x[r], min(200, V // 2)).indices] = False
        allowed[r, int(rng.integers(V))] = True  # no row is empty
    return ops.pack_mask(allowed).contiguous()


def _history(rng, B, V, H):
    if not H:
        return None
    ids = (rng.zipf(1.1, size=(B, H)).astype(np.int64) - 1) % V
    return torch.from_numpy(rng.permutation(V)[ids].astype(np.int32)).to(DEV)


def _prepare_sample(case, g, rng):
    B, V = case["B"], case["V"]
    x = _logits(g, rng, B, V, case["dist"]).to(_dt(case))
    mask = _masks(g, rng, x.float(), case["mask"])
    hist = _history(rng, B, V, case["H"])
    noise = None
    if case["noise"] == "icdf":
        noise = torch.from_numpy(rng.random((B, 2), dtype=np.float32)).to(DEV)
    mode = N.NOISE_GUMBEL if case["noise"] == "gumbel" else N.NOISE_ICDF
    ctx = ops.Context(0, max_rows=B, max_vocab=V)
    call = ctx.bind_sample(x, _params(case, rng, B), mask=mask, history=hist, noise_mode=mode,
                           noise=noise)
    return dict(op="sample", ctx=ctx, call=call)


def _prepare_verify(case, g, rng):
    B, k, V, Vd = case["B"], case["k"], case["V"], case["Vd"]
    x = _logits(g, rng, B * (k + 1), V, "zipf").reshape(B, k + 1, V).to(_dt(case))
    dl = table = None
    if Vd:  # drafts sampled from a draft model that leans towards the target
        table = torch.randperm(V, device=DEV, generator=g)[:Vd].sort().values
        dl = 1.25 * torch.randn(B, k, Vd, device=DEV, generator=g)
        dl = (dl + 0.8 * x[:, :k].float()[:, :, table]).to(_dt(case))
        q = torch.softmax(dl.float() / case["T"], dim=-1).reshape(B * k, Vd)
        drafts = table[torch.multinomial(q, 1, generator=g).reshape(B, k)].to(torch.int32)
        table = table.to(torch.int32).contiguous()
    else:  # argmax drafts of a model that is right about two times in three
        drafts = x[:, :k].float().argmax(-1)
        other = torch.randint(0, V, (B, k), device=DEV, generator=g)
        keep = torch.rand(B, k, device=DEV, generator=g) < 0.66
        drafts = torch.where(keep, drafts, other).to(torch.int32)
    mode = N.NOISE_GUMBEL if case["noise"] == "gumbel" else N.NOISE_ICDF
    ctx = ops.Context(0, max_rows=B * (k + 1), max_vocab=V)
    call = ctx.bind_verify(x.contiguous(), drafts.contiguous(), _params(case, rng, B),
                           draft_logits=dl, draft_to_full=table, noise_mode=mode)
    return dict(op="verify", ctx=ctx, call=call)


def _head_inputs(case, seed):
    g = _gen(seed)
    B, K, V = case["B"], case["K"], case["V"]
    x = (2.0 * torch.randn(B, K, device=DEV, generator=g)).to(torch.bfloat16)
    nw = (1.0 + 0.1 * torch.randn(K, device=DEV, generator=g)).to(torch.bfloat16)
    w = torch.empty(V, K, dtype=torch.bfloat16, device=DEV)
    for a in range(0, V, 16_384):
        b = min(V, a + 16_384)
        w[a:b] = 0.05 * torch.randn(b - a, K, device=DEV, generator=g)
    return x, nw, w


def _vocabulary(rng, count):
    """Byte strings of a byte-level BPE vocabulary: the single bytes, then pieces of 3 to 64
    bytes (mean about 6.5), a third with a leading space, some with quotes, backslashes or
    UTF-8 continuation bytes."""
    n = count - 256
    lens = np.minimum(64, 2 + rng.geometric(0.22, size=n))
    end = np.cumsum(lens)
    alpha = np.frombuffer(b"abcdefghijklmnopqrstuvwxyzABCDEFGHIJKLMNOPQRSTUVWXYZ0123456789"
                          b"_.,:;-+=()[]{}<>/!?'", dtype=np.uint8)
    data = alpha[rng.integers(len(alpha), size=int(end[-1]))]
    start = end - lens
    data[start[rng.random(n) < 0.33]] = 0x20
    odd = np.nonzero(rng.random(n) < 0.08)[0]
    special = np.frombuffer(b"\"\\\x80\xa0\xc3\xe4", dtype=np.uint8)
    data[start[odd] + rng.integers(lens[odd])] = special[rng.integers(6, size=len(odd))]
    raw = data.tobytes()
    return [bytes([b]) for b in range(256)] + [raw[a:b] for a, b in zip(start.tolist(),
                                                                        end.tolist())]


def _prepare_grammar(case, rng):
    B, V = case["B"], case["V"]
    nt, fl, in_string = workloads.json_object_dfa()
    grammar = DeviceGrammar(_vocabulary(rng, V - 271), V, eos=(V - 273, V - 275), cache_slots=0)
    grammar.set_dfa(nt, fl)
    # half of the requests are inside a string, the others anywhere in the object
    live = np.nonzero(fl & 2)[0]
    keys = np.where(rng.random(B) < 0.5, in_string, live[rng.integers(len(live), size=B)])
    keys = torch.from_numpy(keys.astype(np.int32)).to(DEV)
    out = torch.empty(B, grammar.words, dtype=torch.int32, device=DEV)
    return dict(op="grammar", grammar=grammar, keys=keys, out=out)


def prepare(case, seed):
    g, rng = _gen(seed), np.random.default_rng(seed)
    op = case["op"]
    if op == "sample":
        return _prepare_sample(case, g, rng)
    if op == "verify":
        return _prepare_verify(case, g, rng)
    if op == "head":
        x, nw, w = _head_inputs(case, seed)
        B, K, V = case["B"], case["K"], case["V"]
        return dict(op=op, x=x, nw=nw, w=w,
                    xn=torch.empty(B, K, dtype=torch.bfloat16, device=DEV),
                    out=torch.empty(B, V, dtype=torch.bfloat16, device=DEV))
    if op == "draft":
        Vd = case["Vd"]
        x = _logits(g, rng, case["B"], Vd, "zipf").to(_dt(case))
        ids = rng.choice(2 * Vd, size=Vd, replace=False)
        table = torch.from_numpy(np.sort(ids).astype(np.int32)).to(DEV)
        return dict(op=op, x=x, table=table)
    return _prepare_grammar(case, rng)


def run(state):
    op = state["op"]
    if op in ("sample", "verify"):
        call = state["call"]
        call()
        # a verify's are the accepted counts and the decided tokens
        return call.out_ids, call.out_status, *([call.status] if op == "verify" else [])
    if op == "head":
        return ops.head_logits(state["x"], state["w"], state["nw"], out=state["out"],
                               xn=state["xn"])
    if op == "draft":
        return ops.draft_argmax(state["x"], state["table"])
    return state["grammar"].masks(state["keys"], out=state["out"])


def work(case):
    op, B = case["op"], case["B"]
    size = 4 if case.get("dtype") == "f32" else 2
    if op == "sample":
        V = case["V"]
        noise = 2 if case["noise"] == "icdf" else 0
        return dict(bytes=workloads.algorithmic_bytes(B, V, size, case["mask"] != "none",
                                                      case["H"], noise), flops=0)
    if op == "verify":
        k, V, Vd = case["k"], case["V"], case["Vd"]
        return dict(bytes=B * ((k + 1) * V + k * Vd) * size + 4 * Vd + B * (4 * k + 48 + 12),
                    flops=0)
    if op == "head":
        K, V = case["K"], case["V"]
        return dict(bytes=2 * (V * K + B * V + B * K + K), flops=2 * B * V * K)
    if op == "draft":
        return dict(bytes=B * case["Vd"] * size + 8 * B, flops=0)
    words = (case["V"] + 31) // 32
    # each token's bytes (mean 6.5) and offset, the words written
    return dict(bytes=int((case["V"] - 271) * 10.5) + 4 * B * words, flops=0)


def tolerance(case):
    if case["op"] == "head":
        # bf16 logits of float32 sums: another order of the sum moves a rounding here and
        # there by one bf16 step (measured against a float32 product: 6e-5, 7.8e-3)
        return dict(rel=2.4e-4, max=3.1e-2)
    return "exact"  # token ids, counts, statuses and mask words


def exact(case, seed):
    """The logits in 64 bits; the other cases return whole numbers only."""
    if case["op"] != "head":
        return None
    x, nw, w = _head_inputs(case, seed)
    x = x.double()
    xn = nw.double() * (x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-6))
    out = torch.empty(case["B"], case["V"], dtype=torch.float64, device=DEV)
    for a in range(0, case["V"], 16_384):
        out[:, a:a + 16_384] = xn @ w[a:a + 16_384].double().T
    return out
