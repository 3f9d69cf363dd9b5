"""Timed cases of the attention framework: what its users have it do, through its public entry points.

Five kinds of pass:

  fwd      one dense attention forward (forward / forward_only / forward_bf16)
  prefill  a causal prompt pass of a grouped-query model with its K/V then written into the paged
           cache (forward_bf16 or forward, kv_append with per-sequence lengths)
  bwd      one attention backward from the saved O and L (backward / backward_bf16)
  varlen   forward and backward of one packed ragged batch (forward_varlen, backward_varlen)
  decode   one generated token: optionally its K/V row appended to the cache, then the paged decode

Sizes are the framework's own benchmark and test shapes, and generic ones of the same ranges.
"""
import importlib.util
import math
import pathlib
import random
import sys

import torch

_PKG = pathlib.Path(__file__).resolve().parent.parent / "flashattn-cuda_amd"
_NAME = "flashattn_cuda_amd"


def _package():
    """The package directory has a hyphen in its name, so it is imported by its path."""
    if _NAME not in sys.modules:
        spec = importlib.util.spec_from_file_location(_NAME, _PKG / "__init__.py",
                                                      submodule_search_locations=[str(_PKG)])
        mod = importlib.util.module_from_spec(spec)
        sys.modules[_NAME] = mod
        spec.loader.exec_module(mod)
    return sys.modules[_NAME]


fa = _package()
DEV = "cuda"
PAGE = 16
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}


def listed():
    return [
        # The benchmark's shortest sequence: one attention call of a small model, bound by latency and launches.
        dict(name="fwd_n1024", kind="fwd", dtype="fp16", B=1, H=8, Hkv=8, N=1024, D=64, causal=False, want_l=True),
        # The headline: forward with L, as a training step calls it.
        dict(name="fwd_n4096", kind="fwd", dtype="fp16", B=1, H=8, Hkv=8, N=4096, D=64, causal=False, want_l=True),
        # The largest forward of the benchmark: a causal batch at the head size of large language models.
        dict(name="fwd_causal_d128", kind="fwd", dtype="fp16", B=4, H=16, Hkv=16, N=4096, D=128, causal=True,
             want_l=True),
        # Serving: the prompts of a small batch through one layer of a grouped-query model, padded to an odd length.
        dict(name="prefill_gqa_bf16", kind="prefill", dtype="bf16", B=2, H=32, Hkv=8, N=1777, D=128, causal=True,
             mix=3),
        # A unit-test sized backward in the float32 tensors that the reference's callers pass.
        dict(name="bwd_fp32_n512", kind="bwd", dtype="fp32", B=2, H=8, Hkv=8, N=512, D=64, causal=False),
        # The backward of the headline.
        dict(name="bwd_n4096", kind="bwd", dtype="fp16", B=1, H=8, Hkv=8, N=4096, D=64, causal=False),
        # The backward of the largest forward.
        dict(name="bwd_causal_d128", kind="bwd", dtype="fp16", B=4, H=16, Hkv=16, N=4096, D=128, causal=True),
        # Training one layer of a grouped-query model in bfloat16.
        dict(name="bwd_gqa_bf16", kind="bwd", dtype="bf16", B=1, H=32, Hkv=8, N=2000, D=128, causal=True),
        # Training on a packed batch of documents of uneven lengths.
        dict(name="varlen_train", kind="varlen", dtype="fp16", S=12, H=8, Hkv=8, lo=100, hi=4096, D=64, causal=True,
             mix=11),
        # Serving: a decode step of a grouped-query model, its new K/V row appended first.
        dict(name="decode_step_gqa", kind="decode", dtype="bf16", B=8, H=32, Hkv=8, D=128, lo=200, hi=4000,
             append=True, mix=5),
        # One user's long conversation: a single sequence, bound by how much of the chip it can use.
        dict(name="decode_one_long", kind="decode", dtype="fp16", B=1, H=32, Hkv=8, D=128, lo=32000, hi=32000,
             append=False, mix=1),
        # The benchmark's decode: 32 sequences of up to 32768 tokens, multi-head K/V, bound by memory.
        dict(name="decode_batch_long", kind="decode", dtype="fp16", B=32, H=32, Hkv=32, D=128, lo=512, hi=32768,
             append=False, mix=5),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _heads(rng):
    H = rng.choice([4, 8, 8, 16, 32])
    return H, H // rng.choice([1, 1, 2, 4])


def draw(rng):
    kind = rng.choice(["fwd", "fwd", "prefill", "bwd", "bwd", "varlen", "decode", "decode"])
    D = rng.choice([64, 128])
    while True:
        H, Hkv = _heads(rng)
        if kind == "fwd":
            c = dict(kind=kind, dtype=rng.choice(["fp16", "fp16", "bf16", "fp32"]), B=rng.choice([1, 1, 2, 4]), H=H,
                     Hkv=Hkv, N=_log(rng, 100, 8192), D=D, causal=rng.random() < 0.5, want_l=rng.random() < 0.7)
            most = 3e11
        elif kind == "prefill":
            c = dict(kind=kind, dtype=rng.choice(["fp16", "bf16"]), B=rng.choice([1, 2, 4]), H=H, Hkv=Hkv,
                     N=_log(rng, 60, 4096), D=D, causal=True, mix=rng.randrange(1000))
            most = 3e11
        elif kind == "bwd":
            c = dict(kind=kind, dtype=rng.choice(["fp16", "fp16", "bf16", "fp32"]), B=rng.choice([1, 1, 2, 4]), H=H,
                     Hkv=Hkv, N=_log(rng, 60, 4096), D=D, causal=rng.random() < 0.5)
            most = 6e11
        elif kind == "varlen":
            c = dict(kind=kind, dtype="fp16", S=rng.randint(2, 24), H=H, Hkv=Hkv, lo=rng.choice([16, 100, 400]),
                     hi=_log(rng, 500, 4096), D=D, causal=rng.random() < 0.5, mix=rng.randrange(1000))
            most = 6e11
        else:
            lo = _log(rng, 50, 8000)
            c = dict(kind=kind, dtype=rng.choice(["fp16", "bf16"]), B=_log(rng, 1, 32), H=H, Hkv=Hkv, D=D, lo=lo,
                     hi=min(32768, lo * rng.choice([1, 4, 16])), append=rng.random() < 0.5, mix=rng.randrange(1000))
            most = 1e12
        if work(c)["flops"] <= most and work(c)["bytes"] <= 4e9:
            return c


def _lens(case):
    """Lengths of the sequences of a ragged case: part of the case, not of its inputs."""
    r = random.Random(case["mix"])
    if case["kind"] == "varlen":
        return [r.randint(case["lo"], case["hi"]) for _ in range(case["S"])]
    if case["kind"] == "prefill":   # prompts padded to N: the longest has N tokens
        return [case["N"]] + [r.randint(max(1, case["N"] // 3), case["N"]) for _ in range(case["B"] - 1)]
    return [r.randint(case["lo"], case["hi"]) for _ in range(case["B"])]


def _randn(g, shape, dtype):
    return torch.randn(shape, generator=g, device=DEV, dtype=dtype)


def _pages(case, lens, g):
    """A page table whose pages are scattered over the pool, as a serving allocator leaves them."""
    need = [-(-n // PAGE) for n in lens]
    perm = torch.randperm(sum(need), generator=g, device=DEV).to(torch.int32)
    table = torch.zeros(len(lens), max(need), dtype=torch.int32, device=DEV)
    at = 0
    for b, n in enumerate(need):
        table[b, :n] = perm[at:at + n]
        at += n
    return table, at


def prepare(case, seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    dt, kind, D, H, Hkv = DTYPES[case["dtype"]], case["kind"], case["D"], case["H"], case["Hkv"]
    st = {"case": case}
    if kind in ("fwd", "prefill", "bwd"):
        B, N = case["B"], case["N"]
        st["q"], st["k"], st["v"] = (_randn(g, (B, h, N, D), dt) for h in (H, Hkv, Hkv))
    if kind == "prefill":
        lens = _lens(case)
        st["table"], n_pages = _pages(case, lens, g)
        st["k_pool"], st["v_pool"] = (torch.zeros(n_pages, Hkv, PAGE, D, dtype=dt, device=DEV) for _ in range(2))
        st["start"] = torch.zeros(B, dtype=torch.int32, device=DEV)
        st["lens"] = torch.tensor(lens, dtype=torch.int32, device=DEV)
    elif kind == "bwd":
        fwd = fa.forward_bf16 if case["dtype"] == "bf16" else fa.forward
        st["o"], st["l"] = fwd(st["q"], st["k"], st["v"], causal=case["causal"])
        if case["dtype"] == "fp32":   # such a caller holds every tensor in float32
            st["o"] = st["o"].float()
        st["do"] = _randn(g, (B, H, N, D), dt)
    elif kind == "varlen":
        lens = _lens(case)
        total = sum(lens)
        st["q"], st["k"], st["v"], st["do"] = (_randn(g, (h, total, D), dt) for h in (H, Hkv, Hkv, H))
        st["cu"] = torch.tensor([0] + lens, dtype=torch.int32, device=DEV).cumsum(0).to(torch.int32)
        st["max"] = max(lens)
    elif kind == "decode":
        lens = _lens(case)
        B = len(lens)
        st["table"], n_pages = _pages(case, lens, g)
        st["q"] = _randn(g, (B, H, D), dt)
        st["k_pool"], st["v_pool"] = (_randn(g, (n_pages, Hkv, PAGE, D), dt) for _ in range(2))
        st["ctx"] = torch.tensor(lens, dtype=torch.int32, device=DEV)
        if case["append"]:   # the new token is the context's last
            st["start"] = st["ctx"] - 1
            st["k"], st["v"] = (_randn(g, (B, Hkv, 1, D), dt) for _ in range(2))
    return st


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "fwd":
        if case["dtype"] == "bf16":
            return fa.forward_bf16(st["q"], st["k"], st["v"], causal=case["causal"], want_L=case["want_l"])
        if case["want_l"]:
            return fa.forward(st["q"], st["k"], st["v"], causal=case["causal"])
        return [fa.forward_only(st["q"], st["k"], st["v"], causal=case["causal"])]
    if kind == "prefill":
        if case["dtype"] == "bf16":
            o, = fa.forward_bf16(st["q"], st["k"], st["v"], causal=True, want_L=False)
        else:
            o = fa.forward_only(st["q"], st["k"], st["v"], causal=True)
        bad = fa.kv_append(st["k"], st["v"], st["k_pool"], st["v_pool"], st["table"], st["start"], st["lens"])
        return [o, st["k_pool"], st["v_pool"], bad]
    if kind == "bwd":
        bwd = fa.backward_bf16 if case["dtype"] == "bf16" else fa.backward
        return bwd(st["q"], st["k"], st["v"], st["o"], st["do"], st["l"], causal=case["causal"])
    if kind == "varlen":
        o, l = fa.forward_varlen(st["q"], st["k"], st["v"], st["cu"], st["max"], causal=case["causal"])
        grads = fa.backward_varlen(st["q"], st["k"], st["v"], o, st["do"], l, st["cu"], st["max"],
                                   causal=case["causal"])
        return [o, l, *grads]
    if case["append"]:
        bad = fa.kv_append(st["k"], st["v"], st["k_pool"], st["v_pool"], st["table"], st["start"])
        o, l = fa.decode_paged(st["q"], st["k_pool"], st["v_pool"], st["table"], st["ctx"])
        return [o, l, st["k_pool"], st["v_pool"], bad]
    return fa.decode_paged(st["q"], st["k_pool"], st["v_pool"], st["table"], st["ctx"])


def work(case):
    """Products of the attention (2 forward, 5 backward, half of them under a causal mask); each input read and each
    output written once: 16-bit operands and O (32-bit where the caller passes such), 32-bit L and gradients."""
    kind, D, H, Hkv = case["kind"], case["D"], case["H"], case["Hkv"]
    e = 4 if case["dtype"] == "fp32" else 2

    def pairs(n):
        return n * (n + 1) / 2 if case.get("causal") else n * n

    if kind in ("fwd", "prefill", "bwd"):
        B, N = case["B"], case["N"]
        qo, kv, rows = B * H * N * D, B * Hkv * N * D, B * H * N
        if kind == "bwd":
            return {"bytes": e * (3 * qo + 2 * kv) + 4 * rows + 4 * (qo + 2 * kv), "flops": 10 * B * H * pairs(N) * D}
        b = e * (qo + 2 * kv) + 2 * qo + (4 * rows if case.get("want_l") else 0)
        if kind == "prefill":
            b += 2 * 2 * sum(_lens(case)) * Hkv * D
        return {"bytes": b, "flops": 4 * B * H * pairs(N) * D}
    lens = _lens(case)
    if kind == "varlen":
        total = sum(lens)
        qo, kv, rows = H * total * D, Hkv * total * D, H * total
        return {"bytes": 2 * (2 * qo + 2 * kv) + 4 * rows + 2 * (3 * qo + 2 * kv) + 4 * rows + 4 * (qo + 2 * kv),
                "flops": 14 * H * sum(pairs(n) for n in lens) * D}
    B = len(lens)
    b = 2 * 2 * sum(lens) * Hkv * D + 2 * 2 * B * H * D + 4 * B * H + 4 * sum(-(-n // PAGE) for n in lens) + 4 * B
    if case["append"]:
        b += 2 * 2 * 2 * B * Hkv * D
    return {"bytes": b, "flops": 4 * H * sum(lens) * D}


def tolerance(case):
    """About four times the largest relative error against 64 bits that the path shows over these ranges (2.9e-4 in
    fp16, 2.3e-3 in bf16): P, dS and the outputs are rounded to 16 bits (11 significant in fp16, 8 in bf16) before
    their products or stores."""
    return {"rel": 1e-2 if case["dtype"] == "bf16" else 1.2e-3}


def _attend(q, k, v, causal):
    """64-bit attention of one head, rows in blocks: (O, L)."""
    n, d = q.shape
    o, l = torch.empty(n, d, dtype=torch.float64, device=q.device), torch.empty(n, dtype=torch.float64, device=q.device)
    kt = k.t().contiguous()
    for r0 in range(0, n, 2048):
        r1 = min(n, r0 + 2048)
        s = (q[r0:r1] @ kt) / math.sqrt(d)
        if causal:
            rows = torch.arange(r0, r1, device=q.device)[:, None]
            s.masked_fill_(torch.arange(n, device=q.device)[None] > rows, -math.inf)
        l[r0:r1] = torch.logsumexp(s, 1)
        o[r0:r1] = (s - l[r0:r1, None]).exp_() @ v
    return o, l


def _gradients(q, k, v, do, causal):
    n, d = q.shape
    dq, dk, dv = torch.empty_like(q), torch.zeros_like(k), torch.zeros_like(v)
    kt, vt = k.t().contiguous(), v.t().contiguous()
    for r0 in range(0, n, 2048):
        r1 = min(n, r0 + 2048)
        s = (q[r0:r1] @ kt) / math.sqrt(d)
        if causal:
            rows = torch.arange(r0, r1, device=q.device)[:, None]
            s.masked_fill_(torch.arange(n, device=q.device)[None] > rows, -math.inf)
        p = torch.softmax(s, 1)
        dp = do[r0:r1] @ vt
        ds = p * (dp - (p * dp).sum(1, keepdim=True)) / math.sqrt(d)
        dv += p.t().contiguous() @ do[r0:r1]
        dk += ds.t().contiguous() @ q[r0:r1]
        dq[r0:r1] = ds @ k
    return dq, dk, dv


def _rounded(t, case):
    """What the path computes with: 16-bit operands, also where the caller passes float32."""
    return (t.half() if case["dtype"] == "fp32" else t).double()


def exact(case, seed):
    st = prepare(case, seed)
    kind, H, Hkv, D = case["kind"], case["H"], case["Hkv"], case["D"]
    group = H // Hkv
    f64 = dict(dtype=torch.float64, device=DEV)

    def heads(q, k, v, do, causal):
        """Forward, and with do the gradients, of [H, n, D] heads."""
        n = q.shape[1]
        o, l = torch.empty(H, n, D, **f64), torch.empty(H, n, **f64)
        dq, dk, dv = torch.empty(H, n, D, **f64), torch.zeros(Hkv, n, D, **f64), torch.zeros(Hkv, n, D, **f64)
        for h in range(H):
            a = [_rounded(x, case) for x in (q[h], k[h // group], v[h // group])]
            if kind != "bwd":
                o[h], l[h] = _attend(*a, causal)
            if do is not None:
                x, y, z = _gradients(*a, _rounded(do[h], case), causal)
                dq[h] = x
                dk[h // group] += y
                dv[h // group] += z
        return o, l, dq, dk, dv

    if kind in ("fwd", "prefill", "bwd"):
        got = [heads(st["q"][b], st["k"][b], st["v"][b], st["do"][b] if kind == "bwd" else None, case["causal"])
               for b in range(case["B"])]
        o, l, dq, dk, dv = (torch.stack(x) for x in zip(*got))
        if kind == "bwd":
            return [dq, dk, dv]
        if kind == "fwd":
            return [o, l] if case["want_l"] else [o]
        return [o, None, None, None]   # the pools are copies, compared as they are
    if kind == "varlen":
        bounds = st["cu"].tolist()
        got = [heads(*(st[x][:, a:b] for x in ("q", "k", "v", "do")), case["causal"])
               for a, b in zip(bounds, bounds[1:])]
        return [torch.cat(x, 1) for x in zip(*got)]
    B = len(_lens(case))
    o, l = torch.empty(B, H, D, **f64), torch.empty(B, H, **f64)
    for b, n in enumerate(_lens(case)):
        pages = st["table"][b, :-(-n // PAGE)].long()
        for hk in range(Hkv):
            k, v = (st[p][pages, hk].reshape(-1, D)[:n].double() for p in ("k_pool", "v_pool"))
            if case["append"]:
                k[n - 1], v[n - 1] = st["k"][b, hk, 0].double(), st["v"][b, hk, 0].double()
            s = st["q"][b, hk * group:(hk + 1) * group].double() @ k.t().contiguous() / math.sqrt(D)
            l[b, hk * group:(hk + 1) * group] = torch.logsumexp(s, 1)
            o[b, hk * group:(hk + 1) * group] = torch.softmax(s, 1) @ v
    return [o, l, None, None, None] if case["append"] else [o, l]
