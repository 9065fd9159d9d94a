"""Work that users of the MLA decode library give it, for timing and comparing builds.

listed() holds the fixed cases and draw() more of the same ranges. A case is
one call of a decode step: one sequence's decode (fp16, bf16, an fp8 cache, or
the fp32 path), a packed or paged batch, or one of the projections around the
decode. "api" says how the call is made: "torch" through the extension's
functions, which allocate the output and the workspace, "c" through the C ABI
with buffers the caller keeps, as a decode loop without an allocator does.
Inputs are N(0, 1) (weights scaled by the square root of their fan-in), as
bench.py and the tests draw them.
"""
import ctypes
import math
import os
import random
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if os.path.join(_ROOT, "ada-mla_amd") not in sys.path:
    sys.path.insert(0, os.path.join(_ROOT, "ada-mla_amd"))

import ada_mla  # noqa: E402
from ada_mla import capi  # noqa: E402

DEV = "cuda:0"
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32, "fp8": torch.float8_e4m3fn}
SCALE = 1.0 / math.sqrt(192.0)  # softmax scale of the decode contract
FP8_SCALE = 1.0


def listed():
    return [
        # the first tokens of a conversation: latency and launches are all there is
        dict(name="short_bf16", kind="decode", dtype="bf16", heads=128, tokens=200, api="c"),
        # the headline decode call: one sequence of ordinary length, all heads
        dict(name="headline_fp16", kind="decode", dtype="fp16", heads=128, tokens=4096, api="c"),
        # a long context, split over the whole chip
        dict(name="long_fp16", kind="decode", dtype="fp16", heads=128, tokens=65536, api="torch"),
        # one rank of an eight-way tensor-parallel model: few heads, a memory stream
        dict(name="few_heads_fp16", kind="decode", dtype="fp16", heads=16, tokens=32768, api="c"),
        # a quantised cache, ragged length
        dict(name="quantised_fp8", kind="decode", dtype="fp8", heads=128, tokens=20011, api="torch"),
        # the full-precision path as a numerical reference, short
        dict(name="short_fp32", kind="decode", dtype="fp32", heads=128, tokens=1024, api="c"),
        # and long, ragged
        dict(name="long_fp32", kind="decode", dtype="fp32", heads=128, tokens=20011, api="torch"),
        # a serving batch of mixed lengths, packed
        dict(name="batch_bf16", kind="batch", dtype="bf16", heads=128, batch=32, shortest=512, longest=16384,
             mix=42, page=0, api="torch"),
        # a larger serving batch of short requests in a paged cache
        dict(name="paged_short_fp16", kind="batch", dtype="fp16", heads=128, batch=64, shortest=1, longest=1500,
             mix=7, page=64, api="torch"),
        # the projections around the decode, at the batch of an ordinary step
        dict(name="absorb_fp16", kind="absorb", dtype="fp16", heads=128, batch=32, api="c"),
        dict(name="project_fp16", kind="project", dtype="fp16", heads=128, batch=32, d_model=5120, api="torch"),
        # and of a full serving batch
        dict(name="project_wide_bf16", kind="project", dtype="bf16", heads=128, batch=160, d_model=5120, api="torch"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: sizes spread over the logarithm of their range, odd ones among them."""
    kind = rng.choice(["decode", "decode", "decode", "fp32", "batch", "batch", "absorb", "project"])
    api = rng.choice(["c", "torch"])
    if kind == "decode":
        heads = rng.choice([16, 32, 48, 64, 128, 256])
        return dict(kind="decode", dtype=rng.choice(["fp16", "bf16", "fp8"]), heads=heads,
                    tokens=_log(rng, 16, min(131072, 128 * 65536 // heads)), api=api)
    if kind == "fp32":
        heads = rng.choice([16, 32, 48, 64, 128])
        return dict(kind="decode", dtype="fp32", heads=heads,
                    tokens=_log(rng, 16, min(65536, 128 * 20011 // heads)), api=api)
    if kind == "batch":
        heads, batch = rng.choice([16, 32, 64, 128]), _log(rng, 2, 128)
        longest = _log(rng, 32, min(16384, 128 * 32 * 16384 // (heads * batch)))
        page = rng.choice([0, 32, 64, 128])
        return dict(kind="batch", dtype=rng.choice(["fp16", "bf16"] if page else ["fp16", "bf16", "fp8"]),
                    heads=heads, batch=batch, shortest=rng.choice([0, 1, longest // 2, longest]), longest=longest,
                    mix=rng.randrange(1 << 30), page=page, api="torch")
    dtype, heads, batch = rng.choice(["fp16", "bf16"]), rng.choice([16, 32, 128]), _log(rng, 1, 256)
    if kind == "absorb":
        return dict(kind="absorb", dtype=dtype, heads=heads, batch=batch, api=api)
    return dict(kind="project", dtype=dtype, heads=heads, batch=batch, d_model=rng.choice([1000, 2048, 4096, 5120, 7168]),
                api=api)


def _lengths(case):
    r = random.Random(case["mix"])
    return [r.randint(case["shortest"], case["longest"]) for _ in range(case["batch"])]


class _Inputs:
    """The inputs of a case, on the GPU, from the seed."""

    def __init__(self, case, seed):
        gen = torch.Generator(device=DEV)
        gen.manual_seed(seed)
        dt = DTYPES[case["dtype"]]
        q_dt = torch.float16 if case["dtype"] == "fp8" else dt

        def normal(*shape, dtype=q_dt, scale=1.0):
            draw_dt = torch.float32 if dtype == torch.float8_e4m3fn else dtype
            t = torch.randn(shape, generator=gen, device=DEV, dtype=draw_dt)
            if scale != 1.0:
                t *= scale
            return t if dtype == draw_dt else t.to(dtype)

        h = case["heads"]
        if case["kind"] == "decode":
            self.q = normal(h, 576)
            self.c = normal(case["tokens"], 576, dtype=dt)
        elif case["kind"] == "batch":
            self.lengths = _lengths(case)
            b, total = case["batch"], sum(self.lengths)
            self.q = normal(b, h, 576)
            cu = [0]
            for n in self.lengths:
                cu.append(cu[-1] + n)
            self.cu_host = cu
            self.cu = torch.tensor(cu, dtype=torch.int32, device=DEV)
            if case["page"]:
                page = case["page"]
                need = [-(-n // page) for n in self.lengths]
                pages = max(1, sum(need))
                order = list(range(pages))
                random.Random(seed).shuffle(order)
                table = [[0] * max(1, max(need)) for _ in range(b)]
                k = 0
                for i, n in enumerate(need):
                    table[i][:n] = order[k:k + n]
                    k += n
                self.table_host = table
                self.table = torch.tensor(table, dtype=torch.int32, device=DEV)
                self.c = normal(pages, page, 576, dtype=dt)
            else:
                self.c = normal(total, 576, dtype=dt)
        elif case["kind"] == "absorb":
            self.q_nope = normal(case["batch"], h, 128)
            self.q_rope = normal(case["batch"], h, 64)
            self.w_uk = normal(h, 128, 512, scale=128 ** -0.5)
        else:
            self.o_star = normal(case["batch"], h, 512)
            self.w_uv = normal(h, 128, 512, scale=512 ** -0.5)
            self.w_o = normal(case["d_model"], h * 128, scale=(h * 128) ** -0.5)


def _c_call(case, x):
    """The C ABI call of a case with the buffers a caller keeps: the arguments, formed once."""
    lib, dtype, h = capi.load(), case["dtype"], case["heads"]
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)

    def buffers(shape, dt, ws_bytes):
        return torch.empty(shape, dtype=dt, device=DEV), torch.empty(max(ws_bytes, 256), dtype=torch.uint8, device=DEV)

    if case["kind"] == "decode":
        n = case["tokens"]
        if dtype == "fp32":
            size = lib.mla_decode_fused_workspace_size(h, n, 0)
            out, ws = buffers((h, 512), torch.float32, size)
            return lib.mla_decode_fused_fp32, (x.q.data_ptr(), x.c.data_ptr(), out.data_ptr(), ws.data_ptr(), size,
                                               h, 576, n, 0, stream), out, ws
        if dtype == "fp8":
            size = lib.mla_decode_split_fp8_workspace_size(1, h, n, 0)
            out, ws = buffers((h, 512), torch.float16, size)
            return lib.mla_decode_split_fp8, (x.q.data_ptr(), x.c.data_ptr(), FP8_SCALE, out.data_ptr(),
                                              ws.data_ptr(), size, h, n, 0, stream), out, ws
        size = lib.mla_decode_split_workspace_size(h, n, 0)
        out, ws = buffers((h, 512), DTYPES[dtype], size)
        return getattr(lib, "mla_decode_split_" + dtype), (x.q.data_ptr(), x.c.data_ptr(), out.data_ptr(),
                                                           ws.data_ptr(), size, h, n, 0, stream), out, ws
    b = case["batch"]
    if case["kind"] == "absorb":
        out, ws = buffers((b, h, 576), DTYPES[dtype], 0)
        return getattr(lib, "mla_absorb_query_" + dtype), (x.q_nope.data_ptr(), x.q_rope.data_ptr(), x.w_uk.data_ptr(),
                                                           out.data_ptr(), b, h, stream), out, ws
    size = lib.mla_project_output_workspace_size(b, h, case["d_model"])
    out, ws = buffers((b, case["d_model"]), DTYPES[dtype], size)
    return getattr(lib, "mla_project_output_" + dtype), (x.o_star.data_ptr(), x.w_uv.data_ptr(), x.w_o.data_ptr(),
                                                         out.data_ptr(), ws.data_ptr(), size, b, h, case["d_model"],
                                                         stream), out, ws


class _State:
    pass


def prepare(case, seed):
    s = _State()
    s.x = x = _Inputs(case, seed)
    s.total = 0
    if case["api"] == "c":
        s.fn, s.args, s.out, s.ws = _c_call(case, x)
        s.call = None
        return s
    if case["kind"] == "decode":
        if case["dtype"] == "fp32":
            s.call = lambda: ada_mla.mla_decode_fused(x.q, x.c)
        elif case["dtype"] == "fp8":
            s.call = lambda: ada_mla.mla_decode_split(x.q, x.c, cache_scale=FP8_SCALE)
        else:
            s.call = lambda: ada_mla.mla_decode_split(x.q, x.c)
    elif case["kind"] == "batch":
        total = sum(x.lengths)
        if case["page"]:
            s.call = lambda: ada_mla.mla_decode_paged(x.q, x.c, x.table, x.cu, total_tokens=total)
        elif case["dtype"] == "fp8":
            s.call = lambda: ada_mla.mla_decode_split_batched(x.q, x.c, x.cu, cache_scale=FP8_SCALE)
        else:
            s.call = lambda: ada_mla.mla_decode_split_batched(x.q, x.c, x.cu)
    elif case["kind"] == "absorb":
        s.call = lambda: ada_mla.mla_absorb_query(x.q_nope, x.q_rope, x.w_uk)
    else:
        s.call = lambda: ada_mla.mla_project_output(x.o_star, x.w_uv, x.w_o)
    return s


def run(state):
    if state.call is not None:
        return state.call()
    status = state.fn(*state.args)
    if status:
        raise RuntimeError("status %d" % status)
    return state.out


def work(case):
    h, e = case["heads"], 4 if case["dtype"] == "fp32" else 2
    if case["kind"] in ("decode", "batch"):
        b = case.get("batch", 1)
        n = sum(_lengths(case)) if case["kind"] == "batch" else case["tokens"]
        ec = 1 if case["dtype"] == "fp8" else e
        return {"bytes": e * b * h * (576 + 512) + ec * n * 576, "flops": 2 * h * n * (576 + 512)}
    b = case["batch"]
    if case["kind"] == "absorb":
        return {"bytes": e * (b * h * (128 + 64 + 576) + h * 128 * 512), "flops": 2 * b * h * 128 * 512}
    d = case["d_model"]
    return {"bytes": e * (b * h * 512 + h * 128 * 512 + d * h * 128 + b * d),
            "flops": 2 * b * (h * 128 * 512 + h * 128 * d)}


def tolerance(case):
    if case["dtype"] == "fp32":
        return {"rel": 1e-5, "max": 4e-4}
    if case["dtype"] == "bf16":  # stored weights, partials and outputs of 8 significant bits
        return {"rel": 1e-2, "max": 0.2}
    if case["dtype"] == "fp8":  # an fp16 query in two fp8 parts
        return {"rel": 4e-3, "max": 0.1}
    return {"rel": 2e-3, "max": 4e-2}


def _attend(q, c):
    if c.shape[0] == 0:
        return torch.zeros(q.shape[0], 512, dtype=torch.float64, device=q.device)
    return torch.softmax(q @ c.t() * SCALE, dim=-1) @ c[:, :512]


def exact(case, seed):
    x = _Inputs(case, seed)
    if case["kind"] == "decode":
        return _attend(x.q.double(), x.c.to(torch.float32).double() * (FP8_SCALE if case["dtype"] == "fp8" else 1.0))
    if case["kind"] == "batch":
        out = []
        for b, n in enumerate(x.lengths):
            if case["page"]:
                ids = x.table_host[b][:max(1, -(-n // case["page"]))]
                c = x.c[torch.tensor(ids, device=DEV)].reshape(-1, 576)[:n]
            else:
                c = x.c[x.cu_host[b]:x.cu_host[b + 1]]
            out.append(_attend(x.q[b].double(), c.to(torch.float32).double()))
        return torch.stack(out)
    if case["kind"] == "absorb":
        up = torch.stack([x.q_nope[:, h].double() @ x.w_uk[h].double() for h in range(case["heads"])], 1)
        return torch.cat([up, x.q_rope.double()], -1)
    o = torch.stack([x.o_star[:, h].double() @ x.w_uv[h].double().t() for h in range(case["heads"])], 1)
    return o.reshape(case["batch"], -1) @ x.w_o.double().t()
