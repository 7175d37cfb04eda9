"""Workloads that this library's rows are timed at, as an engine calls them: operands and
launch scratch built once, then one row launch a pass on the engine's stream.

Every case names one row of the C ABI and its sizes:

  norm    rmsnorm_quant_fp8: M rows of n (residual added in place, bf16 normed row out)
  gemm    gemm_nt_q: Y[M, N] = A[M, K] . W[N, K]^T at dtype mxfp4a8 / fp8a8 / mxfp4a16, on the
          row the resolver picks for M; rblk is fp8a8's weight scale grid (1: per row, 128:
          the 128 x 128 blocks of a checkpoint)
  gated   gemm_nt_q_gated at fp8a8 (silu): [M, N] gate_up, closed into [M, N / 2] codes
  logits  logits_gemm_e4m3: bf16 rows against a joined e4m3 lm_head

The sizes are those of the 27B-class model that bench.py and the tests use: hidden 5376, MLP
21504, q/k/v joined 8192, attention output 4096 -> 5376, vocabulary 262144.
"""
import math

import torch

import libr3d_amd as R

HIDDEN, MLP, QKV, VOCAB = 5376, 21504, 8192, 262144


def listed():
    return [
        # a decode step's norm: the smallest call there is, launch and latency
        dict(name="norm_decode_m4", op="norm", M=4, n=HIDDEN),
        # the same norm over one prefill chunk
        dict(name="norm_prefill_m2048", op="norm", M=2048, n=HIDDEN),
        # one sequence decoding: a gate or up projection with per-channel scales
        dict(name="decode_fp8_gate_m1", op="gemm", dtype="fp8a8", M=1, N=MLP, K=HIDDEN, rblk=1),
        # four sequences decoding: the down projection (long K, few rows)
        dict(name="decode_mxfp4_down_m4", op="gemm", dtype="mxfp4a8", M=4, N=HIDDEN, K=MLP),
        # an odd batch of decoding sequences: the joined q/k/v projection
        dict(name="decode_mxfp4_qkv_m13", op="gemm", dtype="mxfp4a8", M=13, N=QKV, K=HIDDEN),
        # a decode batch past 16 sequences, or ten sequences verifying four drafted tokens each
        dict(name="skinny_fp8_down_m40", op="gemm", dtype="fp8a8", M=40, N=HIDDEN, K=MLP, rblk=128),
        # the MLP's first half for a batch of 24: projection, gate and quantiser in one call
        dict(name="gated_fp8_m24", op="gated", M=24, N=MLP, K=HIDDEN, rblk=128),
        # a short prompt, or one chunk of a chunked prefill, through the down projection
        dict(name="prefill_fp8_down_m512", op="gemm", dtype="fp8a8", M=512, N=HIDDEN, K=MLP, rblk=128),
        # a prompt of no round length through the joined q/k/v projection
        dict(name="prefill_mxfp4_qkv_m1000", op="gemm", dtype="mxfp4a8", M=1000, N=QKV, K=HIDDEN),
        # a full prefill chunk through a gate or up projection, bf16 activations in
        dict(name="prefill_a16_gate_m2048", op="gemm", dtype="mxfp4a16", M=2048, N=MLP, K=HIDDEN),
        # the same chunk with e4m3 weights and per-channel scales
        dict(name="prefill_fp8_gate_m2048", op="gemm", dtype="fp8a8", M=2048, N=MLP, K=HIDDEN, rblk=1),
        # the lm_head for a decode batch of 16
        dict(name="logits_m16", op="logits", M=16, N=VOCAB, K=HIDDEN),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _plane(rng):
    """A weight plane [N, K]: K whole 128-column groups, N of any residue, up to the MLP's."""
    while True:
        n = _log_int(rng, 512, MLP)
        if rng.random() < 0.7:
            n = max(128, n // 128 * 128)
        k = 128 * _log_int(rng, 8, MLP // 128)
        if n * k >= 1 << 22 and n * k <= MLP * HIDDEN:
            return n, k


def draw(rng):
    op = rng.choice(["norm", "decode", "decode", "skinny", "gated", "prefill", "prefill", "logits"])
    if op == "norm":
        return dict(op="norm", M=_log_int(rng, 1, 4096), n=128 * _log_int(rng, 8, 64))
    if op == "logits":
        return dict(op="logits", M=_log_int(rng, 1, 32), N=_log_int(rng, 32000, VOCAB),
                    K=128 * _log_int(rng, 8, HIDDEN // 128))
    N, K = _plane(rng)
    if op == "gated":
        return dict(op="gated", M=rng.randint(1, 64), N=max(256, N // 256 * 256), K=K,
                    rblk=rng.choice([1, 128]))
    M = {"decode": lambda: rng.randint(1, 16), "skinny": lambda: rng.randint(17, 128),
         "prefill": lambda: _log_int(rng, 129, 2048)}[op]()
    dtype = rng.choice(["mxfp4a8", "fp8a8"] + (["mxfp4a16"] if op == "prefill" else []))
    case = dict(op="gemm", dtype=dtype, M=M, N=N, K=K)
    if dtype == "fp8a8":
        case["rblk"] = rng.choice([1, 128])
    return case


# ------------------------------------------------------------------------------- inputs

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda")


def _e4m3(x):
    return x.clamp(-448.0, 448.0).to(torch.float8_e4m3fn)


def _quant_act(x):
    """bf16 rows -> e4m3 codes and one f32 scale per 128 columns (amax onto 448)."""
    M, K = x.shape
    g = x.float().view(M, K // 128, 128)
    s = g.abs().amax(2).clamp_min(1e-30) / 448.0
    return _e4m3(g / s[:, :, None]).view(M, K).view(torch.uint8), s


def _fp8_weights(g, N, K, rblk):
    """N(0, 0.02) weights as e4m3 codes with bf16 scales: one per output channel, repeated
    along K, or one per 128 x 128 block."""
    w = _randn(g, N, K) * 0.02
    if rblk == 1:
        s = (w.abs().amax(1) / 448.0).bfloat16()
        return (_e4m3(w / s.float()[:, None]).view(torch.uint8),
                s[:, None].expand(N, K // 128).contiguous())
    pad = -N % 128
    blk = torch.nn.functional.pad(w, (0, 0, 0, pad)).view(-1, 128, K // 128, 128)
    s = (blk.abs().amax((1, 3)) / 448.0).bfloat16()
    q = blk / s.float()[:, None, :, None]
    return _e4m3(q.view(-1, K)[:N]).view(torch.uint8), s


def _mxfp4_weights(g, N, K):
    """Uniform e2m1 codes, two a byte, with E8M0 scales of 2^-8 .. 2^0 per 32 columns."""
    b = torch.randint(0, 256, (N, K // 2), generator=g, device="cuda", dtype=torch.uint8)
    s = torch.randint(119, 128, (N, K // 32), generator=g, device="cuda", dtype=torch.uint8)
    return b, s


def _head(g, N, K):
    """e4m3 codes [N, K] of N(0, 0.02) weights and a bf16 scale per (row, 128 columns)."""
    codes = torch.empty(N, K, dtype=torch.uint8, device="cuda")
    scale = torch.empty(N, K // 128, dtype=torch.bfloat16, device="cuda")
    for n in range(0, N, 32768):
        w = (_randn(g, min(32768, N - n), K) * 0.02).view(-1, K // 128, 128)
        s = (w.abs().amax(2) / 448.0).bfloat16()
        codes[n:n + len(w)] = _e4m3(w / s.float()[:, :, None]).view(-1, K).view(torch.uint8)
        scale[n:n + len(w)] = s
    return codes, scale


def _inputs(case, seed):
    g = _gen(seed)
    if case["op"] == "norm":
        M, n = case["M"], case["n"]
        return dict(x=_randn(g, M, n).bfloat16(), residual=(4 * _randn(g, M, n)).bfloat16(),
                    w=(1 + 0.1 * _randn(g, n)).bfloat16())
    M, N, K = case["M"], case["N"], case["K"]
    x = _randn(g, M, K).bfloat16()
    if case["op"] == "logits":
        codes, scale = _head(g, N, K)
        return dict(x=x, b=codes, bs=scale)
    if case.get("dtype") == "mxfp4a16":
        b, bs = _mxfp4_weights(g, N, K)
        return dict(x=x, b=b, bs=bs)
    a, s = _quant_act(x)
    b, bs = (_mxfp4_weights(g, N, K) if case.get("dtype") == "mxfp4a8"
             else _fp8_weights(g, N, K, case["rblk"]))
    return dict(a=a, s=s, b=b, bs=bs)


# --------------------------------------------------------------------------- the calls

def _empty(shape, dtype):
    return torch.empty(shape, dtype=dtype, device="cuda")


def _scratch(row, ops):
    """The launch scratch the row's hook asks for, as an engine's arena hands it over."""
    need = R.row_scratch_bytes(row, ops)
    if need > 0:
        ops.set_scratch(_empty((need,), torch.uint8), need)


def prepare(case, seed):
    t = _inputs(case, seed)
    if case["op"] == "norm":
        M, n = case["M"], case["n"]
        q, scale = _empty((M, n), torch.uint8), _empty((M, n // 128), torch.float32)
        out = _empty((M, n), torch.bfloat16)
        row = "rmsnorm_quant_fp8"
        ops = R.RmsNormQuantOperands(t["x"], t["residual"], t["w"], q, scale, out, n=n, M=M)
        result = (t["residual"], q, scale, out)
    elif case["op"] == "logits":
        M, N, K = case["M"], case["N"], case["K"]
        header, codes_at, scale_at, size = R.head_header(N, K)
        blob = _empty((size,), torch.uint8)
        blob[:len(header)] = torch.from_numpy(header).cuda()
        blob[codes_at:codes_at + N * K] = t["b"].view(-1)
        blob[scale_at:scale_at + 2 * t["bs"].numel()] = t["bs"].view(torch.uint8).view(-1)
        y = _empty((M, N), torch.float32)
        row = "logits_gemm_e4m3"
        ops = R.LogitsOperands(t["x"], blob, y, n_vocab=N, n_embd=K)
        R.forget_head(blob)          # a head joined at this address before is another head
        result = y
    elif case["op"] == "gated":
        M, N, K = case["M"], case["N"], case["K"]
        q, scale = _empty((M, N // 2), torch.uint8), _empty((M, N // 256), torch.float32)
        row = "gemm_nt_q_gated_fp8a8"
        ops = R.GatedGemmOperands(t["a"], t["s"], t["b"], t["bs"], q, scale, N=N, K=K, M=M)
        _scratch(row, ops)
        result = (q, scale)
    else:
        M, N, K, dtype = case["M"], case["N"], case["K"], case["dtype"]
        y = _empty((M, N), torch.bfloat16)
        ops = R.GemmOperands(t["x"] if dtype == "mxfp4a16" else t["a"], t.get("s"), t["b"], t["bs"],
                             y, dtype=dtype, N=N, K=K, M=M)
        row = R.resolve("gemm_nt_q", {"dtype": dtype, "M": M, "N": N, "K": K,
                                      "group": 128 if dtype == "fp8a8" else 32})["name"]
        _scratch(row, ops)
        result = y
    return dict(launch=R.row_launcher(row), ops=ops, result=result,
                stream=torch.cuda.current_stream().cuda_stream)


def run(state):
    rc = state["launch"](state["ops"], state["stream"])
    if rc != R.RAD_OK:
        raise RuntimeError("the row refused the launch: %d" % rc)
    return state["result"]


# ------------------------------------------------------------------ what a pass must do

def work(case):
    M = case["M"]
    if case["op"] == "norm":
        n = case["n"]
        return {"bytes": M * n * (2 + 2 + 2 + 1 + 2) + M * (n // 128) * 4 + 2 * n, "flops": 0}
    N, K = case["N"], case["K"]
    if case["op"] == "logits":
        return {"bytes": N * K + N * (K // 128) * 2 + M * K * 2 + M * N * 4, "flops": 2 * M * N * K}
    dtype = case.get("dtype", "fp8a8")
    if dtype == "fp8a8":
        w = N * K + (N if case["rblk"] == 1 else -(-N // 128)) * (K // 128) * 2
    else:
        w = N * K // 2 + N * K // 32
    a = M * K * 2 if dtype == "mxfp4a16" else M * K + M * (K // 128) * 4
    y = M * (N // 2) + M * (N // 256) * 4 if case["op"] == "gated" else M * N * 2
    return {"bytes": w + a + y, "flops": 2 * M * N * K}


def tolerance(case):
    if case["op"] == "norm":
        return "exact"               # codes, scales and rows are bit-exact by contract
    if case["op"] == "logits":
        return {"rel": 5e-7}         # f32 sums: measured 1e-7 against 64 bits
    if case["op"] == "gated":
        # codes of a bf16 plane: a plane value one ulp off moves a code now and then, or its
        # group's scale
        return {"rel": 1.2e-2, "differ": 0.01}   # measured 3e-3 against 64 bits
    return {"rel": 7e-3, "max": 4e-2}        # bf16 results: measured 1.7e-3 against 64 bits


# ------------------------------------------------------------- the same in 64-bit torch

def _codes64(c):
    return c.view(torch.float8_e4m3fn).double()


def _weights64(case, b, bs):
    """The dequantised weights [N, K]."""
    if case.get("dtype", "fp8a8") != "fp8a8":
        lut = torch.tensor([0, .5, 1, 1.5, 2, 3, 4, 6], dtype=torch.float64, device="cuda")
        lut = torch.cat([lut, -lut])
        w = torch.stack([lut[(b & 15).long()], lut[(b >> 4).long()]], 2).view(len(b), -1)
        return w * torch.exp2(bs.double() - 127).repeat_interleave(32, 1)
    s = bs.double().repeat_interleave(128, 1)
    if case.get("rblk", 1) == 128:
        s = s.repeat_interleave(128, 0)[:len(b)]
    return _codes64(b) * s


def _mxfp8_64(x):
    """bf16 rows after the mxfp4a16 row's quantiser: e4m3 codes under a power of two per 32
    columns, the least that brings the block's largest value to 448 or below."""
    M, K = x.shape
    g = x.double().view(M, K // 32, 32)
    e = torch.ceil(torch.log2(g.abs().amax(2).clamp_min(2.0 ** -126) / 448.0)).clamp(-127, 127)
    s = torch.exp2(e)[:, :, None]
    return (_e4m3((g / s).float()).double() * s).view(M, K)


def _by_rows(a, t, case):
    """a [M, K] against every weight row, some rows of the plane at a time."""
    out = []
    for n in range(0, case["N"], 8192):
        bs = t["bs"]
        bs = bs[n // 128:(n + 8192) // 128] if case.get("rblk", 1) == 128 else bs[n:n + 8192]
        out.append(a @ _weights64(case, t["b"][n:n + 8192], bs).T)
    return torch.cat(out, 1)


def exact(case, seed):
    t = _inputs(case, seed)
    if case["op"] == "norm":
        n = case["n"]
        r = t["x"].double() + t["residual"].double()
        y = r * torch.rsqrt(r.square().mean(1, keepdim=True) + 1e-6) * t["w"].double()
        return (r, None, y.view(-1, n // 128, 128).abs().amax(2) / 448.0, y)
    if "x" in t:
        a = _mxfp8_64(t["x"]) if case["op"] == "gemm" else t["x"].double()
    else:
        a = _codes64(t["a"]) * t["s"].double().repeat_interleave(128, 1)
    y = _by_rows(a, t, case)
    if case["op"] == "gated":
        gate, up = y.chunk(2, 1)
        h = gate * torch.sigmoid(gate) * up
        return (None, h.view(len(h), -1, 128).abs().amax(2) / 448.0)
    return y
