"""What is measured: the products and conversions a user of this framework has it do.

Every product goes through the GGML operator boundary (``weft_amd.ggml``), as a
graph executor calls it: a forward step of one layer kind over ``layers``
weight matrices, each with its own activations and outputs.  Row dequantize
goes through ``weft_amd.runtime.compile``, asynchronously (a program that feeds
the result to its next kernel does not wait for it).

Weights are records of random payload bytes with the scale fields at the
magnitudes GGML's quantizers give an N(0, 0.02) matrix; activations are N(0, 1).
"""
from __future__ import annotations

import math

import numpy as np
import torch

from weft_amd import _lib, ggml, kernels
from weft_amd.runtime import Buffer, compile as compile_kernel

# (elements, bytes) of a record, GGML type id, activation format
FORMATS = {
    "q4_0": (32, 18, ggml.Q4_0, "q8_0"), "q4_1": (32, 20, ggml.Q4_1, "q8_1"),
    "mxfp4": (32, 17, ggml.MXFP4, "q8_0"), "nvfp4": (64, 36, ggml.NVFP4, "q8_0"),
    "q4_k": (256, 144, ggml.Q4_K, "q8_k"), "q5_k": (256, 176, ggml.Q5_K, "q8_k"),
    "q6_k": (256, 210, ggml.Q6_K, "q8_k"), "iq2_xxs": (256, 66, ggml.IQ2_XXS, "q8_k"),
    "iq2_xs": (256, 74, ggml.IQ2_XS, "q8_k"),
}
ACT = {"q8_0": (32, 34), "q8_1": (32, 36), "q8_k": (256, 292)}

# GGML's IQ2 grids as 2-bit codes of (8, 25, 43), eight a row, four hex digits a row
IQ2XXS_GRID = (
    "0000000200050008000a00110014002000220028002a00410044005000580061006400800082008a00a20101010401100115014001840198"
    "020002020222028204010404041004210424044004420448046004810484049004a405000502050805200546056905800591060906100640"
    "068406a40800080508080814082808410844085008520888090409400a020a14100110041010102110401060108410901095110011081120"
    "1150115a1180122412451400140814201425144914801518156216001616180118041810184018811900190519a01a5120002002200a2044"
    "20612080208221292148220022022401240424102440245625002541256426902808282028942a4440014004401040184021402440404048"
    "4056406040814084409041004120416141804185420142104248425642684400440844204480449945124524460048014804481048404845"
    "49004958496149824a454a9050005008501150195020508050885104514251a4529154905492550a56015654580058115819586459405a08"
    "6004601060406068610061556218626064006405651065126584684280008002800a80418082810481188140821184018404841084158440"
    "8460850085468594860986408660880289048a11900490109024904090a1911691809245940094229444955198819920a002a050a085a109"
    "a200a418a850a904"
)
IQ2XS_GRID = (
    "0000000200050008000a00110014001600190020002200250028004100440046004900500052005500580061006400800082008500880091"
    "0094009900a001010104010601090110011201150118011a0121012401400142014501480151015401600168018101840190020002020205"
    "020802110214022002410244025002550280028a040104040406040904100412041504180421042404400442044504480451045404560460"
    "04810484049005000502050505080511051405200541054405500561058006010604061006260640064206840800080208050808080a0811"
    "0814082008250841084408500858088008a008aa0901090409100940098109890a000a200a280a960aa01001100410061009101010121015"
    "1018102110241040104210451048105110541060106a10811084109011001102110511081111111411201141114411501180119411961201"
    "1204120612101240126014001402140514081411141414201441144414491450146414801501150415101540160016141649180118041810"
    "18121840185418861900190519661a511aa92000200220052008200a201120142020204120442050208020a0210121042110214021482165"
    "22002222228022a82401240424102429244025002541255225992601261a26a628002808280a28202855288828a2296829902a082a202a82"
    "2a882a8a40014004400640094010401240154018402140244040404240454048404a40514054406040654081408440904100410241054108"
    "4111411441204141414441504180418541a24201420442104212422942404400440244054408441144144419442044414444445044804494"
    "45014504451045244540459a4600460a464446504801480448104840484548544862490049114944495049694a0450005002500550085011"
    "50145020502850415044505050805101510451105115514051425200524452aa540154045410542154405460548154a15500550855805588"
    "5621566856a158005814584158505899591a594059425a85600160046010604060546062608660a961006224624a62926400641665106540"
    "654565a46801686a69256a066a546a628000800280058008801180148020802a8041804480508080808280a880aa81018104810681108140"
    "81518159820082208280828282a082a8840184048410841284158440846084898500854485a58618866a880088088825885a8880888288a8"
    "89068a228a808a888a968aa890019004901090409056908491009122916492569289940094059444945094589529959095929641985198a6"
    "99499a159a60a000a002a008a00aa020a02aa0a0a151a159a1a6a200a202a208a22aa280a2a0a440a495a665a698a80aa820a822a828a8a0"
    "a8a8a904a984a986aa28aa2aaa91aaaa"
)
KVALUES = (0, 1, 2, 3, 4, 6, 8, 12, 0, -1, -2, -3, -4, -6, -8, -12)


# ------------------------------------------------------------------- cases
def _mm(name, fmt, n, k, m, layers):
    return {"name": name, "kind": "mul_mat", "fmt": fmt, "n": n, "k": k, "m": m, "layers": layers}


def listed():
    return [
        # one token through two small attention projections: latency and launches
        _mm("decode_small", "iq2_xxs", 4096, 4096, 1, 2),
        # one token through the FFN up projections of eight layers (the benchmark's headline shape)
        _mm("decode_up", "q4_k", 11008, 4096, 1, 8),
        # one token through FFN down projections, kept in six bits: 43 superblocks a row
        _mm("decode_down", "q6_k", 4096, 11008, 1, 8),
        # eight sequences decoded together
        _mm("batch_decode", "q4_k", 11008, 4096, 8, 4),
        # a short prompt, odd token and row counts
        _mm("prefill_short", "q5_k", 4101, 4096, 37, 4),
        # a prompt chunk of 512 tokens: the benchmark's Q4_K and MXFP4 prefill
        _mm("prefill", "q4_k", 4096, 4096, 512, 2),
        _mm("prefill_mxfp4", "mxfp4", 4096, 4096, 512, 2),
        # the same chunk through a six-bit down projection (odd superblock count)
        _mm("prefill_down", "q6_k", 4096, 11008, 512, 1),
        # a long prompt through an up projection: the largest product
        _mm("prefill_long", "q4_0", 11008, 4096, 2048, 1),
        # mixture of experts, top 2 of 8: a prompt chunk, and four sequences decoded together
        {"name": "moe_prefill", "kind": "mul_mat_id", "fmt": "q4_k", "n": 14336, "k": 4096, "m": 512,
         "experts": 8, "used": 2, "layers": 1},
        {"name": "moe_decode", "kind": "mul_mat_id", "fmt": "mxfp4", "n": 14336, "k": 4096, "m": 4,
         "experts": 8, "used": 2, "layers": 1},
        # a weight matrix to fp32 (for a dense library product)
        {"name": "dequant", "kind": "dequantize", "fmt": "q4_k", "n": 11008, "k": 4096, "layers": 1},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """Another case of the same ranges: any format, matrices of 512 .. 14336
    rows (odd ones among them) and 1024 .. 14336 columns, 1 .. 2048 tokens."""
    fmt = rng.choice(sorted(FORMATS))
    kind = rng.choice(["decode", "decode", "batch", "batch", "short", "short", "prefill", "prefill", "prefill",
                       "moe_decode", "moe_prefill", "dequantize"])
    k = 256 * max(4, min(56, round(_log_uniform(rng, 1024, 14336) / 256)))
    n = _log_uniform(rng, 512, 14336)
    if rng.random() < 0.5:
        n = max(512, n // 64 * 64)
    if kind == "dequantize":
        return {"kind": "dequantize", "fmt": fmt, "n": n, "k": k, "layers": 1}
    if kind.startswith("moe"):
        experts = rng.choice([4, 8, 16])
        while n * k * experts > 8 * 14336 * 4096:
            n //= 2
        m = rng.randint(1, 8) if kind == "moe_decode" else _log_uniform(rng, 128, 512)
        return {"kind": "mul_mat_id", "fmt": fmt, "n": n, "k": k, "m": m, "experts": experts, "used": 2, "layers": 1}
    m = {"decode": (1, 1), "batch": (2, 15), "short": (16, 64), "prefill": (65, 2048)}[kind]
    m = _log_uniform(rng, *m)
    if kind == "prefill":
        # at most the work of 512 tokens through a 4096 x 11008 projection
        m = max(65, min(m, 512 * 4096 * 11008 // (n * k)))
    return _mm_unnamed(fmt, n, k, m, 1 if kind == "prefill" else 4)


def _mm_unnamed(fmt, n, k, m, layers):
    c = _mm("", fmt, n, k, m, layers)
    del c["name"]
    return c


# ------------------------------------------------------------------ inputs
def _weights(fmt, rows, k, gen):
    """rows x k weight records on the GPU, uint8 (rows, row bytes)."""
    elems, nbytes, _, _ = FORMATS[fmt]
    nrec = k // elems
    rec = torch.randint(0, 256, (rows, nrec, nbytes), dtype=torch.uint8, device="cuda", generator=gen)

    def f16(lo, hi, at):
        v = torch.rand((rows, nrec, 1), device="cuda", generator=gen) * (hi - lo) + lo
        rec[:, :, at:at + 2] = v.half().view(torch.uint8)

    if fmt in ("q4_0", "iq2_xxs", "iq2_xs"):
        f16(2e-3, 8e-3, 0)
    elif fmt == "q4_1":
        f16(4e-3, 8e-3, 0)
        f16(-6e-2, -3e-2, 2)
    elif fmt in ("q4_k", "q5_k"):
        f16(1e-4, 3e-4, 0)
        f16(1e-4, 3e-4, 2)
    elif fmt == "q6_k":
        f16(2e-5, 6e-5, 208)
    elif fmt == "mxfp4":
        rec[:, :, 0] = torch.randint(118, 123, (rows, nrec), dtype=torch.uint8, device="cuda", generator=gen)
    else:
        rec[:, :, 0:4] = torch.randint(0x20, 0x40, (rows, nrec, 4), dtype=torch.uint8, device="cuda", generator=gen)
    return rec.view(rows, nrec * nbytes)


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 2654435761 % (1 << 63))


def _inputs(case, seed):
    """Per layer: the weights (experts stacked), and the activations and expert choices of a product."""
    gen = _generator(seed)
    out = []
    for _ in range(case["layers"]):
        w = _weights(case["fmt"], case.get("experts", 1) * case["n"], case["k"], gen)
        x = ids = None
        if case["kind"] != "dequantize":
            x = torch.randn((case["m"], case["k"]), device="cuda", generator=gen)
        if case["kind"] == "mul_mat_id":
            score = torch.rand((case["m"], case["experts"]), device="cuda", generator=gen)
            ids = score.topk(case["used"], dim=1).indices.to(torch.int32).contiguous()
        out.append((w, x, ids))
    return out


def _iq2_grid(fmt):
    code = "".join(IQ2XXS_GRID if fmt == "iq2_xxs" else IQ2XS_GRID)
    v = np.array([int(code[i:i + 4], 16) for i in range(0, len(code), 4)])
    return np.array([8, 25, 43], np.int8)[(v[:, None] >> (2 * np.arange(8))) & 3]


def _signs():
    i = np.arange(128)
    parity = sum((i >> b) & 1 for b in range(7)) & 1
    s = i | (parity << 7)
    return np.where((s[:, None] >> np.arange(8)) & 1, -1, 1).astype(np.int8)


def _e8m0_half():
    e = np.arange(256, dtype=np.uint32)
    return np.where(e < 2, np.uint32(0x00200000) << e, (e - 1) << 23).astype(np.uint32).view(np.float32)


def _ue4m3_half():
    c = np.arange(256)
    ex, mant = (c >> 3) & 15, c & 7
    v = np.where(ex == 0, mant / 1024.0, (8 + mant) * np.ldexp(1.0, ex.astype(np.int32) - 11)).astype(np.float32)
    v[[0, 0x7F]] = 0.0
    return v


def _tables(fmt):
    """The table arguments of row_dequantize, as the kernel takes them."""
    if fmt in ("iq2_xxs", "iq2_xs"):
        return _iq2_grid(fmt), _signs()
    if fmt == "mxfp4":
        return np.array(KVALUES, np.int8), _e8m0_half()
    if fmt == "nvfp4":
        return np.array(KVALUES, np.int8), _ue4m3_half()
    return ()


def prepare(case, seed):
    n, k = case["n"], case["k"]
    _, _, type_id, act = FORMATS[case["fmt"]]
    calls, outs, keep = [], [], []
    if case["kind"] == "dequantize":
        fn = compile_kernel(getattr(kernels, "row_dequantize_" + case["fmt"]))
        fn.synchronize = False
        encoding = {a["name"]: a["encoding"] for a in fn.metadata["arguments"]}
        tables = [torch.from_numpy(t.reshape(-1)).cuda() for t in _tables(case["fmt"])]
        for w, _, _ in _inputs(case, seed):
            y = torch.empty(n * k, device="cuda")
            args = [Buffer(w.view(-1), shape=(n * k,), encoding=encoding["W"]), *tables, y]
            calls.append(args)
            outs.append(y)
            keep += [w, tables]
        return {"kind": case["kind"], "fn": fn, "calls": calls, "outs": outs, "keep": keep}
    m = case["m"]
    for w, x, ids in _inputs(case, seed):
        if case["kind"] == "mul_mat":
            y = torch.empty((m, n), device="cuda")
            s0 = ggml.tensor(type_id, [k, n], w.data_ptr())
            s1 = ggml.tensor(ggml.F32, [k, m], x.data_ptr())
            dst = ggml.tensor(ggml.F32, [n, m], y.data_ptr())
            size = ggml.mul_mat_work_size(s0, s1)
            work = torch.zeros(size, dtype=torch.uint8, device="cuda")
            calls.append((s0, s1, dst, work.data_ptr(), size))
        else:
            used = case["used"]
            y = torch.empty((m, used, n), device="cuda")
            s0 = ggml.tensor(type_id, [k, n, case["experts"]], w.data_ptr())
            s1 = ggml.tensor(ggml.F32, [k, 1, m], x.data_ptr())
            sid = ggml.tensor(ggml.I32, [used, m], ids.data_ptr())
            dst = ggml.tensor(ggml.F32, [n, used, m], y.data_ptr())
            size = ggml.mul_mat_id_work_size(s0, s1, sid)
            work = torch.zeros(size, dtype=torch.uint8, device="cuda")
            calls.append((s0, s1, sid, dst, work.data_ptr(), size))
        outs.append(y)
        keep += [w, x, ids, work]
    return {"kind": case["kind"], "calls": calls, "outs": outs, "keep": keep}


def run(state):
    _lib.set_stream(torch.cuda.current_stream().cuda_stream)
    if state["kind"] == "mul_mat":
        for call in state["calls"]:
            ggml.mul_mat(*call)
    elif state["kind"] == "mul_mat_id":
        for call in state["calls"]:
            ggml.mul_mat_id(*call)
    else:
        for call in state["calls"]:
            state["fn"](*call)
    return state["outs"]


# ------------------------------------------------------------- work, limits
def work(case):
    n, k, layers = case["n"], case["k"], case["layers"]
    elems, nbytes, _, _ = FORMATS[case["fmt"]]
    matrix = n * (k // elems) * nbytes
    if case["kind"] == "dequantize":
        return {"bytes": layers * (matrix + 4 * n * k), "flops": 0}
    m = case["m"]
    if case["kind"] == "mul_mat":
        return {"bytes": layers * (matrix + 4 * m * k + 4 * m * n), "flops": layers * 2 * m * n * k}
    e, u = case["experts"], case["used"]
    touched = e * (1 - (1 - u / e) ** m)  # experts that some token chose, on average
    return {"bytes": layers * (touched * matrix + 4 * m * k + 4 * m * u * n), "flops": layers * 2 * m * u * n * k}


def tolerance(case):
    if case["kind"] == "dequantize":
        return "exact"  # every value one rounded expression of the record
    # exact integer partial sums, scaled and added in fp32: 0.6e-7 .. 1.5e-7 off 64 bits,
    # twice that between two orders of the sum
    return {"rel": 1e-6, "max": 2e-5}


# ---------------------------------------------------------------- 64 bits
def _f16(rec, at):
    return rec[..., at:at + 2].contiguous().view(torch.float16)[..., 0].double()


def _u16(rec, lo, count):
    b = rec[..., lo:lo + 2 * count].to(torch.int64).unflatten(-1, (count, 2))
    return b[..., 0] | (b[..., 1] << 8)


def _nibbles(b):
    """Low nibbles of a run of bytes, then the high ones."""
    return torch.cat([b & 15, b >> 4], -1)


def _scale_min(rec):
    """The eight 6-bit scales and mins of a Q4_K / Q5_K record."""
    s = rec[..., 4:16].to(torch.int64)
    sc = torch.cat([s[..., 0:4] & 63, (s[..., 8:12] & 15) | ((s[..., 0:4] >> 6) << 4)], -1)
    mn = torch.cat([s[..., 4:8] & 63, (s[..., 8:12] >> 4) | ((s[..., 4:8] >> 6) << 4)], -1)
    return sc.double(), mn.double()


def _dequantize(fmt, w, k):
    """(rows, k) weights in float64, and the (rows, k / 32) block minimum of Q4_1 (else None)."""
    elems, nbytes, _, _ = FORMATS[fmt]
    rows = w.shape[0]
    rec = w.view(rows, k // elems, nbytes)
    low = None
    if fmt in ("q4_0", "q4_1"):
        q = _nibbles(rec[..., nbytes - 16:]).double()
        v = (q - 8 if fmt == "q4_0" else q) * _f16(rec, 0)[..., None]
        low = _f16(rec, 2) if fmt == "q4_1" else None
    elif fmt == "mxfp4":
        d = torch.from_numpy(_e8m0_half().astype(np.float64)).to(w.device)
        kv = torch.tensor(KVALUES, dtype=torch.float64, device=w.device)
        v = kv[_nibbles(rec[..., 1:]).long()] * d[rec[..., 0].long()][..., None]
    elif fmt == "nvfp4":
        d = torch.from_numpy(_ue4m3_half().astype(np.float64)).to(w.device)
        kv = torch.tensor(KVALUES, dtype=torch.float64, device=w.device)
        q = _nibbles(rec[..., 4:].unflatten(-1, (4, 8)))
        v = kv[q.long()] * d[rec[..., :4].long()][..., None]
    elif fmt in ("q4_k", "q5_k"):
        sc, mn = _scale_min(rec)
        q = _nibbles(rec[..., nbytes - 128:].unflatten(-1, (4, 32))).unflatten(-1, (2, 32)).flatten(-3, -2).long()
        if fmt == "q5_k":
            bit = torch.arange(8, device=w.device)[:, None]
            q = q + (((rec[..., None, 16:48].long() >> bit) & 1) << 4)
        v = (_f16(rec, 0)[..., None] * sc)[..., None] * q - (_f16(rec, 2)[..., None] * mn)[..., None]
    elif fmt == "q6_k":
        ql = rec[..., :128].long().unflatten(-1, (2, 2, 32))
        qh = rec[..., 128:192].long().unflatten(-1, (2, 1, 32))
        q4 = torch.cat([ql & 15, ql >> 4], -2)
        q = (q4 | (((qh >> (2 * torch.arange(4, device=w.device)[:, None])) & 3) << 4)) - 32
        sc = rec[..., 192:208].contiguous().view(torch.int8).double()
        v = q.flatten(-3).unflatten(-1, (16, 16)) * (_f16(rec, 208)[..., None] * sc)[..., None]
    else:
        grid = torch.from_numpy(_iq2_grid(fmt).astype(np.float64)).to(w.device)
        sign = torch.from_numpy(_signs().astype(np.float64)).to(w.device)
        if fmt == "iq2_xxs":
            b = rec[..., 2:].long().unflatten(-1, (8, 8))
            meta = b[..., 4] | (b[..., 5] << 8) | (b[..., 6] << 16) | (b[..., 7] << 24)
            row = b[..., :4]
            sgn = (meta[..., None] >> (7 * torch.arange(4, device=w.device))) & 127
            sc = (0.5 + (meta >> 28).double())[..., None].expand(*row.shape)
        else:
            q = _u16(rec, 2, 32).unflatten(-1, (8, 4))
            row, sgn = q & 511, q >> 9
            s = rec[..., 66:74].long()
            sc = torch.stack([s & 15, s & 15, s >> 4, s >> 4], -1).double() + 0.5
        d = (_f16(rec, 0)[..., None, None] * sc * 0.25)[..., None]
        v = d * grid[row] * sign[sgn]
    return v.reshape(rows, k), low


def _activation(fmt, x):
    """x (m, k) as the activation format keeps it, in float64, and Q8_1's block sums (else None)."""
    act = FORMATS[fmt][3]
    x = x.cpu().numpy()
    m, k = x.shape
    b = x.reshape(m, -1, ACT[act][0])
    sums = None
    with np.errstate(divide="ignore", invalid="ignore"):
        if act == "q8_k":
            at = np.abs(b).argmax(-1)[..., None]
            top = np.take_along_axis(b, at, -1)
            inv = np.where(top != 0, np.float32(-127) / top, np.float32(0)).astype(np.float32)
            q = np.minimum(np.rint(inv * b), 127)
            d = np.where(inv != 0, np.float32(1) / inv, np.float32(0)).astype(np.float32)
        else:
            d = (np.abs(b).max(-1, keepdims=True) / np.float32(127)).astype(np.float32)
            inv = np.where(d != 0, np.float32(1) / d, np.float32(0)).astype(np.float32)
            t = (b * inv).astype(np.float64)
            q = np.trunc(t + np.copysign(0.5, t))
            if act == "q8_1":
                sums = (q.sum(-1).astype(np.float32) * d[..., 0]).astype(np.float16).astype(np.float64)
            d = d.astype(np.float16)
    xq = torch.from_numpy((q * d.astype(np.float64)).reshape(m, k))
    return xq, None if sums is None else torch.from_numpy(sums)


def _product(fmt, w, x, k):
    """x . w^T over the quantized operands, in float64."""
    xq, sums = _activation(fmt, x)
    out = []
    for lo in range(0, w.shape[0], 4096):
        wd, low = _dequantize(fmt, w[lo:lo + 4096], k)
        y = xq.to(w.device) @ wd.T
        if low is not None:
            y += sums.to(w.device) @ low.T
        out.append(y)
    return torch.cat(out, 1)


def exact(case, seed):
    n, k, fmt = case["n"], case["k"], case["fmt"]
    outs = []
    for w, x, ids in _inputs(case, seed):
        if case["kind"] == "dequantize":
            y = torch.empty((n, k), dtype=torch.float64, device=w.device)
            for lo in range(0, n, 2048):
                v, low = _dequantize(fmt, w[lo:lo + 2048], k)
                if low is not None:
                    v = v + low.repeat_interleave(32, 1)
                y[lo:lo + 2048] = v
            outs.append(y.view(-1))
        elif case["kind"] == "mul_mat":
            outs.append(_product(fmt, w, x, k))
        else:
            y = torch.empty((case["m"], case["used"], n), dtype=torch.float64, device=w.device)
            for e in range(case["experts"]):
                t, s = (ids == e).nonzero(as_tuple=True)
                if len(t):
                    y[t, s] = _product(fmt, w[e * n:(e + 1) * n], x[t], k)
            outs.append(y)
    return outs
