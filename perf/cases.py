"""The framework's work as cases that can be timed and compared.

Each case is one call, or one training step, that a program built on this
package makes, through the package's own entry points:

  step       SparseLinearFunction forward and backward of both perspectives,
             autograd summing the two weight grads (a training step's FT part)
  eval       SparseLinearFunction forward of both perspectives without grads
  composed   ComposedFeatureTransformer forward and backward
  transform  transform_inputs (the FT and the post-FT epilogue) forward and backward
  q16        QuantizedFeatureTransformer, both perspectives, int16
  encode     encode_batch: positions to index rows
  ranger     the fused Ranger22 update of the FT's tables
  export     int16 quantization and LEB128 codes of an export table

Index rows are either drawn uniformly over the table (`rows` = "uniform", the
benchmark's rows) or encoded from random positions, as the trainer's loader
makes them (`rows` = "encoded").  Every input is made on the GPU from the seed.
"""

import math
import os
import sys

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
for _p in (os.path.join(ROOT, "stockfish-trainer_amd"), ROOT):
    if _p not in sys.path:
        sys.path.insert(0, _p)

from sft_amd import _native  # noqa: E402
from sft_amd.encode import encode_batch, parse_feature_set  # noqa: E402
from sft_amd.quantized import QuantizedFeatureTransformer, quantize_weight_i16  # noqa: E402
from src.model.modules.feature_transformer import SparseLinearFunction  # noqa: E402
from src.model.modules.features import get_feature_cls  # noqa: E402
from src.model.transform_inputs import transform_inputs  # noqa: E402
from src.ranger22.fused_update import get_fused_full_update  # noqa: E402

HALFKA, THREATS = "HalfKAv2_hm^", "Full_Threats+HalfKAv2_hm^"
TABLE_ROWS = {HALFKA: 24576, THREATS: 60720 + 24576}
VIRTUAL_ROWS = 768
PSQT = 8


def listed():
    return [
        # The smallest step: a smoke test's or a debugging run's; launches and host work.
        {"name": "step_tiny", "kind": "step", "B": 300, "N": 517, "K": 32, "lo": 0, "hi": 32, "L": 136},
        # Scoring a handful of positions with a trained table: latency.
        {"name": "eval_b256", "kind": "eval", "B": 256, "N": 23232, "K": 32, "lo": 16, "hi": 32, "L": 1048},
        # The ordinary training batch of one GPU among several.
        {"name": "step_halfka_b16384", "kind": "step", "B": 16384, "N": 23232, "K": 32, "lo": 16, "hi": 32, "L": 1048},
        # The large training batch of the benchmark.
        {"name": "step_halfka_b65536", "kind": "step", "B": 65536, "N": 23232, "K": 32, "lo": 16, "hi": 32, "L": 1048},
        # The largest: the threat feature set, 160 slots over a table beyond any L2.
        {"name": "step_threats_b65536", "kind": "step", "B": 65536, "N": 85296, "K": 160, "lo": 32, "hi": 160, "L": 1048},
        # A small network (L1 = 128) at the large batch.
        {"name": "step_narrow_b65536", "kind": "step", "B": 65536, "N": 23232, "K": 32, "lo": 16, "hi": 32, "L": 136},
        # The module as the trainer builds it, over loader-made rows, at a ragged small batch (an epoch's last one).
        {"name": "composed_halfka_b5003", "kind": "composed", "set": HALFKA, "B": 5003, "L1": 1040},
        # The model's whole input stage over loader-made rows at the large batch.
        {"name": "transform_halfka_b65536", "kind": "transform", "set": HALFKA, "B": 65536, "L1": 1040},
        # Integer inference over the exported table: a large evaluation batch.
        {"name": "q16_b65536", "kind": "q16", "B": 65536, "N": 22528, "K": 32, "lo": 16, "hi": 32, "L": 1040},
        # The loader's encoding of a batch for the threat feature set.
        {"name": "encode_threats_b65536", "kind": "encode", "set": THREATS, "B": 65536},
        # The optimizer step of the HalfKAv2_hm table, its virtual rows and the bias.
        {"name": "ranger_halfka", "kind": "ranger", "rows": 24576, "vrows": 768, "L": 1048},
        # Writing a network: the HalfKAv2_hm export table to int16 and to LEB128 codes.
        {"name": "export_halfka", "kind": "export", "rows": 22528, "L": 1040},
    ]


def _log_int(rng, lo, hi):
    """An integer of [lo, hi], uniform over its logarithm, odd as often as even."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["step", "step", "eval", "composed", "transform", "q16", "encode", "ranger", "export"])
    if kind in ("step", "eval"):
        if rng.random() < 0.25:  # the threat set's slots and table
            K, hi, N = 160, rng.randint(96, 160), rng.randint(60720, 85296)
        else:
            K, hi, N = 32, rng.randint(20, 32), rng.randint(704, 24576)
        return {"kind": kind, "B": _log_int(rng, 16, 60000), "N": N, "K": K, "lo": rng.randint(0, hi), "hi": hi,
                "L": 8 * rng.randint(17, 131)}
    if kind in ("composed", "transform"):
        return {"kind": kind, "set": HALFKA if rng.random() < 0.7 else THREATS, "B": _log_int(rng, 64, 50000),
                "L1": 8 * rng.randint(32, 130)}
    if kind == "q16":
        return {"kind": kind, "B": _log_int(rng, 16, 65536), "N": rng.randint(704, 22528), "K": 32,
                "lo": rng.randint(0, 20), "hi": rng.randint(20, 32), "L": 8 * rng.randint(64, 130)}
    if kind == "encode":
        return {"kind": kind, "set": rng.choice([HALFKA, THREATS]), "B": _log_int(rng, 64, 65536)}
    if kind == "ranger":
        return {"kind": kind, "rows": _log_int(rng, 768, 60720), "vrows": 768, "L": 8 * rng.randint(17, 131)}
    return {"kind": kind, "rows": _log_int(rng, 704, 60720), "L": 8 * rng.randint(16, 130)}


# ------------------------------------------------------------------ inputs ----
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed & 0x7FFFFFFF)


def _randn(g, *shape, scale=1.0):
    return torch.randn(*shape, generator=g, device="cuda").mul_(scale)


def _uniform_rows(g, B, N, K, lo, hi):
    """int32 [B, K]: per row U{lo..hi} distinct features, ascending, then -1."""
    spread = torch.rand(B, hi, generator=g, device="cuda", dtype=torch.float64).mul_(N - hi + 1).long()
    vals = spread.sort(dim=1).values + torch.arange(hi, device="cuda")
    count = torch.randint(lo, hi + 1, (B, 1), generator=g, device="cuda")
    order = torch.rand(B, hi, generator=g, device="cuda").argsort(dim=1).argsort(dim=1)
    vals = torch.where(order < count, vals, N).sort(dim=1).values
    idx = torch.full((B, K), -1, dtype=torch.int32, device="cuda")
    idx[:, :hi] = torch.where(vals < N, vals, -1).int()
    return idx


def _positions(g, B):
    """uint8 boards [B, 64] and sides to move [B]: both kings and up to 15 more
    pieces a side on distinct random squares (no pawns on the back ranks)."""
    squares = torch.rand(B, 64, generator=g, device="cuda").argsort(dim=1)[:, :32]
    # up to 8 pawns, then knights, bishops, rooks and a queen or two
    army = torch.tensor([0, 0, 1, 2, 3, 0, 0, 4, 0, 3, 0, 2, 0, 1, 0], device="cuda")
    types = torch.cat([torch.tensor([5, 5], device="cuda"), army, army]).expand(B, 32)
    colors = torch.tensor([0, 1] + [0] * 15 + [1] * 15, device="cuda")
    left = torch.randint(0, 16, (B, 2), generator=g, device="cuda")
    slot = torch.arange(15, device="cuda")
    on = torch.cat([torch.ones(B, 2, dtype=torch.bool, device="cuda"), slot < left[:, :1], slot < left[:, 1:]], dim=1)
    back = (squares < 8) | (squares >= 56)
    types = torch.where((types == 0) & back, 1, types)
    boards = torch.full((B, 64), 255, dtype=torch.uint8, device="cuda")
    boards.scatter_(1, squares, torch.where(on, 2 * types + colors, 255).to(torch.uint8))
    stm = torch.randint(0, 2, (B,), generator=g, device="cuda").to(torch.uint8)
    return boards, stm


def _module(c, g):
    """The composed module with random tables as training meets them (virtual rows included)."""
    m = get_feature_cls(c["set"])(c["L1"] + PSQT).cuda()
    with torch.no_grad():
        for p in m.parameters():
            # pre-activations spread over the clamp's range [0, 1]
            p.copy_(_randn(g, *p.shape, scale=0.05) if p.dim() == 2 else _randn(g, *p.shape, scale=0.1).add_(0.3))
    return m


def prepare(case, seed):
    c, g = case, _gen(seed)
    s = {"kind": c["kind"], "case": c}
    if c["kind"] in ("step", "eval"):
        s["idx"] = [_uniform_rows(g, c["B"], c["N"], c["K"], c["lo"], c["hi"]) for _ in range(2)]
        s["W"] = _randn(g, c["N"], c["L"], scale=0.01)
        sigma = math.sqrt(1.0 / c["N"])
        s["bias"] = torch.rand(c["L"], generator=g, device="cuda").mul_(2 * sigma).sub_(sigma)
        if c["kind"] == "step":
            s["W"].requires_grad_(True)
            s["bias"].requires_grad_(True)
            s["grad"] = [_randn(g, c["B"], c["L"]) for _ in range(2)]
    elif c["kind"] in ("composed", "transform"):
        s["module"] = _module(c, g)
        s["params"] = list(s["module"].parameters())
        s["batch"] = encode_batch(*_positions(g, c["B"]), c["set"])
        if c["kind"] == "composed":
            s["grad"] = [_randn(g, c["B"], c["L1"] + PSQT) for _ in range(2)]
        else:
            s["grad"] = [_randn(g, c["B"], c["L1"]), _randn(g, c["B"], 1)]
    elif c["kind"] == "q16":
        s["idx"] = [_uniform_rows(g, c["B"], c["N"], c["K"], c["lo"], c["hi"]) for _ in range(2)]
        wq = quantize_weight_i16(_randn(g, c["N"], c["L"], scale=0.1), 127.0)
        bq = quantize_weight_i16(_randn(g, c["L"], scale=0.3), 127.0)
        pq = torch.randint(-2000, 2000, (c["N"], PSQT), generator=g, device="cuda", dtype=torch.int32)
        s["tables"] = (wq, bq, pq)
        s["ft"] = QuantizedFeatureTransformer(wq, bq, pq)
    elif c["kind"] == "encode":
        s["boards"], s["stm"] = _positions(g, c["B"])
    elif c["kind"] == "ranger":
        s["update"] = {n: get_fused_full_update(n) for n in (1, 2)}
        # a step's scalars, as the optimizer computes them (lr, 1/sqrt(bias correction), eps, ...)
        s["scalars"] = torch.tensor([8e-4, 1.02, 1e-8, 2e-5, 0.62, 2.0, -1.0, 8e-4, 0.999, 0.001, 0.81, 0.19],
                                    device="cuda")
        s["tensors"] = []
        for shape in ((c["rows"], c["L"]), (c["vrows"], c["L"]), (c["L"],)):
            p, grad = _randn(g, *shape, scale=0.05), _randn(g, *shape, scale=1e-3)
            var = _randn(g, *shape, scale=1e-3).square_().add_(1e-8)
            s["tensors"].append((p, grad, var, _randn(g, *shape, scale=1e-3), _randn(g, *shape, scale=1e-3)))
    else:
        # normal weights (int16 codes of one and two bytes): their quantiles in random order, so that the
        # codes of every seed take as many bytes
        n = c["rows"] * c["L"]
        at = torch.randperm(n, generator=g, device="cuda").double().add_(0.5).div_(n)
        s["W"] = torch.erfinv(at.mul_(2).sub_(1)).mul_(0.1 * math.sqrt(2.0)).float().view(c["rows"], c["L"])
    return s


# --------------------------------------------------------------------- run ----
def run(state):
    s = state
    kind = s["kind"]
    if kind == "step":
        outs = [SparseLinearFunction.apply(i, s["W"], s["bias"]) for i in s["idx"]]
        dW, db = torch.autograd.grad(outs, [s["W"], s["bias"]], s["grad"])
        return {"out": [o.detach() for o in outs], "dW": dW, "db": db}
    if kind == "eval":
        with torch.no_grad():
            return [SparseLinearFunction.apply(i, s["W"], s["bias"]) for i in s["idx"]]
    if kind == "composed":
        outs = s["module"](s["batch"]["white"], s["batch"]["black"])
        grads = torch.autograd.grad(outs, s["params"], s["grad"])
        return {"out": [o.detach() for o in outs], "grads": list(grads)}
    if kind == "transform":
        b = s["batch"]
        outs = transform_inputs(s["module"], s["case"]["L1"], b["us"], b["white"], b["black"], b["psqt_indices"])
        grads = torch.autograd.grad(outs, s["params"], s["grad"])
        return {"out": [o.detach() for o in outs], "grads": list(grads)}
    if kind == "q16":
        return s["ft"](*s["idx"])
    if kind == "encode":
        return encode_batch(s["boards"], s["stm"], s["case"]["set"])
    if kind == "ranger":
        for p, grad, var, cur, prev in s["tensors"]:
            s["update"][p.dim()](p, grad, var, cur, prev, s["scalars"])
        return [(p, var, cur) for p, _, var, cur, _ in s["tensors"]]
    q = quantize_weight_i16(s["W"], 255.0)
    return {"q": q, "codes": _native.leb128_encode(q.view(-1))}


# -------------------------------------------------------------------- work ----
def work(case):
    """Each input read once, each output written once; one add per gathered or scattered element."""
    c = case
    kind = c["kind"]
    if kind in ("step", "eval"):
        n = (c["lo"] + c["hi"]) / 2
        slots = 2 * c["B"] * n
        touched = c["N"] * -math.expm1(-slots / c["N"])  # table rows that some position reads
        nbytes = 8 * c["B"] * c["K"] + 4 * touched * c["L"] + 8 * c["B"] * c["L"]
        if kind == "eval":
            return {"bytes": nbytes, "flops": slots * c["L"]}
        return {"bytes": nbytes + 8 * c["B"] * c["L"] + 4 * c["N"] * c["L"], "flops": 2 * slots * c["L"]}
    if kind in ("composed", "transform"):
        L, B, K = c["L1"] + PSQT, c["B"], parse_feature_set(c["set"])[1]
        table = 4 * L * (TABLE_ROWS[c["set"]] + VIRTUAL_ROWS)
        outs = 8 * B * L if kind == "composed" else 4 * B * (c["L1"] + 1)
        n = 17 if c["set"] == HALFKA else 17 + 30
        return {"bytes": 8 * B * K + 2 * table + 2 * outs, "flops": 4 * B * n * L}
    if kind == "q16":
        n = (c["lo"] + c["hi"]) / 2
        touched = c["N"] * -math.expm1(-2 * c["B"] * n / c["N"])
        row = 2 * c["L"] + 4 * PSQT
        return {"bytes": 8 * c["B"] * c["K"] + touched * row + 2 * c["B"] * row, "flops": 2 * c["B"] * n * (c["L"] + PSQT)}
    if kind == "encode":
        return {"bytes": c["B"] * (65 + 8 * parse_feature_set(c["set"])[1] + 20), "flops": 0}
    if kind == "ranger":
        n = (c["rows"] + c["vrows"] + 1) * c["L"]
        return {"bytes": 32 * n, "flops": 20 * n}
    n = c["rows"] * c["L"]
    return {"bytes": n * (4 + 2 + 1.2), "flops": n}


def tolerance(case):
    kind = case["kind"]
    if kind in ("q16", "encode", "export"):
        return "exact"
    if kind == "ranger":
        return {"rel": 2e-7}  # about 4e-8 from 64 bits
    if kind == "transform":
        # a pre-activation at a bound of the clamp may round to its other side, which turns its whole
        # grad on or off: about 1e-4 from 64 bits
        return {"rel": 4e-4}
    return {"rel": 8e-7}  # about 2e-7 from 64 bits


# ------------------------------------------------------------------- exact ----
def _gather64(idx, table, bias):
    """bias + sum of the rows that idx selects, in 64 bits."""
    B, K = idx.shape
    L = table.shape[1]
    padded = torch.cat([table, table.new_zeros(1, L)])
    at = torch.where(idx < 0, table.shape[0], idx).long()
    out = torch.empty(B, L, dtype=table.dtype, device=table.device)
    step = max(1, (1 << 28) // (K * L))
    for b in range(0, B, step):
        out[b:b + step] = padded[at[b:b + step]].sum(dim=1) + bias
    return out


def _scatter64(idx, grad, rows):
    """Per table row, the sum of the grad rows of the positions that select it, in 64 bits."""
    B, K = idx.shape
    L = grad.shape[1]
    out = torch.zeros(rows + 1, L, dtype=torch.float64, device=grad.device)
    at = torch.where(idx < 0, rows, idx).long()
    step = max(1, (1 << 27) // (K * L))
    for b in range(0, B, step):
        rows_b = grad[b:b + step].double().repeat_interleave(K, dim=0)
        out.index_add_(0, at[b:b + step].reshape(-1), rows_b)
    return out[:rows]


def _merged64(module):
    """The merged table in 64 bits and how its grad splits over the parameters."""
    return torch.cat([w.detach().double() if v is None else
                      w.detach().double() + v.detach().double().repeat(w.shape[0] // v.shape[0], 1)
                      for w, v in (f.table_blocks() for f in module.features)])


def _param_grads64(module, dW, db):
    """Grads of the module's parameters from the merged table's and the bias's."""
    grads, start = {id(module.bias): db}, 0
    for w, v in (f.table_blocks() for f in module.features):
        part = dW[start:start + w.shape[0]]
        grads[id(w)] = part
        if v is not None:
            grads[id(v)] = part.view(-1, v.shape[0], part.shape[1]).sum(dim=0)
        start += w.shape[0]
    return [grads[id(p)] for p in module.parameters()]


def exact(case, seed):
    c = case
    s = prepare(c, seed)
    kind = c["kind"]
    if kind in ("step", "eval"):
        W, bias = s["W"].detach().double(), s["bias"].detach().double()
        outs = [_gather64(i, W, bias) for i in s["idx"]]
        if kind == "eval":
            return outs
        dW = sum(_scatter64(i, d, c["N"]) for i, d in zip(s["idx"], s["grad"]))
        return {"out": outs, "dW": dW, "db": sum(d.double().sum(dim=0) for d in s["grad"])}
    if kind in ("composed", "transform"):
        m, b = s["module"], s["batch"]
        W, bias = _merged64(m), m.bias.detach().double()
        pre = [_gather64(i, W, bias) for i in (b["white"], b["black"])]
        if kind == "composed":
            outs, grads = pre, [d.double() for d in s["grad"]]
        else:
            leaves = [p.requires_grad_(True) for p in pre]
            outs = _epilogue64(leaves, c["L1"], b["us"].double(), b["psqt_indices"])
            grads = torch.autograd.grad(outs, leaves, [d.double() for d in s["grad"]])
            outs = [o.detach() for o in outs]
            pre = leaves = None
        dW = sum(_scatter64(i, d, W.shape[0]) for i, d in zip((b["white"], b["black"]), grads))
        return {"out": outs, "grads": _param_grads64(m, dW, sum(d.sum(dim=0) for d in grads))}
    if kind == "ranger":
        return [_ranger64([t.double() for t in ts], s["scalars"].double()) for ts in s["tensors"]]
    return None  # whole numbers and bytes


def _epilogue64(pre, L1, us, psqt):
    half = L1 // 2
    prod = [p[:, :half].clamp(0, 1) * p[:, half:L1].clamp(0, 1) for p in pre]
    side = us.bool()
    l0 = torch.cat([torch.where(side, prod[0], prod[1]), torch.where(side, prod[1], prod[0])], dim=1) * (127 / 128)
    k = psqt.unsqueeze(1)
    return [l0, (pre[0][:, L1:].gather(1, k) - pre[1][:, L1:].gather(1, k)) * (us - 0.5)]


def _ranger64(tensors, scalars):
    p, g, var, cur, prev = tensors
    lr, bc2, eps, nl, noise, pa, pb, size, b2, ob2, b1, ob1 = scalars
    var = var * b2 + g * g * ob2
    cur = cur * b1 + g * ob1
    norm = p.norm(dim=1, keepdim=True) if p.dim() == 2 else p.norm()
    fix = nl * (1 - 1 / (norm + eps))
    p = p * (1 - lr * fix) - (cur * pa + prev * pb) * noise / (var.sqrt() * bc2 + eps) * size
    return p, var, cur
