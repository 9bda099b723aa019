"""Performance cases of the attention path: what a program that uses this framework has it do.

Five kinds of call, each through the public Python entry points with the plan, planes, scratch
tables and output buffers that a program keeps from one layer to the next:

* ``text``    one gated full-attention layer over packed causal records, bf16 qkv rows
              (``TextAttention.forward``); with ``fp32`` the same layer on f32 rows, the rerun of a
              record whose f16 operands overflowed;
* ``prefix``  the same layer where new tokens attend to keys that a prefix-cache entry holds;
* ``layer``   the QKV projection with the K/V prologue in its epilogue, then the attention core
              (``TextAttention.project`` and ``forward(stage="core")``);
* ``vision``  the vision tower's bidirectional attention over packed images;
* ``omni``    the Omni decoder's FP32 attention (``OmniAttention.prep`` and ``attention``).

``exact`` restates each in float64 with plain torch.
"""
import ctypes
import math

import numpy as np
import torch

from cleffa_amd import AttnPlan, TextAttention, VisionAttention, vision_positions
from cleffa_amd.omni import OmniAttention, OmniPlan

HD, N_ROT, THETA, EPS = 256, 64, 1e7, 1e-6          # text: head dim, rotary dims, frequency base
VIS_HD, VIS_THETA = 72, 1e4
OMNI_HD, OMNI_THETA = 128, 1e6
DEVICE = "cuda"


def listed():
    """The workloads C1-C4 and S and the Omni benchmark of bench.py, and the calls at the ends
    of the range. ``lens`` are the new tokens of each record, ``cached`` the keys that each
    record's prefix-cache entry already holds."""
    return [
        # one short prompt alone: nothing to fill the GPU with, launches and host work count
        {"name": "text_one_short", "kind": "text", "lens": "37", "nh": 16, "nkv": 4},
        # a full micro-batch of very short prompts (workload S)
        {"name": "text_short_batch", "kind": "text", "lens": "256x16", "nh": 24, "nkv": 4},
        # the ordinary micro-batch: eight requests of mixed length, 4,096 tokens (C1, seed 0)
        {"name": "text_packed", "kind": "text", "lens": "1160,890,730,425,472,136,179,104", "nh": 24, "nkv": 4},
        # one long document (C2)
        {"name": "text_long", "kind": "text", "lens": "16384", "nh": 24, "nkv": 4},
        # four requests that continue a cached prefix by 512 tokens each (C3)
        {"name": "prefix_packed", "kind": "prefix", "lens": "4x512", "cached": "4x2048", "nh": 16, "nkv": 4},
        # a short question on a cached document: prefix-cache requests run alone
        {"name": "prefix_question", "kind": "prefix", "lens": "45", "cached": "4091", "nh": 24, "nkv": 4},
        # four images of 32 x 32 patches (C4)
        {"name": "vision_packed", "kind": "vision", "grids": "4x32:32", "heads": 16},
        # the ordinary micro-batch with every product in FP32
        {"name": "fp32_packed", "kind": "text", "lens": "1160,890,730,425,472,136,179,104", "nh": 24, "nkv": 4, "fp32": True,
         "out": "f32"},
        # the rerun of one record after an overflow
        {"name": "fp32_rerun", "kind": "text", "lens": "425", "nh": 24, "nkv": 4, "fp32": True, "out": "f32"},
        # the Omni decoder on a long recording (bench.py's size)
        {"name": "omni_long", "kind": "omni", "lens": "16344", "nh": 32, "nkv": 4},
        # the QKV projection and the core over the ordinary micro-batch, hidden size 5,120
        {"name": "layer_packed", "kind": "layer", "lens": "1160,890,730,425,472,136,179,104", "nh": 24, "nkv": 4, "hidden": 5120},
        # the same for one short prompt: the projection reads all of its weights for few rows
        {"name": "layer_short", "kind": "layer", "lens": "61", "nh": 24, "nkv": 4, "hidden": 5120},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _split(rng, total, n):
    """n record lengths, mixed, that sum to about total."""
    w = [rng.uniform(0.1, 1.0) for _ in range(n)]
    return [max(1, int(total * x / sum(w))) for x in w]


def _texts(lens):
    return ",".join(str(n) for n in lens)


def draw(rng):
    kind = rng.choice(["text", "text", "text", "prefix", "prefix", "vision", "fp32", "fp32", "omni", "layer"])
    nh, nkv = rng.choice([(16, 4), (24, 4), (24, 4), (32, 4), (8, 2), (16, 8)])
    if kind == "vision":
        c = {"kind": "vision", "heads": 16,
             "grids": ",".join("%d:%d" % (2 * rng.randint(4, 32), 2 * rng.randint(4, 32)) for _ in range(rng.randint(1, 6)))}
        if rng.random() < 0.3:
            c["out"] = "f16"
        return c
    if kind == "omni":
        total = _log(rng, 64, 8192)
        return {"kind": "omni", "nh": rng.choice([32, 16]), "nkv": 4, "lens": _texts(_split(rng, total, rng.choice([1, 1, 2, 5])))}
    if kind == "layer":
        return {"kind": "layer", "nh": nh, "nkv": nkv, "hidden": rng.choice([2560, 4096, 5120]),
                "lens": _texts(_split(rng, _log(rng, 16, 6000), rng.choice([1, 3, 8])))}
    if kind == "prefix":
        n = rng.choice([1, 1, 1, 2, 5])
        new, cached = [_log(rng, 8, 700) for _ in range(n)], [_log(rng, 200, 12000 // n) for _ in range(n)]
        # every record but the last ends at a multiple of 8 keys
        cached = [c if r == n - 1 else c + (-(c + new[r])) % 8 for r, c in enumerate(cached)]
        return {"kind": "prefix", "nh": nh, "nkv": nkv, "lens": _texts(new), "cached": _texts(cached)}
    if kind == "fp32":
        lens = _split(rng, _log(rng, 32, 6000), rng.choice([1, 1, 4, 9]))
        return {"kind": "text", "fp32": True, "nh": nh, "nkv": nkv, "lens": _texts(lens), "out": rng.choice(["f32", "bf16"])}
    lens = _split(rng, _log(rng, 24, 15000), rng.choice([1, 1, 3, 8, 30]))
    c = {"kind": "text", "nh": nh, "nkv": nkv, "lens": _texts(lens)}
    if rng.random() < 0.3:
        c["out"] = rng.choice(["f16", "f32"])
    if rng.random() < 0.2:
        c["plain"] = True          # no norms, rotary or gate
    elif rng.random() < 0.3:
        c["image"] = rng.randint(4, 24)   # an image span of that many merged rows and columns
    return c


# ---- what a case says

def _ints(text):
    """"4x512,7" -> [512, 512, 512, 512, 7]"""
    out = []
    for part in str(text).split(","):
        n, x, v = part.partition("x")
        out += [int(v)] * int(n) if x else [int(n)]
    return out


def _grids(text):
    """"2x32:24" -> [(32, 24), (32, 24)] (rows, columns of patches)"""
    out = []
    for part in text.split(","):
        n, x, v = part.partition("x")
        r, c = (v if x else n).split(":")
        out += [(int(r), int(c))] * (int(n) if x else 1)
    return out


def _cu(lens):
    return np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)


def _positions(case):
    """[T][3] rotary positions (temporal, row, column) of the new tokens."""
    lens = _ints(case["lens"])
    cached = _ints(case["cached"]) if "cached" in case else [0] * len(lens)
    side = case.get("image", 0)
    rows = []
    for n, L in zip(lens, cached):
        p = np.repeat(np.arange(L, L + n)[:, None], 3, axis=1)
        if side and n >= 8 + side * side:   # tokens 8 .. 8 + side^2 are an image's
            y, x = np.divmod(np.arange(side * side), side)
            p[8:8 + side * side] = 8 + np.stack([0 * y, y, x], axis=1)
            p[8 + side * side:] = (8 + side + np.arange(n - 8 - side * side))[:, None]
        rows.append(p)
    return np.concatenate(rows).astype(np.int32)


def _vision_pos(grids):
    """[P][2] (row, column) of each patch, in 2 x 2 merge windows row by row."""
    out = []
    for r, c in grids:
        p = np.arange(r * c)
        win, within = p // 4, p % 4
        out.append(np.stack([win // (c // 2) * 2 + within // 2, win % (c // 2) * 2 + within % 2], axis=1))
    return np.concatenate(out).astype(np.int32)


def _pairs(case):
    """(query, key) pairs under the mask."""
    if case["kind"] == "vision":
        return sum((r * c) ** 2 for r, c in _grids(case["grids"]))
    lens = _ints(case["lens"])
    cached = _ints(case["cached"]) if "cached" in case else [0] * len(lens)
    return sum(n * L + n * (n + 1) // 2 for n, L in zip(lens, cached))


def work(case):
    kind, pairs = case["kind"], _pairs(case)
    if kind == "vision":
        P, E = sum(r * c for r, c in _grids(case["grids"])), case["heads"] * VIS_HD
        return {"bytes": P * 4 * E * 2 + 3 * E * 4 + P * 8, "flops": 4 * VIS_HD * case["heads"] * pairs}
    nh, nkv, T = case["nh"], case["nkv"], sum(_ints(case["lens"]))
    if kind == "omni":
        return {"bytes": T * (2 * nh + 2 * nkv) * OMNI_HD * 4 + T * 12, "flops": 4 * OMNI_HD * nh * pairs}
    row, size = 2 * (nh + nkv) * HD, 4 if case.get("fp32") else 2
    out = {"bf16": 2, "f16": 2, "f32": 4}[case.get("out", "bf16")]
    # plain attention reads no gate columns
    read = row - (nh * HD if case.get("plain") else 0)
    w = {"bytes": T * (read * size + nh * HD * out + 12), "flops": 4 * HD * nh * pairs}
    if kind == "prefix":    # the cached rows are read, the new rows written
        w["bytes"] += (sum(_ints(case["cached"])) + T) * nkv * HD * 2 * 2
    if kind == "layer":     # X and W in, qkv rows out instead of in
        w["bytes"] += (T + row) * case["hidden"] * 2
        w["flops"] += 2 * T * row * case["hidden"]
    return w


def tolerance(case):
    """Four times the errors measured against ``exact`` over the listed cases: relative 2-norm, and the
    largest difference in units of the outputs' root mean square (or the value itself)."""
    if case["kind"] == "omni" or (case.get("fp32") and case.get("out") == "f32"):
        return {"rel": 2e-6, "max": 1.6e-4}     # measured 3.6e-7 to 4.4e-7, largest 3.9e-5
    if case["kind"] == "vision":
        return {"rel": 2e-2, "max": 0.1}        # 5.5e-3, 2.6e-2 (bf16 Q and K)
    if case["kind"] == "layer":
        return {"rel": 1.3e-2, "max": 0.5}      # 3.3e-3, 1.2e-1 (through bf16 qkv rows)
    return {"rel": 9e-3, "max": 0.3}            # 1.8e-3 to 2.4e-3, 7.5e-2


# ---- inputs

def _gen(seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(1000003 * seed + 17)
    return g


def _randn(g, *shape):
    return torch.randn(shape, generator=g, device=DEVICE, dtype=torch.float32)


def _outliers(g, nh, nkv):
    """Per-column scale of the qkv rows: 2% of the query and key channels are 8 times larger."""
    row = 2 * (nh + nkv) * HD
    cols = torch.arange(row, device=DEVICE)
    qk = torch.where(cols < 2 * nh * HD, cols % (2 * HD) < HD, cols < (2 * nh + nkv) * HD)
    pick = torch.rand(row, generator=g, device=DEVICE) < 0.02
    return torch.where(pick & qk, 8.0, 1.0)


def _norm_weight(g, n):
    return 1.0 + 0.1 * _randn(g, n)


def _text_inputs(case, seed):
    nh, nkv, T = case["nh"], case["nkv"], sum(_ints(case["lens"]))
    g, row = _gen(seed), 2 * (nh + nkv) * HD
    x = {"pos3": torch.from_numpy(_positions(case)).to(DEVICE)}
    if case["kind"] == "layer":
        x["X"] = _randn(g, T, case["hidden"]).to(torch.bfloat16)
        x["W"] = (_randn(g, row, case["hidden"]) * (case["hidden"] ** -0.5 * _outliers(g, nh, nkv))[:, None]).to(torch.bfloat16)
    else:
        x["qkv"] = _randn(g, T, row)
        if not case.get("plain"):
            x["qkv"] *= _outliers(g, nh, nkv)
        if not case.get("fp32"):
            x["qkv"] = x["qkv"].to(torch.bfloat16)
    x["q_norm"], x["k_norm"] = (None, None) if case.get("plain") else (_norm_weight(g, HD), _norm_weight(g, HD))
    if case["kind"] == "prefix":   # keys of RMS-normalised rows, times the norm weights; values N(0, 1)
        L = sum(_ints(case["cached"])) + T
        k = _randn(g, nkv, L, HD)
        x["k_cache"] = (k * torch.rsqrt(k.square().mean(-1, keepdim=True)) * x["k_norm"]).to(torch.float16)
        x["v_cache"] = _randn(g, nkv, L, HD).to(torch.bfloat16)
    return x


def _prefix_cu(case):
    return _cu([n + L for n, L in zip(_ints(case["lens"]), _ints(case["cached"]))])


def _cached_rows(case):
    """Mask over the key rows: True where the row was cached before the call."""
    keep = np.zeros(int(_prefix_cu(case)[-1]), bool)
    for k0, L in zip(_prefix_cu(case)[:-1], _ints(case["cached"])):
        keep[k0:k0 + L] = True
    return torch.from_numpy(keep).to(DEVICE)


def _vision_inputs(case, seed):
    g, E, P = _gen(seed), case["heads"] * VIS_HD, sum(r * c for r, c in _grids(case["grids"]))
    return {"qkv": _randn(g, P, 3 * E).to(torch.bfloat16), "bias": 0.1 * _randn(g, 3 * E)}


def _omni_inputs(case, seed):
    g, T = _gen(seed), sum(_ints(case["lens"]))
    return {"qkv": _randn(g, T, (case["nh"] + 2 * case["nkv"]) * OMNI_HD), "q_norm": _norm_weight(g, OMNI_HD),
            "k_norm": _norm_weight(g, OMNI_HD), "pos3": torch.from_numpy(_positions(case)).to(DEVICE)}


def prepare(case, seed):
    kind = case["kind"]
    if kind == "vision":
        grids = _grids(case["grids"])
        cu = _cu([r * c for r, c in grids])
        s = _vision_inputs(case, seed)
        att = VisionAttention(case["heads"], VIS_HD, VIS_THETA, device=DEVICE)
        plan = AttnPlan(cu, causal=False, device=DEVICE)
        s.update(case=case, att=att, plan=plan, pos2=torch.from_numpy(vision_positions(cu, [c for _, c in grids])).to(DEVICE),
                 scratch=att.scratch(plan.T, plan.kvT), out_dtype=case.get("out", "bf16"),
                 ovf=torch.zeros(plan.T, dtype=torch.int32, device=DEVICE))
        s["out"] = torch.empty((plan.T, att.E), dtype=torch.float16 if s["out_dtype"] == "f16" else torch.bfloat16, device=DEVICE)
        return s
    if kind == "omni":
        s = _omni_inputs(case, seed)
        att = OmniAttention(case["nh"], case["nkv"], OMNI_THETA, EPS, device=DEVICE)
        plan = OmniPlan(_cu(_ints(case["lens"])), device=DEVICE)
        s.update(case=case, att=att, plan=plan, planes=att.planes(plan.T), status=torch.zeros(1, dtype=torch.int32, device=DEVICE),
                 out=torch.empty((plan.T, case["nh"] * OMNI_HD), dtype=torch.float32, device=DEVICE))
        return s
    s = _text_inputs(case, seed)
    nh, nkv = case["nh"], case["nkv"]
    att = TextAttention(nh, nkv, HD, 0 if case.get("plain") else N_ROT, EPS, THETA, device=DEVICE)
    plan = AttnPlan(_cu(_ints(case["lens"])), _prefix_cu(case) if kind == "prefix" else None, device=DEVICE)
    k, v = att.planes(plan.kvT, fp32=bool(case.get("fp32")))
    if kind == "prefix":
        kc, vc = s.pop("k_cache"), s.pop("v_cache")
        keep = _cached_rows(case)
        k.zero_()
        v.zero_()
        k[:, :kc.shape[1]] = kc * keep[None, :, None]
        v[:, :, :vc.shape[1]] = vc.transpose(1, 2) * keep
    s.update(case=case, att=att, plan=plan, k_plane=k, vt_plane=v, out_dtype=case.get("out", "bf16"), gate=not case.get("plain"),
             rope_cs=None if case.get("plain") else att.rope_table(plan.T),
             ovf=torch.zeros(plan.T, dtype=torch.int32, device=DEVICE))
    if kind == "layer":
        s["qkv"] = torch.empty((plan.T, att.row), dtype=torch.bfloat16, device=DEVICE)
    s["out"] = torch.empty((plan.T, nh * HD), device=DEVICE,
                           dtype={"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}[s["out_dtype"]])
    return s


def run(s):
    kind, att, plan = s["case"]["kind"], s["att"], s["plan"]
    if kind == "vision":
        att.forward(s["qkv"], s["bias"], s["pos2"], plan, out=s["out"], out_dtype=s["out_dtype"], ovf=s["ovf"], scratch=s["scratch"])
        return {"out": s["out"], "ovf": s["ovf"]}
    if kind == "omni":
        Q, K, V, status = att.prep(s["qkv"], s["q_norm"], s["k_norm"], s["pos3"], planes=s["planes"], status=s["status"])
        att.attention(Q, K, V, plan, out=s["out"])
        return {"out": s["out"], "status": status}
    if kind == "layer":
        att.project(s["X"], s["W"], plan, s["q_norm"], s["k_norm"], s["pos3"], qkv=s["qkv"], k_plane=s["k_plane"],
                    vt_plane=s["vt_plane"], kvT=plan.kvT, ovf=s["ovf"], rope_cs=s["rope_cs"])
    att.forward(s["qkv"], s["q_norm"], s["k_norm"], s["pos3"], plan, out=s["out"], out_dtype=s["out_dtype"], gate=s["gate"],
                k_plane=s["k_plane"], vt_plane=s["vt_plane"], kvT=plan.kvT, ovf=s["ovf"], rope_cs=s["rope_cs"],
                stage="core" if kind == "layer" else "prefill")
    if kind == "layer":
        return {"out": s["out"], "qkv": s["qkv"], "ovf": s["ovf"]}
    if kind == "prefix":
        return {"out": s["out"], "k_plane": s["k_plane"], "vt_plane": s["vt_plane"], "ovf": s["ovf"]}
    return {"out": s["out"], "ovf": s["ovf"]}


# ---- the same in 64 bits

def _inv_freq(theta, n):
    """1 / theta^(2j / n) in f32: the frequency table is an FP32 input of the model."""
    powf = ctypes.CDLL("libm.so.6").powf
    powf.restype, powf.argtypes = ctypes.c_float, [ctypes.c_float, ctypes.c_float]
    f = [np.float32(1) / np.float32(powf(theta, np.float32(2 * j) / np.float32(n))) for j in range(n // 2)]
    return torch.from_numpy(np.array(f, dtype=np.float32)).to(DEVICE)


def _rms(x, w):
    return x if w is None else x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def _turn(x, cos, sin):
    """Rotates dims (i, i + n) of the last axis's first 2n, n = cos.shape[-1]."""
    n = cos.shape[-1]
    a, b = x[..., :n], x[..., n:2 * n]
    return torch.cat([a * cos - b * sin, b * cos + a * sin, x[..., 2 * n:]], -1)


def _attend(q, k, v, scale, cu_q, cu_k, causal):
    """softmax(scale q k^T) v for q [T][nh][d], k, v [Tk][nkv][d], record by record, head by head."""
    group = q.shape[1] // k.shape[1]
    out = torch.empty(q.shape[0], q.shape[1], v.shape[2], dtype=torch.float64, device=q.device)
    for r in range(len(cu_q) - 1):
        q0, q1, k0, k1 = int(cu_q[r]), int(cu_q[r + 1]), int(cu_k[r]), int(cu_k[r + 1])
        for i0 in range(q0, q1, 4096):
            i1 = min(q1, i0 + 4096)
            last = k1 - (q1 - i1) if causal else k1
            if causal:
                qpos = torch.arange(i0, i1, device=q.device) - q0 + (k1 - k0) - (q1 - q0)
                hide = torch.arange(last - k0, device=q.device)[None, :] > qpos[:, None]
            for h in range(q.shape[1]):
                s = (q[i0:i1, h] @ k[k0:last, h // group].T) * scale
                if causal:
                    s.masked_fill_(hide, -math.inf)
                out[i0:i1, h] = torch.softmax(s, -1) @ v[k0:last, h // group]
    return out


def _batched_records(case):
    """Records of one length without cached keys, as (records, length), or None."""
    lens = _ints(case["lens"])
    return (len(lens), lens[0]) if len(set(lens)) == 1 and len(lens) > 16 and "cached" not in case else None


def _exact_text(case, seed):
    x, nh, nkv = _text_inputs(case, seed), case["nh"], case["nkv"]
    qkv = x["X"].double() @ x["W"].double().T if case["kind"] == "layer" else x["qkv"].double()
    T = qkv.shape[0]
    qg = qkv[:, :2 * nh * HD].view(T, nh, 2, HD)
    q, gate = _rms(qg[:, :, 0], x["q_norm"]), qg[:, :, 1]
    k = _rms(qkv[:, 2 * nh * HD:(2 * nh + nkv) * HD].view(T, nkv, HD), x["k_norm"])
    v = qkv[:, (2 * nh + nkv) * HD:].view(T, nkv, HD)
    if not case.get("plain"):   # pair i turns by position axis i % 3; the angle is an FP32 product
        axis = torch.arange(N_ROT // 2, device=DEVICE) % 3
        ang = (x["pos3"][:, axis].float() * _inv_freq(THETA, N_ROT)).double()[:, None]
        q, k = _turn(q, ang.cos(), ang.sin()), _turn(k, ang.cos(), ang.sin())
    cu_q = cu_k = _cu(_ints(case["lens"]))
    planes = {}
    if case["kind"] == "prefix":
        cu_k, keep = _prefix_cu(case), _cached_rows(case)
        kk, vv = x["k_cache"].double().transpose(0, 1).contiguous(), x["v_cache"].double().transpose(0, 1).contiguous()
        kk[~keep], vv[~keep] = k, v
        k, v = kk, vv
        # the planes end with whole 64-key tiles from each record's first key
        rows = max(int(a) + -(-int(b - a) // 64) * 64 for a, b in zip(cu_k[:-1], cu_k[1:]))
        planes = {"k_plane": torch.zeros(nkv, rows, HD, dtype=torch.float64, device=DEVICE),
                  "vt_plane": torch.zeros(nkv, HD, rows, dtype=torch.float64, device=DEVICE)}
        planes["k_plane"][:, :k.shape[0]] = k.transpose(0, 1)
        planes["vt_plane"][:, :, :v.shape[0]] = v.permute(1, 2, 0)
    same = _batched_records(case)
    if same:   # many records of one length at once
        B, n = same
        qh, kh, vh = (t.reshape(B, n, -1, HD).transpose(1, 2) for t in
                      (q, k.repeat_interleave(nh // nkv, 1), v.repeat_interleave(nh // nkv, 1)))
        s = (qh @ kh.transpose(2, 3)) / 16
        s.masked_fill_(torch.ones(n, n, dtype=torch.bool, device=DEVICE).triu(1), -math.inf)
        out = (torch.softmax(s, -1) @ vh).transpose(1, 2).reshape(T, nh, HD)
    else:
        out = _attend(q, k, v, HD ** -0.5, cu_q, cu_k, True)
    if not case.get("plain"):
        out = out * torch.sigmoid(gate)
    res = {"out": out.reshape(T, nh * HD), "ovf": None, **planes}
    if case["kind"] == "layer":
        res["qkv"] = qkv
    return res


def _exact_vision(case, seed):
    x, heads, grids = _vision_inputs(case, seed), case["heads"], _grids(case["grids"])
    cu = _cu([r * c for r, c in grids])
    qkv = (x["qkv"].double() + x["bias"].double()).view(-1, 3, heads, VIS_HD)
    pos = torch.from_numpy(_vision_pos(grids)).to(DEVICE).float()
    f = _inv_freq(VIS_THETA, VIS_HD // 2)   # 18 frequencies: the row turns pairs 0-17, the column 18-35
    ang = torch.cat([pos[:, :1] * f, pos[:, 1:] * f], 1).double()[:, None]
    q, k = _turn(qkv[:, 0], ang.cos(), ang.sin()), _turn(qkv[:, 1], ang.cos(), ang.sin())
    return {"out": _attend(q, k, qkv[:, 2], VIS_HD ** -0.5, cu, cu, False).reshape(-1, heads * VIS_HD), "ovf": None}


def _exact_omni(case, seed):
    x, nh, nkv = _omni_inputs(case, seed), case["nh"], case["nkv"]
    cu = _cu(_ints(case["lens"]))
    qkv = x["qkv"].double().view(-1, nh + 2 * nkv, OMNI_HD)
    pair = torch.arange(OMNI_HD // 2, device=DEVICE)
    freq = OMNI_THETA ** (-2.0 * pair.double() / OMNI_HD)
    ang = (x["pos3"][:, torch.where(pair < 60, pair % 3, 0)].double() * freq)[:, None]
    q = _turn(_rms(qkv[:, :nh], x["q_norm"]), ang.cos(), ang.sin())
    k = _turn(_rms(qkv[:, nh:nh + nkv], x["k_norm"]), ang.cos(), ang.sin())
    return {"out": _attend(q, k, qkv[:, nh + nkv:], OMNI_HD ** -0.5, cu, cu, True).reshape(-1, nh * OMNI_HD), "status": None}


def exact(case, seed):
    return {"vision": _exact_vision, "omni": _exact_omni}.get(case["kind"], _exact_text)(case, seed)
