"""FP32 text mode (qkv_type CLEF_HIP_QKV_F32: the reference's FP32 attention kernels,
metal/clef.metal:250-654, dispatched at clef_metal.m:1330-1413) against the float64 oracle and
the oracle's scalar FP32 restatement, through the C ABI.

Bound (the FP32 kernels' own, bench/vision_attention_bench.m:144-157 style): max-abs error
against float64 within max(5e-5, 2x the FP32 control's), mean-abs within 2x the control's."""
import numpy as np
import pytest
import torch

from cleffa_amd import AttnPlan, TextAttention, workloads
from tests.helpers import errors, oracle_text

pytestmark = pytest.mark.gpu


def _say(*a):
    print(*a, flush=True)


def _fp32(w, seed=11):
    """The workload with f32 qkv rows: bf16 values given full 24-bit mantissas."""
    g = torch.Generator().manual_seed(seed)
    q = w["qkv"].float()
    q = q * (1.0 + 2.0 ** -9 * torch.randn(q.shape, generator=g))
    return dict(w, qkv=q.contiguous())


def _run(w, out_dtype="f32", ovf=None, plan=None, **kw):
    att = TextAttention(w["nh"], w["nkv"], w["hd"], w["n_rot"], rope_theta=w.get("theta", 1e7))
    plan = plan or AttnPlan(w["cu_seqlens"], causal=True)
    d = lambda t: None if t is None else t.cuda()
    out = att.forward(d(w["qkv"]), d(w["q_norm"]), d(w["k_norm"]), d(w["pos3"]), plan, out_dtype=out_dtype,
                      gate=w.get("gate", True), ovf=ovf, **kw)
    torch.cuda.synchronize()
    return out, plan


def _check_fp32(got, w, rows=None, what=""):
    want = oracle_text(w, rows=rows)
    ctrl = oracle_text(w, rows=rows, precision="f32")
    mx, mean = errors(got, want)
    cmx, cmean = errors(ctrl, want)
    _say(f"[fp32] {what}: max_abs {mx:.3g} mean_abs {mean:.3g} (f32 control {cmx:.3g} / {cmean:.3g})")
    assert mx <= max(5e-5, 2 * cmx), f"{what}: max_abs {mx:.3g}, control {cmx:.3g}"
    assert mean <= 2 * cmean + 1e-7, f"{what}: mean_abs {mean:.3g}, control {cmean:.3g}"


@pytest.mark.parametrize("name", ["C0", "C1"])
def test_fp32_configs(name):
    _say(f"[fp32] {name}")
    w = _fp32(workloads.config(name, seed=0))
    out, _ = _run(w)
    _check_fp32(out.cpu().numpy(), w, what=name)


def test_fp32_gqa_widths_and_edges():
    """Group sizes 1, 3, 5, 8 with ragged records of 1, 2, 15,
    16, 17, 31, 33, 127, 129 tokens: every row offset of the 16-row groups and 32-key tiles."""
    lengths = [1, 2, 15, 16, 17, 31, 33, 127, 129]
    for nh, nkv in ((2, 2), (6, 2), (5, 1), (16, 2)):
        _say(f"[fp32] nh {nh} nkv {nkv}")
        w = workloads.text_inputs(lengths, nh, nkv, seed=nh)
        w.update(gate=True, theta=1e7)
        w = _fp32(w)
        out, _ = _run(w)
        _check_fp32(out.cpu().numpy(), w, what=f"{nh}/{nkv}")


def test_fp32_c2_sampled_rows():
    _say("[fp32] C2 sampled rows")
    w = _fp32(workloads.config("C2", seed=0))
    out, _ = _run(w)
    rows = np.array([0, 1, 15, 16, 127, 128, 4095, 8191, 12000, 16383], np.int32)
    _check_fp32(out.cpu().numpy()[rows], w, rows=rows, what="C2")


def test_fp32_packing_invariance_bitwise():
    """Each record's output is bitwise the same packed with others as run alone
    (bench/attention_bench.m:263-308): key tiles start at the record's first key."""
    lengths = [1] * 8 + [2, 9, 31, 32, 33, 63, 65, 263]
    w = _fp32(dict(workloads.text_inputs(lengths, 8, 2, seed=4), gate=True, theta=1e7))
    packed, _ = _run(w)
    cu = w["cu_seqlens"]
    for r, n in enumerate(lengths):
        a, b = int(cu[r]), int(cu[r + 1])
        wr = dict(w, qkv=w["qkv"][a:b].clone(), pos3=w["pos3"][a:b].clone(),
                  cu_seqlens=np.array([0, n], np.int32), lengths=[n])
        alone, _ = _run(wr)
        assert torch.equal(alone.view(torch.int32), packed[a:b].view(torch.int32)), f"record {r} (len {n})"


def test_fp32_16bit_outputs_are_rounded_f32():
    """bf16 / f16 outputs are round-to-nearest-even of the f32 output (act16, clef.metal:98-106)."""
    w = _fp32(dict(workloads.text_inputs([300, 77], 8, 2, seed=6), gate=True, theta=1e7))
    f32, _ = _run(w)
    for dt, tdt in (("bf16", torch.bfloat16), ("f16", torch.float16)):
        o, _ = _run(w, out_dtype=dt)
        assert torch.equal(o.view(torch.int16), f32.to(tdt).view(torch.int16)), dt


def test_fp32_f16_overflow_flags_isolated():
    """Odd records' V x 1e5: their f16 outputs saturate and flag the record's first row; the
    other records' outputs are unchanged (bench/attention_bench.m:256-261)."""
    lengths = [100, 150, 64, 200]
    nh, nkv, hd = 8, 2, 256
    w = _fp32(dict(workloads.text_inputs(lengths, nh, nkv, seed=3), gate=False, theta=1e7))
    vcol = 2 * nh * hd + nkv * hd
    cu = w["cu_seqlens"]
    q = w["qkv"].clone()
    for r in (1, 3):
        q[cu[r]:cu[r + 1], vcol:] *= 1e5
    ovf = torch.zeros(int(cu[-1]), dtype=torch.int32, device="cuda")
    out, _ = _run(dict(w, qkv=q), out_dtype="f16", ovf=ovf)
    clean, _ = _run(w, out_dtype="f16")
    want = np.zeros(int(cu[-1]), np.int32)
    want[cu[1]] = want[cu[3]] = 1
    assert np.array_equal(ovf.cpu().numpy(), want)
    assert torch.isfinite(out.float()).all()
    for r in (0, 2):
        a, b = cu[r], cu[r + 1]
        assert torch.equal(out[a:b].view(torch.int16), clean[a:b].view(torch.int16))


def test_fp32_prefix_equals_full_pass_bitwise():
    """A prefix-cache pass (queries = a record's last tokens, keys = cached rows + new rows) gives
    bitwise the full pass's rows (tests/test_prefix_attention.m semantics), with the FP32 planes
    of the full pass as the cache."""
    nh, nkv = 8, 2
    full_len, new = 328, 72                 # cached 256 rows (a multiple of 8)
    w = _fp32(dict(workloads.text_inputs([full_len], nh, nkv, seed=8), gate=True, theta=1e7))
    att = TextAttention(nh, nkv, 256, 64, rope_theta=1e7)
    plan = AttnPlan(w["cu_seqlens"], causal=True)
    kp, vp = att.planes(plan.kvT, fp32=True)
    d = lambda t: t.cuda()
    full = att.forward(d(w["qkv"]), d(w["q_norm"]), d(w["k_norm"]), d(w["pos3"]), plan, out_dtype="f32",
                       k_plane=kp, vt_plane=vp, kvT=plan.kvT)
    # prefix pass over the same planes: its prologue rewrites rows 256..327 with the same values
    cq = np.array([0, new], np.int32)
    ck = np.array([0, full_len], np.int32)
    pplan = AttnPlan(cq, ck, causal=True)
    a = full_len - new
    part = att.forward(d(w["qkv"][a:].clone()), d(w["q_norm"]), d(w["k_norm"]), d(w["pos3"][a:].clone()), pplan,
                       out_dtype="f32", k_plane=kp, vt_plane=vp, kvT=plan.kvT)
    torch.cuda.synchronize()
    assert torch.equal(part.view(torch.int32), full[a:].view(torch.int32))


@pytest.mark.parametrize("nh,nkv", [(12, 1), (16, 1), (9, 1), (24, 2)])
def test_fp32_wide_groups(nh, nkv):
    """Groups of more than 8 q heads (12 and 16 per kv head, whose items hold two heads, or more where a record is
    short; 9, whose items hold one or three; 12 per kv head over two kv heads) against float64 within
    the FP32 bound, with ragged records."""
    _say(f"[fp32] wide group {nh}/{nkv}")
    w = _fp32(dict(workloads.text_inputs([1, 17, 40, 130, 300], nh, nkv, seed=nh), gate=True, theta=1e7))
    out, _ = _run(w)
    _check_fp32(out.cpu().numpy(), w, what=f"{nh}/{nkv}")


def test_fp32_repeated_passes_agree_bitwise():
    """The same pass gives the same bits every time, with other passes between (whose workgroups leave other
    values in LDS and registers)."""
    _say("[fp32] repeated passes")
    w = _fp32(dict(workloads.text_inputs([700, 33, 129, 1, 260], 24, 4, seed=3), gate=True, theta=1e7))
    other = _fp32(dict(workloads.text_inputs([70, 400], 24, 4, seed=4), gate=True, theta=1e7))
    one, _ = _run(w)
    for _ in range(5):
        _run(other)
        out, _ = _run(w)
        assert torch.equal(out.view(torch.int32), one.view(torch.int32))


FP32_GEOMETRIES = [(24, 4), (16, 4), (8, 2), (4, 1), (6, 2), (12, 4), (16, 8), (10, 5), (2, 2), (5, 1), (14, 2),
                   (9, 1), (24, 2), (7, 1)]


@pytest.mark.parametrize("seed", range(24))
def test_fp32_random_pass(seed):
    """Seeded random packed passes in the FP32 mode (ragged records around the 16-row groups
    and 32-key tiles; group widths 1-12: items of one or two heads of a group, of more where a record is
    short; with and without the norms, rotary and gate) against float64 within the FP32 bound."""
    rng = np.random.default_rng(5000 + seed)
    n = int(rng.integers(1, 5))
    lengths = [int(x) for x in rng.choice([1, 2, 15, 16, 17, 31, 33, 64, 65, 127, 129, 300], size=n)]
    nh, nkv = FP32_GEOMETRIES[int(rng.integers(len(FP32_GEOMETRIES)))]
    norm = bool(rng.integers(2))
    n_rot = 64 if norm and rng.integers(3) else 0
    gate = bool(rng.integers(2))
    _say(f"[fp32] random seed {seed}: lengths {lengths} heads {nh}/{nkv} norm {norm} rot {n_rot} gate {gate}")
    w = workloads.text_inputs(lengths, nh, nkv, n_rot=n_rot, seed=seed, norm=norm)
    w.update(gate=gate, theta=1e7)
    w = _fp32(w)
    out, _ = _run(w)
    _check_fp32(out.cpu().numpy(), w, what=f"random {seed}")


@pytest.mark.parametrize("which", ["v_inf", "v_big", "v_small", "q_big", "k_minus"])
def test_fp32_values_without_bf16_parts(which):
    """Infinities and magnitudes above bf16's overflow threshold (3.39e38) have no bf16 parts: rows
    that see one run on the FP32 matrix instructions, against float64 (infinite and NaN outputs included); records
    beside theirs stay bit for bit what they are alone. Values of 1e-28 keep their relative precision."""
    _say(f"[fp32] values {which}")
    lengths, nh, nkv, hd = [40, 70, 21], 8, 2, 256
    plain = which in ("q_big", "k_minus")
    w = workloads.text_inputs(lengths, nh, nkv, n_rot=0 if plain else 64, seed=9, norm=not plain, outlier_frac=0)
    w = _fp32(dict(w, gate=True, theta=1e7))
    q = w["qkv"].clone()
    kcol, vcol, row = 2 * nh * hd, (2 * nh + nkv) * hd, 40 + 33
    if which == "v_inf":
        q[row, vcol + 5], q[row + 20, vcol + hd + 9] = float("inf"), float("-inf")
    elif which == "v_big":
        q[row, vcol + 5] = 3.395e38
    elif which == "v_small":
        q[:, vcol:] *= 1e-28
    elif which == "q_big":      # head 1 (kv head 0), against keys near 0 in that dim: finite scores
        q[row, 2 * hd + 3] = 3.395e38
        q[:, kcol + 3] = 1e-38
    else:                       # scores of minus infinity for one key: no weight
        for h in range(nh // nkv):
            q[:, 2 * h * hd + 7] = q[:, 2 * h * hd + 7].abs() + 0.1
        q[row, kcol + 7] = float("-inf")
    w = dict(w, qkv=q)
    got = _run(w)[0].cpu().numpy()
    with np.errstate(all="ignore"):
        want = oracle_text(w)
    fine = np.isfinite(want)
    assert np.array_equal(got[~fine], want[~fine].astype(np.float32), equal_nan=True)
    unit = 1e-28 if which == "v_small" else 1.0
    assert (np.abs(got[fine] - want[fine]) / np.maximum(np.abs(want[fine]), unit)).max() < 2e-5
    cu = w["cu_seqlens"]
    for r in (0, 2):
        a, b = int(cu[r]), int(cu[r + 1])
        alone, _ = _run(dict(w, qkv=q[a:b].clone(), pos3=w["pos3"][a:b].clone(), cu_seqlens=np.array([0, b - a], np.int32)))
        assert np.array_equal(alone.cpu().numpy().view(np.uint32), got[a:b].view(np.uint32))


# Equal operands whose parts the products leave out (m l) all have one sign: 2^-24 of each product at 0x1.00ff8p+0.
# Below 1.16, so that e^(-64 x^2), which the test reads the scores from, is a normal FP32 number.
REPEATED = np.array([float.fromhex("0x1.00ff8p+0"), float.fromhex("0x1.00ff7ep+0"), float.fromhex("0x1.01017ep+0"), 1.1, 1.15], np.float32)


def test_fp32_repeated_operands():
    """Products whose rounding errors add up. Scores: key 0's, 4 x^2 256 / 16, against a key of score 0,
    whose V alone is not zero: the output's relative error is the score's. Bound on that of the score: 8 steps
    and their sum's roundings, the left-out terms, Q's scale and its product, 12 x 2^-24 of it (the
    FP32 matrix instructions' 64 steps gave 16). P . V: constant V over 32 keys, one tile: 6 roundings at full size,
    the left-out terms, 12 of the sum of P and the output's, 20 x 2^-24."""
    _say("[fp32] repeated operands")
    n = len(REPEATED)
    x = torch.from_numpy(REPEATED).repeat_interleave(2)[:, None]
    qkv = torch.zeros(2 * n, 4 * 256)
    qkv[:, :256] = 4 * x
    qkv[0::2, 512:768] = x[0::2]
    qkv[1::2, 768:] = 1
    w = dict(qkv=qkv, q_norm=None, k_norm=None, pos3=torch.zeros(2 * n, 3, dtype=torch.int32), nh=1, nkv=1, hd=256, n_rot=0, gate=False,
             cu_seqlens=np.arange(0, 2 * n + 1, 2, dtype=np.int32))
    o = _run(w)[0].cpu().numpy()[1::2].astype(np.float64)
    s = 4 * REPEATED.astype(np.float64)[:, None] ** 2 * 16
    assert (np.abs(np.log(1 / o - 1) - s) / s).max() < 12 * 2.0 ** -24
    qkv = torch.randn(32 * n, 4 * 256, generator=torch.Generator().manual_seed(3))
    qkv[:, 768:] = torch.from_numpy(REPEATED).repeat_interleave(32)[:, None]
    w = dict(w, qkv=qkv, pos3=torch.zeros(32 * n, 3, dtype=torch.int32), cu_seqlens=np.arange(0, 32 * n + 1, 32, dtype=np.int32))
    v = qkv[:, 768:].numpy().astype(np.float64)
    assert (np.abs(_run(w)[0].cpu().numpy() - v) / v).max() < 20 * 2.0 ** -24


def _every_magnitude(n, seed):
    """[n][256] f32 of both signs over FP32's whole range, subnormals included: 24-bit values times 2^e."""
    rng = np.random.default_rng(seed)
    e = rng.integers(-149, 105, (n, 256))
    return np.ldexp(rng.integers(1 << 22, 1 << 24, (n, 256)) * rng.choice([-1.0, 1.0], (n, 256)), e).astype(np.float32)


def test_fp32_one_key_gives_its_value_back():
    """A row that sees one key gives that key's V: probability 1, the sum of V's three parts (or, from 2^55
    on, the plain path). Exact for every magnitude, so the parts lose no bit of any of them."""
    _say("[fp32] one key")
    n = 4096
    V = _every_magnitude(n, 1)
    qkv = torch.zeros(n, 4 * 256)
    qkv[:, 3 * 256:] = torch.from_numpy(V)
    w = dict(qkv=qkv, q_norm=None, k_norm=None, pos3=torch.zeros(n, 3, dtype=torch.int32), nh=1, nkv=1, hd=256, n_rot=0, gate=False,
             cu_seqlens=np.arange(n + 1, dtype=np.int32))
    got = _run(w)[0].cpu().numpy()
    assert np.array_equal(got.view(np.uint32), V.view(np.uint32))


def test_fp32_small_probabilities_keep_their_precision():
    """Probabilities near 2^-124 of a large V beside a likely key whose V is nothing: the output is
    theirs. Bound: the exponent's FP32 rounding, 2^-24 x 124, three times over, is 2.2e-5."""
    _say("[fp32] small probabilities")
    qkv = torch.zeros(64, 4 * 256)
    rng = np.random.default_rng(2)
    qkv[:, 0] = 32.0                                                      # Q
    qkv[1:, 2 * 256] = torch.from_numpy(rng.uniform(-43.2, -42.8, 63))    # K: scores of -86, 2^-124
    qkv[0, 3 * 256:] = 1e-38
    qkv[1:, 3 * 256:] = torch.from_numpy(rng.uniform(0.5e10, 1e10, (63, 256)))
    w = dict(qkv=qkv, q_norm=None, k_norm=None, pos3=torch.zeros(64, 3, dtype=torch.int32), nh=1, nkv=1, hd=256, n_rot=0, gate=False,
             cu_seqlens=np.array([0, 64], np.int32))
    got, want = _run(w)[0].cpu().numpy(), oracle_text(w)
    assert (np.abs(got - want) / np.abs(want)).max() < 2.2e-5


BAD_VALUES = ["v_inf", "v_nan", "v_big", "k_inf", "k_nan", "q_inf", "q_nan"]


def _with_bad_value(w, which, row):
    """The workload with one infinite, NaN or huge element in pass row `row`: in kv head 1's V or K, or in
    head 1's Q. Returns it and the heads that meet it."""
    nh, nkv, hd = w["nh"], w["nkv"], w["hd"]
    q = w["qkv"].clone()
    value = {"inf": float("inf"), "nan": float("nan"), "big": 3e38}[which[2:]]
    col = {"v": (2 * nh + nkv + 1) * hd + 5, "k": (2 * nh + 1) * hd + 99, "q": 2 * hd + 77}[which[0]]
    q[row, col] = value
    group = nh // nkv
    return dict(w, qkv=q), range(1, 2) if which[0] == "q" else range(group, 2 * group)


@pytest.mark.parametrize("which", BAD_VALUES)
@pytest.mark.parametrize("nh,nkv", [(24, 4), (10, 2)])
def test_fp32_rows_that_do_not_see_a_value_keep_their_bits(nh, nkv, which):
    """A value that takes the plain path changes only the rows and heads that see it: every other output
    has the bits of the same pass without it, also in the rows just before it."""
    _say(f"[fp32] rows beside {which}, heads {nh}/{nkv}")
    w = _fp32(dict(workloads.text_inputs([300, 70], nh, nkv, seed=2), gate=True, theta=1e7))
    row = 150
    bad, heads = _with_bad_value(w, which, row)
    clean, got = (_run(x)[0].view(torch.int32).view(370, nh, 256).clone() for x in (w, bad))
    sees = torch.zeros(370, nh, dtype=torch.bool, device="cuda")
    sees[row:(row + 1 if which[0] == "q" else 300), list(heads)] = True
    assert torch.equal(got[~sees], clean[~sees])


@pytest.mark.parametrize("which", ["v_inf", "v_big", "q_nan"])
def test_fp32_bad_values_without_a_causal_mask(which):
    """Without the mask every row of the record sees a bad key: the affected heads against float64, the
    others with the bits of the clean pass."""
    _say(f"[fp32] {which} without a causal mask")
    nh, nkv, T = 6, 2, 110
    w = _fp32(dict(workloads.text_inputs([70, 40], nh, nkv, seed=3), gate=False, theta=1e7))
    bad, heads = _with_bad_value(w, which, 30)
    plan = AttnPlan(w["cu_seqlens"], causal=False)
    clean, got = (_run(x, plan=plan)[0].cpu().numpy().reshape(T, nh, 256) for x in (w, bad))
    with np.errstate(all="ignore"):
        want = oracle_text(bad, causal=False).reshape(T, nh, 256)
    sees = np.zeros((T, nh), bool)
    sees[(slice(30, 31) if which == "q_nan" else slice(0, 70)), list(heads)] = True
    assert np.array_equal(got[~sees].view(np.uint32), clean[~sees].view(np.uint32))
    fine = np.isfinite(want)
    assert np.array_equal(got[~fine], want[~fine].astype(np.float32), equal_nan=True)
    assert (np.abs(got[fine] - want[fine]) / np.maximum(np.abs(want[fine]), 1)).max() < 2e-5


@pytest.mark.parametrize("gate", [True, False])
def test_fp32_plain_rows_in_16_bits(gate):
    """Rows on the plain path give bf16 and f16 outputs as the others do: the f32 output rounded, f16 saturated
    and its record flagged, the other record's rows and flag untouched."""
    _say(f"[fp32] plain rows in 16 bits, gate {gate}")
    w = _fp32(dict(workloads.text_inputs([100, 70], 8, 2, seed=6), gate=gate, theta=1e7))
    w, _ = _with_bad_value(w, "v_big", 60)
    f32 = _run(w)[0]
    assert (f32[60:100].abs() > 65504).any() and torch.isfinite(f32).all()
    assert torch.equal(_run(w, out_dtype="bf16")[0].view(torch.int16), f32.to(torch.bfloat16).view(torch.int16))
    ovf = torch.zeros(170, dtype=torch.int32, device="cuda")
    f16 = _run(w, out_dtype="f16", ovf=ovf)[0]
    assert torch.equal(f16.view(torch.int16), f32.clamp(-65504, 65504).to(torch.float16).view(torch.int16))
    assert ovf.nonzero().flatten().tolist() == [0]


@pytest.mark.parametrize("which", BAD_VALUES)
def test_fp32_bad_values_agree_bitwise_over_item_sizes(which):
    """A record that holds such a value has the same bits alone (four-wave items), in a pass of eight-wave items,
    and as the continuation of a cached prefix, whose 16-row groups start elsewhere."""
    _say(f"[fp32] {which} over item sizes")
    nh, nkv, n, new = 24, 4, 304, 84
    w = _fp32(dict(workloads.text_inputs([n] + [257] * 30, nh, nkv, seed=5), gate=True, theta=1e7))
    w, _ = _with_bad_value(w, which, 250)
    packed, _ = _run(w)
    att = TextAttention(nh, nkv, 256, 64, rope_theta=1e7)
    plan = AttnPlan(np.array([0, n], np.int32))
    kp, vp = att.planes(plan.kvT, fp32=True)
    alone, _ = _run(dict(w, qkv=w["qkv"][:n].clone(), pos3=w["pos3"][:n].clone()), plan=plan, k_plane=kp, vt_plane=vp, kvT=plan.kvT)
    assert torch.equal(alone.view(torch.int32), packed[:n].view(torch.int32))
    a = n - new
    part, _ = _run(dict(w, qkv=w["qkv"][a:n].clone(), pos3=w["pos3"][a:n].clone()),
                   plan=AttnPlan(np.array([0, new], np.int32), np.array([0, n], np.int32)), k_plane=kp, vt_plane=vp, kvT=plan.kvT)
    assert torch.equal(part.view(torch.int32), packed[a:n].view(torch.int32))


@pytest.mark.parametrize("nh,nkv", [(24, 4), (15, 3), (16, 2)])
def test_fp32_item_sizes_agree_bitwise(nh, nkv):
    """A record gives the same bits in a pass large enough for eight-wave items as in a small pass, whose
    items hold rows in four waves (and packed with short records, whose items take more heads)."""
    _say(f"[fp32] item sizes {nh}/{nkv}")
    lengths = [300, 5, 17, 40, 81, 97, 128] + [257] * 30
    w = _fp32(dict(workloads.text_inputs(lengths, nh, nkv, seed=2), gate=True, theta=1e7))
    packed, _ = _run(w)
    cu = w["cu_seqlens"]
    for r in range(8):
        a, b = int(cu[r]), int(cu[r + 1])
        alone, _ = _run(dict(w, qkv=w["qkv"][a:b].clone(), pos3=w["pos3"][a:b].clone(), cu_seqlens=np.array([0, b - a], np.int32)))
        assert torch.equal(alone.view(torch.int32), packed[a:b].view(torch.int32)), f"record {r}"


def test_fp32_without_rope_table():
    """The core evaluates the angles itself when no cos / sin table is given: the same bits."""
    _say("[fp32] no rope table")
    w = _fp32(dict(workloads.text_inputs([200, 33], 8, 2, seed=12), gate=True, theta=1e7))
    att, plan = TextAttention(8, 2, 256, 64, rope_theta=1e7), AttnPlan(w["cu_seqlens"])
    d = [w[k].cuda() for k in ("qkv", "q_norm", "k_norm", "pos3")]
    kp, vp = att.planes(plan.kvT, fp32=True)
    kw = dict(out_dtype="f32", k_plane=kp, vt_plane=vp, kvT=plan.kvT)
    with_table = att.forward(*d, plan, rope_cs=att.rope_table(plan.T), **kw)
    without = att.forward(*d, plan, stage="core", **kw)
    torch.cuda.synchronize()
    assert torch.equal(with_table.view(torch.int32), without.view(torch.int32))


@pytest.mark.parametrize("nh,nkv,lengths", [(16, 8, [64] * 12), (16, 4, [64] * 7 + [1] * 13), (32, 4, [9] * 40 + [130, 33]), (15, 3, [45] * 10),
                                            (24, 4, [64] * 16), (3, 1, [40] * 45), (2, 1, [70] * 150)])
def test_fp32_short_records_with_idle_workgroups(nh, nkv, lengths):
    """Passes of short records, whose blocks are followed by idle workgroups: every row is written, and each record
    has the bits it has alone."""
    _say(f"[fp32] short records {nh}/{nkv} {len(lengths)} x {lengths[0]}")
    w = _fp32(dict(workloads.text_inputs(lengths, nh, nkv, seed=8), gate=True, theta=1e7))
    got = _run(w, out=torch.full((sum(lengths), nh * 256), float("nan"), device="cuda"))[0].view(torch.int32)
    cu = w["cu_seqlens"]
    for r in sorted({0, 1, len(lengths) // 2, len(lengths) - 1}):
        a, b = int(cu[r]), int(cu[r + 1])
        alone, _ = _run(dict(w, qkv=w["qkv"][a:b].clone(), pos3=w["pos3"][a:b].clone(), cu_seqlens=np.array([0, b - a], np.int32)))
        assert torch.equal(alone.view(torch.int32), got[a:b])
    assert torch.isfinite(got.view(torch.float32)).all()
