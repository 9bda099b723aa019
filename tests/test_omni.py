"""Omni decoder attention (hd 128, FP32): the oracle's prep pinned against transformers' Qwen3-Omni
RMSNorm and interleaved M-RoPE, and on the GPU the checks of tests/test_omni_attention.m: FP64
prep and attention tolerances, packed-versus-single byte equality, flat scores, poisoned inputs
reported, the output guard, large positions, f32 angles and a long constant-value row."""
import numpy as np
import pytest
import torch

from cleffa_amd import _lib
from cleffa_amd.omni import OmniAttention, OmniPlan, omni_rope_table
from oracle import oracle

HF = "transformers.models.qwen3_omni_moe.modeling_qwen3_omni_moe"


def _hf_prep(qkv, nh, nkv, qn, kn, pos3, exact, theta=1e6, eps=1e-6):
    """Q, K through transformers' Qwen3-Omni modules: RMSNorm(head_dim), the interleaved M-RoPE
    frequency layout (mrope_section 24/20/20) and apply_rotary_pos_emb. exact: angles in float64."""
    import importlib
    hf = importlib.import_module(HF)
    T = qkv.shape[0]
    x = torch.from_numpy(qkv.astype(np.float32)).view(T, nh + 2 * nkv, 128)
    norm = hf.Qwen3OmniMoeThinkerTextRMSNorm(128, eps=eps)
    with torch.no_grad():
        norm.weight.copy_(torch.from_numpy(qn))
        q = norm(x[:, :nh]).double()
        norm.weight.copy_(torch.from_numpy(kn))
        k = norm(x[:, nh:nh + nkv]).double()
    if exact:
        inv = torch.tensor([theta ** (-2.0 * i / 128.0) for i in range(64)], dtype=torch.float64)
        pos = torch.from_numpy(pos3.T.astype(np.float64))            # (3, T)
    else:
        inv = (1.0 / (theta ** (torch.arange(0, 128, 2, dtype=torch.float) / 128))).float()
        pos = torch.from_numpy(pos3.T.astype(np.float32))
    freqs = pos[:, :, None] * inv[None, None, :]                     # (3, T, 64)
    freqs = hf.Qwen3OmniMoeThinkerTextRotaryEmbedding.apply_interleaved_mrope(None, freqs[:, None], [24, 20, 20])[0]
    emb = torch.cat((freqs, freqs), dim=-1).double()
    q, k = hf.apply_rotary_pos_emb(q, k, emb.cos(), emb.sin(), unsqueeze_dim=1)   # cos (T, 1, 128)
    return q.permute(1, 0, 2).numpy(), k.permute(1, 0, 2).numpy()


def _inputs(T, nh, nkv, seed, pos_max=3000):
    rng = np.random.default_rng(seed)
    qkv = rng.standard_normal((T, (nh + 2 * nkv) * 128)).astype(np.float32)
    qn = (1 + 0.2 * rng.standard_normal(128)).astype(np.float32)
    kn = (1 + 0.2 * rng.standard_normal(128)).astype(np.float32)
    pos3 = rng.integers(0, pos_max, size=(T, 3)).astype(np.int32)
    return qkv, qn, kn, pos3


@pytest.mark.parametrize("exact", [True, False])
def test_oracle_prep_matches_transformers(exact):
    nh, nkv, T = 4, 2, 40
    qkv, qn, kn, pos3 = _inputs(T, nh, nkv, seed=1)
    inv = omni_rope_table(1e6)[:64]
    Q, K, V = oracle.omni_prep(qkv, nh, nkv, qn, kn, pos3, theta=1e6, exact=exact, inv_freq=inv)
    hq, hk = _hf_prep(qkv, nh, nkv, qn, kn, pos3, exact)
    assert np.abs(Q - hq).max() < 2e-6 and np.abs(K - hk).max() < 2e-6
    np.testing.assert_array_equal(V, qkv.reshape(T, nh + 2 * nkv, 128)[:, nh + nkv:].transpose(1, 0, 2))


def test_oracle_prep_axes_and_pairs():
    """Position (p, 0, 0) turns exactly the temporal pairs (i % 3 == 0 below 60, and 60-63); every
    pair (i, i + 64) keeps its length."""
    nh, nkv, T = 1, 1, 3
    qkv, qn, kn, _ = _inputs(T, nh, nkv, seed=2)
    Q0, _, _ = oracle.omni_prep(qkv, nh, nkv, qn, kn, np.zeros((T, 3), np.int32))
    for axis in range(3):
        pos = np.zeros((T, 3), np.int32)
        pos[:, axis] = 77
        Q, _, _ = oracle.omni_prep(qkv, nh, nkv, qn, kn, pos)
        moved = np.abs(Q[0] - Q0[0])[:, :64].max(0) > 1e-9
        want = np.array([(i < 60 and i % 3 == axis) or (i >= 60 and axis == 0) for i in range(64)])
        np.testing.assert_array_equal(moved, want)
        r0 = Q0[0][:, :64] ** 2 + Q0[0][:, 64:] ** 2
        r1 = Q[0][:, :64] ** 2 + Q[0][:, 64:] ** 2
        assert np.abs(r0 - r1).max() < 1e-12


def test_rope_table():
    t = omni_rope_table(1e6)
    f = 1e6 ** (-np.arange(64) * 2 / 128.0)
    assert np.abs(t[64:128].astype(np.float64) + t[128:].astype(np.float64) - f).max() <= 1e-15 * 1
    # the f32 table is C's 1 / powf(theta, 2j / 128) (clef_metal.m:177); libm's powf is within an ulp
    np.testing.assert_allclose(t[:64], 1.0 / 1e6 ** (np.arange(64) * 2 / 128.0), rtol=2.5e-7, atol=0)


def test_plan_blocks():
    p = OmniPlan([0, 33, 33, 40], device="cpu")
    b = p.blocks_host
    assert p.n_blk == 4 and (np.diff(b[:, 4]) <= 0).all()
    assert sorted(map(tuple, b[:, :5].tolist())) == [(0, 16, 0, 0, 16), (16, 16, 16, 0, 32), (32, 1, 32, 0, 33),
                                                      (33, 7, 0, 33, 7)]
    assert p.pairs() == 33 * 34 // 2 + 7 * 8 // 2


def test_abi_rejects_bad_heads():
    import ctypes
    lib = _lib.load()
    a = _lib.OmniAttnArgs()
    a.nh, a.nkv, a.T, a.kvT, a.scale, a.n_blk = 24, 4, 8, 40, 0.1, 1
    err = ctypes.create_string_buffer(256)
    assert not lib.clef_hip_omni_attention(ctypes.byref(a), None, err, 256)
    assert "head counts" in err.value.decode()
    a.nh, a.kvT = 32, 20
    assert not lib.clef_hip_omni_attention(ctypes.byref(a), None, err, 256)
    assert "kvT" in err.value.decode()


# ---------------------------------------------------------------- GPU: tests/test_omni_attention.m

def _sample(i):
    return (np.sin(np.asarray(i, dtype=np.float32) * np.float32(0.37)) * np.float32(0.7)).astype(np.float32)


def _run(length, packed, mode, rope_exact=True, pos_base=0):
    """One case of tests/test_omni_attention.m:run: nh 8, nkv 1; packed puts a 7-token record
    before and a 3-token record after. mode 1 sharp norms, 2 flat scores, 3-5 a NaN / +inf / -inf
    input, 6 flat scores with constant V."""
    nh, nkv = 8, 1
    before, after = (7, 3) if packed else (0, 0)
    T, row = before + length + after, (nh + 2 * nkv) * 128
    starts = np.array([0 if t < before else before if t < before + length else before + length for t in range(T)])
    local = np.arange(T) - starts
    norms = ((8.0 if mode == 1 else 1.0) + _sample(np.arange(256) + 3) * np.float32(0.2)).astype(np.float32)
    qkv = _sample(local[:, None] * row + np.arange(row)[None, :])
    if mode in (2, 6):
        qkv[:, :(nh + nkv) * 128] = 0
    if mode == 6:
        qkv[:, (nh + nkv) * 128:] = (np.float32(0.1234567) + np.arange(128, dtype=np.float32) * np.float32(1e-4))
    if 3 <= mode <= 5:
        qkv[before + length - 1, 0] = {3: np.nan, 4: np.inf, 5: -np.inf}[mode]
    pos3 = np.stack([pos_base + local + 5, pos_base + 2 * local + 1, pos_base + 3 * local + 2], 1).astype(np.int32)
    cu = np.array(sorted({0, before, before + length, T}), np.int32)
    att = OmniAttention(nh, nkv, theta=1e6, rope_exact=rope_exact)
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    plan = OmniPlan(cu)
    out = torch.full((T * nh * 128 + 32,), float("nan"), device="cuda")
    o = out[: T * nh * 128].view(T, nh * 128)
    Q, K, V, status = att.prep(d(qkv), d(norms[:128]), d(norms[128:]), d(pos3))
    att.attention(Q, K, V, plan, out=o)
    torch.cuda.synchronize()
    return dict(qkv=qkv, norms=norms, pos3=pos3, cu=cu, before=before, T=T, nh=nh, nkv=nkv,
                Q=Q.cpu().numpy(), K=K.cpu().numpy(), out=out.cpu().numpy(), status=int(status.item()))


def _check_fp64(r, length, sharp, rope_exact):
    nh, nkv, T, before = r["nh"], r["nkv"], r["T"], r["before"]
    inv = omni_rope_table(1e6)[:64]
    Q, K, V = oracle.omni_prep(r["qkv"], nh, nkv, r["norms"][:128], r["norms"][128:], r["pos3"], theta=1e6,
                               exact=rope_exact, inv_freq=inv)
    tol = 1e-5 if sharp else 2e-6
    assert np.abs(r["Q"][:, :T] - Q).max() < tol, "RMS/RoPE mismatch (Q)"
    assert np.abs(r["K"][:, :T] - K).max() < tol, "RMS/RoPE mismatch (K)"
    assert (r["K"][:, T:T + 32] == 0).all(), "kv slack rows not zeroed"
    want = oracle.attention(Q, K, V, r["cu"], None, True, 128 ** -0.5, None)
    got = r["out"][: T * nh * 128].reshape(T, nh * 128)
    err = np.abs(got[before:before + length] - want[before:before + length]).max()
    assert np.isfinite(got).all() and err < (3e-4 if sharp else 3e-6), f"attention FP64 max err {err:.3g}"
    assert np.isnan(r["out"][T * nh * 128:]).all(), "output guard overwritten"
    return err


@pytest.mark.gpu
@pytest.mark.parametrize("mode", [0, 1, 2])
def test_omni_fp64_and_packing(mode):
    print(f"[omni] mode {mode}", flush=True)
    for length in (1, 31, 32, 33, 127, 128, 129):
        single, packed = _run(length, False, mode), _run(length, True, mode)
        assert single["status"] == 0 and packed["status"] == 0
        _check_fp64(single, length, mode == 1, True)
        _check_fp64(packed, length, mode == 1, True)
        n = length * 8 * 128
        b = packed["before"] * 8 * 128
        assert np.array_equal(single["out"][:n].view(np.uint32), packed["out"][b:b + n].view(np.uint32)), \
            f"packing changed output bytes at length {length}"


@pytest.mark.gpu
@pytest.mark.parametrize("mode", [3, 4, 5])
def test_omni_nonfinite_reported(mode):
    print(f"[omni] poison mode {mode}", flush=True)
    for length, packed in ((1, False), (33, True)):
        r = _run(length, packed, mode)
        t = r["before"] + length - 1
        assert not np.isfinite(r["Q"][0, t, 0]), "non-finite Q was hidden"
        assert r["status"] != 0, "non-finite attention was not reported"


@pytest.mark.gpu
def test_omni_large_positions_and_f32_angles():
    print("[omni] large positions", flush=True)
    for mode in (0, 1):
        for length in (1, 65, 129):
            single, packed = _run(length, False, mode, pos_base=65000), _run(length, True, mode, pos_base=65000)
            _check_fp64(single, length, mode == 1, True)
            n, b = length * 8 * 128, packed["before"] * 8 * 128
            assert np.array_equal(single["out"][:n].view(np.uint32), packed["out"][b:b + n].view(np.uint32))
    _check_fp64(_run(33, False, 0, rope_exact=False), 33, False, False)
    _check_fp64(_run(33, True, 1, rope_exact=False), 33, True, False)


@pytest.mark.gpu
def test_omni_long_flat():
    """8,193 keys of one constant V row: every output equals that row within 6e-8, and the
    packed run matches the single one byte for byte."""
    print("[omni] long flat", flush=True)
    res = []
    for packed in (False, True):
        r = _run(8193, packed, 6)
        T, b = r["T"], r["before"]
        got = r["out"][: T * 8 * 128].reshape(T, 8, 128)[b:b + 8193]
        want = r["qkv"][b, (8 + 1) * 128:]
        assert np.abs(got - want[None, None, :]).max() < 6e-8, "long accumulation lost constant values"
        res.append(got.copy())
    assert np.array_equal(res[0].view(np.uint32), res[1].view(np.uint32))


def _planes(T, nh, nkv, seed):
    """Q, K, V planes [heads][T][128] as the prologue leaves them (RMS-normalised rows), f32."""
    rng = np.random.default_rng(seed)
    Q, K, V = (rng.standard_normal((n, T, 128)).astype(np.float32) for n in (nh, nkv, nkv))
    return [x / np.sqrt((x.astype(np.float64) ** 2).mean(-1, keepdims=True)).astype(np.float32) for x in (Q, K)] + [V]


def _attend(Q, K, V, cu):
    """The attention kernel on given planes (slack rows and rows between records as they come)."""
    nh, T, _ = Q.shape
    nkv = K.shape[0]
    att, plan = OmniAttention(nh, nkv), OmniPlan(cu)
    q, k, v = att.planes(T)
    q.copy_(torch.from_numpy(Q))
    for dst, src in ((k, K), (v, V)):
        dst.zero_()
        dst[:, :T].copy_(torch.from_numpy(src))
    out = torch.full((T, nh * 128), float("nan"), device="cuda")
    att.attention(q, k, v, plan, out=out)
    torch.cuda.synchronize()
    return out.cpu().numpy()


def _reference(Q, K, V, cu):
    with np.errstate(all="ignore"):
        return oracle.attention(*[x.astype(np.float64) for x in (Q, K, V)], np.asarray(cu, np.int32), None, True, 128 ** -0.5, None)


@pytest.mark.gpu
@pytest.mark.parametrize("nh,nkv", [(8, 1), (8, 2), (6, 3), (3, 3)])
def test_omni_group_widths_and_tile_edges(nh, nkv):
    """Every group width (8, 4, 2, 1 heads) over records that end on, before and after 32-key
    tiles. Bound: the scores' FP32 rounding (|s| up to ~40 in exponents of 2, 5 roundings of 2^-24
    each: 1.2e-5 of P at most, averaged over keys) leaves outputs of size ~1 within 3e-6, as the
    reference's tests ask."""
    print(f"[omni] widths {nh}/{nkv}", flush=True)
    lens = [1, 16, 17, 31, 32, 33, 48, 63, 64, 65, 95, 96, 97, 130, 257]
    cu = np.concatenate([[0], np.cumsum(lens)])
    Q, K, V = _planes(int(cu[-1]), nh, nkv, seed=nh)
    got, want = _attend(Q, K, V, cu), _reference(Q, K, V, cu)
    assert np.abs(got - want).max() < 3e-6
    alone = _attend(Q[:, :lens[0]], K[:, :lens[0]], V[:, :lens[0]], [0, lens[0]])
    assert np.array_equal(alone.view(np.uint32), got[:lens[0]].view(np.uint32))


@pytest.mark.gpu
@pytest.mark.parametrize("nh,nkv", [(8, 1), (4, 1)])
@pytest.mark.parametrize("which", ["v_inf", "v_big", "v_small", "k_minus", "q_big"])
def test_omni_values_without_bf16_parts(nh, nkv, which):
    """Infinities and magnitudes above bf16's overflow threshold (3.39e38) have no bf16 parts: rows that
    see one run on the FP32 and FP64 matrix instructions, and every record stays bit for bit what it is alone."""
    print(f"[omni] values {which} {nh}/{nkv}", flush=True)
    lens = [40, 70, 21]
    cu = np.concatenate([[0], np.cumsum(lens)])
    Q, K, V = _planes(int(cu[-1]), nh, nkv, seed=5)
    row = 40 + 33
    if which == "v_inf":
        V[0, row, 5], V[0, row + 20, 9] = np.inf, -np.inf
    elif which == "v_big":       # finite in FP32, above bf16's largest
        V[0, row, 5] = np.float32(3.395e38)
    elif which == "v_small":     # parts near the subnormals: relative to V, not to the others
        V[:] *= np.float32(1e-28)
    elif which == "k_minus":     # scores of minus infinity for that key: no weight
        Q[:, :, 7], K[0, row, 7] = np.abs(Q[:, :, 7]) + np.float32(0.1), -np.inf
    else:
        Q[1, row, 3], K[0, :, 3] = np.float32(3.395e38), np.float32(1e-38)
    got, want = _attend(Q, K, V, cu), _reference(Q, K, V, cu)
    fine = np.isfinite(want)
    assert np.array_equal(got[~fine], want[~fine].astype(np.float32), equal_nan=True)
    scale = np.abs(V[np.isfinite(V) & (np.abs(V) < 1e30)]).max() if which != "v_big" else 1.0
    big = np.maximum(np.abs(want[fine]), scale)
    assert (np.abs(got[fine] - want[fine]) / big).max() < 3e-6
    for r in range(3):
        a, b = cu[r], cu[r + 1]
        alone = _attend(Q[:, a:b], K[:, a:b], V[:, a:b], [0, b - a])
        assert np.array_equal(alone.view(np.uint32), got[a:b].view(np.uint32))


@pytest.mark.gpu
@pytest.mark.parametrize("which", ["v_inf", "v_nan", "v_big", "k_inf", "k_nan", "q_inf", "q_nan"])
def test_omni_rows_that_do_not_see_a_value_keep_their_bits(which):
    """A value that takes the plain path changes only the rows and heads that see it, at every group width and
    where a small pass splits a group of 8 heads; and its record has the same bits in a large pass."""
    value = np.float32({"inf": np.inf, "nan": np.nan, "big": 3e38}[which[2:]])
    for nh, nkv in ((16, 2), (8, 2), (4, 2), (2, 2)):
        print(f"[omni] rows beside {which}, heads {nh}/{nkv}", flush=True)
        T, row, group = 180, 101, nh // nkv
        Q, K, V = _planes(T, nh, nkv, seed=nh)
        clean = _attend(Q, K, V, [0, T])
        sees = np.zeros((T, nh, 128), bool)
        if which[0] == "q":
            Q[1, row, 77] = value
            sees[row, 1] = True
        else:
            (V if which[0] == "v" else K)[1, row, 99] = value
            sees[row:, group:] = True
        got = _attend(Q, K, V, [0, T])
        sees = sees.reshape(T, -1)
        assert np.array_equal(got.view(np.uint32)[~sees], clean.view(np.uint32)[~sees])
        more = [np.concatenate(x, axis=1) for x in zip((Q, K, V), _planes(2400, nh, nkv, seed=9))]
        packed = _attend(*more, np.concatenate([[0], T + np.arange(0, 2401, 100)]))
        assert np.array_equal(packed[:T].view(np.uint32), got.view(np.uint32))


@pytest.mark.gpu
@pytest.mark.parametrize("nh,nkv", [(8, 1), (4, 1), (1, 1)])
def test_omni_repeated_operands(nh, nkv):
    """Products whose rounding errors add up: equal operands, whose left-out parts all have one sign (2^-24 of
    each product at 0x1.00ff8p+0). Scores: key 0's, 4 x^2 128 / sqrt(128), against a key of score 0, whose V
    alone is not zero: the output's relative error is the score's; 4 steps and their sum's roundings, the
    left-out terms, Q's scale and its product: 8 x 2^-24. P . V: constant V over 200 keys: 6 FP32 roundings of
    a tile's sum, its left-out terms, 12 of the sum of P, the output's: 20 x 2^-24."""
    for x in (float.fromhex("0x1.00ff8p+0"), float.fromhex("0x1.00ff7ep+0"), float.fromhex("0x1.01017ep+0"), 1.1, 1.3):
        x = np.float32(x)
        print(f"[omni] repeated {x!r} {nh}/{nkv}", flush=True)
        Q, K, V = np.full((nh, 2, 128), 4 * x, np.float32), np.full((nkv, 2, 128), x, np.float32), np.ones((nkv, 2, 128), np.float32)
        K[:, 1] = 0
        V[:, 0] = 0
        o = _attend(Q, K, V, [0, 2])[1].astype(np.float64)
        s = 4 * float(x) ** 2 * 128 ** 0.5
        assert (np.abs(np.log(1 / o - 1) - s) / s).max() < 8 * 2.0 ** -24
        Q, K, V = _planes(200, nh, nkv, seed=7)
        V[:] = x
        assert (np.abs(_attend(Q, K, V, [0, 200]) - float(x)) / x).max() < 20 * 2.0 ** -24


@pytest.mark.gpu
@pytest.mark.parametrize("nh,nkv", [(8, 1), (8, 2), (2, 2)])
def test_omni_one_key_gives_its_value_back(nh, nkv):
    """A row that sees one key gives that key's V, exactly, for every magnitude of FP32 (24-bit values times
    2^e, subnormals included): the three parts of V lose no bit, and the plain path none of the largest."""
    print(f"[omni] one key {nh}/{nkv}", flush=True)
    n, rng = 2048, np.random.default_rng(1)
    V = np.ldexp(rng.integers(1 << 22, 1 << 24, (nkv, n, 128)) * rng.choice([-1.0, 1.0], (nkv, n, 128)),
                 rng.integers(-149, 105, (nkv, n, 128))).astype(np.float32)
    Q, K, _ = _planes(n, nh, nkv, seed=4)
    got = _attend(Q, K, V, np.arange(n + 1)).reshape(n, nh, 128)
    want = V.transpose(1, 0, 2).repeat(nh // nkv, axis=1)
    assert np.array_equal(got.view(np.uint32), np.ascontiguousarray(want).view(np.uint32))


@pytest.mark.gpu
def test_omni_small_probabilities_keep_their_precision():
    """Probabilities near 2^-124 of a large V beside a likely key whose V is nothing: the output is
    theirs. Bound: the exponent's FP32 rounding, 2^-24 x 124, three times over, is 2.2e-5."""
    Q, K, V = (np.zeros((1, 64, 128), np.float32) for _ in range(3))
    rng = np.random.default_rng(2)
    Q[0, :, 0] = 32.0
    K[0, 1:, 0] = rng.uniform(-30.5, -30.3, 63)      # scores of -86
    V[0, 0] = 1e-38
    V[0, 1:] = rng.uniform(0.5e10, 1e10, (63, 128))
    got, want = _attend(Q, K, V, [0, 64]), _reference(Q, K, V, [0, 64])
    assert (np.abs(got - want) / np.abs(want)).max() < 2.2e-5


@pytest.mark.gpu
@pytest.mark.parametrize("nh,nkv", [(8, 1), (4, 1)])
@pytest.mark.parametrize("big", [1e36, 1.1e37, 2e37, 1e38, 3.3e38])
def test_omni_sums_of_large_values_stay_finite(nh, nkv, big):
    """Equal scores over values whose plain sum leaves FP32's range: the output is their mean, finite.
    Bound: FP32 sums of 32 equally signed values (32 roundings of 2^-24 at most), FP64 across tiles,
    one rounding of the output: 33 x 2^-24 = 2e-6 of the largest value."""
    print(f"[omni] values of {big:g} {nh}/{nkv}", flush=True)
    T = 100
    Q, K, V = _planes(T, nh, nkv, seed=3)
    Q[:] = 0
    V = (big * np.random.default_rng(1).uniform(0.9, 1.0, V.shape)).astype(np.float32)
    got, want = _attend(Q, K, V, [0, 33, T]), _reference(Q, K, V, [0, 33, T])
    assert np.isfinite(got).all()
    assert np.abs(got - want).max() < 2e-6 * big


@pytest.mark.gpu
def test_omni_split_groups_agree_bitwise():
    """A small pass runs a group of 8 heads as two workgroups of 4: a record's bytes are those it
    has in a pass large enough for one workgroup per group, at both sides of the rule (2 x 16-row
    blocks x kv heads against 256 CUs)."""
    nh, nkv = 32, 4
    lens = [33, 495, 512, 513] + [200] * 12
    cu = np.concatenate([[0], np.cumsum(lens)])
    Q, K, V = _planes(int(cu[-1]), nh, nkv, seed=11)
    packed = _attend(Q, K, V, cu)
    for r in range(4):
        print(f"[omni] split groups, {lens[r]} tokens", flush=True)
        a, b = cu[r], cu[r + 1]
        alone = _attend(Q[:, a:b], K[:, a:b], V[:, a:b], [0, b - a])
        assert np.array_equal(alone.view(np.uint32), packed[a:b].view(np.uint32))
