"""Calls of several to many token rows at the edges of their kernels' tiles, against the CPU oracle:
final_norm_and_logits around 16 and 32 rows, sliding_attention around the row count from which it runs
on the matrix cores and its 16-row blocks, the full-attention pages around their 4-row blocks, the
full-attention projections past 16 rows, and the GEMM's row tiles. Gate: the reference's atol / rtol
1e-2 (gate_rope for rotated heads); running_max and running_sum as in test_gpu_full.py."""
import numpy as np
import pytest

from gpu_util import gate, gate_rope, need_gpu, say
from kat_inputs import unbf
from moa_amd import prng, synth
from oracle import oracle as O

pytestmark = pytest.mark.gpu
TS, TF = 1024, 512


@pytest.mark.parametrize("M", [2, 16, 32, 33])
def test_logits_rows(M):
    """Sampled vocabulary rows of every token row against the oracle, and the one-row call's bits."""
    need_gpu()
    from test_gpu_logits import check_sampled, lm_head, run_gpu
    say(f"logits M={M}")
    d = synth.cfg_logits(seed=M, M=M)
    got = run_gpu(d, lm_head(0))
    check_sampled(d, lm_head(0), got, f"logits M{M}", seed=M)
    for m in {M // 2, M - 1}:
        one = dict(input=d["input"][m:m + 1], rms_weight=d["rms_weight"])
        assert np.array_equal(run_gpu(one, lm_head(0))[0], got[m]), f"row {m}"


@pytest.mark.parametrize("M,kind", [(5, "causal"), (6, "causal"), (16, "scattered"), (17, "causal"), (40, "scattered"),
                                    (33, "empty"), (6, "empty"), (130, "causal"), (270, "scattered")])
def test_sliding_attention_rows(M, kind):
    """Causal rows from position 20 (whole tiles of slots valid for nobody), random masks, and masks that
    leave single slots, whole rows and whole tiles out."""
    need_gpu()
    from test_gpu_attention import run_gpu, run_oracle
    say(f"attention M={M} {kind}")
    d = synth.cfg_attention(seed=M, M=M, pos=20 + np.arange(M), q_std=0.5)
    rng = np.random.default_rng(M)
    if kind != "causal":
        d["mask"] = (rng.random((M, TS)) < 0.3).astype(np.float32) * np.float32(-2.5)  # any non-zero value counts
    if kind == "empty":
        d["mask"][:, 64:700] = 0.0
        d["mask"][3] = 0.0
        d["mask"][M - 1] = 0.0
        d["mask"][M - 1, 1023] = 1.0
    got = run_gpu(d)
    gate(run_oracle(d), got, f"attention M{M} {kind}")
    if kind == "empty":
        assert not got[3].any()
        v = d["v_cache"].reshape(TS, 8, 256)[1023]
        assert np.array_equal(got[M - 1], np.repeat(v[:, None, :], 2, axis=1))


def check_pages(d, got, label):
    gm, gs, go = got
    wm, ws, wo = O.full_attention_pages(d["q"], d["k_pages"], d["v_pages"], d["masks"])
    fin = np.isfinite(wm)
    assert np.array_equal(np.isfinite(gm), fin), label
    assert np.all(np.abs(gm[fin] - wm[fin]) <= 1e-3 * (1.0 + np.abs(wm[fin]))), f"{label}: running_max"
    assert np.all(np.abs(gs - ws) <= 1e-3 * np.abs(ws)), f"{label}: running_sum"
    gate(wo, go, f"{label} out")


@pytest.mark.parametrize("P,M,kind", [(3, 7, "causal"), (3, 8, "causal"), (6, 13, "scattered"), (12, 2, "causal"), (10, 3, "causal"), (11, 3, "causal"),
                                      (2, 66, "empty"), (1, 24, "scattered")])
def test_full_attention_rows(P, M, kind):
    need_gpu()
    from test_gpu_full import fused_gpu
    say(f"full attention P={P} M={M} {kind}")
    d = synth.cfg_full_attention(seed=P * M, M=M, P=P, pos=P * TF - M - 100 + np.arange(M), q_std=0.3)
    rng = np.random.default_rng(M)
    if kind != "causal":
        d["masks"] = (rng.random(d["masks"].shape) < 0.3).astype(np.float32)
    if kind == "empty":
        d["masks"][0, :, :200] = 0.0  # the first tiles: nobody's
        d["masks"][:, 3] = 0.0        # a row with no valid slot beside rows with some
        d["masks"][1, 40:] = 0.0
    got = fused_gpu(d)
    check_pages(d, got, f"pages P{P} M{M} {kind}")
    if kind == "empty":
        assert np.all(got[0][3] == -np.inf) and not got[1][3].any() and not got[2][3].any()


def test_one_page_call_of_many_rows():
    """Past 16 rows the per-page calls share a pass over the page: 19 rows, two pages, against the oracle
    and the 16-row call of the same rows."""
    need_gpu()
    from test_gpu_full import check_state, pages_gpu
    say("full attention, per page, M=19")
    d = synth.cfg_full_attention(seed=19, M=19, P=2, q_std=0.3)
    rng = np.random.default_rng(19)
    d["masks"] = (rng.random(d["masks"].shape) < 0.4).astype(np.float32)
    d["masks"][0, 4] = 0.0
    d["masks"][:, 6] = 0.0
    check_state(d, "pages M19")
    few = pages_gpu(dict(d, q=d["q"][:16], masks=np.ascontiguousarray(d["masks"][:, :16])))
    many = pages_gpu(d)
    gate(few[2], many[2][:16], "pages: 19 rows and 16")


@pytest.mark.parametrize("P,M", [(1, 17), (3, 6), (12, 3)])
def test_running_max_has_the_same_bits_in_every_kernel(P, M):
    """A score is summed in one order whichever kernel computes it: rows of a call that shares passes over
    the pages, and each row by itself, page by page (one-row kernels) and over all pages."""
    need_gpu()
    from test_gpu_full import fused_gpu, pages_gpu
    say(f"running max P={P} M={M}")
    d = synth.cfg_full_attention(seed=7 * P + M, M=M, P=P, pos=P * TF - M - 3 + np.arange(M), q_std=1.0)
    many = (fused_gpu(d), pages_gpu(d))
    for m in range(M):
        one = dict(d, q=np.ascontiguousarray(d["q"][m:m + 1]), masks=np.ascontiguousarray(d["masks"][:, m:m + 1]))
        for got in (fused_gpu(one), pages_gpu(one)):
            for w in many:
                assert np.array_equal(w[0][m].reshape(-1), got[0].reshape(-1)), f"row {m}"


@pytest.mark.parametrize("M,pos", [(17, 600), (65, 30)])
def test_full_projection_rows(M, pos):
    need_gpu()
    from moa_amd import ops
    from test_gpu_full import out_gpu, out_oracle, qkv_gpu, qkv_oracle
    say(f"full qkv and output M={M}")
    d = synth.cfg_full_qkv(seed=M, M=M, pos=pos)
    gq, gk, gv = qkv_gpu(d, M)
    assert ops.device_errors() == 0
    wq, wk, wv = qkv_oracle(d, M)
    s = np.arange(pos % TF, pos % TF + M)
    gate_rope(wq, gq, f"full q_out M{M}", 512)
    gate_rope(wk[s], gk[s], f"full k M{M}", 512)
    gate(wv[s], gv[s], f"full v M{M}")
    keep = np.setdiff1d(np.arange(TF), s)
    assert np.array_equal(gk[keep], d["k_cache"][keep]) and np.array_equal(gv[keep], d["v_cache"][keep])
    o = synth.cfg_full_o(seed=M, M=M)
    o["running_sum"][M - 1, 0] = 0.0  # a head with no valid slot
    gate(out_oracle(o), out_gpu(o), f"full output M{M}")


def test_full_qkv_rows_past_the_page_write_nothing():
    need_gpu()
    from moa_amd import _lib, ops
    from test_gpu_full import qkv_gpu, qkv_oracle
    say("full qkv: 20 rows, the last 8 past the page")
    d = synth.cfg_full_qkv(seed=20, M=20, pos=500)
    gq, gk, gv = qkv_gpu(d, 20)
    assert ops.device_errors() == _lib.DEVERR_KV_OFFSET
    wq, wk, wv = qkv_oracle(dict(d, x=d["x"][:12]), 12)
    gate_rope(wq, gq[:12], "full q_out rows 0-11", 512)
    assert not gq[12:].any()
    gate_rope(wk[500:], gk[500:], "full k slots 500-511", 512)
    assert np.array_equal(gk[:500], d["k_cache"][:500]) and np.array_equal(gv[:500], d["v_cache"][:500])


ROWS = [17, 64, 65, 128, 129]  # the GEMM's 64-, 128- and 256-row tiles


def picked(M):
    return sorted({0, 31, min(32, M - 1), M // 2, M - 1})


@pytest.mark.parametrize("M", ROWS)
def test_projection_row_tiles(M):
    need_gpu()
    from test_gpu_o import run_gpu as o_gpu, run_oracle as o_oracle
    from test_gpu_qkv import run_gpu as qkv_gpu, run_oracle as qkv_oracle
    say(f"qkv and o M={M}")
    rows = picked(M) if M > 31 else list(range(M))
    d = synth.cfg_qkv(M, M=M, pos=1024 - M // 2)
    q, kc, vc = qkv_gpu(d, M)
    qe, kce, vce = qkv_oracle(d, M)
    ss = (1024 - M // 2 + np.arange(M)) % 1024
    gate_rope(np.asarray(qe).reshape(M, -1), np.asarray(q).reshape(M, -1), f"qkv M{M} q", 256)
    gate_rope(np.asarray(kce).reshape(1024, -1)[ss], np.asarray(kc).reshape(1024, -1)[ss], f"qkv M{M} k", 256)
    gate(np.asarray(vce).reshape(1024, -1)[ss], np.asarray(vc).reshape(1024, -1)[ss], f"qkv M{M} v")
    o = synth.cfg_o(M, M=M)
    few = dict(o, x=o["x"][rows].copy(), residual=o["residual"][rows].copy())
    gate(o_oracle(few), o_gpu(o)[rows], f"o M{M}")


@pytest.mark.parametrize("M", ROWS)
@pytest.mark.parametrize("fmt", ["fp8", "mxfp4", "nvfp4"])
def test_ffn_row_tiles(fmt, M):
    need_gpu()
    import test_gpu_ffn as F
    say(f"ffn {fmt} M={M}")
    if fmt == "nvfp4":
        d = synth.ref_ffn_inputs(0)
        d["residual"] = prng.f32_to_bf16_bits(
            np.random.default_rng(M).standard_normal((M, 3840)).astype(np.float32))
    else:
        d = (synth.cfg_ffn_fp8 if fmt == "fp8" else synth.cfg_ffn_mxfp4)(M, M=M)
    rows = picked(M) if M > 31 else list(range(0, M, 4))
    got = getattr(F, "gpu_" + fmt)(d).reshape(M, -1)
    want = getattr(F, "oracle_" + fmt)(dict(d, residual=d["residual"][rows].copy()))
    assert np.all(np.isfinite(unbf(got.reshape(-1))))
    gate(np.asarray(want).reshape(len(rows), -1), got[rows], f"ffn {fmt} M{M}", atol=F.FFN_ATOL)


@pytest.mark.parametrize("M", [520, 769])
def test_o_sums_of_long_chunks_run_in_one_chain(M):
    """Past 512 rows the sliding O adds a column's 4096 products into one f32 chain, so a row's bits are those
    that O has always given. The odd columns' sums stand midway between two bf16 values after the first product
    ((1 + 2^-5)(1 + 2^-3), the lower of the two even); every later product is 2^-30, so the 16 that one matrix
    instruction adds are under half an f32 step of that sum and leave it. Summed apart from it, as by a second k
    split, 2048 of them are 2^-19 and push the rounding up. So the row with them and the row without must agree."""
    need_gpu()
    from test_gpu_o import run_gpu as o_gpu
    say(f"o M={M}: sums in one chain")
    d = synth.cfg_o(3, M=M)
    x = np.zeros((M, 4096), np.float32)
    x[:, 0] = 1.0 + 2.0 ** -5
    x[1::2, 1:] = 2.0 ** -24
    w = np.full((3840, 4096), 0x08, np.uint8)  # E4M3 2^-6
    w[:, 0] = 0x38                              # 1
    w[1::2, 0] = 0x39                           # 1.125
    d.update(x=prng.f32_to_bf16_bits(x), o_weight=w, o_weight_scale=np.ones(3840, np.float32),
             residual=np.zeros((M, 3840), np.uint16))
    got = o_gpu(d)
    assert not np.array_equal(got[0, 0::2], got[0, 1::2])
    assert np.array_equal(got, np.broadcast_to(got[0], got.shape))


def test_qkv_heads_bits_in_every_call_size():
    """Rows with one non-zero input have projections of one product, the same in any order of summation; the head
    norms' sums of squares are added in one order too, so a 300-row call and 16-row calls agree in every bit."""
    need_gpu()
    from test_gpu_qkv import run_gpu as qkv_gpu
    say("qkv: 300 rows and 16 at a time")
    M, pos = 300, 40
    d = synth.cfg_qkv(5, M=M, pos=pos)
    x = np.zeros((M, 3840), np.float32)
    x[np.arange(M), 11 * np.arange(M)] = 1.0 + np.arange(M) / 512.0
    d["x"] = prng.f32_to_bf16_bits(x)
    q, k, v = qkv_gpu(d, M)
    q = np.asarray(q).reshape(M, -1)
    for m in range(0, M, 16):
        n = min(16, M - m)
        few = dict(d, x=np.ascontiguousarray(d["x"][m:m + n]), rope_offset=(pos + m) * 256 * 2,
                   kv_offset=(pos + m) * 8 * 256 * 2)
        qf, kf, vf = qkv_gpu(few, n)
        at = slice(pos + m, pos + m + n)
        assert np.array_equal(q[m:m + n], np.asarray(qf).reshape(n, -1)), f"q of rows {m} .."
        assert np.array_equal(np.asarray(k)[at], np.asarray(kf)[at]), f"k of rows {m} .."
        assert np.array_equal(np.asarray(v)[at], np.asarray(vf)[at]), f"v of rows {m} .."


@pytest.mark.parametrize("M", [3, 6, 130])
def test_sliding_attention_weights_keep_their_f32_bits(M):
    """Three slots with scores 0, 0 and -s: out = (p - hi - lo) / (2 + p) with p = exp(-s) on a value of 1 and
    hi, lo, the bf16 parts of p nearest first, as the other slots' values with their signs turned. Only bits of
    p below its first 16 are left. Bound: the largest f32 step of |s log2 e| < 1 and of exp2's result is 2^-24,
    two of each and three sums of as much below 1 stay under 2^-21 in the numerator (2^-18 here); bf16 output."""
    need_gpu()
    from test_gpu_attention import run_gpu
    say(f"attention M={M}: bits of the weights")
    s = 77.0 / 128.0
    bf = lambda x: float(unbf(prng.f32_to_bf16_bits(np.array([x], np.float32)))[0])
    p = float(np.exp(np.float64(-s)))
    hi = bf(p)
    lo = bf(p - hi)
    d = synth.cfg_attention(seed=M, M=M)
    k = np.zeros((TS, 8, 256), np.float32)
    v = np.zeros((TS, 8, 256), np.float32)
    q = np.zeros((M, 8, 2, 256), np.float32)
    q[..., 0] = 1.0
    k[9, :, 0] = -s
    v[5], v[9], v[20] = -hi, 1.0, -lo
    mask = np.zeros((M, TS), np.float32)
    mask[:, [5, 9, 20]] = 1.0
    d.update(q=prng.f32_to_bf16_bits(q), k_cache=prng.f32_to_bf16_bits(k), v_cache=prng.f32_to_bf16_bits(v), mask=mask)
    got = unbf(run_gpu(d).reshape(-1)).astype(np.float64)
    want = (p - hi - lo) / (2.0 + p)
    assert abs(want) > 2.0 ** -20
    assert np.all(np.abs(got - want) <= 2.0 ** -21 / (2.0 + p) + 2.0 ** -8 * abs(want)), (got.min(), got.max(), want)


@pytest.mark.parametrize("M", [130, 260])
def test_sliding_attention_row_does_not_depend_on_its_neighbours(M):
    """A row with valid slots in every other 32-slot tile keeps its bits whichever tiles the other rows of the
    call need."""
    need_gpu()
    from test_gpu_attention import run_gpu
    say(f"attention M={M}: a row beside others")
    d = synth.cfg_attention(seed=M, M=M, q_std=0.1)
    sparse = (np.arange(TS) // 32 % 2 == 0).astype(np.float32)
    d["mask"] = np.broadcast_to(sparse, (M, TS)).copy()
    alone = run_gpu(d)
    d["mask"] = np.ones((M, TS), np.float32)
    rows = [0, 21, M - 1]
    d["mask"][rows] = sparse
    beside = run_gpu(d)
    for m in rows:
        assert np.array_equal(alone[m], beside[m]), f"row {m}"
