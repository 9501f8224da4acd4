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


def long_pages(P, M, kind):
    """Pages whose scores grow from tile to tile, so that a row's reference moves several times over a workgroup's
    tiles. scattered: random masks, tile 5 of every page and all of page 1 nobody's, a row with one late slot and a
    row with none."""
    rng = np.random.default_rng(1000 * P + M)
    grow = np.linspace(0.3, 1.0, P * 8, dtype=np.float32).reshape(P, 8, 1, 1)
    k = rng.standard_normal((P, 8, 64, 512), np.float32) * grow
    masks = synth.full_masks(P, P * TF - M - 100 + np.arange(M))
    if kind == "scattered":
        masks = (rng.random((P, M, TF), np.float32) < 0.3).astype(np.float32)
        masks[:, :, 320:384] = 0.0
        masks[1] = 0.0
        masks[:, M // 2] = 0.0
        masks[P - 1, M // 2, 500] = 1.0
        masks[:, M - 2] = 0.0
    b = prng.f32_to_bf16_bits
    return dict(q=b(rng.standard_normal((M, 16, 512), np.float32)), k_pages=b(k.reshape(P, TF, 512)),
                v_pages=b(rng.standard_normal((P, TF, 512), np.float32)), masks=masks)


@pytest.mark.parametrize("P,M,kind", [(6, 200, "causal"), (6, 200, "scattered"), (20, 40, "scattered"), (40, 130, "causal"),
                                      (64, 130, "scattered")])
def test_full_attention_rows_over_many_tiles(P, M, kind):
    """On 256 CUs 10, 7, 46 and 64 tiles per workgroup (200, 40, 130 and 130 rows): the pipeline beyond its first
    tiles, tiles left out between others, repeated rescaling and every pass over the mask bits. 130 rows of 64 pages
    are two launches, of 128 rows and of 2."""
    need_gpu()
    from test_gpu_full import fused_gpu
    say(f"full attention P={P} M={M} {kind}")
    d = long_pages(P, M, kind)
    got = fused_gpu(d)
    rows = sorted({0, 3, 4, M // 2, min(127, M - 3), M - 2, M - 1})
    few = dict(d, q=np.ascontiguousarray(d["q"][rows]), masks=np.ascontiguousarray(d["masks"][:, rows]))
    check_pages(few, [x[rows] for x in got], f"pages P{P} M{M} {kind}")
    if kind == "scattered":
        assert np.all(got[0][M - 2] == -np.inf) and not got[1][M - 2].any() and not got[2][M - 2].any()
        assert np.all(got[1][M // 2] == 1.0)
        assert np.array_equal(got[2][M // 2].reshape(16, 512), np.broadcast_to(d["v_pages"][P - 1, 500], (16, 512)))


@pytest.mark.parametrize("M", [129, 256, 257, 300])
def test_full_projection_row_tiles(M):
    """The 256-row tile in one and two row blocks, QKV with two splits and one, O on 64 and 128 weight rows, and the
    division by the sums over XCD-ordered rows."""
    need_gpu()
    from moa_amd import ops
    from test_gpu_full import out_gpu, out_oracle, qkv_gpu, qkv_oracle
    say(f"full qkv and output M={M}")
    pos, rows = 5, sorted({0, 31, 63, 64, 127, 128, min(256, M - 1), M - 1})
    d = synth.cfg_full_qkv(seed=M, M=M, pos=pos)
    gq, gk, gv = qkv_gpu(d, M)
    assert ops.device_errors() == 0
    for m in rows:
        one = dict(d, x=d["x"][m:m + 1], rope_offset=(pos + m) * 1024, kv_offset=(pos + m) * 1024)
        wq, wk, wv = qkv_oracle(one, 1)
        gate_rope(wq, gq[m:m + 1], f"full q_out M{M} row {m}", 512)
        gate_rope(wk[pos + m], gk[pos + m], f"full k M{M} row {m}", 512)
        gate(wv[pos + m], gv[pos + m], f"full v M{M} row {m}")
    keep = np.setdiff1d(np.arange(TF), pos + np.arange(M))
    assert np.array_equal(gk[keep], d["k_cache"][keep]) and np.array_equal(gv[keep], d["v_cache"][keep])
    o = synth.cfg_full_o(seed=M, M=M)
    o["running_sum"][M - 1, 0] = 0.0  # heads with no valid slot
    o["running_sum"][64, 15] = 0.0
    few = dict(o, x=o["x"][rows].copy(), running_sum=o["running_sum"][rows].copy(), residual=o["residual"][rows].copy())
    gate(out_oracle(few), out_gpu(o)[rows], f"full output M{M}")


def test_full_output_call_of_two_chunks():
    """1030 rows are a chunk of 1024 and one of 6: the first chunk's bits are those of a 1024-row call, and the last
    rows use their own sums."""
    need_gpu()
    from test_gpu_full import out_gpu, out_oracle
    say("full output: 1030 rows")
    o = synth.cfg_full_o(seed=30, M=1030)
    o["running_sum"][1027, 2] = 0.0
    part = lambda lo, hi: dict(o, **{k: np.ascontiguousarray(o[k][lo:hi]) for k in ("x", "running_sum", "residual")})
    got = out_gpu(o)
    assert np.array_equal(got[:1024], out_gpu(part(0, 1024)))
    gate(out_oracle(part(1024, 1030)), got[1024:], "full output, rows 1024 .. 1029")


def test_full_qkv_call_of_two_chunks_past_the_page():
    """520 rows from slot 0 are a chunk of 512 and one of 8, whose rows fall past the page: the page and q_out of
    the first 512 are those of a 512-row call, and the others write nothing and are reported."""
    need_gpu()
    from moa_amd import _lib, ops
    from test_gpu_full import qkv_gpu
    say("full qkv: 520 rows")
    d = synth.cfg_full_qkv(seed=52, M=520, pos=0)
    gq, gk, gv = qkv_gpu(d, 520)
    assert ops.device_errors() == _lib.DEVERR_KV_OFFSET
    hq, hk, hv = qkv_gpu(dict(d, x=np.ascontiguousarray(d["x"][:512])), 512)
    assert ops.device_errors() == 0
    assert np.array_equal(gq[:512], hq) and np.array_equal(gk, hk) and np.array_equal(gv, hv)
    assert not gq[512:].any()


def test_graph_replays_of_many_rows_match_eager():
    """The calls of many rows captured in one graph: every replay gives the eager bits."""
    need_gpu()
    from gpu_util import dev, host, torch
    from moa_amd import ops
    ops.init(0)
    up = lambda d, *skip: {k: dev(v) for k, v in d.items() if isinstance(v, np.ndarray) and k not in skip}
    i32 = lambda v: torch.tensor([int(v)], dtype=torch.int32, device="cuda")
    bits = lambda *shape: torch.zeros(shape, dtype=torch.int16, device="cuda")
    f32 = lambda n: torch.zeros(n, device="cuda")
    at = up(synth.cfg_attention(9, M=40, pos=300 + np.arange(40)))
    qv = synth.cfg_qkv(9, M=40, pos=1000)
    Q, ffn, o = up(qv), up(synth.cfg_ffn_fp8(9, M=40)), up(synth.cfg_o(9, M=40))
    fq = synth.cfg_full_qkv(9, M=20, pos=30)
    F, fo = up(fq), up(synth.cfg_full_o(9, M=20))
    fa, pg = up(synth.cfg_full_attention(9, M=66, P=2, q_std=0.3)), up(synth.cfg_full_attention(8, M=19, P=2, q_std=0.3))
    lg, lm = up(synth.cfg_logits(9, M=24)), synth.lm_head_device(9)
    kv, ro, fkv, fro = i32(qv["kv_offset"]), i32(qv["rope_offset"]), i32(fq["kv_offset"]), i32(fq["rope_offset"])
    outs = dict(attn=bits(40, 4096), q=bits(40, 4096), kc=bits(*Q["k_cache"].shape), vc=bits(*Q["v_cache"].shape),
                res=bits(40, 3840), fq=bits(20, 8192), fk=bits(*F["k_cache"].shape), fv=bits(*F["v_cache"].shape),
                fres=bits(20, 3840), fmax=f32(66 * 16), fsum=f32(66 * 16), fout=bits(66, 8192), pmax=f32(19 * 16),
                psum=f32(19 * 16), pout=bits(19, 8192), logits=bits(24, synth.W))
    t = outs

    def step():
        for n, x in (("kc", Q["k_cache"]), ("vc", Q["v_cache"]), ("res", o["residual"]), ("fk", F["k_cache"]),
                     ("fv", F["v_cache"]), ("fres", fo["residual"])):
            t[n].copy_(x)
        ops.sliding_attention(at["q"], at["k_cache"], at["v_cache"], at["mask"], t["attn"])
        ops.sliding_project_qkv(Q["x"], Q["q_weight"], Q["k_weight"], Q["v_weight"], Q["q_weight_scale"],
                                Q["k_weight_scale"], Q["v_weight_scale"], Q["input_rms_weight"], Q["q_rms_weight"],
                                Q["k_rms_weight"], kv, ro, Q["cos"], Q["sin"], t["kc"], t["vc"], t["q"])
        ops.sliding_attention_output_feedforward_fp8(
            o["x"], o["post_attn_rms_weight"], o["o_weight"], o["o_weight_scale"], t["res"], ffn["pre_ff_rms_weight"],
            ffn["up_weight"], ffn["gate_weight"], ffn["down_weight"], ffn["up_weight_scale"], ffn["gate_weight_scale"],
            ffn["down_weight_scale"], ffn["post_ff_rms_weight"], ffn["layer_scalar"])
        ops.full_project_qkv(F["x"], F["q_weight"], F["k_weight"], F["q_weight_scale"], F["k_weight_scale"],
                             F["input_rms_weight"], F["q_rms_weight"], F["k_rms_weight"], fkv, fro, F["cos"], F["sin"],
                             t["fk"], t["fv"], t["fq"])
        ops.full_attention_output(fo["x"], fo["running_sum"], fo["post_attn_rms_weight"], fo["o_weight"],
                                  fo["o_weight_scale"], t["fres"])
        ops.full_attention(fa["q"], fa["k_pages"], fa["v_pages"], fa["masks"], t["fmax"], t["fsum"], t["fout"])
        for p, call in enumerate((ops.full_attention_first_page, ops.full_attention_page)):
            call(pg["q"], pg["k_pages"][p], pg["v_pages"][p], pg["masks"][p], t["pmax"], t["psum"], t["pout"])
        ops.final_norm_and_logits(lg["input"], lg["rms_weight"], lm, t["logits"])

    def read():
        return {n: host(x).copy() for n, x in t.items()}

    step()
    want = read()
    assert ops.device_errors() == 0 and all(w.any() for w in want.values())
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        step()
    for replay in range(4):
        say(f"graph replay {replay}")
        for x in t.values():
            x.fill_(0)  # eager work between replays
        torch.cuda.synchronize()
        g.replay()
        for n, got in read().items():
            assert np.array_equal(want[n], got), f"replay {replay}: {n} differs from the eager result"
        step()
        for n, got in read().items():
            assert np.array_equal(want[n], got), f"eager after replay {replay}: {n}"
    assert ops.device_errors() == 0
