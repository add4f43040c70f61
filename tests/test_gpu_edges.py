"""Kernels at the edges of their geometry (group counts at and just past the
lane layouts, partial tiles, the smallest and largest row counts), against the
oracle."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest
import torch

from maxuna_amd import ops
from maxuna_amd._lib import lib
from maxuna_amd.gguf import ExpertStack, GgmlDType
from maxuna_amd.synth import LayerSpec, build_layer, make_x, synth_stack, tensor_key

from tests.gpu_util import assert_close, check_ids, dev_f32, dev_u32, host, rel_l2, selection_margin

pytestmark = pytest.mark.gpu

# f32-class arithmetic (24-bit activation grid, exact integer plane sums, a few
# f32 roundings per sub-block): the bound the precision tests hold decode layers to
F32_CLASS = 1e-5


def layer_against_oracle(orc, spec, t, seed, bound):
    layer = build_layer(spec, seed=seed)
    x = make_x(spec, seed + 1, t)
    out, ids, w = layer.block.forward(torch.from_numpy(x).cuda(), return_routing=True)
    out, ids = host(out), host(ids)
    want, oid, _ = orc.moe_layer(spec, layer.keys, layer.router_t, layer.bias, x)
    logits = x.astype(np.float64) @ layer.router.T.astype(np.float64)
    assert check_ids(ids, oid, selection_margin(logits, layer.bias, spec.top_k)) == 0
    r = rel_l2(out, want)
    print(f"{spec} t={t}: rel-L2 {r:.2e}", flush=True)
    assert r <= bound


# hidden: groups per row at the lane layouts' ends (16 | 32 | 64 lanes of one
# group, 32 lanes of three, 64 lanes of two and more) and just past them; ff 544
# and 96 leave partial passes and workgroups
GU_ROWS = [
    (GgmlDType.Q4_K, 256), (GgmlDType.Q4_K, 1280), (GgmlDType.Q4_K, 2304), (GgmlDType.Q4_K, 4352),
    (GgmlDType.Q4_K, 6400), (GgmlDType.Q4_K, 8448), (GgmlDType.Q4_K, 12544), (GgmlDType.Q5_K, 2048),
    (GgmlDType.Q5_K, 6144), (GgmlDType.Q5_K, 8192), (GgmlDType.Q5_K, 8448), (GgmlDType.Q6_K, 512),
    (GgmlDType.Q6_K, 2304), (GgmlDType.Q6_K, 4352), (GgmlDType.Q6_K, 6400), (GgmlDType.Q6_K, 8448),
    (GgmlDType.Q8_0, 32), (GgmlDType.Q8_0, 544), (GgmlDType.Q8_0, 1056), (GgmlDType.Q8_0, 2080),
    (GgmlDType.Q8_0, 3104), (GgmlDType.Q8_0, 4128), (GgmlDType.Q8_0, 6688),
]


@pytest.mark.parametrize("dt,hidden", GU_ROWS, ids=lambda v: str(getattr(v, "name", v)))
def test_decode_gate_up_row_widths(orc, dt, hidden):
    for t, ff in ((1, 544), (3, 96)):
        spec = LayerSpec(hidden, ff, 12, 3, dt, GgmlDType.Q8_0, shared=True)
        layer_against_oracle(orc, spec, t, 4200 + t, F32_CLASS)


@pytest.mark.parametrize("dt,hidden", [GU_ROWS[i] for i in (6, 10, 13, 14, 15)], ids=lambda v: str(getattr(v, "name", v)))
def test_decode_gate_up_wide_rows_passes(orc, dt, hidden):
    """Rows contracted group by group, four and eight passes a wave: each row's copy follows
    the last read of the row before it in the same buffer."""
    for t, ff in ((1, 4160), (3, 2112)):
        spec = LayerSpec(hidden, ff, 12, 3, dt, GgmlDType.Q8_0, shared=True)
        layer_against_oracle(orc, spec, t, 4220 + t, F32_CLASS)


# k / ff: groups per row at the lane layouts' ends and just past them
DOWN_ROWS = [
    (GgmlDType.Q4_K, 512), (GgmlDType.Q4_K, 768), (GgmlDType.Q4_K, 1280), (GgmlDType.Q4_K, 2304),
    (GgmlDType.Q4_K, 4352), (GgmlDType.Q4_K, 8448), (GgmlDType.Q5_K, 1024), (GgmlDType.Q5_K, 2048),
    (GgmlDType.Q5_K, 4096), (GgmlDType.Q6_K, 512), (GgmlDType.Q6_K, 768), (GgmlDType.Q6_K, 1024),
    (GgmlDType.Q6_K, 1280), (GgmlDType.Q6_K, 1792), (GgmlDType.Q6_K, 2304), (GgmlDType.Q6_K, 3328),
    (GgmlDType.Q6_K, 8192), (GgmlDType.Q8_0, 32), (GgmlDType.Q8_0, 544), (GgmlDType.Q8_0, 800),
    (GgmlDType.Q8_0, 1056), (GgmlDType.Q8_0, 1568), (GgmlDType.Q8_0, 2080), (GgmlDType.Q8_0, 3104),
    (GgmlDType.Q8_0, 4128), (GgmlDType.Q8_0, 8224),
]


@pytest.mark.parametrize("dt,ff", DOWN_ROWS, ids=lambda v: str(getattr(v, "name", v)))
def test_decode_down_row_widths(orc, dt, ff):
    # hidden 288: a last tile of 8 rows at 16 or 64 rows a workgroup
    for t in (1, 2, 3, 7):
        spec = LayerSpec(288, ff, 12, 3, GgmlDType.Q8_0, dt, shared=True)
        layer_against_oracle(orc, spec, t, 4300 + t, F32_CLASS)


@pytest.mark.parametrize("dt,k", DOWN_ROWS, ids=lambda v: str(getattr(v, "name", v)))
def test_mul_mv_row_widths(orc, dt, k):
    rng = np.random.default_rng(k)
    for n_out, t in ((1, 1), (5, 1), (333, 1), (4099, 1)):
        st = synth_stack(dt, 1, n_out, k, tensor_key(4400, 0, n_out))
        x = rng.standard_normal((t, k)).astype(np.float32)
        got = host(ops.mul_mv(st.buffer, dt, n_out, k, dev_f32(x)))
        w = orc.dequantize(int(dt), host(st.buffer), n_out * k).reshape(n_out, k)
        r = rel_l2(got, x.astype(np.float64) @ w.astype(np.float64).T)
        print(f"{dt.name} [{n_out} x {k}] t={t}: rel-L2 {r:.2e}", flush=True)
        assert r <= F32_CLASS


# rows at and just past the ends of the lane layouts of three and six groups
THREES = [
    (GgmlDType.Q4_K, 3072), (GgmlDType.Q4_K, 3328), (GgmlDType.Q4_K, 6144), (GgmlDType.Q5_K, 4352),
    (GgmlDType.Q5_K, 6144), (GgmlDType.Q5_K, 12288), (GgmlDType.Q6_K, 4352), (GgmlDType.Q6_K, 6144),
    (GgmlDType.Q6_K, 8448), (GgmlDType.Q6_K, 12288), (GgmlDType.Q8_0, 4128), (GgmlDType.Q8_0, 6144),
    (GgmlDType.Q8_0, 12288), (GgmlDType.Q8_0, 12320),
]


@pytest.mark.parametrize("dt,k", THREES, ids=lambda v: str(getattr(v, "name", v)))
def test_mul_mv_id_grids(orc, dt, k):
    """One batch a wave, whole rounds of workgroups and rounds that share a wave's batches
    unevenly: 2, 26 and 330 pairs of a row count that no batch divides."""
    rng = np.random.default_rng(k)
    e, n_out, top_k = 3, 197, 2
    st = synth_stack(dt, e, n_out, k, tensor_key(4460, 0, k))
    w = orc.dequantize(int(dt), host(st.buffer), e * n_out * k).reshape(e, n_out, k).astype(np.float64)
    for t in (1, 13, 165):
        x = rng.standard_normal((t, 1, k)).astype(np.float32)
        ids = np.stack([rng.permutation(e)[:top_k] for _ in range(t)])
        got = host(ops.mul_mv_id(st, dev_f32(x), dev_u32(ids)))
        y = x[:, 0].astype(np.float64) @ w.reshape(e * n_out, k).T
        want = y.reshape(t, e, n_out)[np.arange(t)[:, None], ids]
        r = rel_l2(got, want)
        print(f"{dt.name} k={k} t={t}: rel-L2 {r:.2e}", flush=True)
        assert r <= F32_CLASS


@pytest.mark.parametrize("dt,ff", [THREES[i] for i in (0, 2, 4, 7, 12)], ids=lambda v: str(getattr(v, "name", v)))
def test_decode_down_rows_of_three(orc, dt, ff):
    for t in (1, 2, 5):
        spec = LayerSpec(288, ff, 12, 3, GgmlDType.Q8_0, dt, shared=True)
        layer_against_oracle(orc, spec, t, 4310 + t, F32_CLASS)


@pytest.mark.parametrize("hidden,ff,top_k,ts", [
    (1024, 512, 3, (3, 4, 5)), (2048, 512, 3, (2, 3, 4)), (5120, 512, 3, (1, 2)), (8192, 512, 3, (1, 2)),
    (4128, 256, 1, (3, 4)), (5120, 512, 5, (1, 2)), (2048, 512, 11, (1, 2, 3, 4)), (1024, 1536, 3, (3, 4, 5))])
def test_decode_down_slots_line(orc, hidden, ff, top_k, ts):
    """Both sides of the slot-per-wave down kernel's lines: one round of its tiles of 16 rows,
    a partly filled second round, two full rounds; few slots (several workgroups per CU), many,
    and Q6_K rows of 1536."""
    for t in ts:
        spec = LayerSpec(hidden, ff, 12, top_k, GgmlDType.Q8_0, GgmlDType.Q6_K, shared=top_k < 11)
        layer_against_oracle(orc, spec, t, 4320 + t, F32_CLASS)


# rows the f32 mat-vec holds: seven groups times a power of two, and rows too wide for
# the mat-vec's two copies in LDS (the narrowest of each type whose scale group is 128 values)
F32_ROWS = [
    (GgmlDType.Q4_K, 1792), (GgmlDType.Q4_K, 7168), (GgmlDType.Q4_K, 14336), (GgmlDType.Q4_K, 20224),
    (GgmlDType.Q5_K, 3584), (GgmlDType.Q5_K, 7168), (GgmlDType.Q5_K, 14336), (GgmlDType.Q5_K, 17920),
    (GgmlDType.Q6_K, 16384), (GgmlDType.Q8_0, 13568),
]


def _no_weight_in_first_group(buffer, dt):
    """Zeroes the weights of the first 32 values of every 256 (of every 128 for Q8_0)."""
    raw = buffer.reshape(-1, dt.type_size)
    if dt in (GgmlDType.Q4_K, GgmlDType.Q5_K):  # the first sub-block's 6-bit scale and minimum
        raw[:, 4] &= 0xC0
        raw[:, 8] &= 0xC0
    elif dt == GgmlDType.Q6_K:  # the first two 16-value groups' scales
        raw[:, 192:194] = 0
    else:  # every fourth block's scale
        raw[::4, 0:2] = 0


@pytest.mark.parametrize("dt,k", F32_ROWS, ids=lambda v: str(getattr(v, "name", v)))
def test_f32_rows_keep_their_precision(orc, dt, k):
    """Activations held in f32: a value of 2^20 that meets only zero weights takes nothing
    from the 127 others of its scale group (the 24-bit block grid would hold those to
    2^-4).  Bound: f32 products and sums, as the precision tests hold the mat-vec to."""
    rng = np.random.default_rng(k)
    e, n_out, t, top_k = 4, 70, 2, 2
    st = synth_stack(dt, e, n_out, k, tensor_key(4450, 0, k))
    _no_weight_in_first_group(st.buffer, dt)
    x = rng.standard_normal((t, 1, k)).astype(np.float32)
    x[..., :: 256 if dt.block_size == 256 else 128] = np.float32(2.0**20)
    ids = np.stack([rng.permutation(e)[:top_k] for _ in range(t)])
    got = host(ops.mul_mv_id(st, dev_f32(x), dev_u32(ids)))
    w = orc.dequantize(int(dt), host(st.buffer), e * n_out * k).reshape(e, n_out, k).astype(np.float64)
    want = np.einsum("tsnk,tk->tsn", w[ids], x[:, 0].astype(np.float64))
    r = rel_l2(got, want)
    print(f"{dt.name} k={k}: rel-L2 {r:.2e}", flush=True)
    assert r <= 2e-6


@pytest.mark.parametrize("dt,ff", [(GgmlDType.Q4_K, 1792), (GgmlDType.Q4_K, 7168), (GgmlDType.Q4_K, 14336),
                                   (GgmlDType.Q5_K, 7168)], ids=lambda v: str(getattr(v, "name", v)))
def test_f32_down_rows_keep_the_layer_in_f32(orc, dt, ff):
    """Layers with such down rows run the f32 mat-vecs below 32 tokens, also at the
    token counts whose experts elsewhere take f16 operands (an error near 5e-4)."""
    spec = LayerSpec(512, ff, 8, 2, GgmlDType.Q4_K, dt, shared=False)
    for t in (1, 5, 20):
        layer_against_oracle(orc, spec, t, 4470 + t, F32_CLASS)


SHORT_ROWS = [(GgmlDType.Q4_K, 256), (GgmlDType.Q5_K, 256), (GgmlDType.Q6_K, 256), (GgmlDType.Q8_0, 256), (GgmlDType.Q8_0, 288)]


@pytest.mark.parametrize("dt,ff", SHORT_ROWS, ids=lambda v: str(getattr(v, "name", v)))
def test_decode_down_short_rows(orc, dt, ff):
    for t in (1, 2, 3, 7):
        spec = LayerSpec(288, ff, 12, 3, GgmlDType.Q8_0, dt, shared=True)
        layer_against_oracle(orc, spec, t, 4340 + t, F32_CLASS)


@pytest.mark.parametrize("dt,k", SHORT_ROWS, ids=lambda v: str(getattr(v, "name", v)))
def test_mul_mv_id_short_rows(orc, dt, k):
    """Few to many batches a wave, row counts that no batch divides.  Bound per output (a short
    dot may cancel to nothing): the activation grid's 2^-23 (1 + 2^-8) of a scale group's largest
    value on every weight of it, and two f32 roundings of the sum of magnitudes."""
    rng = np.random.default_rng(k)
    e, top_k, group = 3, 2, 128 if k % 128 == 0 else 32
    for n_out, t in ((1, 1), (5, 2), (333, 9), (2049, 40)):
        st = synth_stack(dt, e, n_out, k, tensor_key(4480, 0, n_out))
        w = orc.dequantize(int(dt), host(st.buffer), e * n_out * k).reshape(e, n_out, k).astype(np.float64)
        x = rng.standard_normal((t, 1, k)).astype(np.float32)
        ids = np.stack([rng.permutation(e)[:top_k] for _ in range(t)])
        got = host(ops.mul_mv_id(st, dev_f32(x), dev_u32(ids)))
        xd, aw = x[:, 0].astype(np.float64), np.abs(w)
        top = np.repeat(np.abs(xd).reshape(t, -1, group).max(-1), group, axis=1)
        pick = lambda y: y.reshape(t, e, n_out)[np.arange(t)[:, None], ids]  # noqa: E731
        err = np.abs(got - pick(xd @ w.reshape(-1, k).T))
        bound = pick((2.0**-23 * (1 + 2.0**-8) * top + 2.0**-23 * np.abs(xd)) @ aw.reshape(-1, k).T)
        print(f"{dt.name} [{n_out} x {k}] t={t}: {np.max(err / bound):.3f} of the bound", flush=True)
        assert np.all(err <= bound)


def _mul_mv_errors(orc, dt, n_out, k, x, off=0):
    """Relative error of each token's row of mul_mv against float64."""
    st = synth_stack(dt, 1, n_out, k, tensor_key(4500, 0, n_out))
    raw = torch.zeros(off + st.nbytes, dtype=torch.uint8, device="cuda")
    raw[off:] = st.buffer
    got = host(ops.mul_mv(raw[off:], dt, n_out, k, dev_f32(x))).astype(np.float64)
    w = orc.dequantize(int(dt), host(st.buffer), n_out * k).reshape(n_out, k).astype(np.float64)
    want = x.astype(np.float64) @ w.T
    return np.linalg.norm(got - want, axis=1) / np.linalg.norm(want, axis=1)


# two f16 pieces carry an activation to 2^-23 of itself, so f32 sums dominate: rows
# of at most 6400 centred products, errors near 2e-7 (bound: 1e-6 per token)
TOKENS = 1e-6


@pytest.mark.parametrize("dt", [GgmlDType.Q4_K, GgmlDType.Q5_K, GgmlDType.Q6_K, GgmlDType.Q8_0], ids=lambda v: v.name)
@pytest.mark.parametrize("k", [256, 512, 1792, 3072, 3328, 6400])
def test_mul_mv_tokens(orc, dt, k):
    """1 to 12 waves a workgroup, and K cut into two and three launches; partial row
    tiles and token groups; weights off 16-byte alignment where the type allows it."""
    rng = np.random.default_rng(k)
    off = 2 if dt in (GgmlDType.Q6_K, GgmlDType.Q8_0) else 0
    for n_out, t in ((1, 2), (15, 3), (16, 16), (17, 17), (333, 5), (4200, 33)):
        err = _mul_mv_errors(orc, dt, n_out, k, rng.standard_normal((t, k)).astype(np.float32), off)
        print(f"{dt.name} [{n_out} x {k}] t={t}: {err.max():.2e}", flush=True)
        assert err.max() <= (TOKENS if n_out > 16 else F32_CLASS)


@pytest.mark.parametrize("dt", [GgmlDType.Q4_K, GgmlDType.Q5_K, GgmlDType.Q6_K, GgmlDType.Q8_0], ids=lambda v: v.name)
@pytest.mark.parametrize("k", [256, 1024, 3072, 3328, 6400])
def test_mul_mv_tokens_taken(orc, dt, k):
    """Calls past the line between a mat-vec per token and the several-token kernel: partial
    row tiles and token groups, 1 to 12 waves, K in up to three launches.  A value of 2^20
    that meets zero weights tells the two apart: the several-token kernel holds its
    neighbours to 2^-40 of it (an error near 1e-6), the block grid to 2^-23 (4e-2)."""
    rng = np.random.default_rng(k)
    for n_out in (17, 333, 4201):
        st = synth_stack(dt, 1, n_out, k, tensor_key(4520, 0, n_out))
        t = int(1e8) * (k // 3073 + 2) // st.nbytes | 1  # (by bytes: the line's measure)
        _no_weight_in_first_group(st.buffer, dt)
        x = rng.standard_normal((t, k)).astype(np.float32)
        x[:, ::256] = np.float32(2.0**20)
        got = host(ops.mul_mv(st.buffer, dt, n_out, k, dev_f32(x)))
        w = orc.dequantize(int(dt), host(st.buffer), n_out * k).reshape(n_out, k).astype(np.float64)
        r = rel_l2(got, x.astype(np.float64) @ w.T)
        print(f"{dt.name} [{n_out} x {k}] t={t}: rel-L2 {r:.2e}", flush=True)
        assert r <= F32_CLASS


@pytest.mark.parametrize("exponent", [-124, -114, 100])
def test_mul_mv_tokens_magnitudes(orc, exponent):
    """Whole calls of very small and very large activations through the several-token kernel,
    with the block scales of centred weights (2e-5): no product of a block's scale and the
    token's power of two may lose bits."""
    rng = np.random.default_rng(5)
    n_out, k, t = 4201, 1024, 143
    st = synth_stack(GgmlDType.Q6_K, 1, n_out, k, tensor_key(4530, 0, 0))
    d = (2e-5 * (0.5 + rng.random(n_out * k // 256))).astype(np.float16)
    st.buffer.reshape(-1, 210)[:, 208:210] = torch.from_numpy(d.view(np.uint8).reshape(-1, 2)).cuda()
    x = (rng.standard_normal((t, k)) * 2.0**exponent).astype(np.float32)
    got = host(ops.mul_mv(st.buffer, GgmlDType.Q6_K, n_out, k, dev_f32(x)))
    w = orc.dequantize(int(GgmlDType.Q6_K), host(st.buffer), n_out * k).reshape(n_out, k).astype(np.float64)
    want = x.astype(np.float64) @ w.T
    r = rel_l2(got.astype(np.float64) * 2.0**-exponent, want * 2.0**-exponent)
    print(f"2^{exponent}: {r:.2e}", flush=True)
    assert r <= TOKENS


def test_mul_mv_tokens_ranges(orc):
    """Tokens of very different magnitudes, super-blocks 2^40 apart, an all-zero token,
    and a token with an Inf: only that token's outputs are not finite."""
    rng = np.random.default_rng(3)
    k, n_out = 1024, 200
    x = rng.standard_normal((6, k)).astype(np.float32)
    x[1] *= np.float32(2.0**-100)
    x[2] *= np.float32(2.0**90)
    x[3, 256:512] *= np.float32(2.0**40)
    x[4] = 0
    for dt in (GgmlDType.Q4_K, GgmlDType.Q6_K):
        err = _mul_mv_errors(orc, dt, n_out, k, x[[0, 1, 2, 3]])
        assert err.max() <= TOKENS, err
        st = synth_stack(dt, 1, n_out, k, 9)
        bad = x.copy()
        bad[5, 700] = np.inf
        got = host(ops.mul_mv(st.buffer, dt, n_out, k, dev_f32(bad)))
        assert np.all(np.isfinite(got[:5])) and np.all(got[4] == 0) and not np.any(np.isfinite(got[5]))


# (gate/up type, down type, hidden, ff): every type on both projections, an odd and an even
# number of super-blocks
SMALL_GROUPED = [
    ("Q4_K", "Q4_K", 512, 768), ("Q4_K", "Q6_K", 1280, 1536), ("Q4_K", "Q6_K", 3072, 1792), ("Q4_K", "Q4_K", 3328, 1024),
    ("Q4_K", "Q5_K", 4352, 512), ("Q4_K", "Q6_K", 6400, 512), ("Q5_K", "Q5_K", 1024, 2304), ("Q5_K", "Q6_K", 3584, 1280),
    ("Q6_K", "Q6_K", 1536, 768), ("Q6_K", "Q5_K", 3840, 512), ("Q6_K", "Q4_K", 5120, 512), ("Q8_0", "Q8_0", 512, 1024),
    ("Q8_0", "Q8_0", 2048, 1280), ("Q8_0", "Q8_0", 2560, 768), ("Q8_0", "Q8_0", 4096, 512), ("Q8_0", "Q8_0", 5632, 512),
]


@pytest.mark.parametrize("gate,down,hidden,ff", SMALL_GROUPED)
def test_few_pairs_small_matrices(orc, gate, down, hidden, ff):
    """Layers of a few pairs per expert, skewed, past the verify tiles, whose matrices are
    small: the grouped GEMM, or the matmuls of few pairs for Q6_K gate/up and where the GEMM
    would have few workgroups, against the oracle's own routing.  f16 operands: the contract's
    bound."""
    spec = LayerSpec(hidden, ff, 40, 4, GgmlDType[gate], GgmlDType[down], shared=hidden % 512 == 0, bias_sigma=0.3)
    layer = build_layer(spec, seed=4600)
    t = 50 if hidden > 4096 else 210 if gate == "Q4_K" else 70
    tried = [w >= 0 for w in few_pairs_words(layer.block, t)]
    assert tried[0] or gate != "Q6_K"
    assert not any(tried) or gate == "Q6_K" or 12 * 40 > 4 * t
    x = make_x(spec, 4601, t)
    out, ids, w = layer.block.forward(torch.from_numpy(x).cuda(), return_routing=True)
    out, ids, w = host(out), host(ids), host(w)
    want, _, _ = orc.moe_layer(spec, layer.keys, layer.router_t, layer.bias, x, ids=ids, w=w)
    assert_close(out, want, what=f"{gate}/{down} {hidden}x{ff}")


def few_pairs_words(block, t):
    """Workspace offsets of the words that say whether the matmuls for few pairs per expert
    took gate/up and down (-1: not tried)."""
    gu, dn = C.c_int64(), C.c_int64()
    lib().mx_moe_few_pairs_words(C.byref(block._c), t, C.byref(gu), C.byref(dn))
    return gu.value, dn.value


def moe_f64(block, x, ids, w):
    """The layer in 64-bit torch from the dequantised stacks and the given routing."""
    def weights(st, e):
        step = st.n_out * st.k // st.dtype.block_size * st.dtype.type_size
        return ops.dequantize(st.buffer[e * step:(e + 1) * step], st.dtype, st.n_out * st.k).double().reshape(st.n_out, st.k)

    def expert(x, gate, up, down, e):
        g, u = x @ weights(gate, e).T, x @ weights(up, e).T
        return (g / (1.0 + torch.exp(-g)) * u) @ weights(down, e).T

    x, ids, w = x.double(), ids.view(torch.int32).long(), w.double()
    out = torch.zeros_like(x)
    b = block.experts
    for e in torch.unique(ids).tolist():
        tok, slot = torch.nonzero(ids == e, as_tuple=True)
        out.index_add_(0, tok, expert(x[tok], b.gate, b.up, b.down, e) * w[tok, slot][:, None])
    if block.shared is not None:
        out += expert(x, block.shared.gate, block.shared.up, block.shared.down, 0)
    return out


# (gate/up type, down type, hidden, ff): the K of both projections through every wave
# layout of the stationary-activation matmuls (2, 4, 6 and 12 waves of one super-block, 8 of
# two, of three and of four; Q8_0 4 and 6 of two in place of 6 and 12 of one), at the ends of
# each: full and partly filled teams and last waves, several teams
GST = [
    ("Q4_K", "Q4_K", 1280, 512), ("Q4_K", "Q6_K", 1536, 1536), ("Q4_K", "Q5_K", 1792, 768), ("Q4_K", "Q4_K", 3072, 1024),
    ("Q4_K", "Q6_K", 3328, 512), ("Q4_K", "Q4_K", 4096, 1280), ("Q4_K", "Q5_K", 4352, 1536), ("Q4_K", "Q6_K", 6144, 1024),
    ("Q4_K", "Q4_K", 6400, 2304), ("Q4_K", "Q6_K", 8192, 3072),
    ("Q5_K", "Q5_K", 1280, 512), ("Q5_K", "Q6_K", 1792, 768), ("Q5_K", "Q5_K", 3072, 1024), ("Q5_K", "Q6_K", 4096, 3328),
    ("Q5_K", "Q5_K", 6144, 2304), ("Q5_K", "Q4_K", 6400, 3328), ("Q5_K", "Q5_K", 4352, 4096), ("Q5_K", "Q4_K", 2048, 4352),
    ("Q6_K", "Q6_K", 1536, 4352), ("Q6_K", "Q4_K", 1792, 8192), ("Q6_K", "Q6_K", 3840, 6400), ("Q6_K", "Q5_K", 5120, 6144),
    ("Q6_K", "Q6_K", 7168, 512), ("Q6_K", "Q5_K", 3072, 6400),
    ("Q8_0", "Q8_0", 1280, 512), ("Q8_0", "Q8_0", 2048, 1024), ("Q8_0", "Q8_0", 2304, 1280), ("Q8_0", "Q8_0", 3072, 2048),
    ("Q8_0", "Q8_0", 3328, 2304), ("Q8_0", "Q8_0", 4096, 3072), ("Q8_0", "Q8_0", 4352, 4096), ("Q8_0", "Q8_0", 6400, 4352),
    ("Q8_0", "Q8_0", 1536, 6400),
]


@pytest.mark.parametrize("gate,down,hidden,ff", GST)
def test_few_pairs_per_expert(gate, down, hidden, ff):
    """Layers whose gate/up and down both run the stationary-activation matmuls (read back from
    the words they write): an expert of every token (several runs), experts of none, the rest
    evenly used with under a run each.  Against 64 bits, all outputs; f16 operands: the
    contract's bound."""
    top_k = 4
    gdt, ddt = GgmlDType[gate], GgmlDType[down]
    # both projections' matrices past the 256 MB from which they are tried
    row = lambda dt, k: k // dt.block_size * dt.type_size  # noqa: E731
    e = max(128, -(-(264 << 20) // min(2 * ff * row(gdt, hidden), hidden * row(ddt, ff))))
    spec = LayerSpec(hidden, ff, e, top_k, gdt, ddt, shared=hidden % 512 == 0, bias_sigma=0.0)
    layer = build_layer(spec, seed=4600)
    bias = torch.zeros(e)
    bias[1], bias[2:6] = 10.0, -10.0
    layer.block.exp_probs_b.copy_(bias)
    # past the tiles' 1280 pairs where the shape has tiles, about 4 pairs per expert (plus the hot one's)
    t = max(40 if (hidden // 256) % 2 or (ff // 256) % 2 or "Q5_K" in (gate, down) or gate != "Q4_K" else 325, e)
    words = few_pairs_words(layer.block, t)
    assert min(words) >= 0, words
    x = torch.from_numpy(make_x(spec, 4601, t)).cuda()
    out, ids, w = layer.block.forward(x, return_routing=True)
    ws = layer.block._ws.cpu()
    assert [int(ws[o:o + 4].view(torch.int32)) for o in words] == [1, 1]
    got = ids.view(torch.int32).cpu()
    assert int((got == 1).sum()) == t and not torch.any((got >= 2) & (got < 6))
    want = moe_f64(layer.block, x, ids, w)
    assert_close(host(out), host(want), what=f"{gate}/{down} {hidden}x{ff} E{e} t{t}")


@pytest.mark.parametrize("gate,hidden", [("Q4_K", 1792), ("Q5_K", 2304), ("Q8_0", 1792)])
def test_few_pairs_gate_up_line(gate, hidden):
    """Gate/up whose K fills part of a CU's waves: taken at 4 pairs per expert, left to the
    grouped GEMM at 30 (read back from the word it writes); both against 64 bits."""
    ff, top_k = 512, 4
    gdt = GgmlDType[gate]
    e = -(-(264 << 20) // (2 * ff * (hidden // gdt.block_size * gdt.type_size)))
    spec = LayerSpec(hidden, ff, e, top_k, gdt, gdt, shared=False, bias_sigma=0.0)
    layer = build_layer(spec, seed=4900)
    for per, taken in ((4, 1), (30, 0)):
        t = per * e // top_k
        x = torch.from_numpy(make_x(spec, 4901, t)).cuda()
        at, _ = few_pairs_words(layer.block, t)
        assert at >= 0
        out, ids, w = layer.block.forward(x, return_routing=True)
        assert int(layer.block._ws[at:at + 4].cpu().view(torch.int32)) == taken
        assert_close(host(out), host(moe_f64(layer.block, x, ids, w)), what=f"{gate} {hidden} t{t}")


def test_few_pairs_per_expert_alignment_rule(orc):
    """Q6_K stacks two bytes off 16-byte alignment take the other grouped kernel: same
    outputs to f16-operand rounding."""
    rng = np.random.default_rng(8)
    t, top_k, e, n_out, k = 400, 4, 224, 2048, 768  # (matrices of 289 MB)
    st = synth_stack(GgmlDType.Q6_K, e, n_out, k, tensor_key(4700, 0, 1))
    raw = torch.zeros(st.nbytes + 2, dtype=torch.uint8, device="cuda")
    raw[2:] = st.buffer
    off = ExpertStack(raw, GgmlDType.Q6_K, e, n_out, k, 2)
    ids = dev_u32(np.argsort(rng.random((t, e)), axis=1)[:, :top_k])
    x = dev_f32(rng.standard_normal((t, 1, k)).astype(np.float32))
    a, b = host(ops.mul_mm_id(st, x, ids)), host(ops.mul_mm_id(off, x, ids))
    assert rel_l2(a, b) <= 1e-6  # (the same products in another order of summation)


@pytest.mark.parametrize("dt", ["Q4_K", "Q5_K", "Q6_K", "Q8_0"])
def test_few_pairs_on_average_many_in_use(orc, dt):
    """3 pairs per expert on average, but 400 on each of two experts: the grouped GEMM
    does the work after the other kernel left it, with the same bits as at an expert count
    whose average sends it there at once."""
    rng = np.random.default_rng(9)
    t, top_k, n_out, k = 400, 2, 2560, 768
    st = synth_stack(GgmlDType[dt], 256, n_out, k, tensor_key(4800, 0, 1))
    few = ExpertStack(st.buffer, GgmlDType[dt], 3, n_out, k)
    ids = dev_u32(np.argsort(rng.random((t, 2)), axis=1))
    x = dev_f32(rng.standard_normal((t, 1, k)).astype(np.float32))
    a, b = host(ops.mul_mm_id(st, x, ids)), host(ops.mul_mm_id(few, x, ids))
    assert np.array_equal(a, b)
