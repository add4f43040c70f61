"""Kernels at the edges of their geometry (group counts at and just past the
lane layouts, partial tiles, the smallest and largest row counts), against the
oracle."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from maxuna_amd import ops
from maxuna_amd.gguf import GgmlDType
from maxuna_amd.synth import LayerSpec, build_layer, make_x, synth_stack, tensor_key

from tests.gpu_util import check_ids, dev_f32, host, rel_l2, selection_margin

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
