"""Kernels at the edges of their geometry (group counts at and just past the
lane layouts, partial tiles, the smallest and largest row counts), against the
oracle."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from maxuna_amd.gguf import GgmlDType
from maxuna_amd.synth import LayerSpec, build_layer, make_x

from .gpu_util import check_ids, host, rel_l2, selection_margin

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
