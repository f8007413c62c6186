"""The 256-row kernel on causal grids past one round of CUs."""
import ctypes
import math

import numpy as np
import pytest
import torch

import oracle
from amdgpu_rustdsl_amd import lib
from tests import gpu_util

pytestmark = pytest.mark.gpu
D = 128

def _bits(out):
    return out.view(torch.int16).cpu().numpy().view(np.uint16)


# (name, B, H, HK, S): square causal grids of more 256-row blocks than CUs; heads that divide over the 8 XCDs and not
CAUSAL = [
    ("H32_gqa", 2, 32, 8, 1300),
    ("H43", 1, 43, 43, 1500),
    ("H8_batches", 17, 8, 8, 513),
]


@pytest.mark.parametrize("case", CAUSAL, ids=[c[0] for c in CAUSAL])
def test_causal_256row_grid(gpu, case):
    """Every row of the causal 256-row grid (heaviest query tiles first): the 256-thread t128 kernel takes every tile
    whole too, on other blocks in another order, so the two must agree bit for bit, whatever the causal_pair field
    says; and the sampled rows meet the emulation's bar (gpu_util.causal_bar)."""
    name, B, H, HK, S = case
    print(f"[case] causal 256-row grid {name}", flush=True)
    assert not lib.uses_split_tiles("vs128", B, H, S, S, causal=True)
    inp = oracle.Inputs(B, H, S, S, HK=HK, causal=True)
    out, used, lse = gpu_util.run(inp, gpu, lse=True)
    assert used[0] == "vs128"
    paired, _, _ = gpu_util.run(inp, gpu, causal_pair=True)
    np.testing.assert_array_equal(out, paired)
    q, k, v, qs, ks, vs = gpu_util.upload(inp, gpu)
    o2 = torch.full((B, S, H, D), float("nan"), dtype=torch.bfloat16, device=gpu)
    a = lib.fill_args(o2.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), qs.data_ptr(), ks.data_ptr(), vs.data_ptr(), B, H, HK, S, S)
    a.flags = lib.FLAG_CAUSAL
    st = torch.cuda.current_stream(gpu).cuda_stream
    assert lib.raw.fmha_mxfp8_launch_t128(ctypes.byref(a), math.ceil(S / 128), H, B, st) == 0
    torch.cuda.synchronize()
    np.testing.assert_array_equal(out, _bits(o2).reshape(-1))
    rows = oracle.first_and_last(S, 64)
    emu = oracle.emulate(inp, rows=rows)
    fig, viol = gpu_util.causal_bar(inp, out, emu, rows)
    print(f"[case] causal 256-row grid {name} causal-bar={fig}", flush=True)
    assert not viol, (viol, fig)
    assert torch.isfinite(lse).all()
