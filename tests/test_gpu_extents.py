"""Keys and values whose sizes pass 32-bit signed arithmetic: a K of 2 GiB and more in one batch, and so many KV heads that a few
rows of one tile do. Each head's output is that of the same head alone, whose tensors are small: both run every tile in the
same order, so bit for bit."""
import pytest
import torch

from amdgpu_rustdsl_amd import ops

pytestmark = pytest.mark.gpu
D = 128


def _inputs(gpu, H, S, SK):
    g = torch.Generator(device=gpu)
    g.manual_seed(H + SK)
    r = lambda n: torch.randn(1, n, H, D, generator=g, device=gpu, dtype=torch.float16).to(torch.float8_e4m3fn).view(torch.uint8)   # noqa: E731
    vs = torch.zeros(1024, device=gpu)
    vs[0] = 0.5
    # scores of about N(0, 0.7): E8M0 2^-2 on both sides
    return r(S), r(SK), r(SK), ops.alloc_scales(1, S, H, gpu, fill=125), ops.alloc_scales(1, SK, H, gpu, fill=125), vs


@pytest.mark.parametrize("H,SK,path,alone", [(128, 131200, "t128", "t128"), (44000, 200, "auto", "t128"), (44000, 385, "auto", "t128")],
                         ids=["k_of_2_gib", "many_heads_short_recipe", "many_heads"])
def test_large_strides(gpu, H, SK, path, alone):
    if torch.cuda.get_device_properties(gpu).total_memory < 64 << 30:
        pytest.skip("takes 20 GB of device memory")
    print(f"[case] extents H{H} SK{SK}", flush=True)
    S = 3
    q, k, v, qs, ks, vs = _inputs(gpu, H, S, SK)
    out = torch.full((1, S, H, D), float("nan"), dtype=torch.bfloat16, device=gpu)
    ops.fmha_fwd_mxfp8(q, k, v, qs, ks, vs, out, path=path)
    torch.cuda.synchronize()
    assert torch.isfinite(out.float()).all()
    for h in (0, 1, H // 2, H - 1):
        one = [x[:, :, h:h + 1].contiguous() for x in (q, k, v)]
        q1, k1 = ops.alloc_scales(1, S, 1, gpu, fill=125), ops.alloc_scales(1, SK, 1, gpu, fill=125)
        ref = torch.full((1, S, 1, D), float("nan"), dtype=torch.bfloat16, device=gpu)
        ops.fmha_fwd_mxfp8(*one, q1, k1, vs, ref, path=alone)
        torch.cuda.synchronize()
        assert torch.equal(out[:, :, h:h + 1].contiguous().view(torch.int16), ref.view(torch.int16)), h
