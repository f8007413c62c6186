"""The 256-row kernel on grids past one round of CUs: split last blocks, and the causal order.

Split last blocks (fmha_fwd_hd128_mxfp8_auto_ws): the whole rounds' blocks must give the uncut kernel's bits; a split
block's ranges start from the softmax reference of its first tile, so P is quantised on the same grid and its rows differ
from the uncut kernel's by the order of the f32 sums and one bf16 rounding (2^-8 of a value, rms of the differences well
under 1e-3). Orders with another reference differ by 3e-2.
"""
import ctypes
import math

import numpy as np
import pytest
import torch

import oracle
from amdgpu_rustdsl_amd import lib
from tests import gpu_util
from tests.test_gpu_packed import _bf16, _guard_untouched, _params, _workspace

pytestmark = pytest.mark.gpu
D = 128

# (name, B, H, HK, S, SK, v_seq32, scale): one block past a round in the most ranges (the last two empty), ragged last
# query tiles and keys, grouped heads, the extensions
TAIL = [
    ("one_block_empty_ranges", 1, 257, 257, 130, 2100, False, 0.0),
    ("ragged_gqa_seq32", 9, 16, 4, 300, 2561, True, 0.0),
    ("scaled", 3, 96, 48, 200, 3000, False, 0.7),
]


def _bits(out):
    return out.view(torch.int16).cpu().numpy().view(np.uint16)


@pytest.mark.parametrize("case", TAIL, ids=[c[0] for c in TAIL])
def test_split_last_blocks(gpu, case):
    name, B, H, HK, S, SK, seq32, scale = case
    print(f"[case] split last blocks {name}", flush=True)
    cus = torch.cuda.get_device_properties(gpu).multi_processor_count
    gx = math.ceil(S / 256)
    blocks = gx * H * B
    if cus != 256:
        pytest.skip("the shapes are one round and a bit of 256 CUs")
    inp = oracle.Inputs(B, H, S, SK, HK=HK, v_seq32=seq32, qk_scale=scale)
    t = gpu_util.upload(inp, gpu)
    st = torch.cuda.current_stream(gpu).cuda_stream
    res = []
    for use_ws in (True, False):
        out = torch.empty(B, S, H, D, dtype=torch.bfloat16, device=gpu)
        out.view(torch.int16).fill_(0x7fc1)
        lse = torch.full((B, H, S), float("nan"), device=gpu)
        p = _params(t, out, lse, B, H, HK, S, SK, False, seq32, scale, "auto", 0)
        need = lib.auto_workspace_bytes(p)
        assert need > 0
        ws = _workspace(need, gpu)
        ran = lib.run_auto_ws(p, ws.data_ptr(), need, st) if use_ws else lib.run_auto(p, None, 0, st)
        torch.cuda.synchronize()
        assert tuple(ran) == ("vs128", 0) and _guard_untouched(ws, need)
        res.append((out, lse))
    (x, xl), (y, yl) = res
    # [B, S, H] mask of the split blocks' rows: block l = (b H + h) gx + query tile, from the last whole round on
    split = np.zeros((B, S, H), dtype=bool)
    for l in range(blocks // cus * cus, blocks):
        b, h, qt = l // gx // H, l // gx % H, l % gx
        split[b, qt * 256:(qt + 1) * 256, h] = True
    assert split.any()
    xb, yb = _bits(x), _bits(y)
    np.testing.assert_array_equal(xb[~split], yb[~split])
    dx = _bf16(x).reshape(x.shape)[split]
    dy = _bf16(y).reshape(y.shape)[split]
    assert not np.isnan(dx).any()
    rel = np.linalg.norm(dx - dy) / np.linalg.norm(dy)
    big = np.max(np.abs(dx - dy) / np.maximum(np.sqrt(np.mean(dy * dy)), np.abs(dy)))
    sl = np.transpose(split, (0, 2, 1))
    xl, yl = xl.cpu().numpy(), yl.cpu().numpy()
    ldiff = np.abs(xl - yl).max()
    print(f"[case] split last blocks {name} need={need} rel={rel:.2e} max={big:.2e} lse={ldiff:.2e}", flush=True)
    np.testing.assert_array_equal(xl[~sl], yl[~sl])
    assert rel <= 1e-3 and big <= 0.02 and ldiff <= 1e-5, (rel, big, ldiff)


# (name, B, H, HK, S, SK): causal grids of more 256-row blocks than CUs with 4 to 8 key tiles; heads that divide over the 8 XCDs
# and not
CAUSAL = [
    ("H32_gqa", 3, 32, 8, 650, 650),
    ("H43", 2, 43, 43, 1000, 1000),
    ("H8_batches", 17, 8, 8, 513, 513),
    ("more_keys", 33, 8, 2, 129, 1024),
]


@pytest.mark.parametrize("case", CAUSAL, ids=[c[0] for c in CAUSAL])
def test_causal_256row_grid(gpu, case):
    """Every row of the causal 256-row grid (heaviest query tiles first): the 256-thread t128 kernel takes every tile
    whole too, on other blocks in another order, so the two must agree bit for bit, also where the caller asks for its
    pairs; and the sampled rows meet the emulation's bar (gpu_util.causal_bar)."""
    name, B, H, HK, S, SK = case
    print(f"[case] causal 256-row grid {name}", flush=True)
    assert not lib.uses_split_tiles("vs128", B, H, S, SK, causal=True)
    inp = oracle.Inputs(B, H, S, SK, HK=HK, causal=True)
    out, used, lse = gpu_util.run(inp, gpu, lse=True)
    assert used[0] == "vs128"
    paired, _, _ = gpu_util.run(inp, gpu, causal_pair=True)
    np.testing.assert_array_equal(out, paired)
    q, k, v, qs, ks, vs = gpu_util.upload(inp, gpu)
    o2 = torch.full((B, S, H, D), float("nan"), dtype=torch.bfloat16, device=gpu)
    a = lib.fill_args(o2.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), qs.data_ptr(), ks.data_ptr(), vs.data_ptr(), B, H, HK, S, SK)
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


@pytest.mark.parametrize("seq32,scale", [(False, 0.0), (True, 0.0), (False, 0.7), (True, 0.7)], ids=["plain", "seq32", "scaled", "scaled_seq32"])
@pytest.mark.parametrize("B,H,HK,S,SK", [(5, 56, 28, 129, 385), (40, 8, 2, 200, 1024), (2, 48, 48, 511, 640)])
def test_causal_256row_grid_forms(gpu, B, H, HK, S, SK, seq32, scale):
    """The 256-row kernel and the pairs it stands in for, over the forms that both take: the same bits and LSE bits."""
    print(f"[case] causal 256-row forms B{B} H{H} S{S} SK{SK} {seq32} {scale}", flush=True)
    inp = oracle.Inputs(B, H, S, SK, HK=HK, causal=True, v_seq32=seq32, qk_scale=scale)
    out, _, lse = gpu_util.run(inp, gpu, lse=True)
    paired, _, plse = gpu_util.run(inp, gpu, lse=True, causal_pair=True)
    np.testing.assert_array_equal(out, paired)
    assert torch.equal(lse, plse) and torch.isfinite(lse).all()


def test_asked_pairing_runs_the_paired_kernel(gpu):
    """causal_pair=True runs the query-tile pairs of the 128-row kernel also where the automatic choice is the 256-row one."""
    from torch.profiler import ProfilerActivity, profile

    inp = oracle.Inputs(40, 8, 300, 520, HK=8, causal=True)
    names = []
    for pair in ("auto", True):
        gpu_util.run(inp, gpu, causal_pair=pair)
        with profile(activities=[ProfilerActivity.CUDA]) as prof:
            gpu_util.run(inp, gpu, causal_pair=pair)
        names.append([e.key for e in prof.key_averages() if "fmha_fwd" in e.key])
    print(f"[case] asked pairing {names}", flush=True)
    assert names == [["fmha_fwd_hd128_mxfp8_pre_vs128"], ["fmha_fwd_hd128_mxfp8_v3_t128"]]
