"""The packed-rows kernel (short query ranges) against the kernels it stands in for, and against float64 attention.

Every share of a key range starts from the softmax reference of the whole range's first tile, so P is quantised on the
same grid as in the path's own kernel: the two outputs differ by the order of the f32 sums and one bf16 rounding (2^-8),
and where the reference is taken over whole tiles also in the first tile's P: the own kernel computes that tile's S on
the start value b = 64 (one f32 step there is 2^-17, 2^-8 of a score in log2 units, 2.7e-3 of a weight) and shifts it,
the packed kernel computes it again on the reference itself, so a few of its P round to the next e4m3 value (2^-3).
That is one tile of at least 8: at most 2.7e-3 / 8 in the LSE, and a few 1e-3 in the outputs. Orders that quantise P
against another running maximum differ by 3e-2 and more, so the bar of 6e-3 separates a share that starts from a wrong
reference.
"""
import ctypes
import math

import numpy as np
import pytest
import torch

import oracle
from amdgpu_rustdsl_amd import lib, ops
from tests import gpu_util

pytestmark = pytest.mark.gpu
D = 128

# (name, B, H, HK, S, SK, causal, v_seq32, scale, lse, path, splits): row counts around the 32-row waves and 128-row
# tiles, group sizes 1 to 16, ragged last tiles, ranges that do not divide into shares
CASES = [
    ("decode_whole_tile_order", 8, 32, 8, 1, 4100, False, False, 0.0, True, "auto", 0),
    ("decode_split_tile_order", 8, 16, 1, 1, 2100, False, False, 0.0, False, "auto", 0),
    ("rows31", 1, 31, 31, 1, 1100, False, False, 0.0, True, "auto", 0),
    ("rows33_group1", 2, 4, 4, 33, 1300, False, True, 0.0, True, "auto", 0),
    ("rows96_group8", 2, 8, 1, 12, 1900, False, False, 0.7, True, "auto", 0),
    ("rows128_group2", 2, 8, 4, 64, 1537, True, False, 0.0, True, "auto", 0),
    ("rows129_group1_is_not_packed", 1, 4, 4, 129, 1537, False, False, 0.0, False, "auto", 0),
    ("forced_path_is_not_packed", 2, 4, 4, 33, 1300, False, False, 0.0, False, "t128", 0),
    ("rows400_group4", 1, 8, 2, 100, 3000, True, True, 0.7, True, "auto", 0),
    ("rows2048_group16", 1, 16, 1, 128, 4100, True, False, 0.0, False, "auto", 0),
    ("causal_share_no_early_row_sees", 1, 2, 1, 120, 2050, True, False, 0.0, True, "auto", 0),
    ("split_decode", 1, 32, 8, 1, 16383, False, False, 0.0, False, "kvsplit", 8),
    ("split_rows28_seq32", 2, 4, 1, 7, 4097, False, True, 0.0, False, "kvsplit", 4),
    ("split_rows128_scaled", 1, 8, 8, 128, 16000, False, False, 0.7, False, "kvsplit", 8),
    ("split_rows512", 1, 16, 2, 64, 6000, False, False, 0.0, False, "kvsplit", 2),
]


def _params(t, out, lse, B, H, HK, S, SK, causal, seq32, scale, path, splits, f32=0):
    q, k, v, qs, ks, vs = t
    p = lib.Params()
    p.o, p.q, p.k, p.v = out.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr()
    p.q_descale, p.k_descale, p.v_descale = qs.data_ptr(), ks.data_ptr(), vs.data_ptr()
    p.lse = lse.data_ptr() if lse is not None else None
    p.B, p.H, p.HK, p.S, p.SK = B, H, HK, S, SK
    p.path = -1 if path == "auto" else lib.PATH_IDS[path]
    p.splits, p.causal, p.v_seq32, p.softmax_scale, p.f32_partials = splits, int(causal), int(seq32), scale, f32
    p.no_check = 1
    return p


def _bf16(out):
    return out.float().cpu().numpy().reshape(-1).astype(np.float64)


GUARD = 4096


def _workspace(need, gpu):
    """`need` bytes of workspace (a NaN pattern) and GUARD bytes behind them, in one allocation."""
    ws = torch.full((need + GUARD,), 0xff, dtype=torch.uint8, device=gpu)
    ws[need:] = 0x5a
    return ws


def _guard_untouched(ws, need):
    return bool((ws[need:] == 0x5a).all())


# the partial format is the KV split's
@pytest.mark.parametrize("case,f32", [(c, f) for c in CASES for f in ((0, 1) if c[10] == "kvsplit" else (0,))],
                         ids=[c[0] + s for c in CASES for s in (("", "-f32") if c[10] == "kvsplit" else ("",))])
def test_packed_matches_own_kernel(gpu, case, f32):
    name, B, H, HK, S, SK, causal, seq32, scale, want_lse, path, splits = case
    print(f"[case] packed {name}", flush=True)
    inp = oracle.Inputs(B, H, S, SK, HK=HK, causal=causal, v_seq32=seq32, qk_scale=scale)
    t = gpu_util.upload(inp, gpu)
    st = torch.cuda.current_stream(gpu).cuda_stream

    def outputs():
        out = torch.empty(B, S, H, D, dtype=torch.bfloat16, device=gpu)
        out.view(torch.int16).fill_(0x7fc1)
        return out, (torch.full((B, H, S), float("nan"), device=gpu) if want_lse else None)

    out, lse = outputs()
    p = _params(t, out, lse, B, H, HK, S, SK, causal, seq32, scale, path, splits, f32)
    need = lib.auto_workspace_bytes(p)
    ws = _workspace(need, gpu)
    ran = lib.run_auto_ws(p, ws.data_ptr(), need, st)
    ref, ref_lse = outputs()
    p2 = _params(t, ref, ref_lse, B, H, HK, S, SK, causal, seq32, scale, path, splits, f32)
    if path != "kvsplit":
        assert (need > 0) == (not name.endswith("is_not_packed")), need
        ran2 = lib.run_auto(p2, None, 0, st)     # no workspace: the path's own kernel
    else:
        # the reference-named pair on the partials that the entry reports (the packed rows cut each of them further)
        parts = lib.kv_partials(B, H, S, SK, splits)
        own = lib.workspace_bytes(B, H, S, parts)
        assert ran.partials == parts and (need > own or (f32 and need == own))   # f32 rows may not pay for more shares
        rows = B * S * H
        buf = torch.empty(lib.workspace_bytes(B, H, S, parts), dtype=torch.uint8, device=gpu)
        a = lib.fill_args(ref.data_ptr(), *(x.data_ptr() for x in t), B, H, HK, S, SK)
        if scale:
            a.softmax_scale = int(np.float32(scale).view(np.uint32))
        ka = lib.KvsplitArgs()
        ctypes.memmove(ctypes.byref(ka), ctypes.byref(a), 0x270)
        ka.ptr_ohat, ka.ptr_lse = buf.data_ptr(), buf.data_ptr() + parts * rows * 512
        fmt = lib.KVS_F32_PARTIALS if f32 else 0
        ka.kvs_splits = parts | fmt | (lib.KVS_V_SEQ32 if seq32 else 0) | (lib.KVS_SCALE if scale else 0)
        ka.kvs_rows_total = rows
        assert lib.raw.fmha_mxfp8_launch_kvsplit(ctypes.byref(ka), math.ceil(S / 256), H, B * parts, st) == 0
        ca = lib.CombineArgs(ka.ptr_ohat, ka.ptr_lse, ref.data_ptr(), rows, 128, parts | fmt)
        assert lib.raw.fmha_mxfp8_launch_combine(ctypes.byref(ca), (rows * 16 + 255) // 256, st) == 0
        ran2 = ("kvsplit", splits)
    torch.cuda.synchronize()
    assert tuple(ran) == tuple(ran2)
    assert _guard_untouched(ws, need)
    x, y = _bf16(out), _bf16(ref)
    assert not np.isnan(x).any()
    rms = np.sqrt(np.mean(y * y))
    rel = np.linalg.norm(x - y) / np.linalg.norm(y)
    big = np.max(np.abs(x - y) / np.maximum(rms, np.abs(y)))
    bits = out.view(torch.int16).cpu().numpy().view(np.uint16).reshape(-1)
    rbits = ref.view(torch.int16).cpu().numpy().view(np.uint16).reshape(-1)
    ours, own = oracle.check_fp64(inp, bits, rows=S), oracle.check_fp64(inp, rbits, rows=S)
    print(f"[case] packed {name} need={need} rel={rel:.2e} max={big:.2e} ours={ours} own={own}", flush=True)
    assert rel <= 6e-3 and big <= 0.06, (rel, big)
    assert ours["mean_err"] <= 1.05 * own["mean_err"] + 1e-7 and ours["bad"] <= own["bad"]
    if want_lse:
        assert torch.isfinite(lse).all() and (lse - ref_lse).abs().max().item() <= 1e-3


def test_workspace_too_small_runs_own_kernel(gpu):
    """Short of the shares' partials the entry takes fewer shares, and with none the path's own kernel: same results."""
    B, H, HK, S, SK = 2, 16, 4, 3, 3000
    inp = oracle.Inputs(B, H, S, SK, HK=HK, causal=True)
    t = gpu_util.upload(inp, gpu)
    st = torch.cuda.current_stream(gpu).cuda_stream
    got = []
    out = torch.empty(B, S, H, D, dtype=torch.bfloat16, device=gpu)
    p = _params(t, out, None, B, H, HK, S, SK, True, False, 0.0, "auto", 0)
    need = lib.auto_workspace_bytes(p)
    one = lib.workspace_bytes(B, H, S, 1)
    assert need > 2 * one
    for size in (need, 2 * one, 2 * one - 1, 0):
        ws = _workspace(size, gpu)
        out.zero_()
        lib.run_auto_ws(p, ws.data_ptr() if size else None, size, st)
        torch.cuda.synchronize()
        assert _guard_untouched(ws, size)
        got.append(_bf16(out))
    for g in got[:-1]:
        assert np.linalg.norm(g - got[-1]) / np.linalg.norm(got[-1]) <= 6e-3
