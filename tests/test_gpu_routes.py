"""Routes a call takes by its rows, its values and the memory there is: the
decode-batch FFN under its own rule, the forms that need less workspace (the
allocation-free entry point, calls recorded in a graph), and rows that are not
finite or span a wide range.
"""
import ctypes as C
import os
import subprocess
import sys

import numpy as np
import pytest
import torch

from conftest import ROOT, rel_l2
from test_gpu_gemm import assert_bf16_close
from test_gpu_tiles import dev, expert, host

pytestmark = pytest.mark.gpu
BF16, F16 = 0, 1


@pytest.fixture(scope="module")
def cl():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    import cascadia_amd

    return cascadia_amd


def gpu_expert(cl, h, i, g, seed):
    flat = cl.fill_bytes(torch.empty(cl.expert_bytes(h, i, g), dtype=torch.uint8, device="cuda"),
                         seed, 1)
    W = cl.ExpertWeights(flat, h, i, g, F16)
    for t in W.slices()[1::2]:
        cl.fill_scales(t.view(torch.int16), seed, 2)
    return flat, W.tiled()


@pytest.mark.parametrize("M,few", [(8, False), (9, True), (16, True), (17, True), (32, True),
                                   (33, False)])
def test_ffn_few_rows_by_default(cl, orc, tuning, M, few):
    """9 .. 32 rows of an FFN of 32 MiB and more, without a variable: the result
    is the forced route's, bit for bit, and within the bar of the oracle."""
    h, i, g = 2048, 11264, 128
    flat = expert(orc, h, i, g, F16, 41)
    W = cl.ExpertWeights(dev(flat), h, i, g, F16).tiled()
    xb = orc.fill_normal_bf16(M, 52, M * h)
    x = dev(xb.view(np.int16).reshape(M, h))
    outs = []
    for rows in (None, "2" if few else "100"):
        if rows:
            tuning("CASCADIA_INT4_FEW_MIN_TOKENS", rows)
        out = torch.empty(M * h, dtype=torch.int16, device="cuda")
        cl.expert_forward(x, *W.slices(), out, group_size=g, scale_dtype=F16,
                          tiling=cl.TILING_MFMA)
        outs.append(host(out).view(np.uint16).reshape(M, h))
    assert np.array_equal(*outs)
    assert_bf16_close(outs[0], orc.cpu_expert_forward(xb, M, flat, h, i, g, F16), f"few M{M}")


@pytest.mark.parametrize("x_f32,M,n,k,g,tiles", [
    # where the skinny kernel's plan is one round of workgroups with all of K in
    # LDS, and the next rows or shapes, where it is not or the tiles are faster
    (True, 24, 4096, 11264, 128, False), (True, 32, 4096, 11264, 128, True),
    (True, 17, 4096, 11264, 32, False), (True, 17, 6144, 8192, 32, True),
    (True, 16, 7168, 8192, 128, False), (True, 17, 7168, 8192, 128, True),
    (True, 40, 8192, 4096, 128, True), (True, 64, 8192, 4096, 128, False),
    (False, 40, 32768, 1536, 128, False), (False, 48, 32768, 1536, 128, True)])
def test_gemm_route_by_default(cl, tuning, x_f32, M, n, k, g, tiles):
    """The route that a GEMM of few rows takes without a variable: the forced
    route's result, bit for bit, and not the other's."""
    packed = cl.fill_bytes(torch.empty(n * k // 2, dtype=torch.uint8, device="cuda"), 16, 1)
    scales = cl.fill_scales(torch.empty(n * (k // g), dtype=torch.int16, device="cuda"), 16, 2)
    pt, st = cl.tile_weights(packed, scales.view(torch.uint8), n, k, g)
    x = cl.fill_normal(torch.empty((M, k), dtype=torch.float32 if x_f32 else torch.bfloat16,
                                   device="cuda"), 16, 3)
    var = "CASCADIA_INT4_F32_TILE_TOKENS" if x_f32 else "CASCADIA_INT4_BF16_TILE_TOKENS"
    ys = {}
    for route, rows in (("default", None), ("tiles", "2"), ("skinny", "100000")):
        if rows:
            tuning(var, rows)
        y = ys[route] = torch.empty((M, n), device="cuda")
        cl.dequant_gemm_int4_multi_auto(pt, st, x, n, k, M, y, group_size=g, scale_dtype=F16,
                                        tiling=cl.TILING_MFMA)
    assert not torch.equal(ys["tiles"], ys["skinny"])
    assert torch.equal(ys["default"], ys["tiles" if tiles else "skinny"])


@pytest.mark.parametrize("h,i,g,M,form", [(1536, 10240, 32, 70, "skinny"),
                                          (1024, 1024, 32, 512, "tiles")])
def test_noalloc_least_form(cl, orc, tuning, h, i, g, M, form):
    """An FFN whose usual form needs more than the static scratch and whose least
    form fits: the skinny kernel, or the tile GEMMs without slices of K."""
    assert cl.ffn_workspace_bytes(h, i, M, g) > 8 << 20
    flat = expert(orc, h, i, g, F16, 43)
    W = cl.ExpertWeights(dev(flat), h, i, g, F16).tiled()
    ex = cl._lib.Expert(*(t.data_ptr() for t in W.slices()), cl.TILING_MFMA)
    xb = orc.fill_normal_bf16(M, 53, M * h)
    x = dev(xb.view(np.int16).reshape(M, h))
    out = torch.empty(M * h, dtype=torch.int16, device="cuda")
    assert cl.lib().cascadia_int4_expert_forward_noalloc(
        h, i, g, F16, C.byref(ex), x.data_ptr(), M, out.data_ptr(),
        torch.cuda.current_stream().cuda_stream) == 0
    got = host(out).view(np.uint16).reshape(M, h)
    assert_bf16_close(got, orc.cpu_expert_forward(xb, M, flat, h, i, g, F16), f"noalloc {form}")
    if form == "skinny":
        tuning("CASCADIA_INT4_FFN_TILE_TOKENS", "100000")
        cl.expert_forward(x, *W.slices(), out, group_size=g, scale_dtype=F16,
                          tiling=cl.TILING_MFMA)
        assert np.array_equal(host(out).view(np.uint16).reshape(M, h), got)


@pytest.mark.parametrize("T,tiles", [(191, False), (199, False), (200, True)])
def test_moe_route_by_default(cl, tuning, T, tiles):
    """From 192 tokens a layer runs on tiles where the experts' mean is 40 rows
    and more: the forced route's result, bit for bit, and not the other's."""
    E, top, h, i, g = 40, 8, 512, 256, 128
    stride = (cl.expert_bytes(h, i, g) + 255) // 256 * 256
    blobs = cl.fill_bytes(torch.empty(stride * E, dtype=torch.uint8, device="cuda"), 18, 1)
    for e in range(E):
        W = cl.ExpertWeights(blobs[e * stride:e * stride + cl.expert_bytes(h, i, g)], h, i, g, F16)
        for t in W.slices()[1::2]:
            cl.fill_scales(t.view(torch.int16), 18, 2)
    ex = cl.MoEExperts.from_crate(blobs, E, h, i, g, F16, stride)
    x = cl.fill_normal(torch.empty((T, h), device="cuda"), 18, 3)
    logits = cl.fill_normal(torch.empty((T, E), device="cuda"), 18, 4)
    out = {}
    for route, tokens in (("default", None), ("tiles", "2"), ("skinny", "100000")):
        if tokens:
            tuning("CASCADIA_INT4_MOE_TILE_TOKENS", tokens)
        out[route] = torch.empty_like(x)
        cl.moe_forward(ex, x, out[route], top_k=top, logits=logits)
    assert not torch.equal(out["tiles"], out["skinny"])
    assert torch.equal(out["default"], out["tiles" if tiles else "skinny"])


SPECIAL = {3: float("nan"), 20: float("inf"), 40: float("-inf"), 63: 3.4028234663852886e38}


@pytest.mark.parametrize("g", [32, 64, 128])
def test_gemm_f32_tiles_not_finite(cl, tuning, g):
    """f32 rows with a NaN, an infinity or the largest finite value (whose hi
    plane is truncated, not rounded to infinity): those rows are not finite, as
    in the skinny kernel, and no other row changes by a bit.  Rows scaled far
    up and down keep their precision."""
    n, k, M = 512, 4096, 100
    packed = cl.fill_bytes(torch.empty(n * k // 2, dtype=torch.uint8, device="cuda"), 14, 1)
    scales = cl.fill_scales(torch.empty(n * (k // g), dtype=torch.int16, device="cuda"), 14, 2)
    scales = scales.view(torch.uint8)
    pt, st = cl.tile_weights(packed, scales, n, k, g)
    clean = cl.fill_normal(torch.empty((M, k), dtype=torch.float32, device="cuda"), 14, 3)
    clean[50] *= 1e30
    clean[51] *= 1e-30
    x = clean.clone()
    for r, v in SPECIAL.items():
        x[r, 100 + r] = v
    ys = {}
    for route, rows in (("tiles", "17"), ("skinny", "100000")):
        tuning("CASCADIA_INT4_F32_TILE_TOKENS", rows)
        for name, t in (("special", x), ("clean", clean)):
            y = ys[route, name] = torch.empty((M, n), device="cuda")
            cl.dequant_gemm_int4_multi_auto(pt, st, t, n, k, M, y, group_size=g, scale_dtype=F16,
                                            tiling=cl.TILING_MFMA)
    rest = [r for r in range(M) if r not in SPECIAL]
    for route in ("tiles", "skinny"):
        assert not torch.isfinite(ys[route, "special"][list(SPECIAL)]).any(), route
        assert torch.equal(ys[route, "special"][rest], ys[route, "clean"][rest]), route
    want = clean.double() @ cl.debug_dequant(packed, scales, n, k, g, F16).double().T
    for r in (0, 50, 51):  # (1e-5: the bar of the f32 tiles)
        assert rel_l2(host(ys["tiles", "clean"][r]), want[r].cpu().numpy()) <= 1e-5, r


@pytest.mark.parametrize("x_f32", [True, False])
@pytest.mark.parametrize("M,h,i,g", [(200, 2048, 1536, 128), (100, 1024, 2048, 64),
                                     (32, 2048, 11264, 128)])
def test_ffn_not_finite(cl, tuning, M, h, i, g, x_f32):
    """The same through an FFN whose gate/up is cut into slices of K (the
    SwiGLU planes and seeds made by the reduce) or is a decode batch's."""
    if M > 32:
        tuning("CASCADIA_INT4_FFN_TILE_TOKENS", "33")
    _, W = gpu_expert(cl, h, i, g, 15)
    clean = cl.fill_normal(torch.empty((M, h), dtype=torch.float32, device="cuda"), 15, 3)
    special = {r: v for r, v in SPECIAL.items() if r < M}
    if not x_f32:
        clean = clean.to(torch.bfloat16)
        special = {r: v for r, v in special.items() if abs(v) != SPECIAL[63]}
    x = clean.clone()
    for r, v in special.items():
        x[r, 100 + r] = v
    outs = []
    for t in (x, clean):
        out = torch.empty_like(t)
        opts = dict(group_size=g, scale_dtype=F16, tiling=cl.TILING_MFMA)
        if x_f32:
            cl.ffn_forward_sparse_f32(t, h, i, *W.slices(), out, 0.0, **opts)
        else:
            cl.expert_forward(t, *W.slices(), out, **opts)
        outs.append(out)
    rest = [r for r in range(M) if r not in special]
    assert not torch.isfinite(outs[0][list(special)]).any()
    assert torch.equal(outs[0][rest], outs[1][rest])
    assert torch.isfinite(outs[1]).all()


CAPTURE = r"""
import os, sys
sys.path.insert(0, sys.argv[1])
import torch
import cascadia_amd as cl

F16, MFMA = 1, cl.TILING_MFMA


def forced(**env):
    os.environ.update(env)
    cl.lib().cascadia_int4_reload_tuning()



def record(call, out):
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        call()
    got = []
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        got.append(out.clone())
    assert all(torch.equal(g, got[0]) for g in got)
    return got[0]


def weights(n, k, g, seed):
    p = cl.fill_bytes(torch.empty(n * k // 2, dtype=torch.uint8, device="cuda"), seed, 1)
    s = cl.fill_scales(torch.empty(n * (k // g), dtype=torch.int16, device="cuda"), seed, 2)
    return p, s.view(torch.uint8)


# 1. an f32 GEMM recorded as the process's first call: no memory is shared yet
n, k, g, M = 3000, 4096, 128, 333
pt, st = cl.tile_weights(*weights(n, k, g, 1), n, k, g)
x = cl.fill_normal(torch.empty((M, k), device="cuda"), 1, 3)
y = torch.empty((M, n), device="cuda")
gemm = lambda: cl.dequant_gemm_int4_multi_auto(pt, st, x, n, k, M, y, group_size=g,
                                               scale_dtype=F16, tiling=MFMA)
recorded = record(gemm, y)

# 2. a MoE layer and an FFN that do not fit what graphs have (nothing) are
# refused; where that is between their least and usual forms' needs, they are
# recorded in the least (a layer of 9.44 / 9.61 MB, an FFN of 2.2 / 10.6 MB,
# and an AXPY whose partials are 9.54 MB)
E, top, h, i, T = 12, 4, 384, 256, 200
per = cl.expert_bytes(h, i, 128)
stride = (per + 255) // 256 * 256
blobs = cl.fill_bytes(torch.empty(stride * E, dtype=torch.uint8, device="cuda"), 2, 1)
for e in range(E):
    W = cl.ExpertWeights(blobs[e * stride:e * stride + per], h, i, 128, F16)
    for t in W.slices()[1::2]:
        cl.fill_scales(t.view(torch.int16), 2, 2)
ex = cl.MoEExperts.from_crate(blobs, E, h, i, 128, F16, stride)
mx = cl.fill_normal(torch.empty((T, h), device="cuda"), 2, 3)
logits = cl.fill_normal(torch.empty((T, E), device="cuda"), 2, 4)
mo = torch.empty_like(mx)
moe = lambda: cl.moe_forward(ex, mx, mo, top_k=top, logits=logits, residual=mx)
H, I, G, R = 1024, 1024, 32, 512
flat = torch.empty(cl.expert_bytes(H, I, G), dtype=torch.uint8, device="cuda")
W = cl.ExpertWeights(cl.fill_bytes(flat, 3, 1), H, I, G, F16)
for t in W.slices()[1::2]:
    cl.fill_scales(t.view(torch.int16), 3, 2)
W = W.tiled()
fx = cl.fill_normal(torch.empty((R, H), dtype=torch.bfloat16, device="cuda"), 3, 3)
fo = torch.empty_like(fx)
ffn = lambda: cl.expert_forward(fx, *W.slices(), fo, group_size=G, scale_dtype=F16, tiling=MFMA)
for call in (moe, ffn):
    try:
        record(call, mo)
        raise SystemExit("a call without memory was recorded")
    except cl.CascadiaInt4Error as e:
        assert e.rc == -2, e
    torch.cuda.synchronize()
ax = 2330 * 32  # slices of 32 active rows, each 1,024 f32
cl.dequant_axpy_int4_active(
    torch.full((64 * 512,), 0x99, dtype=torch.uint8, device="cuda"),
    torch.zeros(64 * 32 * 2, dtype=torch.uint8, device="cuda"),
    torch.ones(64, device="cuda"), torch.zeros(ax, dtype=torch.int32, device="cuda"), 64, 1024,
    torch.zeros(1024, device="cuda"))
assert cl.lib().cascadia_int4_axpy_workspace_bytes(1024, ax) == 9543680
moe_recorded, ffn_recorded = record(moe, mo), record(ffn, fo)

# the eager calls: other forms, the same sums
rel = lambda a, b: float((a.double() - b.double()).norm() / b.double().norm())
gemm(), moe(), ffn()
torch.cuda.synchronize()
print("recorded / eager: gemm %.2e moe %.2e ffn %.2e" % (rel(recorded, y), rel(moe_recorded, mo),
                                                         rel(ffn_recorded, fo)))
assert 0 < rel(recorded, y) <= 1e-5
assert 0 < rel(moe_recorded, mo) <= 1e-3 and 0 < rel(ffn_recorded, fo) <= 1e-3
# and the recorded forms are the skinny kernel's, bit for bit
forced(CASCADIA_INT4_F32_TILE_TOKENS="100000", CASCADIA_INT4_MOE_TILE_TOKENS="100000")
gemm(), moe()
torch.cuda.synchronize()
assert torch.equal(recorded, y) and torch.equal(moe_recorded, mo)
print("ok")
"""


def test_recorded_forms_in_a_fresh_process(cl):
    """Calls without a workspace recorded before any eager call has made room for
    them: in a process of its own, whose first library call is a recorded one."""
    r = subprocess.run([sys.executable, "-c", CAPTURE, ROOT], capture_output=True, text=True,
                       timeout=110, env={**os.environ, "PYTHONDONTWRITEBYTECODE": "1"})
    assert r.returncode == 0 and r.stdout.rstrip().endswith("ok"), (r.stdout, r.stderr[-3000:])
