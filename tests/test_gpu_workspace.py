"""Caller workspaces: a size asked for n rows serves every call of fewer, no call
writes past it, and the Python entry points refuse a smaller one.
"""
import ctypes as C

import pytest
import torch

pytestmark = pytest.mark.gpu
F16 = 1


@pytest.fixture(scope="module")
def cl():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    import cascadia_amd

    return cascadia_amd


@pytest.mark.parametrize("h,i,g", [(4096, 14336, 128), (7168, 2048, 32), (4096, 4096, 128),
                                   (5120, 8192, 64), (2048, 1024, 32), (512, 256, 256),
                                   (96, 160, 32)])
def test_sizes_do_not_fall_with_more_rows(cl, h, i, g):
    """(more rows can take fewer slices of K, so smaller partials)"""
    L = cl.lib()
    packed = torch.empty(1024, dtype=torch.uint8, device="cuda").data_ptr()
    segs = (cl._lib.OvSegment * 2)(cl._lib.OvSegment(packed, packed, i, 1),
                                   cl._lib.OvSegment(packed, packed, 48, 0))
    E, k = 24, 4
    moe = cl._lib.MoeLayer(h, i, g, F16, 1, E, 256, 1 << 40,
                           cl._lib.Expert(256, 256, 256, 256, 256, 256, 1), i)
    lay = cl._lib.Layout(i, h, g, F16, 1)
    sizes = {
        "gemm f32": lambda n: L.cascadia_int4_gemm_workspace_bytes(C.byref(lay), 1, n),
        "gemm bf16": lambda n: L.cascadia_int4_gemm_workspace_bytes(C.byref(lay), 0, n),
        "ffn": lambda n: L.cascadia_int4_ffn_workspace_bytes(h, i, g, n),
        "sparse": lambda n: L.cascadia_int4_ffn_sparse_workspace_bytes(h, i, g, n),
        "axpy": lambda n: L.cascadia_int4_ffn_sparse_axpy_workspace_bytes(h, i, g, n),
        "ov": lambda n: L.cascadia_int4_ov_gemv_workspace_bytes(segs, 2, h, g, n),
        "moe": lambda n: L.cascadia_int4_moe_workspace_bytes(C.byref(moe), k, n),
    }
    rows = [*range(1, 140), *range(140, 1100, 13), 384, 385, 511, 512, 677, 678, 1024, 2048]
    for name, size in sizes.items():
        last = 0
        for n in sorted(set(rows)):
            b = size(n)
            assert b >= last, f"{name}: {n} rows ask for {b} bytes, fewer for {last}"
            last = b
        assert last > 0 or name.startswith("gemm"), name  # (a GEMM may need none)


def guarded(nbytes):
    """A workspace of nbytes between two guards."""
    t = torch.full((nbytes + 2 * 65536,), 0xA5, dtype=torch.uint8, device="cuda")
    return t, t[65536:65536 + nbytes]


def test_largest_workspace_serves_fewer_rows(cl):
    """3072 x 1536: 896 rows need more than 1,024.  Calls of fewer rows over the
    workspace of 1,024 leave the bytes around it alone and equal the calls over
    a workspace of their own."""
    h, i, g, n_max = 3072, 1536, 128, 1024
    flat = cl.fill_bytes(torch.empty(cl.expert_bytes(h, i, g), dtype=torch.uint8, device="cuda"), 3, 1)
    W = cl.ExpertWeights(flat, h, i, g, F16)
    for s in W.slices()[1::2]:
        cl.fill_scales(s.view(torch.int16), 3, 2)
    W = W.tiled()
    whole, ws = guarded(cl.ffn_workspace_bytes(h, i, n_max, g))
    for n in (16, 128, 200, 384, 896, 1024):
        print(f"{n} rows", flush=True)
        x = cl.fill_normal(torch.empty((n, h), dtype=torch.bfloat16, device="cuda"), 3, n)
        out, want = torch.empty_like(x), torch.empty_like(x)
        call = dict(group_size=g, scale_dtype=F16, tiling=cl.TILING_MFMA)
        cl.expert_forward(x, *W.slices(), out, workspace=ws, **call)
        own = torch.empty(cl.ffn_workspace_bytes(h, i, n, g), dtype=torch.uint8, device="cuda")
        cl.expert_forward(x, *W.slices(), want, workspace=own, **call)
        assert torch.equal(out, want)
        assert bool((whole[:65536] == 0xA5).all()) and bool((whole[-65536:] == 0xA5).all())


def test_small_workspaces_are_refused(cl):
    h, i, g, n = 512, 256, 32, 40
    flat = torch.zeros(cl.expert_bytes(h, i, g), dtype=torch.uint8, device="cuda")
    W = cl.ExpertWeights(flat, h, i, g, F16).tiled()
    xb = torch.zeros((n, h), dtype=torch.bfloat16, device="cuda")
    xf = xb.float()
    call = dict(group_size=g, scale_dtype=F16, tiling=cl.TILING_MFMA)
    short = torch.empty(cl.ffn_workspace_bytes(h, i, n, g) - 1, dtype=torch.uint8, device="cuda")
    with pytest.raises(ValueError, match="workspace"):
        cl.expert_forward(xb, *W.slices(), torch.empty_like(xb), workspace=short, **call)
    with pytest.raises(ValueError, match="workspace"):
        cl.ffn_forward_sparse_f32(xf, h, i, *W.slices(), torch.empty_like(xf), 0.0,
                                  workspace=short, **call)
    with pytest.raises(ValueError, match="workspace"):
        cl.ffn_forward_sparse_f32(xf, h, i, *W.slices(), torch.empty_like(xf), 0.3,
                                  workspace=short[:4096], **call)
    E, k = 12, 4
    per = cl.expert_bytes(h, i, g)
    stride = (per + 255) // 256 * 256
    ex = cl.MoEExperts(torch.zeros(stride * E, dtype=torch.uint8, device="cuda"), E, h, i, g, F16,
                       shared=cl.ExpertWeights(flat, h, i, g, F16))
    short = torch.empty(cl.moe_workspace_bytes(ex, k, n) - 1, dtype=torch.uint8, device="cuda")
    logits = torch.zeros((n, E), device="cuda")
    with pytest.raises(ValueError, match="workspace"):
        cl.moe_forward(ex, xf, torch.empty_like(xf), top_k=k, logits=logits, workspace=short)
