"""GPU parity of the MFMA-tile GEMMs (grouped.hip) against the CPU oracle.

They run an expert FFN of many tokens (65 and more; expert_forward for bf16
rows, ffn_forward_sparse_f32 at tau 0 for f32 rows: the shared expert) and
every MoE layer of 65 tokens or more: routing, grouping into 128-row chunks,
the grouped gate/up with the SwiGLU epilogue into hi / lo planes, the grouped
down, the slot-order combine.  Groups of 32 and 64 columns take the
transposed-fragment steps, 128 the plain ones.  Bars as for the other
kernels: bf16 outputs rel-L2 <= 1e-3 and within one bf16 ulp of the oracle
(+ 1e-5 max|y|); f32 outputs rel-L2 <= 1e-3, max-abs <= 2e-2; MoE layers as in
test_gpu_moe.check_layer.
"""
import numpy as np
import pytest
import torch

from conftest import REL_L2_TOL, rel_l2
from test_gpu_gemm import assert_bf16_close, assert_f32_close
from test_gpu_moe import build, check_layer

pytestmark = pytest.mark.gpu
BF16, F16 = 0, 1


@pytest.fixture(scope="module")
def cl():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    import cascadia_amd

    return cascadia_amd


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def host(t):
    torch.cuda.synchronize()
    return t.cpu().numpy()


def expert(orc, h, i, g, sdt, seed):
    flat = orc.fill_bytes(seed, 50, orc.expert_bytes(h, i, g)).copy()
    offs, sizes = orc.expert_offsets(h, i, g)
    for s_ in (1, 3, 5):
        flat[offs[s_]:offs[s_] + sizes[s_]] = orc.fill_scales(seed, 51 + s_, sizes[s_] // 2,
                                                              sdt).view(np.uint8)
    return flat


@pytest.mark.parametrize("M", [65, 130, 257])
@pytest.mark.parametrize("h,i,g,sdt", [(512, 384, 32, F16), (1024, 768, 64, BF16),
                                       (768, 1280, 128, F16), (512, 256, 256, BF16)])
def test_expert_forward_tiles(cl, orc, tuning, M, h, i, g, sdt):
    """expert_forward over M rows on the tile GEMMs (bf16 rows, bf16 out;
    the tile threshold lowered to 65 rows)."""
    tuning("CASCADIA_INT4_FFN_TILE_TOKENS", "65")
    flat = expert(orc, h, i, g, sdt, M + g)
    W = cl.ExpertWeights(dev(flat), h, i, g, sdt).tiled()
    xb = orc.fill_normal_bf16(M, 52, M * h)
    out = torch.empty(M * h, dtype=torch.int16, device="cuda")
    cl.expert_forward(dev(xb.view(np.int16).reshape(M, h)), *W.slices(), out, group_size=g,
                      scale_dtype=sdt, tiling=cl.TILING_MFMA)
    want = orc.cpu_expert_forward(xb, M, flat, h, i, g, sdt)
    assert_bf16_close(host(out).view(np.uint16).reshape(M, h), want, f"tiles M{M} G{g}")


@pytest.mark.parametrize("n,k,g,sdt,M", [
    # one to four k-blocks (fewer than the pipeline's stages, and one more), a
    # single 16-row weight tile, the 32- and 64-column edges of a wave, ragged
    # rows around the 32 / 64 / 128-row edges, groups of several k-blocks
    (16, 128, 32, F16, 64), (17, 128, 128, F16, 65), (255, 256, 64, BF16, 96),
    (257, 384, 32, BF16, 127), (272, 512, 128, F16, 129), (31, 768, 256, F16, 161),
    (1000, 1536, 512, BF16, 300), (4097, 1024, 64, F16, 70)])
def test_gemm_tile_edges(cl, orc, n, k, g, sdt, M):
    """gemm_int4_bf16 (bf16 out) and bf16-in / f32-out over tiled weights at
    the tile kernel's edges, against the oracle."""
    packed = orc.fill_bytes(n + M, 1, n * k // 2)
    scales = orc.fill_scales(n + M, 2, n * (k // g), sdt).view(np.uint8).copy()
    pt, st = cl.tile_weights(dev(packed), dev(scales), n, k, g)
    xb = orc.fill_normal_bf16(k, M, M * k)
    xd = dev(xb.view(np.int16))
    want = orc.gemm_multi(packed, scales, orc.bf16_to_f32(xb), n, k, M, g, sdt)
    ys = torch.empty(M * n, dtype=torch.float32, device="cuda")
    cl.dequant_gemm_int4_multi_auto(pt, st, xd, n, k, M, ys, group_size=g, scale_dtype=sdt,
                                    tiling=cl.TILING_MFMA)
    assert_f32_close(host(ys).reshape(M, n), want, f"f32 out {n}x{k} G{g} M{M}")
    yb = torch.empty(M * n, dtype=torch.int16, device="cuda")
    cl.gemm_int4_bf16(pt, st, xd, n, k, M, yb, group_size=g, scale_dtype=sdt,
                      tiling=cl.TILING_MFMA)
    assert_bf16_close(host(yb).view(np.uint16).reshape(M, n), orc.f32_to_bf16(want),
                      f"bf16 out {n}x{k} G{g} M{M}")


@pytest.mark.parametrize("n,k,g,sdt,M", [
    (16, 128, 128, BF16, 17), (33, 384, 32, F16, 63), (300, 1024, 64, BF16, 64),
    (1000, 4096, 32, BF16, 65), (257, 2048, 256, F16, 130)])
def test_gemm_f32_tiles(cl, orc, tuning, n, k, g, sdt, M):
    """f32 rows over tiled weights as two planes through the tile GEMM, whole
    and with K split (long K, few tiles), against the oracle.  The planes hold x
    to 2^-18 of its size and the sums are f32: 1e-5 of the result's norm."""
    tuning("CASCADIA_INT4_F32_TILE_TOKENS", "17")
    packed = orc.fill_bytes(n + M, 3, n * k // 2)
    scales = orc.fill_scales(n + M, 4, n * (k // g), sdt).view(np.uint8).copy()
    pt, st = cl.tile_weights(dev(packed), dev(scales), n, k, g)
    xs = orc.fill_normal_f32(k, M, M * k)
    want = orc.gemm_multi(packed, scales, xs, n, k, M, g, sdt)
    ys = torch.empty(M * n, dtype=torch.float32, device="cuda")
    cl.dequant_gemm_int4_multi_auto(pt, st, dev(xs), n, k, M, ys, group_size=g, scale_dtype=sdt,
                                    tiling=cl.TILING_MFMA)
    got = host(ys).reshape(M, n)
    assert_f32_close(got, want, f"f32 tiles {n}x{k} G{g} M{M}")
    assert rel_l2(got, want) <= 1e-5


@pytest.mark.parametrize("g,mean", [(32, 0.0), (64, 0.0), (64, 1.0), (128, 0.0), (128, 1.0)])
def test_gemm_f32_tiles_lose_no_precision(cl, tuning, g, mean):
    """The tile GEMM's f32 result is no further from 64 bits than the skinny
    kernel's, whose planes add up apart, also where the zero point's share of a
    group's sum is large (rows of mean 1)."""
    n, k, M = 1024, 4096, 64
    packed = cl.fill_bytes(torch.empty(n * k // 2, dtype=torch.uint8, device="cuda"), 11, 1)
    scales = cl.fill_scales(torch.empty(n * (k // g), dtype=torch.int16, device="cuda"), 11, 2, F16)
    x = cl.fill_normal(torch.empty((M, k), dtype=torch.float32, device="cuda"), 11, 3) + mean
    scales = scales.view(torch.uint8)
    want = x.double() @ cl.debug_dequant(packed, scales, n, k, g, F16).double().T
    pt, st = cl.tile_weights(packed, scales, n, k, g)
    err = {}
    for route, rows in (("tiles", "17"), ("skinny", "100000")):
        tuning("CASCADIA_INT4_F32_TILE_TOKENS", rows)
        ys = torch.empty((M, n), dtype=torch.float32, device="cuda")
        cl.dequant_gemm_int4_multi_auto(pt, st, x, n, k, M, ys, group_size=g, scale_dtype=F16,
                                        tiling=cl.TILING_MFMA)
        err[route] = rel_l2(host(ys), want.cpu().numpy())
    assert err["tiles"] <= err["skinny"], err


@pytest.mark.parametrize("n", [1001, 1002, 1003, 4097])
@pytest.mark.parametrize("M,g", [(64, 128), (77, 32)])
def test_gemm_split_any_columns(cl, tuning, n, M, g):
    """K is cut into slices whatever the columns (few tiles, long K): f32 and
    bf16 rows, f32 and bf16 outputs, nothing written past the last column."""
    k = 8192
    tuning("CASCADIA_INT4_F32_TILE_TOKENS", "17")
    packed = cl.fill_bytes(torch.empty(n * k // 2, dtype=torch.uint8, device="cuda"), 17, 1)
    scales = cl.fill_scales(torch.empty(n * (k // g), dtype=torch.int16, device="cuda"), 17, 2)
    scales = scales.view(torch.uint8)
    pt, st = cl.tile_weights(packed, scales, n, k, g)
    x = cl.fill_normal(torch.empty((M, k), device="cuda"), 17, 3)
    W = cl.debug_dequant(packed, scales, n, k, g, F16).double()
    # the partials of at least two slices, beside the f32 rows' planes
    assert cl.gemm_workspace_bytes(n, k, M, True, g, cl.TILING_MFMA) >= 4 * M * k + 8 * M * n
    for dt in (torch.float32, torch.bfloat16):
        xd = x.to(dt)
        want = (xd.double() @ W.T).cpu().numpy()
        opts = dict(group_size=g, scale_dtype=F16, tiling=cl.TILING_MFMA)
        buf = torch.full((M * n + 8,), 7.0, device="cuda")
        cl.dequant_gemm_int4_multi_auto(pt, st, xd, n, k, M, buf[:M * n], **opts)
        assert rel_l2(host(buf[:M * n]).reshape(M, n), want) <= 1e-5
        assert bool((buf[M * n:] == 7.0).all())
        if dt == torch.bfloat16:
            out = torch.full((M * n + 8,), 7.0, dtype=dt, device="cuda")
            cl.gemm_int4_bf16(pt, st, xd, n, k, M, out[:M * n], **opts)
            # one rounding to 8 bits: at most 2^-9 of each value
            assert rel_l2(host(out[:M * n].float()).reshape(M, n), want) <= 2 ** -9
            assert bool((out[M * n:] == 7.0).all())


def shifted(t):
    """The same bytes two past a 16-byte boundary."""
    s = torch.empty(t.numel() + 16, dtype=torch.uint8, device="cuda")[2:2 + t.numel()]
    return s.copy_(t)


@pytest.mark.parametrize("g", [32, 128])
def test_scales_aligned_to_two_bytes(cl, tuning, g):
    """Scales need two bytes' alignment only; the kernels that load them into LDS
    four bytes at a time leave such calls to the skinny kernel."""
    n, k, M = 1024, 2048, 100
    packed = cl.fill_bytes(torch.empty(n * k // 2, dtype=torch.uint8, device="cuda"), 12, 1)
    scales = cl.fill_scales(torch.empty(n * (k // g), dtype=torch.int16, device="cuda"), 12, 2, F16)
    pt, st = cl.tile_weights(packed, scales.view(torch.uint8), n, k, g)
    x = cl.fill_normal(torch.empty((M, k), dtype=torch.float32, device="cuda"), 12, 3)
    opts = dict(group_size=g, scale_dtype=F16, tiling=cl.TILING_MFMA)
    ys = [torch.empty((M, n), device="cuda") for _ in range(2)]
    tuning("CASCADIA_INT4_F32_TILE_TOKENS", "17")
    cl.dequant_gemm_int4_multi_auto(pt, shifted(st), x, n, k, M, ys[0], **opts)
    tuning("CASCADIA_INT4_F32_TILE_TOKENS", "100000")
    cl.dequant_gemm_int4_multi_auto(pt, st, x, n, k, M, ys[1], **opts)
    assert torch.equal(ys[0], ys[1])
    h, i = 1024, 512
    flat = cl.fill_bytes(torch.empty(cl.expert_bytes(h, i, g), dtype=torch.uint8, device="cuda"),
                         13, 1)
    W = cl.ExpertWeights(flat, h, i, g, F16)
    for t in W.slices()[1::2]:
        cl.fill_scales(t.view(torch.int16), 13, 2)
    W = W.tiled()
    xb = x[:, :h].to(torch.bfloat16).contiguous()
    for m, var in ((16, "CASCADIA_INT4_FEW_MIN_TOKENS"), (100, "CASCADIA_INT4_FFN_TILE_TOKENS")):
        outs = [torch.empty((m, h), dtype=torch.bfloat16, device="cuda") for _ in range(2)]
        tuning(var, "2")
        cl.expert_forward(xb[:m], *[shifted(t) if j % 2 else t for j, t in enumerate(W.slices())],
                          outs[0], **opts)
        tuning(var, "100000")
        cl.expert_forward(xb[:m], *W.slices(), outs[1], **opts)
        assert torch.equal(outs[0], outs[1]), f"{m} rows"


def test_gemm_f32_capture(cl, orc):
    """An f32 GEMM without a workspace, of a shape not seen before, is recorded in
    the skinny kernel's form (a process whose first call is recorded:
    test_recorded_forms_in_a_fresh_process); replays and eager calls between
    them, on the tile route, are both within the bar."""
    n, k, g, M = 3000, 4096, 128, 333
    packed = orc.fill_bytes(5, 5, n * k // 2)
    scales = orc.fill_scales(5, 6, n * (k // g), F16).view(np.uint8).copy()
    pt, st = cl.tile_weights(dev(packed), dev(scales), n, k, g)
    xs = orc.fill_normal_f32(5, 7, M * k)
    xd = dev(xs)
    want = orc.gemm_multi(packed, scales, xs, n, k, M, g, F16)
    ys = torch.empty(M * n, dtype=torch.float32, device="cuda")
    call = lambda: cl.dequant_gemm_int4_multi_auto(  # noqa: E731
        pt, st, xd, n, k, M, ys, group_size=g, scale_dtype=F16, tiling=cl.TILING_MFMA)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call()
    for _ in range(3):
        ys.zero_()
        graph.replay()
        assert_f32_close(host(ys).reshape(M, n), want, "replay")
        call()
        assert_f32_close(host(ys).reshape(M, n), want, "eager")


@pytest.mark.parametrize("M,h,i,g", [(33, 2048, 1024, 32), (100, 1024, 2048, 64),
                                     (161, 2048, 1536, 128)])
def test_ffn_split_tiles(cl, orc, tuning, M, h, i, g):
    """An FFN whose gate/up and down split K (few tiles): the SwiGLU and the
    planes' seeds made by the reduce, bf16 and f32 rows."""
    tuning("CASCADIA_INT4_FFN_TILE_TOKENS", "33")
    flat = expert(orc, h, i, g, F16, M + g)
    W = cl.ExpertWeights(dev(flat), h, i, g, F16).tiled()
    xb = orc.fill_normal_bf16(M, 52, M * h)
    out = torch.empty(M * h, dtype=torch.int16, device="cuda")
    cl.expert_forward(dev(xb.view(np.int16).reshape(M, h)), *W.slices(), out, group_size=g,
                      scale_dtype=F16, tiling=cl.TILING_MFMA)
    assert_bf16_close(host(out).view(np.uint16).reshape(M, h),
                      orc.cpu_expert_forward(xb, M, flat, h, i, g, F16), f"split M{M} G{g}")
    x = orc.fill_normal_f32(8, M, M * h).reshape(M, h)
    of = torch.empty((M, h), dtype=torch.float32, device="cuda")
    cl.ffn_forward_sparse_f32(dev(x), h, i, *W.slices(), of, 0.0, group_size=g, scale_dtype=F16,
                              tiling=cl.TILING_MFMA)
    want = np.stack([orc.ffn_forward_f32(x[t], flat, h, i, g, F16)[0] for t in range(M)])
    assert_f32_close(host(of), want, f"split f32 M{M} G{g}")


@pytest.mark.parametrize("M,h,i,g,sdt", [(2, 384, 256, 32, F16), (16, 2048, 1152, 32, BF16),
                                         (17, 640, 1024, 64, F16), (9, 4096, 1536, 128, BF16),
                                         (32, 1536, 4608, 128, F16), (31, 2048, 512, 256, F16)])
def test_ffn_few_rows(cl, orc, tuning, M, h, i, g, sdt):
    """The kernel of a decode batch (2 .. 32 rows): one and two M-tiles, K of an
    odd number of blocks, both GEMMs with and without K slices."""
    tuning("CASCADIA_INT4_FEW_MIN_TOKENS", "2")
    flat = expert(orc, h, i, g, sdt, M + g)
    W = cl.ExpertWeights(dev(flat), h, i, g, sdt).tiled()
    xb = orc.fill_normal_bf16(M, 52, M * h)
    x = dev(xb.view(np.int16).reshape(M, h))
    out = torch.empty(M * h, dtype=torch.int16, device="cuda")
    cl.expert_forward(x, *W.slices(), out, group_size=g, scale_dtype=sdt, tiling=cl.TILING_MFMA)
    want = orc.cpu_expert_forward(xb, M, flat, h, i, g, sdt)
    assert_bf16_close(host(out).view(np.uint16).reshape(M, h), want, f"few M{M} G{g}")


@pytest.mark.parametrize("M,g", [(65, 32), (100, 64), (200, 128)])
def test_ffn_f32_tiles(cl, orc, tuning, M, g):
    """The f32-in / f32-out FFN (the shared expert) over M rows: x split into
    hi / lo planes, both planes through every MFMA."""
    tuning("CASCADIA_INT4_FFN_TILE_TOKENS", "65")
    h, i, sdt = 512, 384, F16
    flat = expert(orc, h, i, g, sdt, 7 + g)
    W = cl.ExpertWeights(dev(flat), h, i, g, sdt).tiled()
    x = orc.fill_normal_f32(8, M, M * h).reshape(M, h)
    out = torch.empty((M, h), dtype=torch.float32, device="cuda")
    cl.ffn_forward_sparse_f32(dev(x), h, i, *W.slices(), out, 0.0, group_size=g, scale_dtype=sdt,
                              tiling=cl.TILING_MFMA)
    want = np.stack([orc.ffn_forward_f32(x[t], flat, h, i, g, sdt)[0] for t in range(M)])
    assert_f32_close(host(out), want, f"ffn f32 tiles M{M} G{g}")


@pytest.mark.parametrize("hot_rows", ["1", "48"])
@pytest.mark.parametrize("T", [65, 200])
@pytest.mark.parametrize("g,mode,shared_inter,thr", [(32, 1, 256, 0.0), (128, 2, 0, 0.0),
                                                     (64, 1, 128, 0.2)])
def test_moe_tiles(cl, orc, tuning, T, g, mode, shared_inter, thr, hot_rows):
    """MoE layers of 65+ tokens (routing by logits; the tile thresholds
    lowered to 65 tokens): every expert on the tile GEMMs (hot_rows 1), or the
    hybrid split -- experts with 48+ rows on tiles, the others on the skinny
    kernels' 16-row chunks."""
    tuning("CASCADIA_INT4_MOE_TILE_TOKENS", "65")
    tuning("CASCADIA_INT4_FFN_TILE_TOKENS", "65")
    tuning("CASCADIA_INT4_MOE_TILE_ROWS", hot_rows)
    E, k, h, i, sdt = 12, 4, 512, 256, F16
    blob, shared, ex = build(cl, orc, E, h, i, g, sdt, 61 + g, shared_inter, True)
    logits = orc.fill_normal_f32(62, T, T * E).reshape(T, E)
    x = orc.fill_normal_f32(63, T, T * h).reshape(T, h)
    out = torch.empty((T, h), dtype=torch.float32, device="cuda")
    ids_o = torch.empty((T, k), dtype=torch.int32, device="cuda")
    w_o = torch.empty((T, k), dtype=torch.float32, device="cuda")
    xd = dev(x)
    cl.moe_forward(ex, xd, out, top_k=k, logits=dev(logits), mode=mode, scale=1.0,
                   threshold=thr, residual=xd, ids_out=ids_o, weights_out=w_o)
    check_layer(orc, host(out), x, blob, shared, shared_inter, E, h, i, g, sdt, host(ids_o),
                host(w_o), thr, f"tiles T={T} G{g} mode={mode}")


@pytest.mark.parametrize("T,E,k,g", [(191, 12, 4, 32), (192, 12, 4, 64), (192, 24, 4, 128),
                                     (216, 24, 4, 32)])
def test_moe_tile_rule(cl, orc, T, E, k, g):
    """Both sides of the default rule's edges: 192 tokens, 36 rows per expert."""
    h, i = 384, 256
    blob, shared, ex = build(cl, orc, E, h, i, g, F16, 67 + g, 128, True)
    logits = orc.fill_normal_f32(62, T, T * E).reshape(T, E)
    x = orc.fill_normal_f32(63, T, T * h).reshape(T, h)
    out = torch.empty((T, h), dtype=torch.float32, device="cuda")
    ids_o = torch.empty((T, k), dtype=torch.int32, device="cuda")
    w_o = torch.empty((T, k), dtype=torch.float32, device="cuda")
    xd = dev(x)
    cl.moe_forward(ex, xd, out, top_k=k, logits=dev(logits), mode=1, scale=1.0, residual=xd,
                   ids_out=ids_o, weights_out=w_o)
    check_layer(orc, host(out), x, blob, shared, 128, E, h, i, g, F16, host(ids_o), host(w_o),
                0.0, f"rule T={T} E={E} G{g}")


def test_moe_tiles_hot_expert(cl, orc, tuning):
    """Given ids sending every token to one expert (300 rows: three 128-row
    chunks, the last partial) plus scattered ones; two calls bit-identical."""
    tuning("CASCADIA_INT4_MOE_TILE_TOKENS", "65")
    E, k, h, i, g, T = 9, 3, 384, 256, 32, 300
    blob, shared, ex = build(cl, orc, E, h, i, g, F16, 71, 128, True)
    rng = np.random.default_rng(3)
    ids = rng.integers(0, E, size=(T, k)).astype(np.int32)
    ids[:, 0] = 4
    ids[:, 1] = np.where(ids[:, 1] == 4, 5, ids[:, 1])
    ids[:, 2] = np.where((ids[:, 2] == 4) | (ids[:, 2] == ids[:, 1]), 0, ids[:, 2])
    ids[:, 1] = np.where(ids[:, 1] == ids[:, 2], 1, ids[:, 1])
    w = rng.random((T, k)).astype(np.float32)
    x = orc.fill_normal_f32(72, T, T * h).reshape(T, h)
    xd = dev(x)
    outs = []
    for _ in range(2):
        o = torch.empty((T, h), dtype=torch.float32, device="cuda")
        cl.moe_forward(ex, xd, o, top_k=k, mode=cl.ROUTE_IDS, ids=dev(ids), weights=dev(w),
                       residual=xd)
        outs.append(host(o))
    assert np.array_equal(outs[0].view(np.uint32), outs[1].view(np.uint32)), "not deterministic"
    check_layer(orc, outs[0], x, blob, shared, 128, E, h, i, g, F16, ids, w, 0.0, "hot expert")


def test_tiles_match_skinny_path(cl, orc, tuning):
    """The same 80-token layer through both paths (the skinny grouped kernels
    forced by a high tile threshold): both within the bar of the oracle and of
    each other."""
    E, k, h, i, g, T = 10, 4, 512, 384, 32, 80
    blob, shared, ex = build(cl, orc, E, h, i, g, F16, 81, 128, True)
    logits = orc.fill_normal_f32(82, T, T * E).reshape(T, E)
    x = orc.fill_normal_f32(83, T, T * h).reshape(T, h)
    xd = dev(x)
    res = []
    for thr_tokens in ("65", "100000"):
        tuning("CASCADIA_INT4_MOE_TILE_TOKENS", thr_tokens)
        tuning("CASCADIA_INT4_FFN_TILE_TOKENS", thr_tokens)
        o = torch.empty((T, h), dtype=torch.float32, device="cuda")
        cl.moe_forward(ex, xd, o, top_k=k, logits=dev(logits), mode=1, scale=2.5,
                       residual=xd)
        res.append(host(o))
    d0, d1 = res[0] - x, res[1] - x
    assert rel_l2(d0, d1) <= REL_L2_TOL
