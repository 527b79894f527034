"""Calls on two streams at once, each with its own workspace and outputs,
equal the same calls made one after another, bit for bit.

The header promises that calls are reentrant for distinct output buffers
when each brings its own workspace (include/cascadia_int4.h).  Here the
expert FFN at one and four tokens (at four tokens both projections split K
across workgroups into partials in the workspace), the f32-in FFN at three
tokens, and MoE layers at
5 and 70 tokens (one prep launch, then separate routing / grouping launches;
the shared expert forks onto the library's side stream) are enqueued on two
streams, alternating, with no synchronisation between them, and every output
is compared with the serial result.

Calls without a workspace use the library's buffer of their stream: multi-row
GEMMs and FFNs on two streams, on more streams than have a buffer of their own,
from two threads on one stream, and beside the replays of a graph.
"""
import threading

import numpy as np
import pytest
import torch

from test_gpu_moe import build

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


def expert(orc, h, i, g, sdt, seed):
    flat = orc.fill_bytes(seed, 60, orc.expert_bytes(h, i, g)).copy()
    offs, sizes = orc.expert_offsets(h, i, g)
    for s_ in (1, 3, 5):
        flat[offs[s_]:offs[s_] + sizes[s_]] = orc.fill_scales(seed, 61 + s_, sizes[s_] // 2,
                                                              sdt).view(np.uint8)
    return flat


def test_two_streams_equal_serial(cl, orc):
    print("two streams: expert FFN M1/M4, f32 FFN, MoE T5/T70", flush=True)
    h, i, g = 1024, 3072, 128
    W = cl.ExpertWeights(dev(expert(orc, h, i, g, F16, 5)), h, i, g, F16).tiled()
    E, mh, mi, k, si = 16, 512, 384, 4, 128
    _, _, ex = build(cl, orc, E, mh, mi, 32, F16, 6, shared_inter=si, tiled=True)

    # each job: (a closure issuing the call on the current stream into its
    # outputs with its workspace, the output tensors)
    def make_jobs():
        jobs = []
        for T in (1, 4):
            x = cl.fill_normal(torch.empty((T, h), dtype=torch.bfloat16, device="cuda"), 7, T)
            out = torch.empty((T, h), dtype=torch.bfloat16, device="cuda")
            ws = torch.empty(cl.ffn_workspace_bytes(h, i, T, g), dtype=torch.uint8, device="cuda")
            jobs.append((lambda x=x, out=out, ws=ws: cl.expert_forward(
                x, *W.slices(), out, group_size=g, scale_dtype=F16, workspace=ws,
                tiling=cl.TILING_MFMA), [out]))
        xf = cl.fill_normal(torch.empty((3, h), dtype=torch.float32, device="cuda"), 8, 3)
        of = torch.empty((3, h), dtype=torch.float32, device="cuda")
        wsf = torch.empty(cl.ffn_sparse_workspace_bytes(h, i, 3, g), dtype=torch.uint8,
                          device="cuda")
        jobs.append((lambda: cl.ffn_forward_sparse_f32(
            xf, h, i, *W.slices(), of, 0.0, group_size=g, scale_dtype=F16, workspace=wsf,
            tiling=cl.TILING_MFMA), [of]))
        for T in (5, 70):
            x = cl.fill_normal(torch.empty((T, mh), dtype=torch.float32, device="cuda"), 9, T)
            lg = cl.fill_normal(torch.empty((T, E), dtype=torch.float32, device="cuda"), 10, T)
            out = torch.empty((T, mh), dtype=torch.float32, device="cuda")
            ids = torch.empty((T, k), dtype=torch.int32, device="cuda")
            wts = torch.empty((T, k), dtype=torch.float32, device="cuda")
            ws = torch.empty(cl.moe_workspace_bytes(ex, k, T), dtype=torch.uint8, device="cuda")
            jobs.append((lambda x=x, lg=lg, out=out, ids=ids, wts=wts, ws=ws: cl.moe_forward(
                ex, x, out, top_k=k, logits=lg, mode=cl.ROUTE_SIGMOID_BIAS, scale=2.5,
                residual=x, ids_out=ids, weights_out=wts, workspace=ws), [out, ids, wts]))
        return jobs

    serial = make_jobs()
    for fn, _ in serial:
        fn()
        torch.cuda.synchronize()
    want = [[t.clone() for t in outs] for _, outs in serial]

    a_jobs, b_jobs = make_jobs(), make_jobs()
    sa, sb = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    for rep in range(6):
        for j in range(len(a_jobs)):
            with torch.cuda.stream(sa):
                a_jobs[j][0]()
            with torch.cuda.stream(sb):
                b_jobs[(j + rep) % len(b_jobs)][0]()
    torch.cuda.synchronize()
    for jobs, name in ((a_jobs, "stream a"), (b_jobs, "stream b")):
        for j, (_, outs) in enumerate(jobs):
            for t, w in zip(outs, want[j]):
                assert torch.equal(t, w), f"{name}, job {j}: differs from the serial call"


def gemm_jobs(cl, rows=(17, 100, 333), n=3072, k=4096, g=32):
    """Calls without a workspace that need one: f32 and bf16 rows through the
    tile GEMM, and an FFN; each (call, output)."""
    packed = cl.fill_bytes(torch.empty(n * k // 2, dtype=torch.uint8, device="cuda"), 21, 1)
    scales = cl.fill_scales(torch.empty(n * (k // g), dtype=torch.int16, device="cuda"), 21, 2)
    pt, st = cl.tile_weights(packed, scales.view(torch.uint8), n, k, g)
    opts = dict(group_size=g, scale_dtype=F16, tiling=cl.TILING_MFMA)
    jobs = []
    for M in rows:
        for dt in (torch.float32, torch.bfloat16):
            x = cl.fill_normal(torch.empty((M, k), dtype=dt, device="cuda"), 22, M)
            y = torch.empty((M, n), dtype=torch.float32, device="cuda")
            jobs.append((lambda x=x, y=y, M=M: cl.dequant_gemm_int4_multi_auto(
                pt, st, x, n, k, M, y, **opts), y))
    h, i, hg = 1024, 3072, 128
    flat = cl.fill_bytes(torch.empty(cl.expert_bytes(h, i, hg), dtype=torch.uint8, device="cuda"),
                         23, 1)
    W = cl.ExpertWeights(flat, h, i, hg, F16)
    for s in W.slices()[1::2]:
        cl.fill_scales(s.view(torch.int16), 23, 2)
    W = W.tiled()
    x = cl.fill_normal(torch.empty((200, h), dtype=torch.bfloat16, device="cuda"), 24, 1)
    out = torch.empty_like(x)
    jobs.append((lambda: cl.expert_forward(x, *W.slices(), out, group_size=hg, scale_dtype=F16,
                                           tiling=cl.TILING_MFMA), out))
    return jobs


def serial_results(jobs):
    want = []
    for fn, out in jobs:
        fn()
        torch.cuda.synchronize()
        want.append(out.clone())
        out.zero_()
    torch.cuda.synchronize()
    return want


@pytest.mark.parametrize("n_streams", [2, 20])
def test_library_workspace_on_streams(cl, n_streams):
    """(20: more streams than the library keeps a buffer for)"""
    print(f"{n_streams} streams without workspaces", flush=True)
    sets = [gemm_jobs(cl, rows=(333,) if n_streams > 2 else (17, 100, 333))
            for _ in range(n_streams)]
    want = serial_results(sets[0])
    streams = [torch.cuda.Stream() for _ in range(n_streams)]
    torch.cuda.synchronize()
    for rep in range(4):
        for j in range(len(want)):
            for s, jobs in zip(streams, sets):
                with torch.cuda.stream(s):
                    jobs[(j + rep) % len(jobs)][0]()
    torch.cuda.synchronize()
    for c, jobs in enumerate(sets):
        for j, (_, out) in enumerate(jobs):
            assert torch.equal(out, want[j]), f"stream {c}, job {j}: differs from the serial call"


@pytest.mark.parametrize("one_stream", [True, False])
def test_library_workspace_from_two_threads(cl, one_stream):
    print(f"two threads, one stream: {one_stream}", flush=True)
    sets = [gemm_jobs(cl), gemm_jobs(cl)]
    want = serial_results(sets[0])
    shared = torch.cuda.Stream()
    streams = [shared, shared if one_stream else torch.cuda.Stream()]
    errors = []

    def work(jobs, stream):
        try:
            with torch.cuda.stream(stream):
                for _ in range(6):
                    for fn, _ in jobs:
                        fn()
        except Exception as e:  # noqa: BLE001 -- reported below
            errors.append(e)

    threads = [threading.Thread(target=work, args=a) for a in zip(sets, streams)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not errors, errors
    for c, jobs in enumerate(sets):
        for j, (_, out) in enumerate(jobs):
            assert torch.equal(out, want[j]), f"thread {c}, job {j}: differs from the serial call"


@pytest.mark.parametrize("own_workspace", [True, False])
def test_graph_replays_beside_eager_calls(cl, own_workspace):
    """A recorded f32 GEMM replayed while eager ones run on another stream; with a
    workspace of its own it is the eager form, bit for bit."""
    n, k, g, M = 3072, 4096, 32, 333
    packed = cl.fill_bytes(torch.empty(n * k // 2, dtype=torch.uint8, device="cuda"), 31, 1)
    scales = cl.fill_scales(torch.empty(n * (k // g), dtype=torch.int16, device="cuda"), 31, 2)
    pt, st = cl.tile_weights(packed, scales.view(torch.uint8), n, k, g)
    opts = dict(group_size=g, scale_dtype=F16, tiling=cl.TILING_MFMA)
    xs = [cl.fill_normal(torch.empty((M, k), device="cuda"), 32, j) for j in range(2)]
    ys = [torch.empty((M, n), device="cuda") for _ in range(2)]
    call = lambda j, **kw: cl.dequant_gemm_int4_multi_auto(  # noqa: E731
        pt, st, xs[j], n, k, M, ys[j], **opts, **kw)
    want = serial_results([(lambda: call(0), ys[0]), (lambda: call(1), ys[1])])
    kw = {}
    if own_workspace:
        kw["workspace"] = torch.empty(cl.gemm_workspace_bytes(n, k, M, True, g, cl.TILING_MFMA),
                                      dtype=torch.uint8, device="cuda")
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call(0, **kw)
    graph.replay()
    torch.cuda.synchronize()
    recorded = ys[0].clone()
    if own_workspace:
        assert torch.equal(recorded, want[0])
    else:  # the form that shares no memory: another order of the same sums
        assert float((recorded - want[0]).norm() / want[0].norm()) <= 1e-5
    sa, sb = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    for rep in range(8):
        ys[0].zero_(), ys[1].zero_()
        torch.cuda.synchronize()
        with torch.cuda.stream(sa):
            graph.replay()
        with torch.cuda.stream(sb):
            call(1)
            call(1)
        torch.cuda.synchronize()
        assert torch.equal(ys[0], recorded), f"replay {rep}"
        assert torch.equal(ys[1], want[1]), f"eager call beside replay {rep}"
