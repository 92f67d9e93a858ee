"""msco_gmm_launch allocates nothing and never synchronises, so a launch can be recorded into a HIP graph: the graph is
replayed several times with eager work and synchronisations in between, and every replay is compared with the eager
result (bit-exact).  Covers the kernels with cross-workgroup state (K split: self-resetting arrival counters) and the
persistent tile kernel."""
import numpy as np
import pytest
import torch

from ms_custom_ops_amd import cabi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("case", ["decode_split_k", "packed_decode", "packed_rows_split_k", "persistent_tile", "small_tile_split_k"])
def test_launch_is_graph_capturable_and_replays_match_eager(device, case):
    from gpu_utils import pack_on_device
    shapes = {"decode_split_k": (16, 4096, 1024, 1, False, False), "packed_decode": (20, 2048, 1024, 4, False, True),
              "packed_rows_split_k": (128, 4096, 256, 1, False, True), "persistent_tile": (2048, 512, 8192, 8, True, False),
              "small_tile_split_k": (128, 2048, 1024, 1, True, False)}
    m, k, n, e, nk, packed = shapes[case]
    g = torch.Generator(device="cuda")
    g.manual_seed(3)
    x = torch.randint(-127, 128, (m, k), dtype=torch.int8, device="cuda", generator=g)
    w = torch.randint(-127, 128, (e, n, k) if nk else (e, k, n), dtype=torch.int8, device="cuda", generator=g)
    if packed:
        w = pack_on_device(w, e, k, n, nk)
    scale = torch.rand(e, n, device="cuda", generator=g) * 9e-3 + 1e-3
    pt = torch.rand(m, device="cuda", generator=g) * 9e-3 + 1e-3
    gl = torch.tensor([(m * (i + 1)) // e for i in range(e)], dtype=torch.int64, device="cuda")
    op = cabi.GmmOp(x_dtype=cabi.DT_I8, out_dtype=cabi.DT_BF16, group_list_dtype=cabi.DT_I64, scale_dtype=cabi.DT_F32,
                    per_token_dtype=cabi.DT_F32, transpose_b=int(nk and not packed),
                    weight_layout=cabi.WL_PACKED if packed else cabi.WL_ROW_MAJOR)
    ws_bytes = op.plan(m, k, n, e)
    if "split_k" in case:
        assert "split_k=1 " not in op.plan_info(), op.plan_info()
    ws = torch.empty(max(ws_bytes, 1), dtype=torch.uint8, device="cuda")
    out = torch.empty((m, n), dtype=torch.int16, device="cuda")
    ins = [x.data_ptr(), w.data_ptr(), None, scale.data_ptr(), gl.data_ptr(), pt.data_ptr(), None, None]
    op.launch(ins, out.data_ptr(), ws.data_ptr(), ws_bytes, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    eager = out.clone()

    graph = torch.cuda.CUDAGraph()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        with torch.cuda.graph(graph, stream=side):
            op.launch(ins, out.data_ptr(), ws.data_ptr(), ws_bytes, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    for replay in range(4):
        out.fill_(0x7FC0)                      # eager work between replays
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager), (case, replay, op.plan_info())
        # an eager launch between replays shares the handle's arrival counters with the graph's launches
        op.launch(ins, out.data_ptr(), ws.data_ptr(), ws_bytes, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        assert torch.equal(out, eager), (case, replay, "eager after replay")
    op.close()


def test_moe_chain_is_graph_capturable(device):
    """Quantising routing -> int8 grouped matmul on its outputs -> un-permutation, recorded as one graph: none of the
    three allocates, clears memory with a memset node or synchronises, and the routing output feeds the matmul's
    group_list on the device.  Every replay must reproduce the eager result bit for bit."""
    rows, hidden, k, e, n = 256, 1024, 2, 8, 512
    g = torch.Generator(device="cuda")
    g.manual_seed(9)
    x = torch.randn((rows, hidden), dtype=torch.bfloat16, device="cuda", generator=g)
    idx = torch.argsort(torch.randn(rows, e, device="cuda", generator=g), dim=1)[:, :k].to(torch.int32).contiguous()
    w = torch.randint(-127, 128, (e, hidden, n), dtype=torch.int8, device="cuda", generator=g)
    wscale = torch.rand(e, n, device="cuda", generator=g) * 9e-3 + 1e-3
    probs = torch.rand((rows, k), dtype=torch.bfloat16, device="cuda", generator=g)
    xq = torch.empty((rows * k, hidden), dtype=torch.int8, device="cuda")
    xs = torch.empty(rows * k, dtype=torch.float32, device="cuda")
    ridx = torch.empty(rows * k, dtype=torch.int32, device="cuda")
    cum = torch.empty(e, dtype=torch.int32, device="cuda")
    y = torch.empty((rows * k, n), dtype=torch.int16, device="cuda")
    out = torch.empty((rows, n), dtype=torch.int16, device="cuda")
    rws_bytes = cabi.moe_init_routing_v2_workspace_bytes(rows, k, e)
    rws = torch.empty(max(rws_bytes, 1), dtype=torch.uint8, device="cuda")
    op = cabi.GmmOp(x_dtype=cabi.DT_I8, out_dtype=cabi.DT_BF16, group_list_dtype=cabi.DT_I32, scale_dtype=cabi.DT_F32,
                    per_token_dtype=cabi.DT_F32)
    ws_bytes = op.plan(rows * k, hidden, n, e)
    ws = torch.empty(max(ws_bytes, 1), dtype=torch.uint8, device="cuda")

    def chain(stream):
        cabi.moe_init_routing_v2_quant(x.data_ptr(), idx.data_ptr(), xq.data_ptr(), xs.data_ptr(), ridx.data_ptr(), cum.data_ptr(), None,
                                       rws.data_ptr(), rws_bytes, rows, hidden, k, e, cabi.DT_BF16, 1, stream)
        op.launch([xq.data_ptr(), w.data_ptr(), None, wscale.data_ptr(), cum.data_ptr(), xs.data_ptr(), None, None], y.data_ptr(),
                  ws.data_ptr(), ws_bytes, stream)
        cabi.moe_token_unpermute(y.data_ptr(), ridx.data_ptr(), probs.data_ptr(), out.data_ptr(), rows, k, n, cabi.DT_BF16, stream)

    chain(torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    eager = out.clone()
    assert eager.ne(0).any()
    graph = torch.cuda.CUDAGraph()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        with torch.cuda.graph(graph, stream=side):
            chain(torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    for replay in range(3):
        for t in (xq, y, out):
            t.fill_(0)                         # eager work between replays
        xs.fill_(0)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager), replay
    op.close()


def _weight_only(m, k, n, e, seed):
    """A weight-only grouped call through the Python operator; plans with 16 to 128 rows per group and a long K split it."""
    import ms_custom_ops_amd as ops
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    x = torch.randn((m, k), dtype=torch.bfloat16, device="cuda", generator=g)
    w = torch.randint(-127, 128, (e, k, n), dtype=torch.int8, device="cuda", generator=g)
    s = (torch.rand(e, n, device="cuda", generator=g) * 1e-3).to(torch.bfloat16)
    gl = torch.tensor([(m * (i + 1)) // e for i in range(e)], dtype=torch.int64, device="cuda")
    return lambda: ops.grouped_matmul_v4_cops([x], [w], antiquant_scale=[s], group_list=gl, split_item=3, group_type=0)[0]


def _dense(m, k, n, seed):
    import ms_custom_ops_amd as ops
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    x = torch.randint(-127, 128, (m, k), dtype=torch.int8, device="cuda", generator=g)
    w = torch.randint(-127, 128, (k, n), dtype=torch.int8, device="cuda", generator=g)
    s = torch.rand(n, device="cuda", generator=g) * 1e-3
    return lambda: ops.quant_batch_matmul(x, w, s)


# (calls whose plan splits K, and one that does not)
_CALLS = [(_weight_only, (816, 6336, 544, 16)), (_dense, (13, 7952, 5392)), (_dense, (40, 4096, 512)), (_dense, (2048, 1024, 1024))]


@pytest.mark.parametrize("call", _CALLS, ids=["weight_only_split_k", "few_rows_split_k", "small_tile_split_k", "tile"])
def test_first_call_of_a_shape_under_capture_and_replays_after_its_plan_is_gone(device, call):
    """Planning allocates and clears arrival counters; inside a capture it has to go through.  70 other shapes then push the plan out of the
    operators' cache (64 plans per process): the recorded launches keep counters of their own, so replays stay right."""
    make, args = call
    f = make(*args, seed=5)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = f()
    eager = f().clone()
    torch.cuda.synchronize()
    assert eager.ne(0).any()

    def replays():
        for _ in range(3):
            out.fill_(7)
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, eager)
            assert torch.equal(f(), eager)

    replays()
    for i in range(70):
        _dense(1 + i % 16, 1024 + 16 * i, 256, seed=i)()
    replays()


def test_graphs_of_one_shape_replayed_side_by_side(device):
    """Two graphs recorded on the same stream from one shape, and eager calls, at the same time on three streams."""
    fs = [_weight_only(816, 6336, 544, 16, seed=s) for s in (1, 2, 3)]
    want = [f().clone() for f in fs]
    torch.cuda.synchronize()
    graphs, outs = [], []
    for f in fs[:2]:
        graphs.append(torch.cuda.CUDAGraph())
        with torch.cuda.graph(graphs[-1]):
            outs.append(f())
    streams = [torch.cuda.Stream() for _ in range(2)]
    torch.cuda.synchronize()
    for _ in range(20):
        for o in outs:
            o.fill_(7)
        torch.cuda.synchronize()
        for g, st in zip(graphs, streams):
            with torch.cuda.stream(st):
                g.replay()
        eager = fs[2]()
        torch.cuda.synchronize()
        assert torch.equal(outs[0], want[0]) and torch.equal(outs[1], want[1]) and torch.equal(eager, want[2])


def test_a_plan_leaves_the_cache_while_a_stream_is_captured(device):
    """Planning 70 shapes inside one capture evicts plans that other calls allocated counters for."""
    f = _dense(13, 7952, 5392, seed=1)
    want = f().clone()
    small = [_dense(1 + i % 16, 1040 + 16 * i, 272, seed=i) for i in range(70)]
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outs = [g() for g in small]
    for _ in range(2):
        for o in outs:
            o.fill_(7)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(o, g()) for o, g in zip(outs, small))
    assert torch.equal(f(), want)
