"""HIP graph capture of C-ABI calls: every entry point of the hot path issues nothing but kernel launches on the
context's stream, so a caller may record them into a graph.  The graph is replayed several times with new operand
contents, eager calls and synchronisations in between, and every replay is compared with the eager result on the
same operands (bit for bit: the operators here are integer ones)."""
import numpy as np
import pytest

from reference_model_amd import Context, capi

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def test_graph_of_the_int8_layer_chain_matches_eager_on_every_replay():
    dev = torch.device("cuda:0")
    ctx = Context(0)
    try:
        stream = torch.cuda.current_stream()
        ctx.set_stream(stream.cuda_stream)
        rng = np.random.default_rng(8)
        n, hw, c = 4, 28, 64
        x = torch.empty((n, hw, hw, c), dtype=torch.int8, device=dev)
        w = torch.from_numpy(rng.integers(-127, 128, (c, 3, 3, c)).astype(np.int8)).to(dev)
        bias = torch.from_numpy(rng.integers(-9999, 9999, c).astype(np.int32)).to(dev)
        mult = torch.from_numpy(rng.integers(1 << 30, 1 << 31, c).astype(np.int32)).to(dev)
        shift = torch.from_numpy(rng.integers(38, 42, c).astype(np.int8)).to(dev)
        wd = torch.from_numpy(rng.integers(-127, 128, (3, 3, c, 1)).astype(np.int8)).to(dev)
        y = torch.empty((n, hw, hw, c), dtype=torch.int8, device=dev)      # CONV2D + RESCALE + CLAMP
        z = torch.empty((n, hw, hw, c), dtype=torch.int8, device=dev)      # DEPTHWISE_CONV2D + RESCALE
        p = torch.empty((n, hw // 2, hw // 2, c), dtype=torch.int8, device=dev)    # MAX_POOL2D
        rows = (hw // 2) * (hw // 2)
        m = torch.empty((n, rows, hw // 2), dtype=torch.int32, device=dev)         # MATMUL [n, rows, c] x [n, c, hw/2]
        pt = torch.empty((n, c, hw // 2), dtype=torch.int8, device=dev)
        d = ctx.conv_desc(capi.INT8, capi.INT32, (n, hw, hw, c), c, 3, 3, (hw, hw), (1, 1, 1, 1), (1, 1), (1, 1), c)
        r = ctx.rescale_desc(capi.INT32, capi.INT8, c, c, 0, -3, True, capi.ROUND_DOUBLE, True, False, False)
        pd = capi.PoolDesc()
        pd.dtype, pd.N, pd.IH, pd.IW, pd.C, pd.OH, pd.OW = capi.INT8, n, hw, hw, c, hw // 2, hw // 2
        pd.kernel[:], pd.stride[:], pd.pad[:] = [2, 2], [2, 2], [0, 0, 0, 0]
        pd.nan_mode, pd.acc_dtype = 1, capi.INT32

        def chain():
            ctx.conv2d_rescale_clamp(d, x, w, bias, -7, 0, r, mult, shift, y, (-100, 100))
            ctx.depthwise_conv2d_rescale_clamp(d, y, wd, bias, 5, 0, r, mult, shift, z, None)
            ctx.max_pool2d(pd, z, p)
            ctx.matmul(capi.INT8, n, rows, c, hw // 2, p, pt, 2, -1, m)

        def fresh_inputs(seed):
            g = np.random.default_rng(seed)
            x.copy_(torch.from_numpy(g.integers(-128, 128, tuple(x.shape)).astype(np.int8)))
            pt.copy_(torch.from_numpy(g.integers(-128, 128, tuple(pt.shape)).astype(np.int8)))

        fresh_inputs(0)
        chain()     # first calls outside the capture: one-time kernel attribute set-up happens here
        assert ctx.sync() == capi.VALID
        kernels = ctx.last_kernel
        graph = torch.cuda.CUDAGraph()
        side = torch.cuda.Stream()
        side.wait_stream(stream)
        with torch.cuda.graph(graph, stream=side):
            ctx.set_stream(side.cuda_stream)
            chain()
        ctx.set_stream(stream.cuda_stream)
        for seed in (1, 2, 3, 4):
            fresh_inputs(seed)
            chain()                                    # eager, on the same operands
            assert ctx.sync() == capi.VALID
            want = [t.clone() for t in (y, z, p, m)]
            for t in (y, z, p, m):
                t.zero_()
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            assert ctx.sync() == capi.VALID
            for got, ref in zip((y, z, p, m), want):
                assert torch.equal(got, ref)
            assert len(torch.unique(y)) > 50 and len(torch.unique(m)) > 50
        assert kernels.startswith("matmul")
    finally:
        ctx.close()


def test_graph_of_transpose_conv_conv3d_and_avg_pool_matches_eager_on_every_replay():
    """TRANSPOSE_CONV2D and CONV3D once through the kernel that reads their operands in place (one launch, no scratch
    buffer) and once through the re-laid-out operands (scratch buffer grown by the eager pass before the capture),
    and AVG_POOL2D."""
    dev = torch.device("cuda:0")
    ctx = Context(0)
    try:
        stream = torch.cuda.current_stream()
        ctx.set_stream(stream.cuda_stream)
        rng = np.random.default_rng(21)
        n, hw, c, oc = 2, 12, 64, 64
        x = torch.empty((n, hw, hw, c), dtype=torch.int8, device=dev)
        wt = torch.from_numpy(rng.integers(-127, 128, (oc, 3, 3, c)).astype(np.int8)).to(dev)
        bias = torch.from_numpy(rng.integers(-9999, 9999, oc).astype(np.int32)).to(dev)
        up = 2 * (hw - 1) + 3
        t_out = torch.empty((n, up, up, oc), dtype=torch.int32, device=dev)
        t_out2 = torch.empty_like(t_out)
        td = capi.TconvDesc()
        td.in_dtype, td.out_dtype = capi.INT8, capi.INT32
        td.N, td.IH, td.IW, td.IC, td.OC, td.KH, td.KW, td.OH, td.OW = n, hw, hw, c, oc, 3, 3, up, up
        td.out_pad[:], td.stride[:], td.bias_len = [0, 0, 0, 0], [2, 2], oc
        v = torch.empty((1, 6, 10, 10, 32), dtype=torch.int8, device=dev)
        w3 = torch.from_numpy(rng.integers(-127, 128, (oc, 3, 3, 3, 32)).astype(np.int8)).to(dev)
        c_out = torch.empty((1, 6, 10, 10, oc), dtype=torch.int32, device=dev)
        c_out2 = torch.empty_like(c_out)
        cd = capi.Conv3dDesc()
        cd.in_dtype, cd.out_dtype = capi.INT8, capi.INT32
        cd.N, cd.ID, cd.IH, cd.IW, cd.IC, cd.OC, cd.KD, cd.KH, cd.KW, cd.OD, cd.OH, cd.OW = 1, 6, 10, 10, 32, oc, 3, 3, 3, 6, 10, 10
        cd.pad[:], cd.stride[:], cd.dilation[:], cd.bias_len = [1] * 6, [1] * 3, [1] * 3, oc
        pd = capi.PoolDesc()
        pd.dtype, pd.N, pd.IH, pd.IW, pd.C, pd.OH, pd.OW = capi.INT8, n, hw, hw, c, hw // 2, hw // 2
        pd.kernel[:], pd.stride[:], pd.pad[:] = [2, 2], [2, 2], [0, 0, 0, 0]
        pd.nan_mode, pd.acc_dtype = 1, capi.INT32
        p_out = torch.empty((n, hw // 2, hw // 2, c), dtype=torch.int8, device=dev)
        names = []

        def chain():
            ctx.set_kernel_choice(capi.KERNEL_AUTO)
            ctx.transpose_conv2d(td, x, wt, bias, -5, 0, t_out)
            names.append(ctx.last_kernel)
            ctx.conv3d(cd, v, w3, bias, 3, 0, c_out)
            names.append(ctx.last_kernel)
            ctx.set_kernel_choice(capi.KERNEL_MFMA)
            ctx.transpose_conv2d(td, x, wt, bias, -5, 0, t_out2)
            ctx.conv3d(cd, v, w3, bias, 3, 0, c_out2)
            ctx.set_kernel_choice(capi.KERNEL_AUTO)
            ctx.avg_pool2d(pd, x, -5, 7, p_out)

        def fresh_inputs(seed):
            g = np.random.default_rng(seed)
            x.copy_(torch.from_numpy(g.integers(-128, 128, tuple(x.shape)).astype(np.int8)))
            v.copy_(torch.from_numpy(g.integers(-128, 128, tuple(v.shape)).astype(np.int8)))

        fresh_inputs(0)
        chain()     # the eager pass sets kernel attributes and grows the scratch buffer
        assert ctx.sync() == capi.VALID
        assert names[:2] == ["transpose_conv2d_slab_i8", "conv3d_slab_i8"]
        graph = torch.cuda.CUDAGraph()
        side = torch.cuda.Stream()
        side.wait_stream(stream)
        with torch.cuda.graph(graph, stream=side):
            ctx.set_stream(side.cuda_stream)
            chain()
        ctx.set_stream(stream.cuda_stream)
        outs = (t_out, t_out2, c_out, c_out2, p_out)
        for seed in (1, 2, 3):
            fresh_inputs(seed)
            chain()
            assert ctx.sync() == capi.VALID
            want = [t.clone() for t in outs]
            assert torch.equal(want[0], want[1]) and torch.equal(want[2], want[3])
            for t in outs:
                t.zero_()
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            assert ctx.sync() == capi.VALID
            for got, ref in zip(outs, want):
                assert torch.equal(got, ref)
            assert len(torch.unique(t_out)) > 50 and len(torch.unique(c_out)) > 50 and len(torch.unique(p_out)) > 20
    finally:
        ctx.close()


@pytest.mark.parametrize("kind", ["int16", "int8"])
def test_a_layer_with_ragged_channels_is_captured(kind):
    """Channel vectors of no whole pieces are copied: eagerly into a buffer of the context, under capture into memory that
    belongs to the capture."""
    dev = torch.device("cuda:0")
    rng = np.random.default_rng(3)
    t = torch.int16 if kind == "int16" else torch.int8
    n, hw, ic, oc = 2, 15, 137, 96
    x = torch.from_numpy(rng.integers(-128, 128, (n, hw, hw, ic))).to(t).to(dev)
    w = torch.from_numpy(rng.integers(-127, 128, (oc, 3, 3, ic)).astype(np.int8)).to(dev)
    acc_t = torch.int64 if kind == "int16" else torch.int32
    bias = torch.from_numpy(rng.integers(-9999, 9999, oc)).to(acc_t).to(dev)
    results = []
    for captured in (False, True):
        ctx = Context(0)
        try:
            out = torch.zeros((n, hw, hw, oc), dtype=acc_t, device=dev)
            d = ctx.conv_desc(capi.INT16 if kind == "int16" else capi.INT8, capi.INT48 if kind == "int16" else capi.INT32, tuple(x.shape),
                              oc, 3, 3, (hw, hw), (1, 1, 1, 1), (1, 1), (1, 1), oc)
            ctx.set_stream(torch.cuda.current_stream().cuda_stream)    # (leaves the context's own stream, outside the capture)
            if captured:
                graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
                side.wait_stream(torch.cuda.current_stream())
                with torch.cuda.graph(graph, stream=side):
                    ctx.set_stream(side.cuda_stream)
                    ctx.conv2d(d, x, w, bias, 0, 0, out)
                for _ in range(2):
                    out.zero_()
                    graph.replay()
                    torch.cuda.synchronize()
            else:
                ctx.conv2d(d, x, w, bias, 0, 0, out)
                assert ctx.sync() == capi.VALID
            torch.cuda.synchronize()
            results.append(out)
        finally:
            ctx.close()
    assert torch.equal(*results) and len(torch.unique(results[0])) > 1000


@pytest.mark.parametrize("kind, shape", [("int8", (1, 1300, 1301, 1303)), ("fp16", (2, 1100, 960, 1003)), ("int8", (1, 130, 250001, 66))])
def test_a_large_ragged_product_is_captured_without_scratch_memory(kind, shape):
    """Products whose operands would be copied into the scratch buffer, on a context whose buffer is empty and cannot grow: the
    kernel that reads any operand where it lies, not an error.  (The last one has too few tiles for the copies in any case.)"""
    dev = torch.device("cuda:0")
    n, h, c, w = shape
    rng = np.random.default_rng(h)
    t, code, out_t = (torch.int8, capi.INT8, torch.int32) if kind == "int8" else (torch.float16, capi.FP16, torch.float32)
    # whole numbers of at most 5: products and sums are exact in fp32
    a, b = (torch.from_numpy(rng.integers(-5, 6, s)).to(t).to(dev) for s in ((n, h, c), (n, c, w)))
    want = torch.from_numpy(np.matmul(a.cpu().numpy().astype(np.float64), b.cpu().numpy().astype(np.float64))).to(out_t).to(dev)
    ctx = Context(0)
    try:
        out = torch.zeros((n, h, w), dtype=out_t, device=dev)
        ctx.set_stream(torch.cuda.current_stream().cuda_stream)    # (leaves the context's own stream, outside the capture)
        graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.graph(graph, stream=side):
            ctx.set_stream(side.cuda_stream)
            ctx.matmul(code, n, h, c, w, a, b, 0, 0, out)
        assert ctx.last_kernel == ("matmul_ragged_i8" if kind == "int8" else "matmul_ragged_f16") and ctx.workspace_bytes() == (0, 0)
        for _ in range(3):
            out.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, want)
        ctx.set_stream(torch.cuda.current_stream().cuda_stream)
        out.zero_()
        ctx.matmul(code, n, h, c, w, a, b, 0, 0, out)    # with room for them
        assert ctx.sync() == capi.VALID and torch.equal(out, want)
        assert ("pad_gemm" in ctx.last_kernel) == (h > 130)
    finally:
        ctx.close()


@pytest.mark.parametrize("kind", ["int8", "fp16", "int16"])
def test_graphs_of_ragged_layers_replay_at_once(kind):
    """Two graphs of one context and eager calls, each on a stream of its own and at the same time: CONV2D layers whose channel
    vectors are padded on the way share no memory."""
    dev = torch.device("cuda:0")
    rng = np.random.default_rng(5)
    t, acc, code, out_code = {"int8": (torch.int8, torch.int32, capi.INT8, capi.INT32), "fp16": (torch.float16, torch.float16, capi.FP16, capi.FP16),
                              "int16": (torch.int16, torch.int64, capi.INT16, capi.INT48)}[kind]
    n, hw, ic, oc = 8, 56, 73, 72
    wt = torch.int8 if kind == "int16" else t
    layers = []
    for _ in range(3):
        x = torch.from_numpy(rng.integers(-9, 10, (n, hw, hw, ic))).to(t).to(dev)
        w = torch.from_numpy(rng.integers(-1, 2, (oc, 3, 3, ic))).to(wt).to(dev)
        bias = torch.from_numpy(rng.integers(-99, 100, oc)).to(acc).to(dev)
        layers.append((x, w, bias, torch.zeros((n, hw, hw, oc), dtype=acc, device=dev)))
    ctx = Context(0)
    try:
        d = ctx.conv_desc(code, out_code, (n, hw, hw, ic), oc, 3, 3, (hw, hw), (1, 1, 1, 1), (1, 1), (1, 1), oc)
        main = torch.cuda.current_stream()
        ctx.set_stream(main.cuda_stream)
        want = []
        for x, w, bias, out in layers:
            ctx.conv2d(d, x, w, bias, 0, 0, out)
            assert ctx.sync() == capi.VALID
            want.append(out.clone())
        kernel, (live, retired) = ctx.last_kernel, ctx.workspace_bytes()
        assert live > 0 and retired == 0
        graphs, streams = [], [torch.cuda.Stream(), torch.cuda.Stream()]
        for layer, side in zip(layers, streams):
            side.wait_stream(main)
            graphs.append(torch.cuda.CUDAGraph())
            with torch.cuda.graph(graphs[-1], stream=side):
                ctx.set_stream(side.cuda_stream)
                for _ in range(4):
                    ctx.conv2d(d, *layer[:3], 0, 0, layer[3])
            assert ctx.last_kernel == kernel
            ctx.set_stream(main.cuda_stream)
        # one block for each capture, of the size an eager call takes; the eager calls' buffer is untouched
        assert ctx.workspace_bytes() == (live, 2 * live)
        for _ in range(20):
            for layer in layers:
                layer[3].zero_()
            torch.cuda.synchronize()
            for graph, side in zip(graphs, streams):
                with torch.cuda.stream(side):
                    graph.replay()
            for _ in range(4):
                ctx.conv2d(d, *layers[2][:3], 0, 0, layers[2][3])
            torch.cuda.synchronize()
            assert all(torch.equal(layer[3], ref) for layer, ref in zip(layers, want))
        assert ctx.sync() == capi.VALID
        del graphs
        ctx.trim_workspace()
        assert ctx.workspace_bytes() == (live, 0)
    finally:
        ctx.close()
