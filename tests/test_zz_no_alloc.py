"""tts_launch_noalloc (the launch for callers that cannot allocate device memory) against tts_launch, through the C ABI.

Both run the same kernels and add the K slices in slice order, so the int8-weight product must come out bit for bit
the same whether its partial tiles sit in the plan's own workspace (tts_launch) or in the library's static scratch
array (tts_launch_noalloc).  Two calls in a row share that array; the second is a smaller problem."""
import pytest
import torch

from conftest import plan_for
from test_planner import compile_ttir

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _inputs(M, N, Kd, seed):
    torch.manual_seed(seed)
    a = torch.randn(M, Kd).half().to(DEV)
    w = torch.randint(-127, 128, (Kd, N), dtype=torch.int8).to(DEV)
    s = (0.001 + 0.009 * torch.rand(N)).half().to(DEV)
    return a, w, s


def _values(a, w, s, c, M, N, Kd):
    # w8a16_matmul(a, w, scale, c, M, N, K, stride_am, stride_wk, stride_cm): the unit inner strides are constants
    return [a.data_ptr(), w.data_ptr(), s.data_ptr(), c.data_ptr(), M, N, Kd, a.stride(0), w.stride(0), c.stride(0)]


def test_noalloc_launch_matches_the_allocating_launch(native):
    plan, _ = plan_for(native, "w8a16_matmul")
    assert plan.family == "gemm_w8a16"
    stream = torch.cuda.current_stream().cuda_stream
    # a split-K shape on the wide kernel (counters and partial tiles), then a smaller one on the same scratch array,
    # then a shape that the narrow kernel and its separate reduce kernel take
    for seed, (M, N, Kd) in enumerate([(16, 2048, 8192), (16, 1024, 4096), (13, 384, 4096)]):
        a, w, s = _inputs(M, N, Kd, seed)
        grid = (1, (N + 127) // 128, 1)
        want = torch.full((M, N), 5.0, dtype=torch.float16, device=DEV)
        got = torch.full((M, N), 7.0, dtype=torch.float16, device=DEV)
        vals = _values(a, w, s, want, M, N, Kd)
        d = plan.describe_launch(grid, vals)
        assert int(d["split"]) > 1, d            # the case that needs scratch memory
        plan.launch(grid, stream, vals)
        torch.cuda.synchronize()
        free_before = torch.cuda.mem_get_info()[0]
        plan.launch_noalloc(grid, stream, _values(a, w, s, got, M, N, Kd))
        torch.cuda.synchronize()
        if seed > 0:                             # the first call on a device looks up the scratch array's address
            assert torch.cuda.mem_get_info()[0] >= free_before
        assert torch.equal(got, want), (M, N, Kd)
        ref = a.double() @ (w.half() * s[None, :]).double()
        assert ((got.double() - ref).norm() / ref.norm()).item() <= 1e-2


def test_noalloc_launch_refuses_a_plan_that_still_has_to_compile(native):
    # a fused map is compiled into a kernel of its own at its first launch, which allocates: the no-allocation launch
    # says so instead of compiling (nothing is dereferenced before the refusal)
    plan, _ = plan_for(native, "gelu_tanh_bias")
    assert plan.family == "fused_map"
    n = 4096
    x = torch.randn(n, device=DEV)
    b = torch.randn(n, device=DEV)
    y = torch.zeros(n, device=DEV)
    stream = torch.cuda.current_stream().cuda_stream
    vals = [x.data_ptr(), b.data_ptr(), y.data_ptr(), n]
    with pytest.raises(NotImplementedError, match="allocates"):
        plan.launch_noalloc((4, 1, 1), stream, vals)
    plan.launch((4, 1, 1), stream, vals)         # compiles
    want = y.clone()
    y.zero_()
    plan.launch_noalloc((4, 1, 1), stream, vals)  # now there is nothing left to allocate
    torch.cuda.synchronize()
    assert torch.equal(y, want) and want.abs().sum().item() > 0


def test_noalloc_launch_runs_a_skinny_matmul_in_k_slices_from_the_static_array(native):
    # a matrix product with too few output tiles for the chip runs in K slices, whose fp32 partial sums tts_launch keeps in
    # the stream's workspace and tts_launch_noalloc in the static array, in as many slices as fit there (8 MiB: eight
    # slices of 128 x 2048); with the same number of slices the results agree bit for bit, both adding them in slice order.
    # A product of which not even two slices fit (1024 x 2048) runs without slices in the call that may not allocate,
    # which changes the order of the sums: within the tolerance of the family
    plan, _ = plan_for(native, "matmul_tiles")
    assert plan.family == "gemm"
    stream = torch.cuda.current_stream().cuda_stream
    for seed, (M, N, Kd, fits) in enumerate([(128, 2048, 8192, True), (64, 1024, 4096, True), (1000, 2048, 4096, False)]):
        torch.manual_seed(seed)
        a = (torch.randn(M, Kd) * 0.1).bfloat16().to(DEV)
        b = (torch.randn(Kd, N) * 0.1).bfloat16().to(DEV)
        want = torch.full((M, N), 5.0, dtype=torch.bfloat16, device=DEV)
        got = torch.full((M, N), 7.0, dtype=torch.bfloat16, device=DEV)
        grid = (((M + 127) // 128) * ((N + 127) // 128), 1, 1)
        plan.launch(grid, stream, [a.data_ptr(), b.data_ptr(), want.data_ptr(), M, N, Kd, Kd, N, N])
        torch.cuda.synchronize()
        assert plan.last_kernel.endswith("K slices"), plan.last_kernel
        # (the entry point's first call on a device looks the static array's address up, which is when the runtime gives
        # the array its memory: free memory is compared around a later call)
        plan.launch_noalloc(grid, stream, [a.data_ptr(), b.data_ptr(), got.data_ptr(), M, N, Kd, Kd, N, N])
        torch.cuda.synchronize()
        got.fill_(7.0)
        free_before = torch.cuda.mem_get_info()[0]
        plan.launch_noalloc(grid, stream, [a.data_ptr(), b.data_ptr(), got.data_ptr(), M, N, Kd, Kd, N, N])
        torch.cuda.synchronize()
        assert torch.cuda.mem_get_info()[0] >= free_before
        assert plan.last_kernel.endswith("K slices") == fits, plan.last_kernel
        ref = a.double() @ b.double()
        assert ((got.double() - ref).norm() / ref.norm()).item() <= 1e-2
        if fits and M * N * 4 * 16 <= (8 << 20):   # (at most 16 slices are ever taken: then both calls took the same number)
            assert torch.equal(got, want), (M, N, Kd)


def test_noalloc_refusal_leaves_a_matmul_with_epilogue_on_its_kernel(native):
    """A matrix product with a fused epilogue needs a compiled kernel and, per launch shape, a device table of tile
    owners: the launch that may not allocate refuses both, and the refusal must not be remembered as "this launch belongs
    to the generic family" -- the same launch through tts_launch afterwards runs the product kernel with its epilogue."""
    import triton
    import triton_shared_amd as tsa
    import extra_kernels as X
    tsa.activate()
    g = torch.Generator(device="cpu").manual_seed(3)
    stream = torch.cuda.current_stream().cuda_stream

    def operands(M, N, K):
        a = torch.randint(-1, 2, (M, K), generator=g).to(torch.bfloat16).to(DEV)
        b = torch.randint(-1, 2, (K, N), generator=g).to(torch.bfloat16).to(DEV)
        return a, b, torch.full((M, N), 7, device=DEV, dtype=torch.bfloat16)

    M, N, K = 512, 768, 96
    a, b, c = operands(M, N, K)
    grid = (triton.cdiv(M, 128), triton.cdiv(N, 128), 1)
    k = X.matmul_leaky[grid[:2]](a, b, c, M, N, K, a.stride(0), b.stride(0), c.stride(0), 0.5, BM=128, BN=128, BK=64)
    torch.cuda.synchronize()
    assert k.function.family == "gemm" and k.function.last_kernel.startswith("gemm_dma_kernel + epilogue")
    want = torch.nn.functional.leaky_relu(a.float() @ b.float(), 0.5)
    assert torch.equal(c.float(), want)
    n_args = len(k.function.arg_kinds)

    def values(a, b, c, M, N, K):
        vals = [a.data_ptr(), b.data_ptr(), c.data_ptr(), M, N, K, a.stride(0), b.stride(0), c.stride(0), 0.5]
        assert len(vals) == n_args, (n_args, k.function.arg_kinds)
        return vals

    # (1) a plan that has compiled nothing yet: refused, then launched the ordinary way on the product kernel
    fresh = native.PlanHandle(k.kernel)
    c.fill_(7)
    with pytest.raises(NotImplementedError, match="allocates"):
        fresh.launch_noalloc(grid, stream, values(a, b, c, M, N, K))
    torch.cuda.synchronize()
    assert torch.all(c == 7)                     # nothing ran
    fresh.launch(grid, stream, values(a, b, c, M, N, K))
    torch.cuda.synchronize()
    assert fresh.last_kernel.startswith("gemm_dma_kernel + epilogue"), fresh.last_kernel
    assert torch.equal(c.float(), want)
    c.fill_(7)
    fresh.launch_noalloc(grid, stream, values(a, b, c, M, N, K))   # kernel compiled, table of this shape built: runs
    torch.cuda.synchronize()
    assert fresh.last_kernel.startswith("gemm_dma_kernel + epilogue") and torch.equal(c.float(), want)
    # (2) the kernel is compiled, but a new shape needs a new table of tile owners: refused, not rebound to the generic
    # family; a smaller problem than the first, as the second call of two in a row
    M2, N2, K2 = 256, 512, 64
    a2, b2, c2 = operands(M2, N2, K2)
    grid2 = (triton.cdiv(M2, 128), triton.cdiv(N2, 128), 1)
    with pytest.raises(NotImplementedError, match="allocates"):
        fresh.launch_noalloc(grid2, stream, values(a2, b2, c2, M2, N2, K2))
    d = fresh.describe_launch(grid2, values(a2, b2, c2, M2, N2, K2))
    assert d["kernel"] == "gemm_mfma", d
    fresh.launch(grid2, stream, values(a2, b2, c2, M2, N2, K2))
    torch.cuda.synchronize()
    assert fresh.last_kernel.startswith("gemm_dma_kernel + epilogue"), fresh.last_kernel
    assert torch.equal(c2.float(), torch.nn.functional.leaky_relu(a2.float() @ b2.float(), 0.5))


@pytest.mark.parametrize("first", ["contiguous", "strided"])
def test_noalloc_launch_of_an_fp32_product_with_an_activation_takes_every_stride(native, first):
    """leaky_relu(A . B) on fp32 operands runs on the matrix kernel where A's rows are contiguous and on the generic one where they are
    not: once either has been launched, the launch that may not allocate runs both, in a size of another tiling too."""
    import triton_shared_amd as tsa
    import extra_kernels as X
    tsa.activate()
    g = torch.Generator(device="cpu").manual_seed(5)
    stream = torch.cuda.current_stream().cuda_stream

    def case(M, N, K, strided):
        a = torch.randint(-2, 3, (M, K), generator=g).float()
        b = torch.randint(-2, 3, (K, N), generator=g).float()
        held = torch.zeros(M, 3 * K, device=DEV)
        at = held[:, ::3] if strided else torch.zeros(M, K, device=DEV)
        at.copy_(a)
        bd, c = b.to(DEV), torch.full((M, N), 7.0, device=DEV)
        grid = (-(-M // 64), -(-N // 64), 1)
        vals = [at.data_ptr(), bd.data_ptr(), c.data_ptr(), M, N, K, at.stride(0), at.stride(1), bd.stride(0), c.stride(0), 0.5]
        return grid, vals, c, torch.nn.functional.leaky_relu(a @ b, 0.5), (held, at, bd)

    ttir = compile_ttir(X.matmul_leaky_any_stride, {"a_ptr": "*fp32", "b_ptr": "*fp32", "c_ptr": "*fp32", **{x: "i32" for x in ("M", "N", "K", "s_am", "s_ak", "s_bk", "s_cm")}, "slope": "fp32",
                                                    **{x: "constexpr" for x in ("BM", "BN", "BK")}}, {"BM": 64, "BN": 64, "BK": 32})
    plan = native.PlanHandle(native.structured_to_plan(native.ttir_to_structured(ttir))[0])
    grid, vals, c, want, keep = case(100, 130, 96, first == "strided")
    plan.launch(grid, stream, vals)
    torch.cuda.synchronize()
    assert torch.equal(c.cpu(), want)
    for M, N, K in [(100, 130, 96), (700, 900, 64)]:
        for strided in (True, False):
            grid, vals, c, want, keep = case(M, N, K, strided)
            plan.launch_noalloc(grid, stream, vals)
            torch.cuda.synchronize()
            assert torch.equal(c.cpu(), want), (M, strided)
            assert plan.last_kernel.startswith("tile_program") == (strided or first == "strided"), plan.last_kernel


def test_noalloc_launch_of_the_tiled_int8_product_asks_for_no_scratch_it_does_not_use(native):
    # 64 rows run on the tiled kernel.  The decode kernels' partial tiles of this width would not fit the static array (9.4 MB in
    # two slices), but nobody reads them; the tiled kernel's own slices do not fit either, and it runs without
    plan, _ = plan_for(native, "w8a16_matmul")
    stream = torch.cuda.current_stream().cuda_stream
    M, N, Kd = 64, 36864, 512
    a, w, s = _inputs(M, N, Kd, 1)
    want, got = (torch.full((M, N), v, dtype=torch.float16, device=DEV) for v in (5.0, 7.0))
    grid = (4, (N + 127) // 128, 1)
    plan.launch(grid, stream, _values(a, w, s, want, M, N, Kd))
    plan.launch_noalloc(grid, stream, _values(a, w, s, got, M, N, Kd))
    torch.cuda.synchronize()
    assert plan.last_kernel == "gemm_w8a16_tile_kernel"
    ref = a.double() @ (w.half() * s[None, :]).double()
    for c in (want, got):   # fp32 sums in two orders, rounded once to fp16
        assert ((c.double() - ref).norm() / ref.norm()).item() <= 2.0 ** -11


def test_recorded_matmul_with_epilogue_runs_on_a_kernel_that_is_compiled(native):
    # a plan that has compiled the any-shape product in 128-row tiles records one that would take 64-row tiles: the recording
    # compiles nothing; outside of it the launch compiles its own
    import triton
    import triton_shared_amd as tsa
    import extra_kernels as X
    tsa.activate()
    g = torch.Generator(device="cpu").manual_seed(4)

    def problem(M, N, K):
        a = torch.randint(-1, 2, (M, K), generator=g).to(torch.bfloat16).to(DEV)
        b = torch.randint(-1, 2, (K, N), generator=g).to(torch.bfloat16).to(DEV)
        c = torch.full((M, N), 7, device=DEV, dtype=torch.bfloat16)
        return a, b, c, (triton.cdiv(M, 128), triton.cdiv(N, 128), 1), [a.data_ptr(), b.data_ptr(), c.data_ptr(), M, N, K, K, N, N, 0.5]

    want = lambda a, b: torch.nn.functional.leaky_relu(a.float() @ b.float(), 0.5).bfloat16()
    a, b, c, grid, values = problem(2900, 2999, 71)
    k = X.matmul_leaky[grid[:2]](a, b, c, *values[3:], BM=128, BN=128, BK=64)
    torch.cuda.synchronize()
    large, small = "gemm_mfma_kernel<128x128x64> + epilogue (hipRTC)", "gemm_mfma_kernel<64x128x64> + epilogue (hipRTC)"
    assert k.function.last_kernel == large and torch.equal(c, want(a, b))
    plan = native.PlanHandle(k.kernel)
    plan.launch(grid, torch.cuda.current_stream().cuda_stream, values)
    a, b, c, grid, values = problem(200, 300, 150)
    assert plan.describe_launch(grid, values)["kernel"] == "gemm_mfma"   # (the table of this shape's tile owners is there then)
    torch.cuda.synchronize()
    graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    with torch.cuda.graph(graph, stream=side):
        plan.launch(grid, torch.cuda.current_stream().cuda_stream, values)
    assert plan.last_kernel == large
    for _ in range(3):
        a.copy_(torch.randint(-1, 2, a.shape, generator=g))
        c.fill_(7)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(c, want(a, b))
    c.fill_(7)
    plan.launch(grid, torch.cuda.current_stream().cuda_stream, values)
    torch.cuda.synchronize()
    assert plan.last_kernel == small and torch.equal(c, want(a, b))


@pytest.mark.parametrize("M,N,Kd", [(976, 1984, 2816), (128, 2048, 4096), (1504, 3072, 4096)])
def test_recorded_matmul_in_k_slices_allocates_nothing(native, M, N, Kd):
    # a product that runs in K slices, first launched on a stream while that stream records a graph: there is no workspace and
    # none is allocated, the product is recorded whole; once an eager launch has left one there, the slices are recorded
    plan, _ = plan_for(native, "matmul_tiles")
    g = torch.Generator().manual_seed(M)
    a = torch.zeros(M, Kd)
    a = a.scatter_(1, torch.randint(0, Kd, (M, 40), generator=g), 1.0).bfloat16().to(DEV)
    b, c = torch.zeros(Kd, N, dtype=torch.bfloat16, device=DEV), torch.zeros(M, N, dtype=torch.bfloat16, device=DEV)
    grid = (((M + 127) // 128) * ((N + 127) // 128), 1, 1)
    launch = lambda: plan.launch(grid, torch.cuda.current_stream().cuda_stream, [a.data_ptr(), b.data_ptr(), c.data_ptr(), M, N, Kd, Kd, N, N])
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    for sliced in (False, True):
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            launch()
        assert plan.last_kernel.endswith("K slices") == sliced, plan.last_kernel
        for _ in range(3):
            b.copy_(torch.randint(-2, 3, (Kd, N), generator=g))
            want = (a.float() @ b.float()).bfloat16()   # sums of at most 40 small integers: exact
            c.fill_(7)
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(c, want)
            c.fill_(7)
            torch.cuda.synchronize()
            with torch.cuda.stream(side):
                launch()
            torch.cuda.synchronize()
            assert plan.last_kernel.endswith("K slices") and torch.equal(c, want)


def test_recorded_launches_of_the_tiled_int8_product_allocate_nothing(native):
    # the first launch on a stream, while it records a graph: nothing to allocate, clear or wait for
    plan, _ = plan_for(native, "w8a16_matmul")
    M, N, Kd = 64, 2048, 4096
    a, w, s = _inputs(M, N, Kd, 2)
    want, got = (torch.zeros(M, N, dtype=torch.float16, device=DEV) for _ in range(2))
    grid = (4, N // 128, 1)
    plan.launch(grid, torch.cuda.current_stream().cuda_stream, _values(a, w, s, want, M, N, Kd))
    torch.cuda.synchronize()
    graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    with torch.cuda.graph(graph, stream=side):
        plan.launch(grid, torch.cuda.current_stream().cuda_stream, _values(a, w, s, got, M, N, Kd))
    for seed in range(3):
        a.copy_(_inputs(M, N, Kd, 10 + seed)[0])
        got.zero_()
        plan.launch(grid, torch.cuda.current_stream().cuda_stream, _values(a, w, s, want, M, N, Kd))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert ((got.double() - want.double()).norm() / want.double().norm()).item() <= 2.0 ** -11   # (the eager launch runs in K slices)


@pytest.mark.parametrize("M,N,Kd", [(4, 24704, 4096), (15, 2048, 6400), (40, 1040, 4096)])
def test_recorded_first_launches_of_the_int8_decode_kernels_allocate_nothing(native, M, N, Kd):
    # products that run in K slices, first launched on a stream while it records a graph: recorded whole, without workspace and
    # counters; an eager launch on the stream then runs in slices, and one recorded after it, too
    plan, _ = plan_for(native, "w8a16_matmul")
    a, w, s = _inputs(M, N, Kd, 3)
    got = torch.zeros(M, N, dtype=torch.float16, device=DEV)
    grid = ((M + 15) // 16, (N + 127) // 128, 1)
    launch = lambda: plan.launch(grid, torch.cuda.current_stream().cuda_stream, _values(a, w, s, got, M, N, Kd))
    assert int(plan.describe_launch(grid, _values(a, w, s, got, M, N, Kd))["split"]) > 1
    launch()                                   # (on another stream)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    for turn in range(2):
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            launch()
        for seed in range(3):
            a.copy_(_inputs(M, N, Kd, 10 + seed)[0])
            ref = a.double() @ (w.half() * s[None, :]).double()
            for run in (graph.replay, launch):
                got.zero_()
                torch.cuda.synchronize()
                with torch.cuda.stream(side):
                    run()
                torch.cuda.synchronize()
                # fp32 sums in two orders, rounded once to fp16
                assert ((got.double() - ref).norm() / ref.norm()).item() <= 2.0 ** -11


@pytest.mark.parametrize("kind", ["softmax loop in slices", "sums in slices", "slices that meet", "int8 weights"])
def test_first_launches_beside_a_stream_that_records(native, kind):
    # a launch that takes a workspace and counters, the first on its stream, while another stream records a graph: it neither fails
    # nor ends the recording
    import triton
    import triton_shared_amd as tsa
    import extra_kernels as X
    from triton_shared_amd.examples import kernels as K
    tsa.activate()
    g = torch.Generator().manual_seed(8)
    if kind == "softmax loop in slices":
        H, seq, D = 2, 1500, 64
        q, k, v = (torch.randn(H, seq, D, generator=g).half().to(DEV) for _ in range(3))
        out = torch.zeros(H, seq, D, dtype=torch.float16, device=DEV)
        launch = lambda: X.attention_fwd[(triton.cdiv(seq, 64), H)](q, k, v, out, D ** -0.5, seq, seq * D, D, BM=64, BN=64, D=D)
        want = torch.nn.functional.scaled_dot_product_attention(q.float().cpu(), k.float().cpu(), v.float().cpu())
    elif kind == "sums in slices":
        rows, cols = 4096, 512
        x = torch.randn(rows, cols, generator=g).to(DEV)
        out = torch.zeros(cols, device=DEV)
        launch = lambda: X.block_column_sums[(1, cols // 64)](x, out, rows, cols, BR=16, BC=64)
        want = x.double().sum(0).cpu()
    elif kind == "slices that meet":
        M, N, Kd = 768, 768, 1536
        a, b = torch.randn(M, Kd, generator=g).bfloat16().to(DEV), torch.randn(Kd, N, generator=g).bfloat16().to(DEV)
        out = torch.zeros(M, N, dtype=torch.bfloat16, device=DEV)
        launch = lambda: K.matmul_tiles[(36,)](a, b, out, M, N, Kd, Kd, 1, N, 1, N, 1, BM=128, BN=128, BK=64, GROUP_M=8)
        want = (a.double() @ b.double()).cpu()
    else:
        M, N, Kd = 15, 2048, 6400
        a, w, s = _inputs(M, N, Kd, 3)
        out = torch.zeros(M, N, dtype=torch.float16, device=DEV)
        launch = lambda: K.w8a16_matmul[(1, 16)](a, w, s, out, M, N, Kd, Kd, 1, N, 1, N, 1, BM=16, BN=128, BK=128)
        want = (a.double() @ (w.half() * s[None, :]).double()).cpu()
    launch()   # (compiles what it needs)
    torch.cuda.synchronize()
    count = torch.zeros(1, device=DEV)
    one, other = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    out.zero_()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=one):
        count.add_(1)
        with torch.cuda.stream(other):
            launch()
        count.add_(1)
    torch.cuda.synchronize()
    assert ((out.double().cpu() - want.double()).norm() / want.double().norm()).item() <= 5e-3   # (16-bit results)
    for turn in range(3):
        out.zero_()
        graph.replay()
        with torch.cuda.stream(other):
            launch()
        torch.cuda.synchronize()
        assert count.item() == 2 * (turn + 1)
        assert ((out.double().cpu() - want.double()).norm() / want.double().norm()).item() <= 5e-3
