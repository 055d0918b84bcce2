"""The prefill GEMM's preparation and tile kernels at the sizes where their dispatch changes.

Bar of a product: rel L2 <= 2e-3 against the oracle (both operands rounded to fp16 once or, at
G = 64, the weights twice); two kernels that form the same sums in the same order: the same bits."""
import numpy as np
import pytest

from conftest import fp16_operand_bound_ok, rel_l2

pytestmark = pytest.mark.gpu


def matmul_dev(gpu, w, x, M, K, N, G, x_offset=0):
    """tqhip_matmul_i4_dev with X x_offset floats past a 16-byte boundary."""
    xb = np.zeros(K * N + 4, np.float32)
    xb[x_offset:x_offset + K * N] = x
    dw, dx, dy = gpu.DeviceBuffer.from_array(w), gpu.DeviceBuffer.from_array(xb), gpu.DeviceBuffer(4 * M * N)
    gpu.lib().tqhip_memset(dy.ptr, 0xFF, 4 * M * N)  # every output must be written
    gpu.matmul_i4_dev(dw, dx.ptr + 4 * x_offset, dy, M, K, N, G)
    gpu.synchronize()
    return dy.download(np.float32, M * N)


# one, two, four and eight 8-element chunks a thread, at and past each limit; past 16384 elements
# and with X off a 16-byte boundary one float at a time
@pytest.mark.parametrize("K", [2048, 2052, 4096, 4100, 8192, 8196, 9728, 16384, 16388])
@pytest.mark.parametrize("G", [64, 128])
def test_x_conversion_by_row_length(gpu, orc, K, G):
    M, N = 33, 35
    w, x = gpu.synth_i4(M, K, G, seed=K), gpu.synth_normal(K * N, seed=K + 1)
    x[K:2 * K] *= 1e-20
    got = matmul_dev(gpu, w, x, M, K, N, G)
    assert np.array_equal(got.view(np.uint32), matmul_dev(gpu, w, x, M, K, N, G, x_offset=1).view(np.uint32))
    assert rel_l2(got, orc.matmul_i4(w, x, M, K, N, G, threads=8)) <= 2e-3


# group sizes other than 64 on the tile kernel: rows and tokens around its three tiles (32 x 32,
# 128 x 64, 256 x 96), a last group that K does not fill, one that leaves the second half of the
# last step without a group (G = 32, K = 1056), groups across step boundaries (G = 96), fewer steps
# than the ring holds
@pytest.mark.parametrize("G", [32, 96, 128, 256])
@pytest.mark.parametrize("M,K,N", [(1, 32, 1), (33, 64, 32), (31, 1056, 33), (129, 100, 128), (257, 1000, 129),
                                   (300, 2560, 200), (4, 4864, 97)])
def test_other_group_sizes(gpu, orc, M, K, N, G):
    w, x = gpu.synth_i4(M, K, G, seed=M + K + G), gpu.synth_normal(K * N, seed=N)
    got, want = matmul_dev(gpu, w, x, M, K, N, G), orc.matmul_i4(w, x, M, K, N, G, threads=8)
    if M * N < 16:  # a handful of outputs: each within the fp16 operands' rounding of its products
        assert fp16_operand_bound_ok(got, want, orc, w, x, M, K, N, G)
    else:
        assert rel_l2(got, want) <= 2e-3


# every count of steps left over after the rounds of the tiles' rings (3 and 4 steps of 64), from
# fewer steps than a ring holds, on grids of several workgroups per CU and repeated: a step whose
# activations were not waited for shows only now and then
@pytest.mark.parametrize("steps", [1, 2, 3, 5, 6, 7, 15])
@pytest.mark.parametrize("N,G", [(40, 64), (128, 64), (20, 128), (128, 128), (200, 64), (200, 32)])
def test_steps_left_over(gpu, orc, steps, N, G):
    M, K = 9728, 64 * steps
    w, x = gpu.synth_i4(M, K, G, seed=steps + N), gpu.synth_normal(K * N, seed=steps)
    want = orc.matmul_i4(w, x, M, K, N, G, threads=16)
    dw, dx, dy = gpu.DeviceBuffer.from_array(w), gpu.DeviceBuffer.from_array(x), gpu.DeviceBuffer(4 * M * N)
    first = None
    for _ in range(8):
        gpu.lib().tqhip_memset(dy.ptr, 0xFF, 4 * M * N)
        gpu.matmul_i4_dev(dw, dx, dy, M, K, N, G)
        gpu.synchronize()
        got = dy.download(np.float32, M * N)
        first = got if first is None else first
        assert np.array_equal(got.view(np.uint32), first.view(np.uint32))
    assert rel_l2(first, want) <= 2e-3


# K slices (kSplitParts, kSplitSeq): few tiles and many steps, with slices of unequal step counts, at
# the tile edges; both tiles that are split, both dequantizations. The device entry point adds the
# slices' partials, the allocation-free one runs the slices one after the other: the same bits,
# and the same again on every repeat (whichever slice arrives last).
@pytest.mark.parametrize("M,K,N,G", [(128, 9728, 40, 64), (129, 4864, 65, 64), (896, 4864, 128, 64), (1, 4160, 33, 64),
                                     (1000, 2560, 256, 128), (40, 9728, 32, 128), (513, 4900, 1, 32),
                                     (4096, 2560, 16, 256), (2560, 9728, 200, 96)])
def test_k_slices(gpu, orc, M, K, N, G):
    w, x = gpu.synth_i4(M, K, G, seed=M + N), gpu.synth_normal(K * N, seed=K)
    want = orc.matmul_i4(w, x, M, K, N, G, threads=16)
    dw, dx, dy = gpu.DeviceBuffer.from_array(w), gpu.DeviceBuffer.from_array(x), gpu.DeviceBuffer(4 * M * N)
    outs = []
    for i in range(7):
        gpu.lib().tqhip_memset(dy.ptr, 0xFF, 4 * M * N)
        if i < 6:
            gpu.matmul_i4_dev(dw, dx, dy, M, K, N, G)
        else:
            assert gpu.matmul_i4_noalloc_dev(dw, dx, dy, M, K, N, G) == gpu.OK
        gpu.synchronize()
        outs.append(dy.download(np.float32, M * N))
        assert np.array_equal(outs[i].view(np.uint32), outs[0].view(np.uint32)), i
    if M * N < 64:
        assert fp16_operand_bound_ok(outs[0], want, orc, w, x, M, K, N, G)
    else:
        assert rel_l2(outs[0], want) <= 2e-3


def test_k_slices_in_a_captured_graph(gpu, orc):
    """Split calls captured into an op graph: replays with new activations, eager work and
    synchronisations between them give the eager bits (the counters are zero after every replay)."""
    shapes = [(896, 4864, 48, 64), (1024, 2560, 20, 128)]
    bufs = [(gpu.DeviceBuffer.from_array(gpu.synth_i4(M, K, G, seed=M)), gpu.DeviceBuffer(4 * K * N),
             gpu.DeviceBuffer(4 * M * N)) for M, K, N, G in shapes]
    ops = [gpu.Op(gpu.OP_I4_MATMUL, w.ptr, x.ptr, y.ptr, M, K, N, G) for (w, x, y), (M, K, N, G) in zip(bufs, shapes)]
    stream = gpu.Stream()
    graph = gpu.OpsGraph(ops, stream)
    try:
        for rep in range(4):
            for (_, x, _), (M, K, N, _) in zip(bufs, shapes):
                x.upload(gpu.synth_normal(K * N, seed=rep + M))
            graph.launch()
            stream.synchronize()
            got = [y.download(np.float32, M * N) for (_, _, y), (M, _, N, _) in zip(bufs, shapes)]
            gpu.run_ops(ops, 1)
            gpu.synchronize()
            for g, (_, _, y), (M, _, N, _) in zip(got, bufs, shapes):
                assert np.array_equal(g.view(np.uint32), y.download(np.float32, M * N).view(np.uint32)), rep
    finally:
        graph.close()


# the few-token kernel's slices: one (short rows), chosen by estimated time, the fewest that their
# length allows (49 steps: 7 of 7; 50: 8), and two rounds of workgroups (tall, short rows)
@pytest.mark.parametrize("M,K,N", [(129, 60, 8), (896, 256, 8), (129, 448, 3), (300, 512, 32), (1, 3136, 8),
                                   (127, 3140, 1), (896, 4864, 8), (129, 16384, 5), (70000, 132, 2)])
def test_few_token_slices(gpu, orc, M, K, N):
    w, x = gpu.synth_i4(M, K, 64, seed=M + K), gpu.synth_normal(K * N, seed=N)
    got = matmul_dev(gpu, w, x, M, K, N, 64)
    assert np.array_equal(got, matmul_dev(gpu, w, x, M, K, N, 64))  # one order of the slices
    assert rel_l2(got, orc.matmul_i4(w, x, M, K, N, 64, threads=8)) <= 2e-3


# the longest row that the few-token kernel's slices cover (255 of 7 steps), and one past it, which
# takes the tiled GEMM; the few-token call after it finds its counters zero
@pytest.mark.parametrize("K", [114240, 114244, 131072])
def test_rows_past_the_few_token_slices(gpu, orc, K):
    M, N, G = 130, 3, 64
    print(f"[few tokens] {M}x{K}x{N}", flush=True)
    w, x = gpu.synth_i4(M, K, G, seed=K), gpu.synth_normal(K * N, seed=K + 1)
    got = matmul_dev(gpu, w, x, M, K, N, G)
    assert rel_l2(got, orc.matmul_i4(w, x, M, K, N, G, threads=16)) <= 2e-3
    dw, dx, dy = gpu.DeviceBuffer.from_array(w), gpu.DeviceBuffer.from_array(x), gpu.DeviceBuffer(4 * M * N)
    assert gpu.matmul_i4_noalloc_dev(dw, dx, dy, M, K, N, G) == gpu.OK
    gpu.synchronize()
    assert np.array_equal(dy.download(np.float32, M * N), got)
    w, x = gpu.synth_i4(896, 4864, G, seed=1), gpu.synth_normal(4864 * 8, seed=2)
    assert rel_l2(matmul_dev(gpu, w, x, 896, 4864, 8, G), orc.matmul_i4(w, x, 896, 4864, 8, G, threads=16)) <= 2e-3
