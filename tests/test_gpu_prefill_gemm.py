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
