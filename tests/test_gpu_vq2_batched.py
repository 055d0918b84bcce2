"""The batched VQ2 product (matmul_vq2 of the "hip" variant, one launch for all tokens) against the
oracle's matvec of every token.

Bar: rel L2 <= 1e-5 and max|err| <= 1e-3 * max|y_ref|, as for the matvec: the same exact products
with fp32 accumulation."""
import numpy as np
import pytest

from conftest import max_abs_rel, rel_l2

pytestmark = pytest.mark.gpu


def product(orc, w, x, M, K, N):
    return np.concatenate([orc.matvec_vq2(w, x[n * K:(n + 1) * K], M, K, threads=8) for n in range(N)])


# rows and tokens around the 32-row and 32 / 64-token tiles; fewer chunks of 8 indices than waves, a
# partial last chunk, index rows that are not dword-aligned (K % 16 != 0); one and two token blocks
# per wave (9000 rows x 64 tokens: a workgroup per CU)
@pytest.mark.parametrize("M,K,N", [(1, 4, 2), (31, 64, 2), (33, 36, 31), (100, 52, 33), (64, 1024, 65), (77, 1000, 5),
                                   (896, 4864, 7), (9000, 272, 33), (9001, 260, 64), (4864, 896, 130)])
def test_matches_oracle(gpu, orc, M, K, N):
    w, x = gpu.synth_vq2(M, K, seed=M + K), gpu.synth_normal(K * N, seed=K + N)
    got, want = gpu.matmul_vq2(w, x, M, K, N), product(orc, w, x, M, K, N)
    assert rel_l2(got, want) <= 1e-5 and max_abs_rel(got, want) <= 1e-3
    again = gpu.matmul_vq2(w, x, M, K, N)
    assert np.array_equal(got.view(np.uint32), again.view(np.uint32))


def test_token_blocks(gpu, orc):
    """More tokens than one block of the workspaces holds (8M floats): the last block has one token."""
    M, K = 260001, 8
    N = (8 << 20) // M + 1
    w, x = gpu.synth_vq2(M, K, seed=1), gpu.synth_normal(K * N, seed=2)
    assert rel_l2(gpu.matmul_vq2(w, x, M, K, N), product(orc, w, x, M, K, N)) <= 1e-5


@pytest.mark.parametrize("K", [896, 52])
def test_non_finite_values_stay_where_they_are(gpu, orc, K):
    """An infinite codebook entry 0 reaches exactly the rows that use it (positions past the row end
    add nothing), a NaN activation exactly its token."""
    M, N = 70, 35
    w, x = gpu.synth_vq2(M, K, seed=3), gpu.synth_normal(K * N, seed=4)
    w[0:8] = np.frombuffer(np.full(4, np.inf, np.float16).tobytes(), np.uint8)
    x[3 * K + 1] = np.nan
    got, want = gpu.matmul_vq2(w, x, M, K, N), product(orc, w, x, M, K, N)
    fin = np.isfinite(want)
    assert np.array_equal(np.isfinite(got), fin) and 0 < np.count_nonzero(fin) < want.size
    assert rel_l2(got[fin], want[fin]) <= 1e-5


def test_no_tokens_and_one_token(gpu):
    w, x = gpu.synth_vq2(40, 64, seed=5), gpu.synth_normal(64, seed=6)
    gpu.lib().tqhip_dispatch_matmul_vq2(w.ctypes.data, x.ctypes.data, None, 40, 64, 0)  # nothing to do
    assert np.array_equal(gpu.matmul_vq2(w, x, 40, 64, 1), gpu.matvec_vq2(w, x, 40, 64))


# rows past 1024 elements, at least 256 per CU: the table taken slab by slab. Rows that are not a whole
# number of slabs (1040, 2000 with an odd number of dwords), one to three batches a wave, more
# workgroups than CUs (200003 rows), the shortest and a long row; and an infinite codebook entry 0,
# which must not reach a row through the zero entries past its end.
@pytest.mark.parametrize("M,K", [(65536, 1040), (65539, 2000), (70001, 1536), (151936, 1088), (200003, 1040),
                                 (66000, 4112)])
def test_long_row_table_matches_oracle(gpu, orc, M, K):
    w, x = gpu.synth_vq2(M, K, seed=M + K), gpu.synth_normal(K, seed=K)
    dx, dy = gpu.DeviceBuffer.from_array(x), gpu.DeviceBuffer(4 * M)
    for entry0 in (None, np.inf):
        if entry0 is not None:
            w[0:8] = np.frombuffer(np.full(4, entry0, np.float16).tobytes(), np.uint8)
        want = orc.matvec_vq2(w, x, M, K, threads=16)
        dw = gpu.DeviceBuffer.from_array(w)
        gpu.lib().tqhip_memset(dy.ptr, 0xFF, 4 * M)  # every row must be written
        gpu.matvec_vq2_dev(dw, dx, dy, M, K)
        got, fin = dy.download(np.float32, M), np.isfinite(want)
        assert np.array_equal(np.isfinite(got), fin) and (entry0 is not None or fin.all())
        assert rel_l2(got[fin], want[fin]) <= 1e-5


# Rows per wave change at 4, 8 and 32 rows per CU (256 CUs), separately for rows of one step (in_dim
# <= 1024) and longer ones; the last two are the largest the rows kernel takes and one past it.
@pytest.mark.parametrize("M,K", [(1024, 16), (1025, 16), (1027, 1024), (1026, 1040), (2051, 2064), (8193, 272),
                                 (8194, 2048), (8191, 3088), (32768, 1024), (32769, 1024)])
def test_rows_per_wave_give_the_bits_of_one_row_at_a_time(gpu, orc, M, K):
    """Each row's bits do not depend on how many rows a wave takes: alone, as a set of two matrices and
    (a sample of rows) in launches of few rows, aligned x or not."""
    w, xs = gpu.synth_vq2(M, K, seed=M + K), gpu.synth_normal(K + 1, seed=K)
    dw, dx = gpu.DeviceBuffer.from_array(w), gpu.DeviceBuffer.from_array(xs)
    cb, idx = w[:2048], w[2048:].reshape(M, K // 4)
    sample = np.unique(np.r_[0:8, M // 2:M // 2 + 8, M - 8:M])
    few = gpu.DeviceBuffer.from_array(np.concatenate([cb, idx[sample].reshape(-1)]))
    w2 = gpu.synth_vq2(40, 2048, seed=3)
    x2 = gpu.synth_normal(2048, seed=4)
    dw2, dx2, dy2 = gpu.DeviceBuffer.from_array(w2), gpu.DeviceBuffer.from_array(x2), gpu.DeviceBuffer(160)
    for off in (0, 1):
        x = xs[off:off + K]
        ptr = dx.ptr + 4 * off
        dy, dfew, dset = gpu.DeviceBuffer(4 * M), gpu.DeviceBuffer(4 * len(sample)), gpu.DeviceBuffer(4 * M)
        gpu.matvec_vq2_dev(dw, ptr, dy, M, K)
        gpu.matvec_vq2_dev(few, ptr, dfew, len(sample), K)
        gpu.matvec_vq2_set_dev([(dw2, dx2, dy2, 40, 2048), (dw, ptr, dset, M, K)])
        gpu.synchronize()
        got = dy.download(np.float32, M)
        want = orc.matvec_vq2(w, x, M, K, threads=16)
        assert rel_l2(got, want) <= 1e-6, rel_l2(got, want)  # fp32 sums of K / 64 terms a lane and 64 lanes
        assert np.array_equal(dset.download(np.float32, M), got)
        assert rel_l2(dy2.download(np.float32, 40), orc.matvec_vq2(w2, x2, 40, 2048)) <= 1e-6
        if M * K <= 4 * (8 << 20):
            assert np.array_equal(dfew.download(np.float32, len(sample)), got[sample])


# few tokens of long rows, which one matvec per token gives faster: up to 2, 4, 6 and 8 tokens at these
# lengths, and one token more
@pytest.mark.parametrize("M,K,most", [(33, 1024, 2), (130, 2560, 4), (70, 9728, 6), (5, 32768, 8)])
def test_few_tokens_of_long_rows(gpu, orc, M, K, most):
    w, x = gpu.synth_vq2(M, K, seed=M), gpu.synth_normal(K * (most + 1), seed=K)
    each = np.concatenate([gpu.matvec_vq2(w, x[n * K:(n + 1) * K], M, K) for n in range(most + 1)])
    for n in (2, most):
        assert np.array_equal(gpu.matmul_vq2(w, x[:n * K], M, K, n).view(np.uint32), each[:n * M].view(np.uint32)), n
    got = gpu.matmul_vq2(w, x, M, K, most + 1)
    assert not np.array_equal(got, each)  # the matrix launch: other sums
    assert rel_l2(got, product(orc, w, x, M, K, most + 1)) <= 1e-5
