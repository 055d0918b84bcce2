"""One launch over a set of i4 matvecs with their own activations (tqhip_matvec_i4_set_dev).

Every output of the set is held to the matvec bar (rel L2 <= 1e-5, max|err| <= 1e-3 of
max|y|) against the oracle, and where tqhip_matvec_i4_dev runs the set kernel on the
same matrix alone (every decode-size launch of the layer), the set output must have
the same bits. Cases: the Qwen2.5-0.5B layer set, the
Qwen3.5-4B layer shapes, the golden fixtures of the reference in one set,
ragged shapes, more than eight matrices, matrices the set kernel does not take
(G != 64, K % 4 != 0, misaligned x, K > 10240), error codes, and a captured op list.
"""
import numpy as np
import pytest

from conftest import golden, golden_names, max_abs_rel, rel_l2

pytestmark = pytest.mark.gpu

QWEN25_LAYER = [("q", 896, 896, "attn"), ("k", 128, 896, "attn"), ("v", 128, 896, "attn"), ("o", 896, 896, "o"),
                ("gate", 4864, 896, "mlp"), ("up", 4864, 896, "mlp"), ("down", 896, 4864, "down")]


def assert_close(got, want, what):
    l2, mx = rel_l2(got, want), max_abs_rel(got, want)
    assert l2 <= 1e-5 and mx <= 1e-3, f"{what}: rel_l2={l2:.3e} max_rel={mx:.3e}"


def assert_close_rows(got, want, orc, w, x, M, K, what):
    """For outputs of a few rows, where one near-cancelled row dominates the relative L2:
    each row within 1e-5 of the size of its own terms, sum_k |w_mk * x_k| (an fp32 dot
    product of K terms stays well inside that), plus the usual bar where M >= 16."""
    wd = orc.dequant_i4_matrix_f64(w, M, K, 64)
    bound = 1e-5 * (np.abs(wd) @ np.abs(x.astype(np.float64)))
    err = np.abs(got.astype(np.float64) - want.astype(np.float64))
    assert np.all(err <= bound), f"{what}: worst row err/bound = {float(np.max(err / bound)):.3f}"
    if M >= 16:
        assert_close(got, want, what)


def build(gpu, spec, G, seed):
    """spec: (name, M, K, x key); matrices sharing a key share the activation vector."""
    xs, mats = {}, []
    for i, (name, M, K, key) in enumerate(spec):
        if key not in xs:
            x = gpu.synth_normal(K, seed=seed + 1000 + len(xs))
            xs[key] = (x, gpu.DeviceBuffer.from_array(x))
        w = gpu.synth_i4(M, K, G, seed=seed + i)
        mats.append((name, M, K, w, xs[key], gpu.DeviceBuffer.from_array(w), gpu.DeviceBuffer(4 * M)))
    return mats


def run_set(gpu, mats, G):
    arr = gpu.i4_set([(dw, x[1], dy, M, K) for _, M, K, _, x, dw, dy in mats])
    for _, M, _, _, _, _, dy in mats:
        gpu.lib().tqhip_memset(dy.ptr, 0xFF, 4 * M)  # every output must be written by the set
    gpu.matvec_i4_set_dev(arr, G)
    gpu.synchronize()
    return [dy.download(np.float32, M) for _, M, _, _, _, _, dy in mats]


def singles(gpu, mats, G):
    out = []
    for _, M, K, _, x, dw, _ in mats:
        dy = gpu.DeviceBuffer(4 * M)
        gpu.matvec_i4_dev(dw, x[1], dy, M, K, G)
        gpu.synchronize()
        out.append(dy.download(np.float32, M))
    return out


def test_qwen25_layer_set(gpu, orc):
    mats = build(gpu, QWEN25_LAYER, 64, seed=40)
    got = run_set(gpu, mats, 64)
    alone = singles(gpu, mats, 64)
    for (name, M, K, w, x, _, _), g, a in zip(mats, got, alone):
        assert_close(g, orc.matvec_i4(w, x[0], M, K, 64, threads=16), name)
        assert np.array_equal(g, a), f"{name}: set output differs from the single launch (the same kernel)"
    # the same set again: bit-identical (deterministic)
    again = run_set(gpu, mats, 64)
    for (name, *_), g, h in zip(mats, got, again):
        assert np.array_equal(g, h), name


def test_qwen35_4b_layer_shapes(gpu, orc):
    """every long-row matrix has >= 2048 rows, so each wave takes two rows. With a
    896x4864 matrix added, the set runs one long row per wave; the rows of a matrix get the same
    bits either way, and the same bits as its single launch."""
    spec = [("qkv_in", 4096, 2560, "attn"), ("o", 2560, 4096, "o"), ("gate", 9728, 2560, "mlp"),
            ("up", 9728, 2560, "mlp"), ("down", 2560, 9728, "down")]
    mats = build(gpu, spec, 64, seed=60)
    got = run_set(gpu, mats, 64)
    alone = singles(gpu, mats, 64)
    for (name, M, K, w, x, _, _), g, a in zip(mats, got, alone):
        assert_close(g, orc.matvec_i4(w, x[0], M, K, 64, threads=16), name)
        assert np.array_equal(g, a), f"{name}: set output differs from the single launch"
    small = build(gpu, [("small_down", 896, 4864, "s")], 64, seed=70)
    mixed = run_set(gpu, mats + small, 64)
    for (name, *_), g, m in zip(mats, got, mixed):
        assert np.array_equal(g, m), f"{name}: two long rows per wave vs one differ"
    _, M, K, w, x, _, _ = small[0]
    assert_close(mixed[-1], orc.matvec_i4(w, x[0], M, K, 64, threads=16), "small_down")


def test_golden_fixtures_in_one_set(gpu):
    """The reference's outputs (tests/golden, written by its compiled ref kernel) for every
    G = 64 fixture, all in one set launch: special fp16 headers and partial groups included."""
    names = [n for n in golden_names("i4_") if n.endswith("_g64") and "pair" not in n and "qkv" not in n]
    assert len(names) >= 6
    mats, wants = [], []
    for n in names:
        f = golden(n)
        M, K, G = (int(v) for v in f["dims"])
        x = np.ascontiguousarray(f["x"], np.float32)
        mats.append((n, M, K, f["w"], (x, gpu.DeviceBuffer.from_array(x)), gpu.DeviceBuffer.from_array(f["w"]),
                     gpu.DeviceBuffer(4 * M)))
        wants.append(f["y"])
    got = run_set(gpu, mats, 64)
    for (n, *_), g, y in zip(mats, got, wants):
        assert_close(g, y, n)


def test_ragged_and_more_than_eight(gpu, orc):
    # rows not a multiple of a workgroup's rows, partial last groups, K just over 1024 (one
    # wave-row slot) and over 2048 (two), single rows; 11 matrices = two launches
    spec = [("a", 1, 64, "a"), ("b", 3, 200, "b"), ("c", 9, 1028, "c"), ("d", 17, 2052, "d"), ("e", 333, 964, "e"),
            ("f", 5, 4, "f"), ("g", 100, 10240, "g"), ("h", 7, 6144, "h"), ("i", 250, 36, "i"), ("j", 13, 1024, "j"),
            ("k", 2, 8196, "k")]
    mats = build(gpu, spec, 64, seed=80)
    got = run_set(gpu, mats, 64)
    for (name, M, K, w, x, _, _), g in zip(mats, got):
        assert_close_rows(g, orc.matvec_i4(w, x[0], M, K, 64, threads=16), orc, w, x[0], M, K, f"{name} {M}x{K}")


def test_matrices_the_set_kernel_does_not_take(gpu, orc):
    """G = 128 (the whole call), K % 4 != 0, K > 10240 and a misaligned x go through the
    single-matrix kernels; the rest of the set still runs."""
    mats = build(gpu, [("odd_k", 40, 70, "a"), ("wide", 24, 12288, "b"), ("ok", 300, 896, "c")], 64, seed=90)
    # a misaligned activation pointer: x offset by one float inside a larger buffer
    K = 896
    xb = gpu.synth_normal(K + 1, seed=95)
    dxb = gpu.DeviceBuffer.from_array(xb)
    w = gpu.synth_i4(64, K, 64, seed=96)
    mats.append(("misaligned", 64, K, w, (xb[1:].copy(), dxb.ptr + 4), gpu.DeviceBuffer.from_array(w),
                 gpu.DeviceBuffer(4 * 64)))
    got = run_set(gpu, mats, 64)
    for (name, M, K, w, x, _, _), g in zip(mats, got):
        assert_close(g, orc.matvec_i4(w, x[0], M, K, 64, threads=16), name)
    mats = build(gpu, [("g128a", 100, 1024, "a"), ("g128b", 33, 640, "b")], 128, seed=97)
    got = run_set(gpu, mats, 128)
    for (name, M, K, w, x, _, _), g in zip(mats, got):
        assert_close(g, orc.matvec_i4(w, x[0], M, K, 128, threads=16), name)


def test_error_codes(gpu):
    lib = gpu.lib()
    arr = gpu.i4_set([(0, 0, 0, 0, 64)])
    assert lib.tqhip_matvec_i4_set_dev(gpu.ctypes.addressof(arr), 1, 64, None) == gpu.EBADSHAPE
    arr = gpu.i4_set([(0, 0, 0, 4, 64)])
    assert lib.tqhip_matvec_i4_set_dev(gpu.ctypes.addressof(arr), 1, 3, None) == gpu.EBADGROUP
    assert lib.tqhip_matvec_i4_set_dev(None, 1, 64, None) == gpu.EBADSHAPE
    assert lib.tqhip_matvec_i4_set_dev(None, 0, 64, None) == gpu.OK  # an empty set launches nothing


def test_set_op_in_a_captured_graph(gpu, orc):
    """TQHIP_OP_I4_SET in an op list: eager run and graph replays agree bit for bit, with new
    activations written before each replay (the replay reads them at replay time)."""
    mats = build(gpu, QWEN25_LAYER, 64, seed=120)
    arr = gpu.i4_set([(dw, x[1], dy, M, K) for _, M, K, _, x, dw, dy in mats])
    ops = [gpu.set_op(arr, 64)]
    stream = gpu.Stream()
    graph = gpu.OpsGraph(ops, stream)
    keys = {}
    for _, _, K, _, x, _, _ in mats:
        keys[id(x)] = (x, K)
    try:
        for rep in range(3):
            for i, (x, K) in enumerate(keys.values()):
                v = gpu.synth_normal(K, seed=130 + 10 * rep + i)
                x[1].upload(v)
                x[0][:] = v
            gpu.run_ops(ops, 1, stream)
            stream.synchronize()
            want = [dy.download(np.float32, M) for _, M, _, _, _, _, dy in mats]
            for _, M, _, _, _, _, dy in mats:
                gpu.lib().tqhip_memset(dy.ptr, 0xFF, 4 * M)
            graph.launch()
            stream.synchronize()
            for (name, M, K, w, x, _, dy), wv in zip(mats, want):
                assert np.array_equal(dy.download(np.float32, M), wv), f"replay {rep}: {name}"
        for (name, M, K, w, x, _, _), wv in zip(mats, want):
            assert_close(wv, orc.matvec_i4(w, x[0], M, K, 64, threads=16), name)
    finally:
        graph.close()


def test_non_finite_activation_stays_in_its_matrix(gpu, orc):
    """A NaN in one activation vector of a set (up's x): every output of the matrices that read it
    is non-finite, as in the reference, and the matrices with other activation vectors are finite
    and unchanged (each workgroup converts only its own matrix's activations)."""
    mats = build(gpu, QWEN25_LAYER, 64, seed=70)
    clean = run_set(gpu, mats, 64)
    x_mlp, dx_mlp = next(m[4] for m in mats if m[0] == "gate")
    poisoned = x_mlp.copy()
    poisoned[100] = np.nan
    dx_mlp.upload(poisoned)
    got = run_set(gpu, mats, 64)
    for (name, M, K, w, x, _, _), g, c in zip(mats, got, clean):
        if name in ("gate", "up"):
            assert not np.any(np.isfinite(orc.matvec_i4(w, poisoned, M, K, 64, threads=16)))
            assert not np.any(np.isfinite(g)), f"{name}: finite outputs from a NaN activation"
        else:
            assert np.array_equal(g, c), f"{name}: changed by another matrix's NaN activation"


SET_SHAPES = [(1, 4), (17, 32), (33, 96), (65, 860), (2048, 1024), (2049, 1028), (31, 2080), (129, 4864), (16, 8224),
              (2050, 10240), (7, 10244)]  # (10244: past the set kernel's rows)


@pytest.mark.parametrize("G", [32, 64, 128])
@pytest.mark.parametrize("M,K", SET_SHAPES)
def test_group_sizes_at_the_edges(gpu, orc, G, M, K):
    """The set kernel's group sizes at the edges of its shapes (row halves, slots, rows that end inside
    a weight group or a block of 64 activations), alone and in a set with a second matrix. Each row
    is held to its rounding: x to 2^-23 of the largest |x| of its 64 (groups of 128 past the set kernel: 2^-22
    of the largest of 128), then at most 16 roundings (the half-group's value, the slots and the wave sum)
    of its terms, each at most scale * 30 * |x|. Half of the activations are ties of that rounding."""
    rng = np.random.default_rng(K * 7 + M + G)
    x = rng.standard_normal(K).astype(np.float32)
    x[::2] = (np.sign(x[::2]) * (np.floor(np.abs(x[::2]) * 2**18) + 0.5) * 2.0**-18).astype(np.float32)
    w = gpu.synth_i4(M, K, G, seed=5)
    w2 = gpu.synth_i4(24, K, G, seed=6)
    got = []
    for mats in ([(w, M)], [(w2, 24), (w, M)]):
        dev = [(gpu.DeviceBuffer.from_array(b), gpu.DeviceBuffer.from_array(x), gpu.DeviceBuffer(4 * m), m, K)
               for b, m in mats]
        if len(mats) == 1:
            gpu.matvec_i4_dev(dev[0][0], dev[0][1], dev[0][2], M, K, G)
        else:
            gpu.matvec_i4_set_dev(gpu.i4_set(dev), G)
        gpu.synchronize()
        got.append(dev[-1][2].download(np.float32, M))
    wd = orc.dequant_i4_matrix_f64(w, M, K, G)
    want = wd @ x.astype(np.float64)
    groups = -(-K // G)
    scale = w.reshape(M, groups, 4 + G // 2)[:, :, :2].copy().view(np.float16)[:, :, 0].astype(np.float64)
    scale = np.repeat(np.abs(scale), G, axis=1)[:, :K]
    block = 64 if K <= 10240 else max(G, 64)
    peak = np.repeat([np.abs(x[b:b + block]).max() for b in range(0, K, block)], block)[:K].astype(np.float64)
    step = 2.0**-23 if K <= 10240 else 2.0**-22
    bound = step * (np.abs(wd) @ peak) + 16 * 2.0**-24 * 30 * (scale @ np.abs(x.astype(np.float64)))
    for y, what in zip(got, ("alone", "in a set")):
        err = np.abs(y - want)
        assert np.all(err <= bound), f"{what}: worst row err/bound = {float(np.max(err / bound)):.3f}"
    if K <= 10240:
        assert np.array_equal(got[0], got[1])


@pytest.mark.parametrize("G", [32, 64, 128])
def test_extreme_activations_by_group_size(gpu, orc, G):
    """Activations whose scaled value is the largest that 24 bits hold, the largest and the smallest
    floats: products of the ends of the range against the oracle, and an infinity or a NaN in every
    row that reads it."""
    M, K = 48, 1344
    w = gpu.synth_i4(M, K, G, seed=9)
    wd = orc.dequant_i4_matrix_f64(w, M, K, G)
    dw, dy = gpu.DeviceBuffer.from_array(w), gpu.DeviceBuffer(4 * M)
    base = np.random.default_rng(1).standard_normal(K).astype(np.float32)
    for peak in (np.float32(1) - np.float32(2.0**-24), np.float32(3e36), np.float32(1e-38), np.float32(2.0**-149)):
        x = (base / np.abs(base).max() * peak).astype(np.float32)
        x[::7] = peak
        gpu.matvec_i4_dev(dw, gpu.DeviceBuffer.from_array(x), dy, M, K, G)
        gpu.synchronize()
        want = wd @ x.astype(np.float64)
        # 1e-6 of the row's terms; a result below the normal floats is held to a few of their last units
        bound = 1e-6 * (np.abs(wd) @ np.abs(x.astype(np.float64))) + 64 * 2.0**-149
        assert np.all(np.abs(dy.download(np.float32, M) - want) <= bound), peak
    for bad in (np.inf, np.nan):
        x = base.copy()
        x[K - 1] = bad
        gpu.matvec_i4_dev(dw, gpu.DeviceBuffer.from_array(x), dy, M, K, G)
        gpu.synchronize()
        assert not np.isfinite(dy.download(np.float32, M)).any()


@pytest.mark.parametrize("offset", [1, 2, 3])
def test_groups_of_32_at_any_weight_address(gpu, orc, offset):
    """Weights that do not start on 4 bytes: the wave-per-row kernel (the same bits as its own entry
    point), alone, as a pair and in a set."""
    M, K, G = 70, 864, 32
    w, x = gpu.synth_i4(M, K, G, seed=2), gpu.synth_normal(K, seed=3)
    dw = gpu.DeviceBuffer.from_array(np.concatenate([np.zeros(offset, np.uint8), w, np.zeros(4, np.uint8)]))
    dx, ys = gpu.DeviceBuffer.from_array(x), [gpu.DeviceBuffer(4 * M) for _ in range(5)]
    p = dw.ptr + offset
    gpu.lib().tqhip_matvec_i4_generic_dev(p, dx.ptr, ys[0].ptr, M, K, G, None)
    gpu.matvec_i4_dev(p, dx, ys[1], M, K, G)
    gpu.matvec_i4_set_dev(gpu.i4_set([(p, dx, ys[2], M, K)]), G)
    gpu.lib().tqhip_matvec_pair_i4_dev(p, p, dx.ptr, ys[3].ptr, ys[4].ptr, M, K, G, None)
    gpu.synchronize()
    got = [y.download(np.float32, M) for y in ys]
    want = orc.matvec_i4(w, x, M, K, G)
    assert np.linalg.norm(got[0] - want) <= 1e-6 * np.linalg.norm(want)  # fp32 sums of 27 groups
    for g in got[1:]:
        assert np.array_equal(g.view(np.uint32), got[0].view(np.uint32))


@pytest.mark.parametrize("G", [32, 128])
@pytest.mark.parametrize("M,K,peak,where", [(65, 864, 300, "tiny scales"), (65, 4864, 3000, "tiny scales"),
                                            (130, 9728, 1e6, "tiny scales"), (65, 2080, 3000, "zero weights")])
def test_an_outlier_costs_only_its_own_group(gpu, orc, G, M, K, peak, where):
    """One activation of every second group far above the others, where it counts for little: its group's
    scales are tiny, or its own weights are 0. Each row is held to its rounding. Groups of 32: x to 2^-31 of
    the largest |x| of its group, and then one rounding of each half-group's value; groups of 128: x to
    2^-23 of the largest of its 64, and the half-group's sums, formed in fp32 (3 roundings of their
    terms); then the slots, the wave sum and the stores' at most 12 roundings of the values."""
    rng = np.random.default_rng(K + G)
    groups = -(-K // G)
    w = gpu.synth_i4(M, K, G, seed=K).reshape(M, groups, 4 + G // 2)
    x = rng.standard_normal(K).astype(np.float32)
    x[::2 * G] = peak
    head = w[:, :, :4].copy().view(np.float16)  # scale, zero
    if where == "tiny scales":
        head[:, ::2, 0] = 6e-8
    else:
        head[:, ::2, 1] = np.rint(head[:, ::2, 1].astype(np.float32))
        w[:, ::2, 4] = (w[:, ::2, 4] & 0xF0) | head[:, ::2, 1].astype(np.uint8)
    w[:, :, :4] = head.view(np.uint8)
    w = np.ascontiguousarray(w).reshape(-1)
    dw, dx, dy = gpu.DeviceBuffer.from_array(w), gpu.DeviceBuffer.from_array(x), gpu.DeviceBuffer(4 * M)
    gpu.matvec_i4_dev(dw, dx, dy, M, K, G)
    gpu.synchronize()
    pad = -K % 64
    wd = np.pad(orc.dequant_i4_matrix_f64(w, M, K, G), ((0, 0), (0, pad)))
    xp = np.pad(x.astype(np.float64), (0, pad))
    scale = np.pad(np.repeat(np.abs(head[:, :, 0].astype(np.float64)), G, axis=1)[:, :K], ((0, 0), (0, pad)))
    block, step = (32, 2.0**-31) if G == 32 else (64, 2.0**-23)
    largest = np.repeat(np.abs(xp).reshape(-1, block).max(1), block)
    halves = np.abs((wd * xp).reshape(M, -1, 32).sum(2)).sum(1)
    bound = step * (np.abs(wd) @ largest) + 12 * 2.0**-24 * halves
    if G == 128:
        bound += 3 * 2.0**-24 * 30 * (scale @ np.abs(xp))
    err = np.abs(dy.download(np.float32, M) - wd @ xp)
    assert np.all(err <= bound), f"worst row err/bound = {float(np.max(err / bound)):.3f}"
    print(f"[outlier] G {G} {M}x{K} {where}: rel L2 {np.linalg.norm(err) / np.linalg.norm(wd @ xp):.2e}, "
          f"worst err/bound {float(np.max(err / bound)):.2f}", flush=True)
