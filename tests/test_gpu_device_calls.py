"""The device-pointer calls against the CPU oracle: every group size, token
counts on both sides of each kernel's range, rows that leave partial tiles,
and K that leaves partial tiles of groups.  Bar: bit-exact."""
import concurrent.futures

import numpy as np
import pytest

from rai_amd.workload import gemv_operands

pytestmark = pytest.mark.gpu


def _bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


def _call(rai, name, out, nib, params, x, rows, cols, m, gs):
    rc = getattr(rai.lib(), name)(out.ptr, nib.ptr, params.ptr, x.ptr, rows, cols, m, gs, None)
    assert rc == 0, rai.lib().rai_last_error()
    assert rai.lib().rai_device_synchronize() == 0
    return out.to_host(np.float32, m * rows)


@pytest.mark.parametrize("name", ["rai_w4a8_matmul_dev", "rai_w4a8_matmul_noalloc_dev"])
@pytest.mark.parametrize("n,m,gs", [(512, 1, 32), (512, 1, 64), (384, 1, 128), (4608, 1, 32), (512, 5, 32),
                                    (320, 70, 64)])
def test_output_over_its_own_input(rai, ora, name, n, m, gs):
    """The output rows may lie on the input rows (the input is quantized
    before anything is written); an infinite and a zero group among them."""
    nib, params, x = gemv_operands(n, n, m, gs, seed=n + m + gs)
    x = x.reshape(m, n)
    x[0, gs // 2] = np.inf
    x[m - 1, gs:2 * gs] = 0.0
    want = ora.w4a8_matmul(nib, params, x, n, n, m, gs)
    dev = rai.DeviceArray.from_host
    buf = dev(np.ascontiguousarray(x, np.float32))
    got = _call(rai, name, buf, dev(nib), dev(params), buf, n, n, m, gs)
    assert np.array_equal(_bits(got).reshape(-1), _bits(want).reshape(-1))


def _tokens(x, m, cols, gs, seed):
    """Ordinary rows, and among them: values so small that the input sums are
    subnormal, a scale past 2^88 in one group, a zero row."""
    x = x.reshape(m, cols).astype(np.float32)
    r = np.random.default_rng(seed)
    x[r.integers(m)] *= np.float32(1e-39)
    x[r.integers(m), :gs] *= np.float32(1e30)
    x[r.integers(m)] = 0.0
    return x


# K: one group, fewer groups than a step or a stage of the kernel, one past a
# stage, several stages with a remainder.
MM = [(32, 32), (32, 96), (32, 544), (32, 1568), (64, 64), (64, 320), (64, 576), (64, 1728),
      (128, 128), (128, 384), (128, 640), (128, 2176)]


def _both_calls(rai, ora, rows, cols, m, gs, specials=(False, True)):
    nib, params, x = gemv_operands(rows, cols, m, gs, seed=rows + cols + m)
    dev = rai.DeviceArray.from_host
    dn, dp, do = dev(nib), dev(params), rai.DeviceArray(4 * m * rows)
    for special in specials:
        if special:
            x = _tokens(x, m, cols, gs, cols + m)
        want = ora.w4a8_matmul(nib, params, x, rows, cols, m, gs)
        xd = dev(np.ascontiguousarray(x, np.float32))
        names = ["rai_w4a8_matmul_dev"]
        if m * cols <= 1 << 20:
            names.append("rai_w4a8_matmul_noalloc_dev")
        for name in names:
            got = _call(rai, name, do, dn, dp, xd, rows, cols, m, gs)
            assert np.array_equal(_bits(got).reshape(-1), _bits(want).reshape(-1)), (name, special)


@pytest.mark.parametrize("gs,cols", MM)
def test_gemm_every_group_size(rai, ora, gs, cols):
    """Enough row and token tiles for the matrix-core GEMM: a last row tile of
    31 rows, a last token tile of one token."""
    _both_calls(rai, ora, 2111, cols, 545, gs)


@pytest.mark.parametrize("gs,cols", [(32, 96), (64, 192), (128, 128)])
@pytest.mark.parametrize("rows,m", [(36097, 33), (72100, 25)])
def test_gemm_many_rows_few_tokens(rai, ora, gs, cols, rows, m):
    _both_calls(rai, ora, rows, cols, m, gs)


@pytest.mark.parametrize("gs,cols", MM)
@pytest.mark.parametrize("rows,m", [(1, 65), (127, 96), (130, 97), (300, 160)])
def test_streamed_kernel_past_64_tokens(rai, ora, gs, cols, rows, m):
    _both_calls(rai, ora, rows, cols, m, gs)


@pytest.mark.parametrize("gs,experts,topk,m", [(32, 8, 3, 70), (64, 16, 2, 150), (128, 5, 5, 65), (32, 64, 8, 97)])
def test_sparse_layer_prefill(rai, ora, gs, experts, topk, m):
    """More than 64 tokens through a sparse layer: every expert's tiles in one
    launch (experts without a token, with one tile and with several)."""
    img = rai.synth_model(256, 2, 4, 4, 64, 512, 500, 256, group_size=gs, num_experts=experts,
                          experts_per_token=topk, seed=gs + m)
    gm, om = rai.RaiModel.from_bytes(img), ora.Model(img, 128)
    h = np.random.default_rng(m).normal(0.0, 1.0, (m, 256)).astype(np.float32)
    h[m // 2:] = h[0] + 1e-3 * h[m // 2:]  # crowd some experts
    got = gm.forward_batch(h, np.arange(m), gm.create_kv_cache(256))
    want = om.forward_batch(h, np.arange(m), om.create_kv(256))
    assert np.array_equal(_bits(got).reshape(-1), _bits(want).reshape(-1))


@pytest.mark.parametrize("experts,topk,m", [(64, 8, 257), (70, 4, 239), (17, 16, 964)])
@pytest.mark.parametrize("hidden", [128, 288])
def test_router_tiles(rai, ora, hidden, experts, topk, m):
    """Router logits in tiles of 16 tokens x 16 experts: whole and ragged tiles
    of both, column chunks that fill the loads in flight and that do not."""
    img = rai.synth_model(hidden, 1, 2, 2, 64, 64, 300, 1024, group_size=32, num_experts=experts,
                          experts_per_token=topk, seed=experts + m)
    gm, om = rai.RaiModel.from_bytes(img), ora.Model(img, 256)
    h = np.random.default_rng(m).normal(0.0, 1.0, (m, hidden)).astype(np.float32)
    got = gm.forward_batch(h, np.arange(m), gm.create_kv_cache(1024))
    want = om.forward_batch(h, np.arange(m), om.create_kv(1024))
    assert np.array_equal(_bits(got).reshape(-1), _bits(want).reshape(-1))


def _table(vocab, hidden, gs, seed):
    r = np.random.default_rng(seed)
    codes = r.integers(0, 256, vocab * hidden, dtype=np.uint8)
    par = np.stack([r.uniform(0.0005, 0.002, (vocab, hidden // gs)), r.normal(0.0, 0.05, (vocab, hidden // gs))], 2)
    return codes, np.ascontiguousarray(par.astype(np.float16)).view(np.uint8).reshape(-1)


# Units of 32 columns: under one chunk of 64, one chunk, one past it, several.
@pytest.mark.parametrize("gs,hidden", [(32, 32), (32, 2048), (32, 2080), (64, 192), (64, 2112), (64, 4096),
                                       (128, 128), (128, 2176), (128, 5120)])
@pytest.mark.parametrize("vocab", [1, 15, 200])
def test_tied_head_every_group_size(rai, ora, gs, hidden, vocab):
    codes, par = _table(vocab, hidden, gs, hidden + vocab)
    h = np.random.default_rng(vocab).normal(0.0, 1.0, hidden).astype(np.float32)
    for scale in (1.0, 1e-39, 1e30):
        hh = (h * np.float32(scale)).astype(np.float32)
        hh[: gs // 2] = 0.0
        want = ora.tied_lm_head(hh, codes, par, vocab, gs)
        assert np.array_equal(_bits(rai.tied_lm_head(hh, codes, par, vocab, gs)), _bits(want)), scale


@pytest.mark.parametrize("m", [1, 4, 9])
def test_tied_logits_of_a_batch(rai, ora, m):
    img = rai.synth_model(256, 1, 4, 4, 64, 512, 333, 64, group_size=32, tied=True, seed=m)
    gm, om = rai.RaiModel.from_bytes(img), ora.Model(img, 128)
    h = np.random.default_rng(m).normal(0.0, 1.0, (m, 256)).astype(np.float32)
    got, want = gm.hidden_to_logits_batch(h, m), om.hidden_to_logits_batch(h, m)
    assert np.array_equal(_bits(got).reshape(-1), _bits(want).reshape(-1))


# One token: the GEMV that quantizes its row (K <= 4096) or takes it quantized;
# K under a chunk of 1024 columns, one past it, several, with odd group counts.
@pytest.mark.parametrize("gs,cols", [(32, 256), (32, 1056), (32, 4096), (32, 4128), (64, 256), (64, 1088), (64, 4096),
                                     (64, 6976), (128, 256), (128, 1152), (128, 3968), (128, 4224), (128, 14336)])
@pytest.mark.parametrize("rows", [1, 6, 17, 530])
def test_one_token_every_group_size(rai, ora, gs, cols, rows):
    nib, params, x = gemv_operands(rows, cols, 1, gs, seed=rows + cols)
    for scale in (1.0, 1e-39, 1e30):
        xs = (x.reshape(-1) * np.float32(scale)).astype(np.float32)
        want = ora.w4a8_matmul(nib, params, xs, rows, cols, 1, gs)
        dev = rai.DeviceArray.from_host
        for name in ("rai_w4a8_matmul_dev", "rai_w4a8_matmul_noalloc_dev"):
            got = _call(rai, name, rai.DeviceArray(4 * rows), dev(nib), dev(params), dev(xs), rows, cols, 1, gs)
            assert np.array_equal(_bits(got), _bits(want).reshape(-1)), (name, scale)


# Every one-token kernel, K ending inside a chunk of 1024 columns (for group 32,
# also one group past it) and on its edge.
@pytest.mark.parametrize("gs,cols", [(32, 1056), (32, 1184), (32, 2048), (32, 4128), (64, 320), (64, 1088), (64, 4160),
                                     (128, 384), (128, 1152), (128, 4224)])
@pytest.mark.parametrize("last", ["sum", "element"])
def test_one_token_infinite_last_group(rai, ora, gs, cols, last):
    """The last group's input sum overflows (finite values), or one of its
    elements is infinite: nothing but that group's own terms sees it."""
    rows = 37
    nib, params, x = gemv_operands(rows, cols, 1, gs, seed=cols + gs)
    x = np.ascontiguousarray(x, np.float32).reshape(-1)
    if last == "sum":
        x[-gs:] = 2e37
    else:
        x[-gs // 2] = np.inf
    want = ora.w4a8_matmul(nib, params, x, rows, cols, 1, gs).reshape(-1)
    if last == "sum":
        assert np.isneginf(want).all()  # every zero point is negative
    dev = rai.DeviceArray.from_host
    for name in ("rai_w4a8_matmul_dev", "rai_w4a8_matmul_noalloc_dev"):
        got = _call(rai, name, rai.DeviceArray(4 * rows), dev(nib), dev(params), dev(x), rows, cols, 1, gs)
        assert np.array_equal(got, want, equal_nan=True), name
    lin = (nib, params, rows, cols, gs)
    for got in rai.w4a8_fused_gate_up(lin, lin, x):
        assert np.array_equal(got, want, equal_nan=True)


@pytest.mark.parametrize("gs", [32, 64, 128])
@pytest.mark.parametrize("hidden,heads,kv,hd,ffn,experts", [(256, 4, 2, 64, 384, 0), (1152, 9, 3, 128, 1280, 0),
                                                            (512, 8, 8, 64, 256, 8)])
def test_decode_steps_every_group_size(rai, ora, gs, hidden, heads, kv, hd, ffn, experts):
    """One-token forward passes (fused norm, rope and quantization) and the
    head, token after token on one cache."""
    img = rai.synth_model(hidden, 2, heads, kv, hd, ffn, 400, 64, group_size=gs, num_experts=experts,
                          experts_per_token=min(experts, 3), seed=gs + hidden)
    gm, om = rai.RaiModel.from_bytes(img), ora.Model(img, 0)
    gk, ok = gm.create_kv_cache(64), om.create_kv(64)
    r = np.random.default_rng(hidden)
    for pos in range(3):
        h = r.normal(0.0, 1.0, (1, hidden)).astype(np.float32)
        got, want = gm.forward_batch(h, [pos], gk), om.forward_batch(h, np.array([pos]), ok)
        assert np.array_equal(_bits(got).reshape(-1), _bits(want).reshape(-1)), pos
        gl, ol = gm.hidden_to_logits_batch(got, 1), om.hidden_to_logits_batch(want, 1)
        assert np.array_equal(_bits(gl).reshape(-1), _bits(ol).reshape(-1)), pos


# 2..64 tokens: one to four token tiles of 16; row counts that take one, two
# and four waves per row tile; K of one group, of a partial step of four groups
# and of several steps; K the register-pipelined kernel does not take.
@pytest.mark.parametrize("gs,cols", [(32, 32), (32, 160), (32, 416), (32, 768), (32, 1056), (64, 64), (64, 320),
                                     (64, 1088), (128, 128), (128, 640), (128, 2688)])
@pytest.mark.parametrize("rows,m", [(1, 2), (17, 4), (70, 9), (50, 16), (33, 17), (40, 64), (5000, 49), (16400, 33)])
def test_small_batches_every_group_size(rai, ora, gs, cols, rows, m):
    if rows > 1000 and cols > 700:
        cols = 4 * gs + gs  # the oracle's time
    _both_calls(rai, ora, rows, cols, m, gs)


# Both sides of the lines between the kernels of 2..64 tokens: the register-
# pipelined one with its ring of two (K an odd multiple of 256) and past 24 tokens,
# the VALU one at two to four tokens.
@pytest.mark.parametrize("gs,rows,cols,m", [
    (32, 70, 256, 12), (32, 70, 768, 64), (32, 1100, 1280, 65), (32, 4097, 1280, 17), (32, 5009, 2816, 2),
    (32, 5009, 2816, 8), (32, 5009, 2816, 9), (32, 16401, 768, 12), (32, 16401, 2816, 11), (32, 16401, 1280, 13),
    (32, 5009, 5376, 4), (32, 5009, 5376, 5), (32, 4999, 5376, 3), (32, 130, 13056, 4),
    (32, 513, 512, 25), (32, 1024, 2048, 64), (32, 2561, 1024, 47), (32, 3073, 512, 64), (32, 200, 4608, 40),
    (32, 1025, 4608, 64), (32, 60, 14336, 33),
    (32, 300, 1056, 2), (32, 5009, 1056, 3), (32, 8209, 96, 4), (64, 200, 192, 2), (64, 200, 1088, 2),
    (64, 5009, 192, 2), (64, 5009, 576, 3), (64, 8209, 2048, 4), (64, 12289, 320, 3), (64, 12305, 4160, 3),
    (128, 200, 2176, 2), (128, 8209, 4224, 3), (128, 8209, 640, 4), (128, 12305, 640, 3)])
def test_small_batch_kernel_lines(rai, ora, gs, rows, cols, m):
    _both_calls(rai, ora, rows, cols, m, gs)


@pytest.mark.parametrize("hidden,ffn", [(1024, 2816), (1280, 1536), (2560, 5376)])
@pytest.mark.parametrize("m", [2, 3, 9, 24, 25, 40, 64])
def test_small_batch_layers_with_tiled_parameters(rai, ora, hidden, ffn, m):
    """Group 32, where a model also holds its parameters in 16-row tiles."""
    img = rai.synth_model(hidden, 1, hidden // 64, 2, 64, ffn, 400, 128, group_size=32, seed=m)
    gm, om = rai.RaiModel.from_bytes(img, max_groups=1024), ora.Model(img, 0)
    h = np.random.default_rng(m).normal(0.0, 1.0, (m, hidden)).astype(np.float32)
    got = gm.forward_batch(h, np.arange(m), gm.create_kv_cache(128))
    want = om.forward_batch(h, np.arange(m), om.create_kv(128))
    assert np.array_equal(_bits(got).reshape(-1), _bits(want).reshape(-1))


@pytest.mark.parametrize("gs", [32, 64, 128])
@pytest.mark.parametrize("m", [2, 9, 40, 100])
def test_small_batch_layers(rai, ora, gs, m):
    """The model path: norm, attention output, silu_mul and head activations
    in the streamed kernel's order."""
    img = rai.synth_model(1152, 2, 9, 3, 128, 1280, 400, 128, group_size=gs, seed=gs + m)
    gm, om = rai.RaiModel.from_bytes(img), ora.Model(img, 0)
    h = np.random.default_rng(m).normal(0.0, 1.0, (m, 1152)).astype(np.float32)
    got = gm.forward_batch(h, np.arange(m), gm.create_kv_cache(128))
    want = om.forward_batch(h, np.arange(m), om.create_kv(128))
    assert np.array_equal(_bits(got).reshape(-1), _bits(want).reshape(-1))
    gl, ol = gm.hidden_to_logits_batch(got, m), om.hidden_to_logits_batch(want, m)
    assert np.array_equal(_bits(gl).reshape(-1), _bits(ol).reshape(-1))


@pytest.mark.parametrize("m", [1, 3, 700, 1100])
def test_host_buffers_of_every_size(rai, m):
    """Hidden states through the pinned staging in one part, several parts and
    several chunks: the batch equals its halves run one after the other, the
    caller's array is left alone, and logits of a batch equal those of a row."""
    H, V = 1024, 30001
    img = rai.synth_model(H, 1, 8, 2, 128, 1024, V, 1200, group_size=64, seed=m)
    gm = rai.RaiModel.from_bytes(img)
    h = np.random.default_rng(m).normal(0.0, 1.0, (m, H)).astype(np.float32)
    keep = h.copy()
    got = gm.forward_batch(h, np.arange(m), gm.create_kv_cache(1200))
    assert np.array_equal(h, keep)
    kv, cut = gm.create_kv_cache(1200), max(1, m // 2)
    parts = [gm.forward_batch(h[a:b], np.arange(a, b), kv) for a, b in ((0, cut), (cut, m)) if b > a]
    assert np.array_equal(_bits(got), _bits(np.concatenate(parts)))
    n = min(m, 130)
    lg = gm.hidden_to_logits_batch(got[:n], n)
    for i in (0, n // 2, n - 1):
        assert np.array_equal(_bits(lg[i]), _bits(gm.hidden_to_logits(got[i])))


def test_logits_past_one_staging_piece(rai):
    """More than 16 MiB of logits in one call: several pieces through one block."""
    n, V = 64, 70001
    gm = rai.RaiModel.from_bytes(rai.synth_model(64, 1, 1, 1, 64, 64, V, 64, group_size=32, seed=1))
    h = np.random.default_rng(1).normal(0.0, 1.0, (n, 64)).astype(np.float32)
    lg = gm.hidden_to_logits_batch(h, n)
    for i in range(n):
        assert np.array_equal(_bits(lg[i]), _bits(gm.hidden_to_logits(h[i]))), i


def test_calls_on_several_threads(rai):
    """Five threads, each with its own model and cache, at once: forward_batch and
    logits through the two staging blocks, the copy threads and the direct
    copies, device-pointer products through the shared scratch blocks."""
    H, m, V = 1024, 600, 3001
    img = rai.synth_model(H, 1, 8, 2, 128, 1024, V, 1200, group_size=64, seed=9)

    def work(seed, models):
        gm = models[seed]
        r = np.random.default_rng(seed)
        h = r.normal(0.0, 1.0, (m, H)).astype(np.float32)
        out = []
        for it in range(4):
            n = m if it % 2 else 40
            y = gm.forward_batch(h[:n], np.arange(n), gm.create_kv_cache(1200))
            out += [y, gm.hidden_to_logits_batch(y[:33], 33)]
            for mm, gs, rows in ((1, 32, 300), (9, 64, 500), (70, 128, 900)):
                nib, params, x = gemv_operands(rows, 640, mm, gs, seed=seed + it)
                dev = rai.DeviceArray.from_host
                out.append(_call(rai, "rai_w4a8_matmul_dev", rai.DeviceArray(4 * mm * rows), dev(nib), dev(params),
                                 dev(x), rows, 640, mm, gs))
        return out

    n = 5
    models = [rai.RaiModel.from_bytes(img) for _ in range(n)]
    want = [work(i, models) for i in range(n)]
    with concurrent.futures.ThreadPoolExecutor(n) as ex:
        got = list(ex.map(lambda i: work(i, models), range(n)))
    for g, w in zip(got, want):
        assert all(np.array_equal(_bits(a), _bits(b)) for a, b in zip(g, w))


def test_rows_past_the_positions_come_back_unchanged(rai):
    """forward_batch of more rows than positions: the others are the input's."""
    gm = rai.RaiModel.from_bytes(rai.synth_model(256, 1, 4, 4, 64, 512, 100, 64, group_size=32, seed=3))
    h = np.random.default_rng(0).normal(0.0, 1.0, (5, 256)).astype(np.float32)
    want = gm.forward_batch(h[:3], np.arange(3), gm.create_kv_cache(64))
    for _ in range(8):  # so that fresh memory of this size is not the input by chance
        np.full_like(h, 7.0)
    got = gm.forward_batch(h, np.arange(3), gm.create_kv_cache(64))
    assert np.array_equal(_bits(got[:3]), _bits(want)) and np.array_equal(_bits(got[3:]), _bits(h[3:]))


@pytest.mark.parametrize("heads,kv,hd", [(4, 1, 64), (3, 3, 128), (6, 3, 64), (8, 1, 128), (5, 1, 64)])
@pytest.mark.parametrize("first,m", [(0, 16), (1, 17), (5, 33), (63, 64), (64, 161), (130, 300), (1, 530)])
def test_prefill_attention(rai, ora, heads, kv, hd, first, m):
    """Scores and PV on the matrix cores: token tiles of 16 with a remainder,
    position tiles of 64 that tokens see whole, in part or not at all, launches
    of 256 tokens, a cache filled before."""
    H = heads * hd
    img = rai.synth_model(H, 1, heads, kv, hd, 128, 64, 640, group_size=32, embed_group_size=32, seed=first + m)
    gm, om = rai.RaiModel.from_bytes(img), ora.Model(img, 0)
    h = np.random.default_rng(m).normal(0.0, 1.0, (first + m, H)).astype(np.float32)
    gk, ok = gm.create_kv_cache(640), om.create_kv(640)
    for a, b in ((0, first), (first, first + m)):
        if b > a:
            got = gm.forward_batch(h[a:b], np.arange(a, b), gk)
            want = om.forward_batch(h[a:b], np.arange(a, b), ok)
            assert np.array_equal(_bits(got).reshape(-1), _bits(want).reshape(-1)), (a, b)


# Query heads per kv head on both sides of the rule between the two PV kernels
# past 160 tokens (5, 6 / 2: matrix cores; 4, 8, 1: streamed in parts of 128),
# behind each softmax of long rows.
@pytest.mark.parametrize("heads,kv,hd", [(5, 1, 64), (6, 2, 128), (4, 1, 64), (8, 1, 64), (3, 3, 64)])
@pytest.mark.parametrize("first", [4101, 8300, 16500])
def test_prefill_attention_of_long_contexts(rai, ora, heads, kv, hd, first):
    H, m = heads * hd, 203
    cap = first + 2 * m
    img = rai.synth_model(H, 1, heads, kv, hd, 128, 64, cap, group_size=32, embed_group_size=32, seed=first)
    gm = rai.RaiModel.from_bytes(img)
    h = np.random.default_rng(first).normal(0.0, 1.0, (first + m, H)).astype(np.float32)
    whole, parts = gm.create_kv_cache(cap), gm.create_kv_cache(cap)
    for kvc in (whole, parts):
        gm.forward_batch(h[:first], np.arange(first), kvc)
    got = gm.forward_batch(h[first:], np.arange(first, first + m), whole)
    cuts = [(first, first + 101), (first + 101, first + m)]
    want = np.concatenate([gm.forward_batch(h[a:b], np.arange(a, b), parts) for a, b in cuts])
    assert np.array_equal(_bits(got), _bits(want))
    if first == 4101 and heads == 5:
        om = ora.Model(img, 0)
        ok = om.create_kv(cap)
        om.forward_batch(h[:first], np.arange(first), ok)
        want = om.forward_batch(h[first:], np.arange(first, first + m), ok)
        assert np.array_equal(_bits(got).reshape(-1), _bits(want).reshape(-1))


@pytest.mark.parametrize("gs", [32, 64, 128])
@pytest.mark.parametrize("rows,cols", [((1, 3, 17), 256), ((16401, 40, 40), 256), ((100, 530), 1152), ((70, 70), 4096),
                                       ((33, 34, 35), 4224)])
def test_fused_projections_of_unequal_rows(rai, ora, gs, rows, cols):
    """One launch for matrices of different heights (and K past it)."""
    lin = []
    for i, r in enumerate(rows):
        nib, params, x = gemv_operands(r, cols, 1, gs, seed=r + i)
        lin.append((nib, params, r, cols, gs))
    x = np.ascontiguousarray(x, np.float32).reshape(-1)
    got = rai.w4a8_fused_qkv(*lin, x) if len(rows) == 3 else rai.w4a8_fused_gate_up(*lin, x)
    for g, p in zip(got, lin):
        assert np.array_equal(_bits(g), _bits(ora.w4a8_matvec(p[0], p[1], x, p[2], p[3], p[4])))
