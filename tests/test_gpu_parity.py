"""GPU parity: the HIP path, called through the C ABI, against the CPU oracle on
the same seeded inputs.  Bar: bit-exact for everything integer (quantized
activations, block sums, int32 block dots, repacked bytes, fp16 decode) and
max-relative error <= 1e-3 on the f32 outputs (the tolerance the benchmark
definition states); the f32 checks also hold a much tighter engineering bound."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from antfly_amd import _lib, kernels, synth  # noqa: E402
from oracle import oracle as O  # noqa: E402
from tests import gpu_util as G  # noqa: E402

Q4, Q8 = _lib.TYPE_Q4_0, _lib.TYPE_Q8_0
RAW, PREP = _lib.LAYOUT_RAW, _lib.LAYOUT_PREPARED
TOL = 1e-3          # stated tolerance on scaled outputs (max-relative, fp32 accumulate)
TIGHT = 2e-5        # what f32 accumulation in a different order actually needs


def smoke_row(fmt, scale, value):
    hb = np.array([scale], dtype=np.float16).view(np.uint8)
    if fmt == Q8:
        return np.concatenate([hb, np.full(32, value, dtype=np.int8).view(np.uint8)])
    nib = (value + 8) & 0xF
    return np.concatenate([hb, np.full(16, nib | (nib << 4), dtype=np.uint8)])


def test_library_smokes():
    print("case: afhip_smoke_q8_0 / afhip_smoke_q4_0", flush=True)
    kernels.smokeQ8_0()
    kernels.smokeQ4_0()


@pytest.mark.parametrize("fmt", [Q8, Q4])
@pytest.mark.parametrize("layout", [RAW, PREP])
def test_reference_gpu_smoke_kat(kats, fmt, layout):
    k = kats["gpu_smoke"]
    print(f"case: gpu_smoke fmt={fmt} layout={layout}", flush=True)
    x = np.stack([np.arange(1, 33), -np.arange(1, 33)]).astype(np.float32)
    w = np.concatenate([smoke_row(fmt, r["scale"], r["value"]) for r in k["weight_rows"]])
    wd = G.prepare(fmt, w, 3, 32) if layout == PREP else G.to_dev(w)
    y = G.linear(fmt, layout, x, wd, 2, 32, 3)
    assert np.abs(y.reshape(-1) - np.array(k["expected"])).max() <= k["tolerance_abs"]


def test_q4_0_nibble_order_kat(kats):
    k = kats["q4_0_nibble_order"]
    blk = np.full(18, k["fill_byte"], dtype=np.uint8)
    blk[0:2] = np.array([k["scale_bits"]], dtype=np.uint16).view(np.uint8)
    blk[2], blk[3] = k["qs0"], k["qs1"]
    x = np.zeros((1, 32), dtype=np.float32)
    x[0, k["input_ones_at"]] = 1.0
    for layout in (RAW, PREP):
        wd = G.prepare(Q4, blk, 1, 32) if layout == PREP else G.to_dev(blk)
        y = G.linear(Q4, layout, x, wd, 1, 32, 1)
        assert abs(y[0, 0] - k["expected"]) <= k["tolerance_abs"]


def test_fp16_decode_all_bit_patterns_on_device():
    bits = np.arange(65536, dtype=np.uint16)
    src = G.to_dev(bits.view(np.int16))
    dst = torch.empty(65536, dtype=torch.float32, device=G.DEV)
    kernels.launchDecodeFp16(G.stream(), G.buf(dst), G.buf(src), 65536)
    torch.cuda.synchronize()
    got = dst.cpu().numpy()
    want = bits.view(np.float16).astype(np.float32)
    nan = np.isnan(want)
    assert np.array_equal(np.isnan(got), nan)
    assert np.array_equal(got[~nan].view(np.uint32), want[~nan].view(np.uint32))


@pytest.mark.parametrize("rows,in_dim", [(1, 32), (3, 256), (5, 14336), (8, 4096), (64, 4096)])
def test_activation_quantizer_bit_exact(rows, in_dim):
    print(f"case: quantize_activations rows={rows} in_dim={in_dim}", flush=True)
    x = synth.activations(100 + rows, rows, in_dim)
    x[0, :32] = 0.0                       # zero block -> scale 1, q 0
    if in_dim >= 64:
        x[rows - 1, 32:64] = [127.0, 0.5, -0.5, 1.5, -1.5, 126.5, -2.5] + [0.25] * 25  # ties
        x[rows - 1, -32:] *= 1e-30        # tiny magnitudes
    if in_dim >= 4096:
        # every half-integer and its two float neighbours, both signs: block max 127 makes
        # the scale and its reciprocal exactly 1, so these hit the rounding rule directly
        k = np.arange(0, 127, dtype=np.float32) + np.float32(0.5)
        edge = np.concatenate([k, np.nextafter(k, np.float32(0)), np.nextafter(k, np.float32(200)),
                               [0.49999997, 0.25, 126.99999, 127.0]]).astype(np.float32)
        edge = np.concatenate([edge, -edge])
        nblk = (edge.size + 30) // 31
        pad = np.zeros(nblk * 31, np.float32)
        pad[: edge.size] = edge
        blocks = np.concatenate([np.full((nblk, 1), 127.0, np.float32), pad.reshape(nblk, 31)], axis=1)
        x[0, 64 : 64 + blocks.size] = blocks.reshape(-1)
    qw, sw, sumw = O.quantize_activation_rows(x, rows, in_dim)
    xd = G.to_dev(x)
    q = torch.empty(rows * in_dim, dtype=torch.int8, device=G.DEV)
    s = torch.empty(rows * in_dim // 32, dtype=torch.float32, device=G.DEV)
    sums = torch.empty(rows * in_dim // 32, dtype=torch.int32, device=G.DEV)
    kernels.launchQuantizeActivations(G.stream(), G.buf(xd), rows, in_dim, G.buf(q), G.buf(s), G.buf(sums))
    torch.cuda.synchronize()
    assert np.array_equal(q.cpu().numpy().reshape(rows, in_dim), qw)
    assert np.array_equal(s.cpu().numpy().view(np.uint32).reshape(rows, -1), sw.view(np.uint32))
    assert np.array_equal(sums.cpu().numpy().reshape(rows, -1), sumw)


@pytest.mark.parametrize("fmt", [Q8, Q4])
@pytest.mark.parametrize("out_dim,in_dim", [(37, 160), (8, 4096), (5, 8224), (130, 32)])
def test_prepare_weight_is_a_pure_repack(fmt, out_dim, in_dim):
    w = synth.weights(fmt, 7, out_dim, in_dim)
    got = G.prepare(fmt, w, out_dim, in_dim).cpu().numpy()
    want = G.numpy_prepare(fmt, w, out_dim, in_dim)
    assert got.size == want.size == kernels.preparedWeightBytes(fmt, out_dim, in_dim)
    assert np.array_equal(got, want)


SHAPES_A = [  # (rows, in_dim, out_dim): all take the activation-quantized route
    (1, 4096, 512), (2, 96, 515), (3, 2048, 640), (4, 4096, 1024), (5, 1120, 513),
    (6, 256, 600), (7, 160, 777), (8, 4096, 512), (9, 256, 512), (17, 512, 530),
    (33, 96, 513), (64, 1056, 640), (130, 256, 1030), (257, 512, 512),
    (16, 14336, 512), (70, 8224, 520),  # long K on the MFMA kernel: many ring stages, a one-block last stage
    (8, 14336, 516), (7, 9216, 512),    # small batch with a long K: one launch with more than 128 KB of LDS
    # the decode kernel with the quantized activations awaited through a counter (several rows, or one long row, and
    # wavefronts that do not quantize): quantizers with a ragged last block set, every row count, one long row in
    # two and four K slices, a wide matrix (full-size workgroups)
    (2, 4096, 4100), (3, 4096, 2052), (4, 4096, 6144), (2, 1120, 3000), (4, 992, 8200), (1, 6144, 1030), (1, 14336, 2050),
    (2, 2080, 14336),
    # ... and the long-K kernel (K > 4096, two to seven rows, sixteen-wavefront workgroups): full and ragged last slice,
    # ragged columns, the most rows the counter form takes
    (2, 8192, 2048), (4, 9216, 4100), (3, 14336, 4096), (7, 8192, 4096), (5, 4128, 2100),
    (2, 14336, 2048), (2, 12288, 4100),  # (two rows take that kernel from K = 12288 on; below, the decode kernel with K slices)
    (2, 11008, 1030), (2, 6144, 4100),
    # (three and four rows on whole 256-value runs of K take the eight-row MFMA kernel where that measured faster; the
    # long-K kernel keeps a K that is not such a multiple, and three rows of Q4_0 on a long K and few columns)
    (4, 8224, 1030), (3, 6144, 2050), (4, 14336, 1030), (2, 14336, 4100), (3, 11008, 4096),
    # the single-shot MFMA kernel (5..64 rows): every count of live result registers, two row tiles, a K
    # that ends inside a wavefront's run of blocks, a second K share of one block, ragged columns
    (24, 4096, 544), (25, 2048, 512), (32, 4128, 513), (48, 320, 520), (12, 3072, 1000),
    # 65 to 128 rows on the tiled GEMM's 32 x 64 tiles: every row remainder of a tile, ragged columns, K ending inside a stage
    # (three row tiles of the single-shot kernel: test_sixty_five_to_ninety_six_rows)
    (70, 512, 8200), (128, 1056, 8192), (97, 256, 8224), (100, 512, 4700), (66, 1024, 6150),
    # the eight-row MFMA kernel (5..8 rows on a grid of at least a workgroup per compute unit): one live
    # wavefront and a ragged last tile; 64-column tiles, ragged; K shares with a short last share; a
    # wavefront with half its blocks
    (8, 512, 8200), (5, 4096, 12290), (7, 9216, 4112), (6, 256, 16416),
    # ... on 16-column tiles (4096 to 4608 columns and one K share): full, ragged last tile, one live wavefront
    (5, 4096, 4096), (8, 1024, 4600), (6, 256, 4100),
    # ... with the column count of a workgroup picked to spread the matrix evenly over the compute units: 56 of a
    # workgroup's 64 columns live (14336), 48 and 40 (three column groups; ragged last tile), 24 (two groups, 6144)
    (8, 512, 14336), (6, 1024, 11008), (5, 256, 10000), (7, 2048, 6144), (8, 256, 9000),
    (5, 8192, 7168),  # ... 56 columns with two K shares (Q4_0)
    # three and four rows on more columns than one round of the decode kernel's workgroups: Q4_0 takes the eight-row kernel
    (4, 256, 16448), (3, 256, 33000), (4, 4096, 28672), (4, 4096, 33000),  # (four rows of 4096 values: from two rounds on)
    (3, 2048, 14400), (4, 2048, 11040),  # ... and Q8_0 on wide matrices with K of 2048 to 4096
    # nine to 32 rows on 64-column tiles: every count of live result registers, ragged columns, one live
    # wavefront with half its blocks, K shares with a short last share
    (9, 512, 12290), (16, 4096, 12288), (17, 256, 12300), (24, 1024, 12352), (32, 512, 12290), (29, 9216, 12288),
    (33, 1024, 12352), (48, 512, 12290), (64, 4096, 12288),  # ... and two row tiles
    # ... on fewer columns, where the K shares fill the grid: four shares and the reduce launch, two shares adding to
    # the result themselves with a ragged last tile (Q4_0), two shares of Q8_0
    (16, 14336, 4096), (12, 8192, 8190), (20, 4096, 8192), (17, 512, 10250),
]


@pytest.mark.parametrize("fmt", [Q8, Q4])
@pytest.mark.parametrize("layout", [RAW, PREP])
@pytest.mark.parametrize("rows,in_dim,out_dim", SHAPES_A)
def test_block_dots_bit_exact_and_outputs_within_tolerance(fmt, layout, rows, in_dim, out_dim):
    print(f"case: route A fmt={fmt} layout={layout} rows={rows} in={in_dim} out={out_dim}", flush=True)
    assert O.uses_activation_quant(rows, in_dim, out_dim)
    x = synth.activations(rows * 1000 + in_dim, rows, in_dim)
    x[0, :32] = 0.0
    w = synth.weights(fmt, out_dim, out_dim, in_dim)
    wd = G.prepare(fmt, w, out_dim, in_dim) if layout == PREP else G.to_dev(w)
    dots = G.block_dots(fmt, layout, x, wd, rows, in_dim, out_dim)
    assert np.array_equal(dots, O.block_dots(fmt, x, w, rows, in_dim, out_dim))
    y = G.linear(fmt, layout, x, wd, rows, in_dim, out_dim)
    y64 = O.linear_act_f64(fmt, x, w, rows, in_dim, out_dim)
    for workers in (1, 8):  # every thread plan of the reference
        ref = O.linear_no_bias(fmt, x, w, rows, in_dim, out_dim, workers=workers)
        err = G.max_rel_err(y, ref.astype(np.float64))
        assert err <= TOL and err <= TIGHT, err
    assert G.max_rel_err(y, y64) <= TIGHT


@pytest.mark.parametrize("rows,in_dim,out_dim,same", [
    # one matrix and a pair on three row tiles of the single-shot kernel: K ending inside a wavefront's run of sixteen blocks,
    # the last K of one share, row and column remainders, the most columns of one round
    (96, 3104, 5500, True), (65, 4096, 5442, True), (70, 3328, 8190, True),
    # a pair there alone: in three rounds, and with a second K share that ends inside a run
    (66, 3104, 10753, False), (95, 5408, 5500, False),
    # ... and both on the GEMM: one step of rows, K or columns past each line
    (97, 3104, 5500, True), (66, 3072, 5500, True), (66, 4128, 5500, True), (66, 5376, 5500, True), (66, 3104, 5440, True),
    (66, 3104, 10752, True)])
def test_sixty_five_to_ninety_six_rows(rows, in_dim, out_dim, same):
    """Q4_0 either side of the lines between the single-shot kernel and the tiled GEMM, against 64-bit sums, with a bias and a
    residual too; a pair's halves have the bits of single calls but where only the pair takes the single-shot kernel."""
    print(f"case: 65 to 96 rows rows={rows} in={in_dim} out={out_dim}", flush=True)
    x = synth.activations(71 * rows + in_dim, rows, in_dim)
    wa, wb = synth.weights(Q4, out_dim, out_dim, in_dim), synth.weights(Q4, out_dim + 1, out_dim, in_dim)
    da, db = G.prepare(Q4, wa, out_dim, in_dim), G.prepare(Q4, wb, out_dim, in_dim)
    y64 = [O.linear_act_f64(Q4, x, w, rows, in_dim, out_dim) for w in (wa, wb)]
    single = [G.linear(Q4, PREP, x, d, rows, in_dim, out_dim) for d in (da, db)]
    for pair_half, one, want in zip(G.linear_pair(Q4, PREP, x, da, db, rows, in_dim, out_dim), single, y64):
        assert G.max_rel_err(one, want) <= TIGHT and G.max_rel_err(pair_half, want) <= TIGHT
        assert np.array_equal(pair_half, one) == same
    bias = synth.activations(72, 1, out_dim)[0]
    assert G.max_rel_err(G.linear_bias(Q4, PREP, x, da, bias, rows, in_dim, out_dim), y64[0] + bias) <= TIGHT
    biased = G.linear_pair_bias(Q4, PREP, x, da, bias, db, -bias, rows, in_dim, out_dim)
    assert G.max_rel_err(biased[0], y64[0] + bias) <= TIGHT and G.max_rel_err(biased[1], y64[1] - bias) <= TIGHT


@pytest.mark.parametrize("fmt", [Q8, Q4])
@pytest.mark.parametrize("rows,in_dim,out_dim", [
    # Q8_0 on 256 units: 128 x 128 tiles ...
    (700, 96, 4097), (700, 544, 4097), (700, 576, 4097), (700, 608, 4097),
    # ... and 64 x 64; the last has fewer 128 x 128 tiles a unit, but six columns of them on four of the eight XCDs
    (1100, 544, 3800), (129, 160, 16385), (257, 672, 10921), (1300, 192, 5630),
    # ... and 64 x 128: 33 to 64 rows on more columns than the single-shot kernel takes (Q4_0 stays on that)
    (64, 2080, 32780), (33, 2112, 32780), (49, 2144, 32769)])
def test_prefill_grids_past_the_compute_units(fmt, rows, in_dim, out_dim):
    """Grids that take the 64 x 128 (Q4_0), 64 x 64, 128 x 128 and 64 x 128 (Q8_0) tiles: row and column remainders, K shorter
    than the ring of four-block stages and ending one, two and three blocks into a stage; f32 sums in another order (TIGHT)."""
    print(f"case: large prefill fmt={fmt} rows={rows} in={in_dim} out={out_dim}", flush=True)
    x = synth.activations(rows + in_dim, rows, in_dim)
    w = synth.weights(fmt, out_dim + 1, out_dim, in_dim)
    y = G.linear(fmt, PREP, x, G.prepare(fmt, w, out_dim, in_dim), rows, in_dim, out_dim)
    assert G.max_rel_err(y, O.linear_act_f64(fmt, x, w, rows, in_dim, out_dim)) <= TIGHT


@pytest.mark.parametrize("fmt", [Q8, Q4])
@pytest.mark.parametrize("rows,in_dim,out_dim", [(97, 1024, 520), (130, 2048, 5632), (333, 1024, 4164), (1300, 512, 5632)])
def test_prefill_pair_in_one_launch(fmt, rows, in_dim, out_dim):
    """Gate and up of a prefill: each half is the single call, bit for bit, on grids that share K out (two launches and their
    sums), on one share and on each wide tile; tile counts that eight XCDs do not divide."""
    print(f"case: prefill pair fmt={fmt} rows={rows} in={in_dim} out={out_dim}", flush=True)
    x = synth.activations(911, rows, in_dim)
    wa, wb = synth.weights(fmt, 912, out_dim, in_dim), synth.weights(fmt, 913, out_dim, in_dim)
    da, db = G.prepare(fmt, wa, out_dim, in_dim), G.prepare(fmt, wb, out_dim, in_dim)
    ya, yb = G.linear_pair(fmt, PREP, x, da, db, rows, in_dim, out_dim)
    assert np.array_equal(ya, G.linear(fmt, PREP, x, da, rows, in_dim, out_dim))
    assert np.array_equal(yb, G.linear(fmt, PREP, x, db, rows, in_dim, out_dim))
    sample = np.r_[0:2, 31:33, rows - 1]
    for got, w in ((ya, wa), (yb, wb)):
        ref = O.linear_no_bias(fmt, x[sample], w, len(sample), in_dim, out_dim, workers=8)
        assert G.max_rel_err(got[sample], ref.astype(np.float64)) <= TIGHT


@pytest.mark.parametrize("fmt", [Q8, Q4])
@pytest.mark.parametrize("rows,in_dim,out_dim", [
    (700, 160, 4097), (257, 672, 10921), (130, 544, 4100),  # the large tiles and 32 x 64
    (130, 1056, 520)])                                      # ... with K shared out over workgroups
def test_prefill_keeps_small_activations(fmt, rows, in_dim, out_dim):
    """Rows scaled by the power of two that takes the smallest product of two scales just above 2^-126 give the same bits scaled:
    every product is a normal number and every sum a multiple of 2^-149, so nothing is rounded that is not in the row of ordinary
    size.  (Packed Q4_0 nibbles are sixteen times their value and the scale products a sixteenth, subnormal here.)"""
    print(f"case: small prefill activations fmt={fmt} rows={rows} in={in_dim} out={out_dim}", flush=True)
    rng = np.random.default_rng(17 * rows + in_dim)
    x = rng.uniform(-1.0, 1.0, (rows, in_dim)).astype(np.float32)
    x[:, ::32] = rng.uniform(1.0, 1.5, x[:, ::32].shape)  # every block's peak: all scales within a factor of three
    w = synth.weights(fmt, out_dim + 3, out_dim, in_dim)
    blocks = w.reshape(out_dim * in_dim // 32, -1)
    blocks[:, :2] = rng.uniform(2.0 ** -8, 2.0 ** -7, len(blocks)).astype(np.float16).view(np.uint8).reshape(-1, 2)
    down = 2.0 ** (-126 + 15)  # the smallest product of two scales is 2^-8 / 127
    x_small = x.copy()
    x_small[::3] = (x[::3].astype(np.float64) * down).astype(np.float32)
    x_small[5] = 0.0
    wd = G.prepare(fmt, w, out_dim, in_dim)
    y = G.linear(fmt, PREP, x, wd, rows, in_dim, out_dim)
    want = y.copy()
    want[::3] = (y[::3].astype(np.float64) * down).astype(np.float32)
    want[5] = 0.0
    assert np.array_equal(G.linear(fmt, PREP, x_small, wd, rows, in_dim, out_dim), want)


@pytest.mark.parametrize("rows,in_dim,out_dim,bias", [
    (77, 2048, 2048, False), (96, 2048, 5632, False), (65, 3584, 2001, False),  # a run a wavefront on one group of columns, on several; two
    (96, 4096, 6145, False), (66, 4096, 1000, True), (80, 4096, 1000, False),   # ... on several, two apart, two K shares
    (70, 14336, 1000, False), (90, 14336, 1000, True),                          # (the GEMM)
    (65, 768, 513, False), (96, 1024, 33001, False), (70, 1792, 9001, False)])  # four wavefronts on K: one run, two
def test_short_prompts_keep_small_activations(rows, in_dim, out_dim, bias):
    """65 to 96 rows of Q4_0: rows scaled by powers of two give the same bits scaled, from scale products just above 2^-126 (as
    test_prefill_keeps_small_activations) to activations of 2^100, and rows of one call do not feel each other.  Rows around 2^87
    whose parts of K differ by a factor of two cross the line above which a row's scales are divided by 16, in either order."""
    print(f"case: small activations, short prompts rows={rows} in={in_dim} out={out_dim} bias={bias}", flush=True)
    rng = np.random.default_rng(19 * rows + in_dim)
    x = rng.uniform(-1.0, 1.0, (rows, in_dim)).astype(np.float32)
    x[:, ::32] = rng.uniform(1.0, 1.5, x[:, ::32].shape)  # every block's peak: all scales within a factor of three
    w = synth.weights(Q4, out_dim + 3, out_dim, in_dim)
    blocks = w.reshape(out_dim * in_dim // 32, -1)
    blocks[:, :2] = rng.uniform(2.0 ** -8, 2.0 ** -7, len(blocks)).astype(np.float16).view(np.uint8).reshape(-1, 2)
    block = np.arange(in_dim) // 32
    doubled = [block // 8 % 2 == 1, 2 * block >= in_dim // 32, 2 * block < in_dim // 32]
    for i, part in enumerate(doubled):
        x[2 + i::6, part] *= 2.0
    factor = np.array([2.0 ** (-126 + 15), 2.0 ** 100, 2.0 ** 86, 2.0 ** 86, 2.0 ** 86, 1.0])[np.arange(rows) % 6]
    scaled = (x.astype(np.float64) * factor[:, None]).astype(np.float32)
    wd = G.prepare(Q4, w, out_dim, in_dim)
    if bias:
        y, got = (G.linear_bias(Q4, PREP, each, wd, np.zeros(out_dim, np.float32), rows, in_dim, out_dim) for each in (x, scaled))
    else:
        y, got = (G.linear(Q4, PREP, each, wd, rows, in_dim, out_dim) for each in (x, scaled))
    want = (y.astype(np.float64) * factor[:, None]).astype(np.float32)
    assert np.array_equal(got, want)
    for half in G.linear_pair(Q4, PREP, scaled, wd, wd, rows, in_dim, out_dim):
        assert np.array_equal(half, want)


def short_chain_sums(dots: np.ndarray, products: np.ndarray, shares: int, wavefronts: int) -> np.ndarray:
    """f32 sums over blocks (the last axis) of products * dots as K shares, runs of eight blocks a wavefront, even and odd blocks of a
    wavefront, then its four (and four) wavefronts make them.  (Fused multiply-adds in float64 rounded to f32: the product of 24 and 20
    bits is exact, a double rounding takes a tie of one in 2^29.)"""
    blocks = dots.shape[-1]
    share_blocks = (blocks + 8 * shares - 1) // (8 * shares) * 8
    total = None
    for begin in range(0, blocks, share_blocks):
        end = min(begin + share_blocks, blocks)
        waves = []
        for part in range(wavefronts):
            mine = [b for first in range(begin + 8 * part, end, 8 * wavefronts) for b in range(first, min(first + 8, end))]
            chains = []
            for odd in (0, 1):
                acc = np.zeros(dots.shape[:-1], np.float32)
                for b in mine[odd::2]:
                    acc = (products[..., b].astype(np.float64) * dots[..., b] + acc).astype(np.float32)
                chains.append(acc)
            waves.append(chains[0] + chains[1])
        halves = [((waves[i] + waves[i + 1]) + waves[i + 2]) + waves[i + 3] for i in range(0, wavefronts, 4)]
        share = halves[0] if wavefronts == 4 else halves[0] + halves[1]
        total = share if total is None else total + share
    return total


@pytest.mark.parametrize("rows,in_dim,out_dim,shares,wavefronts", [
    (77, 4096, 2048, 1, 8), (65, 3584, 2559, 1, 8), (96, 2304, 1500, 1, 8),  # two runs, one group of columns (a pair: two)
    (70, 6144, 700, 2, 8), (66, 4352, 1000, 2, 8), (80, 8192, 1279, 2, 8),   # ... on two K shares
    (77, 2048, 2730, 1, 4), (96, 1792, 8201, 1, 4),                          # ... of four wavefronts, several groups
    (77, 2048, 2048, 1, 8), (65, 768, 513, 1, 4)])                           # one run
def test_short_prompts_add_up_in_short_chains(rows, in_dim, out_dim, shares, wavefronts):
    """65 to 96 rows of Q4_0 where the GEMM shares K out: no chain of additions longer than eight blocks, bit for bit the sums in that
    order, from the plain call, a pair and a call with a bias."""
    print(f"case: short chains rows={rows} in={in_dim} out={out_dim}", flush=True)
    x = synth.activations(6100 + rows, rows, in_dim)
    w = [synth.weights(Q4, 6101 + i, out_dim, in_dim) for i in range(2)]
    wd = [G.prepare(Q4, each, out_dim, in_dim) for each in w]
    got = [G.linear(Q4, PREP, x, wd[0], rows, in_dim, out_dim)]
    got += [G.linear_pair(Q4, PREP, x, wd[1], wd[0], rows, in_dim, out_dim)[1]]
    got += [G.linear_bias(Q4, PREP, x, wd[0], np.zeros(out_dim, np.float32), rows, in_dim, out_dim)]
    sample, columns = np.r_[0, 31:34, rows - 1], np.r_[0:32, out_dim - 65:out_dim]
    _, row_scales, _ = O.quantize_activation_rows(x[sample], len(sample), in_dim)
    blocks = w[0].reshape(out_dim, -1, 18)[columns]
    scales = blocks[..., :2].copy().view(np.float16)[..., 0].astype(np.float32)
    want = short_chain_sums(O.block_dots(Q4, x[sample], blocks.reshape(-1), len(sample), in_dim, len(columns)),
                            row_scales[:, None, :] * scales[None], shares, wavefronts)
    for y in got:
        assert np.array_equal(y[np.ix_(sample, columns)], want)


SHAPES_B = [(1, 32, 3), (2, 64, 600), (3, 96, 11), (4, 4096, 100), (1, 64, 4096), (12, 128, 40)]


@pytest.mark.parametrize("fmt", [Q8, Q4])
@pytest.mark.parametrize("layout", [RAW, PREP])
@pytest.mark.parametrize("rows,in_dim,out_dim", SHAPES_B)
def test_f32_route_matches_oracle(fmt, layout, rows, in_dim, out_dim):
    print(f"case: route B fmt={fmt} layout={layout} rows={rows} in={in_dim} out={out_dim}", flush=True)
    assert not O.uses_activation_quant(rows, in_dim, out_dim)
    x = synth.activations(rows + in_dim, rows, in_dim)
    w = synth.weights(fmt, 3 * out_dim, out_dim, in_dim)
    wd = G.prepare(fmt, w, out_dim, in_dim) if layout == PREP else G.to_dev(w)
    y = G.linear(fmt, layout, x, wd, rows, in_dim, out_dim)
    ref = O.linear_no_bias(fmt, x, w, rows, in_dim, out_dim)
    dense = O.dequantize(fmt, w).reshape(out_dim, in_dim).astype(np.float64)
    y64 = x.astype(np.float64) @ dense.T
    assert G.max_rel_err(y, ref.astype(np.float64)) <= TIGHT
    assert G.max_rel_err(y, y64) <= TIGHT


@pytest.mark.parametrize("fmt", [Q8, Q4])
@pytest.mark.parametrize("rows,in_dim,out_dim", [(16, 2048, 256), (77, 544, 256), (17, 96, 511), (8, 512, 511), (9, 512, 457), (3, 64, 5000),
                                                 (1, 32, 4096), (300, 2048, 511), (2100, 64, 70),
                                                 # either side of the lines: 4096 outputs up to K = 512, 4864 at 704, 6144 from 1024 on
                                                 (16, 512, 256), (39, 512, 105), (19, 704, 256), (16, 704, 304), (24, 1024, 256),
                                                 (24, 4096, 256), (23, 4096, 267)])
def test_f32_route_on_many_outputs(fmt, rows, in_dim, out_dim):
    """From 4096 outputs on (6144 from K = 1024 on) the f32 route runs on the matrix cores: row and column remainders, K shorter than
    and not a multiple of what its wavefronts take together, one and four column tiles a workgroup; a pair is one launch with the
    bits of two calls.  Activations are split exactly and summed in f32, so the error is that of f32 sums (TIGHT), also next to
    10^6 times larger ones; an infinity stays in its row and reaches it as the reference's does."""
    print(f"case: f32 route rows={rows} in={in_dim} out={out_dim} fmt={fmt}", flush=True)
    assert not O.uses_activation_quant(rows, in_dim, out_dim)
    x = synth.activations(5 * rows + in_dim, rows, in_dim)
    x[rows // 2, ::7] *= 1e6
    x[0, :3] = [1e36, 1e-38, 0.0]  # (times a quant of 127 still finite in f32)
    wa, wb = synth.weights(fmt, 3 * out_dim, out_dim, in_dim), synth.weights(fmt, 3 * out_dim + 1, out_dim, in_dim)
    da, db = G.prepare(fmt, wa, out_dim, in_dim), G.prepare(fmt, wb, out_dim, in_dim)
    ya, yb = G.linear_pair(fmt, PREP, x, da, db, rows, in_dim, out_dim)
    for w, y in ((wa, ya), (wb, yb)):
        y64 = x.astype(np.float64) @ O.dequantize(fmt, w).reshape(out_dim, in_dim).astype(np.float64).T
        assert G.max_rel_err(y, y64) <= TIGHT
    assert np.array_equal(G.linear(fmt, PREP, x, da, rows, in_dim, out_dim), ya)
    assert np.array_equal(G.linear(fmt, PREP, x, db, rows, in_dim, out_dim), yb)
    x[rows - 1, 5] = np.inf
    y = G.linear(fmt, PREP, x, da, rows, in_dim, out_dim)
    with np.errstate(invalid="ignore"):
        want = x[-1].astype(np.float64) @ O.dequantize(fmt, wa).reshape(out_dim, in_dim).astype(np.float64).T
    assert np.array_equal(np.isnan(y[-1]), np.isnan(want)) and np.array_equal(np.isposinf(y[-1]), np.isposinf(want))
    assert np.array_equal(y[:-1], ya[:-1])


@pytest.mark.parametrize("fmt", [Q8, Q4])
@pytest.mark.parametrize("rows,in_dim,out_dim", [(48, 544, 256), (2100, 64, 70)])  # one and four column tiles a workgroup
def test_f32_route_keeps_small_activations(fmt, rows, in_dim, out_dim):
    """Activations near the bottom of f32's range, next to rows of ordinary size: below 2^-110 the last of an activation's three
    bf16 parts is a subnormal and leaves bits behind.  Largest outputs are about 2^-123 (2^-124 activations): subnormal roundings
    of 2^-150, one a block and sum, are 2^-26 of that each, 4e-7 for 17 blocks and 16 wavefront sums -- under TIGHT."""
    print(f"case: small activations rows={rows} in={in_dim} out={out_dim} fmt={fmt}", flush=True)
    x = synth.activations(9 * rows + in_dim, rows, in_dim)
    x[::3] *= np.float32(2.0 ** -116)
    x[1::3] = (x[1::3].astype(np.float64) * 2.0 ** -124).astype(np.float32)
    x[2, 3] = np.float32(1e-40)  # a lone one among ordinary values
    w = synth.weights(fmt, 3 * out_dim, out_dim, in_dim)
    y = G.linear(fmt, PREP, x, G.prepare(fmt, w, out_dim, in_dim), rows, in_dim, out_dim)
    y64 = x.astype(np.float64) @ O.dequantize(fmt, w).reshape(out_dim, in_dim).astype(np.float64).T
    assert G.max_rel_err(y, y64) <= TIGHT


@pytest.mark.parametrize("fmt", [Q8, Q4])
@pytest.mark.parametrize("rows", [6, 12])  # 12 rows forced onto the GEMV kernels: activations quantized by their own kernel
def test_forced_dispatch_kinds_agree(fmt, rows):
    """A plan may force any kernel family; all of them compute the same op."""
    in_dim, out_dim = 512, 640
    x = synth.activations(77, rows, in_dim)
    w = synth.weights(fmt, 78, out_dim, in_dim)
    wd = G.prepare(fmt, w, out_dim, in_dim)
    want = O.block_dots(fmt, x, w, rows, in_dim, out_dim)
    base = G.linear(fmt, PREP, x, wd, rows, in_dim, out_dim)
    for dispatch in (0, 1, 2, 3):
        assert np.array_equal(G.block_dots(fmt, PREP, x, wd, rows, in_dim, out_dim, dispatch), want)
        y = G.linear(fmt, PREP, x, wd, rows, in_dim, out_dim, dispatch)
        assert G.max_rel_err(y, base.astype(np.float64)) <= TIGHT


# ---- two matmuls that share X (linearNoBiasPair, ops/ops.zig:909) ----------------

PAIR_SHAPES = [  # rows, in_dim, out_dim: fused GEMV, small-batch GEMV with K slices, ragged columns, MFMA GEMM, f32 route
    (1, 4096, 1024), (2, 512, 514), (4, 2048, 640), (5, 8224, 513), (8, 4096, 512), (12, 256, 530), (40, 512, 640),
    (3, 64, 100), (20, 2048, 300),  # the last: MFMA GEMM with K shared out over workgroups, both matrices through one scratch
    (6, 512, 8200), (7, 9216, 4112),  # the eight-row MFMA kernel, one launch over both matrices; with K shares
    (20, 512, 12290),                 # the 32-row MFMA kernel on 64-column tiles, both matrices
    (4, 512, 8200), (3, 256, 16500),  # four and three rows whose two matrices together exceed one (two) rounds of the decode kernel
    (12, 9216, 520),                  # the eight-row kernel on two groups of eight rows (Q8_0; Q4_0 on a long K), both matrices
]


@pytest.mark.parametrize("fmt", [Q8, Q4])
@pytest.mark.parametrize("layout", [RAW, PREP])
@pytest.mark.parametrize("rows,in_dim,out_dim", PAIR_SHAPES)
def test_pair_equals_two_single_ops(fmt, layout, rows, in_dim, out_dim):
    """Each half of a pair is bit-identical to the single op on that matrix where both take the same kernel (and so
    equal to the oracle within the single op's bound), within that bound of it otherwise; the op is the engine's
    two-call fallback fused."""
    print(f"case: pair fmt={fmt} layout={layout} rows={rows} in={in_dim} out={out_dim}", flush=True)
    x = synth.activations(510 + rows, rows, in_dim)
    wa = synth.weights(fmt, 511, out_dim, in_dim)
    wb = synth.weights(fmt, 512, out_dim, in_dim)
    da = G.prepare(fmt, wa, out_dim, in_dim) if layout == PREP else G.to_dev(wa)
    db = G.prepare(fmt, wb, out_dim, in_dim) if layout == PREP else G.to_dev(wb)
    ya, yb = G.linear_pair(fmt, layout, x, da, db, rows, in_dim, out_dim)
    sa, sb = G.linear(fmt, layout, x, da, rows, in_dim, out_dim), G.linear(fmt, layout, x, db, rows, in_dim, out_dim)
    # Three and four rows of Q4_0: the pair's two matrices together may exceed one (two) rounds of the decode kernel's
    # workgroups (64 columns a compute unit, 256 units) where one matrix does not; the pair then runs on the eight-row
    # MFMA kernel and a single op on the decode kernel -- the same block dots, another f32 summation order.
    one_round = 256 * 64 * (1 if rows == 4 and rows * in_dim < 16384 else 2)
    routes_differ = (fmt == Q4 and layout == PREP and rows in (3, 4) and in_dim <= 4096 and in_dim % 256 == 0 and
                     out_dim <= one_round < 2 * out_dim)
    if routes_differ:
        assert G.max_rel_err(ya, sa.astype(np.float64)) <= TIGHT and G.max_rel_err(yb, sb.astype(np.float64)) <= TIGHT
    else:
        assert np.array_equal(ya, sa)
        assert np.array_equal(yb, sb)
    ref_b = O.linear_no_bias(fmt, x, wb, rows, in_dim, out_dim, workers=8)
    assert G.max_rel_err(yb, ref_b.astype(np.float64)) <= TIGHT


# ---- the benchmark configurations at full size ---------------------------------

FULL = [
    ("C1", Q8, [1], 4096, 4096),
    ("C4", Q8, [128, 512, 2048], 4096, 4096),
    ("C4-q4", Q4, [128], 4096, 4096),
    ("C2", Q4, [1, 2, 4, 8], 4096, 14336),
    ("C3", Q4, [1, 5], 14336, 4096),
    ("C5-qkv", Q4, [1, 5], 4096, 6144),   # the decode-step sweep: attention projections at one and five rows
    ("C5-o", Q4, [1, 5], 4096, 4096),
]
# element-wise relative error over outputs above 1e-3 of their row maximum (information; the gate
# is the row-normalised figure): collected here and printed by the last full-size case
ELEMENTWISE = {}


@pytest.mark.parametrize("name,fmt,row_list,in_dim,out_dim", FULL)
def test_full_size_decode_configs(name, fmt, row_list, in_dim, out_dim):
    w = synth.weights(fmt, 1234, out_dim, in_dim)
    wd = G.prepare(fmt, w, out_dim, in_dim)
    prepared = O.Prepared(fmt, w, out_dim, in_dim)
    for rows in row_list:
        print(f"case: {name} fmt={fmt} rows={rows} in={in_dim} out={out_dim}", flush=True)
        x = synth.activations(4321 + rows, rows, in_dim)
        y = G.linear(fmt, PREP, x, wd, rows, in_dim, out_dim)
        ref = prepared.linear(x, rows, workers=8)
        err = G.max_rel_err(y, ref.astype(np.float64))
        assert err <= TOL and err <= TIGHT, err
        ELEMENTWISE[(name, rows)] = G.elementwise_rel_err(y, ref.astype(np.float64))
        print(f"  row-normalised max-rel {err:.2e}, element-wise (|want| > 1e-3 row max) {ELEMENTWISE[(name, rows)]:.2e}", flush=True)
        assert ELEMENTWISE[(name, rows)] <= 100 * TOL  # cancellation near zero amplifies by at most 1/floor
        # block dots on a slice of output columns and rows (the full tensor is rows x out x in/32 ints)
        sub, rsub = 64, min(rows, 40)
        wsub = w[: sub * (in_dim // 32) * O.BLOCK_BYTES[fmt]]
        wsub_d = G.prepare(fmt, wsub, sub, in_dim)
        dots = G.block_dots(fmt, PREP, x[:rsub], wsub_d, rsub, in_dim, sub,
                            dispatch=-1 if rows <= 8 else 3)  # rows >= 9: the MFMA kernel
        assert np.array_equal(dots, O.block_dots(fmt, x[:rsub], wsub, rsub, in_dim, sub))
        # linearity in X is NOT a property of this op (activations are re-quantized);
        # scaling X by a power of two is: scales double, int8 values stay.
        y2 = G.linear(fmt, PREP, x * 2.0, wd, rows, in_dim, out_dim)
        assert np.array_equal(y2, y * 2.0)
    prepared.close()


@pytest.mark.parametrize("rows", [1, 5])
def test_full_size_gate_up_pair(rows):
    """The decode step's gate + up projections as the one pair call the engine makes
    (architectures/gpt.zig:5398-5440): each half bit-identical to the single op on that
    matrix, one half against the oracle."""
    in_dim, out_dim = 4096, 14336
    print(f"case: C5 pair rows={rows} in={in_dim} out={out_dim}", flush=True)
    x = synth.activations(8800 + rows, rows, in_dim)
    wa = synth.weights(Q4, 8801, out_dim, in_dim)
    wb = synth.weights(Q4, 8802, out_dim, in_dim)
    da, db = G.prepare(Q4, wa, out_dim, in_dim), G.prepare(Q4, wb, out_dim, in_dim)
    ya, yb = G.linear_pair(Q4, PREP, x, da, db, rows, in_dim, out_dim)
    assert np.array_equal(ya, G.linear(Q4, PREP, x, da, rows, in_dim, out_dim))
    assert np.array_equal(yb, G.linear(Q4, PREP, x, db, rows, in_dim, out_dim))
    prepared = O.Prepared(Q4, wb, out_dim, in_dim)
    ref = prepared.linear(x, rows, workers=8)
    prepared.close()
    err = G.max_rel_err(yb, ref.astype(np.float64))
    assert err <= TOL and err <= TIGHT, err


@pytest.mark.parametrize("fmt_name,fmt", [("q4_0", Q4), ("q8_0", Q8)])
@pytest.mark.parametrize("case,rows,in_dim,out_dim", [("k256_n64", 5, 256, 64), ("k96_n512", 5, 96, 512)])
def test_committed_tiny_vectors(fmt_name, fmt, case, rows, in_dim, out_dim):
    """The HIP path against tests/golden/tiny_vectors.npz (no oracle call): quantized activations,
    scales, sums and int32 block dots bit-exact, outputs within tolerance."""
    import os

    g = np.load(os.path.join(os.path.dirname(__file__), "golden", "tiny_vectors.npz"), allow_pickle=False)
    key = f"{fmt_name}_{case}_"
    x, w = g[key + "x"], g[key + "w_raw"]
    print(f"case: tiny vectors {key}", flush=True)
    xd = G.to_dev(x)
    q = torch.empty(rows * in_dim, dtype=torch.int8, device=G.DEV)
    s = torch.empty(rows * in_dim // 32, dtype=torch.float32, device=G.DEV)
    sums = torch.empty(rows * in_dim // 32, dtype=torch.int32, device=G.DEV)
    kernels.launchQuantizeActivations(G.stream(), G.buf(xd), rows, in_dim, G.buf(q), G.buf(s), G.buf(sums))
    torch.cuda.synchronize()
    assert np.array_equal(q.cpu().numpy().reshape(rows, in_dim), g[key + "qx"])
    assert np.array_equal(s.cpu().numpy().view(np.uint32).reshape(rows, -1), g[key + "sx"].view(np.uint32))
    assert np.array_equal(sums.cpu().numpy().reshape(rows, -1), g[key + "sumx"])
    for layout in (RAW, PREP):
        wd = G.prepare(fmt, w, out_dim, in_dim) if layout == PREP else G.to_dev(w)
        assert np.array_equal(G.block_dots(fmt, layout, x, wd, rows, in_dim, out_dim), g[key + "block_dots"])
        y = G.linear(fmt, layout, x, wd, rows, in_dim, out_dim)
        assert G.max_rel_err(y, g[key + "y_op"].astype(np.float64)) <= TIGHT


@pytest.mark.parametrize("fmt,rows,in_dim,out_dim,pair", [(Q4, 29, 9216, 12288, False), (Q8, 20, 2048, 12290, True),
                                                          (Q4, 20, 512, 12290, True), (Q4, 12, 8192, 12352, True), (Q4, 40, 8192, 12288, True)])
def test_thirty_two_row_kernel_with_k_shares_and_pairs(fmt, rows, in_dim, out_dim, pair):
    """On this chip the 32-row kernel's grid bound (one workgroup per compute unit) keeps launches with
    K shares or two matrices on the older kernel; with the bound lifted they take the 32-row kernel and
    must give what the older kernel gives to f32 summation order, and the oracle's result within its bound."""
    print(f"case: 32-row kernel, bound lifted fmt={fmt} rows={rows} in={in_dim} out={out_dim} pair={pair}", flush=True)
    x = synth.activations(5100 + rows, rows, in_dim)
    wa = synth.weights(fmt, 5101, out_dim, in_dim)
    da = G.prepare(fmt, wa, out_dim, in_dim)
    db = G.prepare(fmt, synth.weights(fmt, 5102, out_dim, in_dim), out_dim, in_dim) if pair else None

    def run():
        if pair:
            return G.linear_pair(fmt, PREP, x, da, db, rows, in_dim, out_dim)
        return (G.linear(fmt, PREP, x, da, rows, in_dim, out_dim),)

    older = run()
    _lib.lib().afhip_tune_batch32_max_workgroups(1000000)
    try:
        got = run()
    finally:
        _lib.lib().afhip_tune_batch32_max_workgroups(-1)
    ref = O.linear_no_bias(fmt, x, wa, rows, in_dim, out_dim, workers=8)
    err = G.max_rel_err(got[0], ref.astype(np.float64))
    assert err <= TOL and err <= TIGHT, err
    for a, b in zip(got, older):
        assert G.max_rel_err(a, b.astype(np.float64)) <= TIGHT
    if pair:  # each half of the pair equals the single op on that matrix, bit for bit
        _lib.lib().afhip_tune_batch32_max_workgroups(1000000)
        try:
            assert np.array_equal(got[0], G.linear(fmt, PREP, x, da, rows, in_dim, out_dim))
            assert np.array_equal(got[1], G.linear(fmt, PREP, x, db, rows, in_dim, out_dim))
        finally:
            _lib.lib().afhip_tune_batch32_max_workgroups(-1)



@pytest.mark.parametrize("fmt,rows,in_dim,out_dim,pair,same", [
    (Q4, 9, 256, 512, False, False), (Q4, 16, 512, 513, True, False), (Q4, 17, 2304, 4095, False, False),  # few columns: one run, two
    (Q4, 32, 4096, 4096, True, False), (Q4, 25, 5632, 2050, True, False), (Q4, 12, 11008, 4096, False, False),  # ... and long K
    (Q4, 64, 14336, 2047, True, False), (Q4, 31, 2048, 8191, True, False), (Q4, 33, 256, 8223, True, False),
    (Q4, 32, 4096, 6145, False, True), (Q4, 16, 3328, 33000, False, True), (Q4, 33, 4096, 4097, True, True),  # column groups
    (Q4, 63, 4096, 14337, True, True), (Q4, 64, 1280, 32001, True, True), (Q4, 9, 2048, 65505, False, True),
    (Q4, 64, 1280, 33001, True, False), (Q4, 65, 2048, 2047, False, False), (Q4, 96, 2048, 5633, True, False),  # ... beyond 64 rows
    (Q4, 77, 4096, 6143, True, True), (Q4, 95, 3584, 10999, True, True), (Q4, 70, 14336, 1000, True, False),
    (Q4, 96, 1024, 33001, True, False), (Q4, 65, 768, 513, True, False),
    (Q8, 17, 256, 545, False, False), (Q8, 17, 1024, 4096, True, False), (Q8, 33, 4096, 1023, True, False),
    (Q8, 48, 1024, 4095, True, False), (Q8, 32, 2048, 8191, False, True), (Q8, 20, 1024, 14000, False, True),
])
def test_column_groups_of_the_thirty_two_row_kernel(fmt, rows, in_dim, out_dim, pair, same):
    """32 rows a workgroup on one and more groups of columns, at the edges of row tiles, column tiles, runs and shares of K: the
    oracle's result, the bits of the kernel it stands in for where the sums have its order (`same`), a pair's halves those of single
    calls, and a call with a bias (two runs in one share) or one whose result lies over X those of the plain call."""
    print(f"case: column groups fmt={fmt} rows={rows} in={in_dim} out={out_dim} pair={pair}", flush=True)
    x = synth.activations(5300 + rows, rows, in_dim)
    w = [synth.weights(fmt, 5301 + i, out_dim, in_dim) for i in range(2 if pair else 1)]
    wd = [G.prepare(fmt, each, out_dim, in_dim) for each in w]
    single = [G.linear(fmt, PREP, x, each, rows, in_dim, out_dim) for each in wd]
    got = G.linear_pair(fmt, PREP, x, wd[0], wd[1], rows, in_dim, out_dim) if pair else single
    _lib.lib().afhip_tune_batch32_max_workgroups(0)
    try:
        older = [G.linear(fmt, PREP, x, each, rows, in_dim, out_dim) for each in wd]
    finally:
        _lib.lib().afhip_tune_batch32_max_workgroups(-1)
    for one, half, old in zip(single, got, older):
        assert np.array_equal(one, half)
        assert np.array_equal(one, old) if same else G.max_rel_err(one, old.astype(np.float64)) <= TIGHT
    zeros = np.zeros(out_dim, np.float32)
    assert np.array_equal(G.linear_bias(fmt, PREP, x, wd[0], zeros, rows, in_dim, out_dim), single[0])
    ws = torch.empty(max(kernels.workspaceBytes(fmt, rows, in_dim, out_dim), 16), dtype=torch.uint8, device=G.DEV)
    room = torch.full((rows * (in_dim + out_dim),), float("nan"), dtype=torch.float32, device=G.DEV)
    room[:rows * in_dim] = torch.from_numpy(x.ravel()).to(G.DEV)
    kernels.launchLinearF32(G.stream(), fmt, PREP, G.buf(room[:rows * out_dim]), G.buf(room[:rows * in_dim]), G.buf(wd[0]), rows, in_dim,
                            out_dim, G.buf(ws))
    torch.cuda.synchronize()
    assert np.array_equal(room[:rows * out_dim].cpu().numpy(), single[0].ravel())
    if 64 < rows < 77:  # a caller that lends what the tiled GEMM needs, and less than the shape's workspace, gets the GEMM
        xd, y = G.to_dev(x), torch.full((rows * out_dim,), float("nan"), dtype=torch.float32, device=G.DEV)
        least = (rows * in_dim + 255) // 256 * 256 + rows * (in_dim // 32) * 8
        assert least < ws.numel()
        ws[least:] = 0xA5  # what is not lent (the column-group kernel's operands, of whole row groups, reach into it)
        kernels.launchLinearF32(G.stream(), fmt, PREP, G.buf(y), G.buf(xd), G.buf(wd[0]), rows, in_dim, out_dim, G.buf(ws[:least]))
        torch.cuda.synchronize()
        assert bool((ws[least:] == 0xA5).all())
        assert G.max_rel_err(y.cpu().numpy().reshape(rows, out_dim), single[0].reshape(rows, out_dim).astype(np.float64)) <= TIGHT
    ref = O.linear_no_bias(fmt, x, w[-1], rows, in_dim, out_dim, workers=8)
    assert G.max_rel_err(got[-1], ref.astype(np.float64)) <= TIGHT


@pytest.mark.parametrize("fmt,rows,in_dim,out_dim,pair", [
    (Q4, 5, 4096, 4096, False), (Q4, 8, 256, 4100, False), (Q4, 7, 1280, 6152, False), (Q4, 6, 3840, 12290, True),
    (Q4, 4, 2048, 16400, False), (Q8, 8, 2048, 4096, False), (Q8, 5, 256, 8200, True), (Q8, 7, 1792, 14336, False),
    (Q8, 6, 4096, 11008, False), (Q8, 8, 3328, 9000, False), (Q8, 3, 4096, 28672, False),
])
def test_eight_row_kernel_quantizes_like_its_quantizer_launch(fmt, rows, in_dim, out_dim, pair):
    """One K share: the workgroups quantize X themselves, unless the result overlaps X -- then the quantizer's launch runs first.
    The two must give the same bits: odd row counts, wavefronts with some or none of their blocks, every tile width, with zero
    blocks, ties, huge and tiny values, infinities and NaNs in X."""
    print(f"case: eight-row kernel's own quantizer fmt={fmt} rows={rows} in={in_dim} out={out_dim} pair={pair}", flush=True)
    x = synth.activations(4200 + rows, rows, in_dim)
    x[0, 32:64] = 0.0
    x[1, :32] = np.arange(32) - 15.5
    x[1, 31] = 127.0
    x[rows - 1, 64:96] *= 1e30
    x[rows - 1, 96:128] *= 1e-38
    x[rows - 1, 128:160] = 1e-45
    x[2, 160:164] = [np.nan, np.inf, -np.inf, 1.0]  # (row 2 alone: the other rows stay numbers)
    x[2, 192:196] = np.nan
    wd = [G.prepare(fmt, synth.weights(fmt, 4300 + i, out_dim, in_dim), out_dim, in_dim) for i in range(2 if pair else 1)]
    ws = torch.empty(max(kernels.workspaceBytes(fmt, rows, in_dim, out_dim), 16), dtype=torch.uint8, device=G.DEV)

    def run(overlap):
        both = torch.full((rows * (in_dim + out_dim),), float("nan"), dtype=torch.float32, device=G.DEV)
        at = 0 if overlap else rows * in_dim  # the (first) result: X's own place, or behind it
        both[:rows * in_dim] = torch.from_numpy(x.ravel()).to(G.DEV)
        xd, y = both[:rows * in_dim], both[at:at + rows * out_dim]
        second = torch.full((rows * out_dim,), float("nan"), dtype=torch.float32, device=G.DEV)
        if pair:
            kernels.launchLinearPairF32(G.stream(), fmt, PREP, G.buf(y), G.buf(second), G.buf(xd), G.buf(wd[0]), G.buf(wd[1]), rows, in_dim,
                                        out_dim, G.buf(ws))
        else:
            kernels.launchLinearF32(G.stream(), fmt, PREP, G.buf(y), G.buf(xd), G.buf(wd[0]), rows, in_dim, out_dim, G.buf(ws))
        torch.cuda.synchronize()
        return y.cpu().numpy().view(np.uint32), second.cpu().numpy().view(np.uint32)

    apart, over = run(False), run(True)
    assert np.array_equal(apart[0], over[0])
    if pair:
        assert np.array_equal(apart[1], over[1])
    y = apart[0].view(np.float32).reshape(rows, out_dim)
    keep = [r for r in range(rows) if r != 2]
    ref = O.linear_no_bias(fmt, x[keep], synth.weights(fmt, 4300, out_dim, in_dim), len(keep), in_dim, out_dim, workers=8)
    assert G.max_rel_err(y[keep], ref.astype(np.float64)) <= TIGHT


@pytest.mark.parametrize("fmt", [Q8, Q4])
@pytest.mark.parametrize("rows,in_dim,out_dim,pair", [(77, 2048, 2048, False), (97, 1024, 1000, True), (129, 1056, 1541, False),
                                                      (161, 3040, 512, True), (400, 1088, 520, False)])
def test_two_k_shares_of_the_prefill_gemm_add_to_the_result(fmt, rows, in_dim, out_dim, pair):
    """A plain call of two K shares clears the result in the quantizer's launch and adds both shares to it.  Whatever the result
    held before, it must be what the reduce launch gives (a call with a bias of zeros, and one whose result overlaps X)."""
    print(f"case: two K shares added fmt={fmt} rows={rows} in={in_dim} out={out_dim} pair={pair}", flush=True)
    x = synth.activations(611, rows, in_dim)
    w = [synth.weights(fmt, 612 + i, out_dim, in_dim) for i in range(2 if pair else 1)]
    wd = [G.prepare(fmt, each, out_dim, in_dim) for each in w]
    want = [G.linear_bias(fmt, PREP, x, each, np.zeros(out_dim, np.float32), rows, in_dim, out_dim) for each in wd]
    ws = torch.empty(max(kernels.workspaceBytes(fmt, rows, in_dim, out_dim), 16), dtype=torch.uint8, device=G.DEV)
    room = torch.full((rows * (in_dim + out_dim),), float("nan"), dtype=torch.float32, device=G.DEV)
    second = torch.full((rows * out_dim,), float("nan"), dtype=torch.float32, device=G.DEV)
    for at in (rows * in_dim, rows * in_dim, 0):  # behind X, once more on the first results, in X's place
        room[:rows * in_dim] = torch.from_numpy(x.ravel()).to(G.DEV)
        xd, y = room[:rows * in_dim], room[at:at + rows * out_dim]
        if pair:
            kernels.launchLinearPairF32(G.stream(), fmt, PREP, G.buf(y), G.buf(second), G.buf(xd), G.buf(wd[0]), G.buf(wd[1]), rows, in_dim,
                                        out_dim, G.buf(ws))
        else:
            kernels.launchLinearF32(G.stream(), fmt, PREP, G.buf(y), G.buf(xd), G.buf(wd[0]), rows, in_dim, out_dim, G.buf(ws))
        torch.cuda.synchronize()
        for got, ref in zip((y, second), want):
            assert np.array_equal(got.cpu().numpy().reshape(rows, out_dim), ref)
    sample = np.r_[0:2, rows - 1]
    ref = O.linear_no_bias(fmt, x[sample], w[0], len(sample), in_dim, out_dim, workers=8)
    assert G.max_rel_err(want[0][sample], ref.astype(np.float64)) <= TIGHT


@pytest.mark.parametrize("fmt", [Q8, Q4])
@pytest.mark.parametrize("rows,in_dim,out_dim", [(77, 2048, 250), (33, 1056, 257), (70, 1088, 500), (530, 1312, 130), (2100, 64, 500),
                                                 (1030, 1024, 510), (18, 5152, 490), (130, 96, 500)])
def test_f32_route_tiles_and_runs_of_blocks(fmt, rows, in_dim, out_dim):
    """One column tile (loads exchanged through LDS) and four: runs of one to eleven blocks a wavefront, the last ones short or
    empty, ragged rows and columns.  Each half of a pair is the single call to the bit, whichever tile each of them takes."""
    print(f"case: f32 route tiles fmt={fmt} rows={rows} in={in_dim} out={out_dim}", flush=True)
    x = synth.activations(711, rows, in_dim)
    x[rows // 2, in_dim // 2:] *= 1e-37  # values that three bf16 parts do not hold
    wa, wb = synth.weights(fmt, 712, out_dim, in_dim), synth.weights(fmt, 713, out_dim, in_dim)
    da, db = G.prepare(fmt, wa, out_dim, in_dim), G.prepare(fmt, wb, out_dim, in_dim)
    ya, yb = G.linear_pair(fmt, PREP, x, da, db, rows, in_dim, out_dim)
    assert np.array_equal(ya, G.linear(fmt, PREP, x, da, rows, in_dim, out_dim))
    assert np.array_equal(yb, G.linear(fmt, PREP, x, db, rows, in_dim, out_dim))
    sample = np.r_[0:2, rows // 2, rows - 2:rows]
    for got, w in ((ya, wa), (yb, wb)):
        ref = O.linear_no_bias(fmt, x[sample], w, len(sample), in_dim, out_dim, workers=8)
        assert G.max_rel_err(got[sample], ref.astype(np.float64)) <= TIGHT


@pytest.mark.parametrize("fmt", [Q8, Q4])
@pytest.mark.parametrize("rows,in_dim,out_dim", [(168, 352, 187), (40, 512, 200), (671, 672, 292), (1090, 1120, 305), (530, 3616, 250),
                                                 (520, 4640, 257), (460, 544, 490)])
def test_f32_route_runs_of_unequal_length(fmt, rows, in_dim, out_dim):
    """Runs of one, two and more blocks a wavefront, some one block longer than the others, on one column tile and on four."""
    test_f32_route_tiles_and_runs_of_blocks(fmt, rows, in_dim, out_dim)
