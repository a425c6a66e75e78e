"""The many-row GEMM (gemm_tile.hip) through lkhip_matmul at the edges of its
tiles and of the rule that picks them, against a float64 product of the
oracle's dequantized weights.  Bound: every product of a 32-column block is
exact, the block sums and the sums over blocks round in f32, so an output is
off by at most (K / 32 + 40) * 2^-24 of the sum of |terms| (40: a block's own
32 sums, the operand split's 2^-22, bias and scale)."""
import numpy as np
import pytest

import oracle
from lokal_amd import Engine, synth
from lokal_amd import kernels as K
from lokal_amd._lib import check, lib
from lokal_amd.config import ModelConfig

pytestmark = pytest.mark.gpu

CASES = [  # type, output rows, columns, activation rows
    (synth.Q8_0, 6061, 64, 33),       # the fewest rows and columns; ragged outputs
    (synth.Q8_0, 1553, 960, 131),     # an odd number of 64-column stages, ragged both ways
    (synth.Q8_0, 200001, 32, 40),     # 32 columns: the general kernel (no whole stage)
    (synth.Q8_0, 32741, 64, 65),      # 64 x 64 tiles
    (synth.Q8_0, 131009, 64, 34),     # 128 x 64 tiles
    (synth.Q8_0, 700, 4864, 300),     # K split over 8-wave blocks
    (synth.F16, 3001, 608, 70),       # a half stage at the end
    (synth.F16, 33000, 96, 67),
    (synth.F16, 131072, 32, 33),
    (synth.F16, 900, 1504, 250),
    (synth.Q4_K, 4001, 256, 50),      # the smallest K
    (synth.Q4_K, 32751, 256, 64),
    (synth.Q4_K, 131007, 256, 33),
    (synth.Q4_K, 1041, 2816, 257),    # an odd number of super-blocks, split
    (synth.Q6_K, 6061, 256, 33),      # 16-column groups of scales (and, Q5_K, mins)
    (synth.Q6_K, 1553, 768, 131),
    (synth.Q6_K, 131007, 256, 33),
    (synth.Q5_K, 32751, 256, 64),
    (synth.Q5_K, 1041, 2816, 257),
    (synth.Q8_0, 4101, 832, 131),     # two wave groups, 13 stages between them
    (synth.Q6_K, 4101, 256, 131),
    (synth.Q8_0, 905, 192, 250),      # four wave groups for three stages
    (synth.Q4_K, 1041, 1792, 380),    # four wave groups, a deep K
    (synth.F16, 1041, 1504, 380),     # one group, a deep K
    (synth.Q8_0, 11771, 960, 17),     # one row of tiles: the fewest rows
    (synth.Q8_0, 16401, 1088, 32),
    (synth.Q4_K, 32001, 256, 24),
    (synth.Q6_K, 11265, 768, 31),
    (synth.F16, 12293, 608, 18),
    (synth.F16, 1100, 4000, 200),     # F16's K split over 8-wave blocks, and below its size
    (synth.F16, 1090, 4000, 160),
    (synth.Q8_0, 8193, 2048, 32),     # one row of tiles, a deep K: the fewest blocks, and fewer
    (synth.Q8_0, 8100, 2048, 32),
    (synth.Q8_0, 1553, 6208, 131),    # rows too wide for the conversion to hold, read twice
    (synth.Q4_K, 1553, 6400, 131),
]


@pytest.mark.parametrize("t,rows,cols,n", CASES)
def test_matmul_tiles_match_float64(t, rows, cols, n):
    data = synth.gen_weight(t, 11, f"w{rows}x{cols}", rows, cols).data
    ref = oracle.dequant_row(t, data, rows * cols).reshape(rows, cols).astype(np.float64)
    rng = np.random.default_rng(rows + cols + n)
    x = rng.standard_normal((n, cols)).astype(np.float32)
    x[1] = 0.0                  # a row of zeros
    x[2] *= np.float32(1e-30)   # rows far from 1, and one of mixed magnitudes
    x[3] *= np.float32(1e30)
    x[4, ::3] *= np.float32(1e-9)
    x[5] = 0.0                  # one-hot: the weight column, bit for bit
    x[5, cols - 1] = 1.0
    bias = rng.standard_normal(rows).astype(np.float32)
    ldx, ldy = cols + 4, rows + 3
    xp = np.full((n, ldx), 7.0, np.float32)
    xp[:, :cols] = x
    w = K.Weight(t, rows, cols, data)
    xd, bd = K.DeviceArray.from_numpy(xp), K.DeviceArray.from_numpy(bias)
    y = K.DeviceArray((n, ldy))
    y.upload(np.full((n, ldy), 3.0, np.float32))
    K.matmul(w, xd, n, y, ldx=ldx, ldy=ldy)
    got = y.numpy()
    assert np.all(got[:, rows:] == 3.0)
    assert np.array_equal(got[5, :rows], ref[:, cols - 1].astype(np.float32))
    want = x.astype(np.float64) @ ref.T
    scale = np.abs(x).astype(np.float64) @ np.abs(ref).T
    bar = (cols / 32 + 40) * 2.0 ** -24
    assert np.max(np.abs(got[:, :rows] - want) / (scale + 1e-300)) < bar
    # accumulate, and a bias
    K.matmul(w, xd, n, y, bias=bd, accumulate=True, ldx=ldx, ldy=ldy)
    twice = y.numpy()[:, :rows]
    assert np.max(np.abs(twice - (2 * want + bias)) / (2 * scale + np.abs(bias) + 1e-300)) < bar


MARKED = [  # a shape of each tile, and of a K split, per type
    (synth.Q6_K, 6061, 256, 33), (synth.Q6_K, 131007, 256, 33), (synth.Q6_K, 1041, 2816, 257),
    (synth.Q6_K, 11265, 768, 31), (synth.Q5_K, 32751, 256, 64), (synth.Q5_K, 1041, 2816, 257),
    (synth.Q8_0, 1553, 960, 131), (synth.Q8_0, 32741, 64, 65), (synth.Q8_0, 700, 4864, 300),
    (synth.F16, 3001, 608, 70), (synth.F16, 33000, 96, 67), (synth.F16, 1100, 4000, 200),
    (synth.Q4_K, 4001, 256, 50), (synth.Q4_K, 32751, 256, 64), (synth.Q4_K, 1041, 2816, 257),
    (synth.Q8_0, 1553, 6208, 131), (synth.Q4_K, 1553, 6400, 131),
]


@pytest.mark.parametrize("t,rows,cols,n", MARKED)
def test_matmul_rows_beyond_the_planes(t, rows, cols, n):
    """Rows that two f16 planes of one scale cannot hold: a large element 2^18 to
    2^100 above the rest, which meets weights of exactly zero in some outputs, and
    infinities.  Finite outputs are off by at most (128 + K / 128 + 2) * 2^-24 of
    the sum of |terms| (f32 sums over a 128-column chunk, then over chunks);
    infinities and NaN are those of the f32 products, and rows beside them keep
    the planes' bound."""
    data = synth.gen_weight(t, 11, f"w{rows}x{cols}", rows, cols).data.copy()
    blk, size = synth.BLK[t]
    raw = data.view(np.uint8).reshape(rows, cols // blk, size)
    if t in (synth.Q4_K, synth.Q5_K):
        raw[..., 2:4] = 0           # no mins: a quant of 0 is a weight of 0
    big = cols - 3
    if t == synth.F16:
        raw[::3, big] = 0
    if t == synth.Q8_0:
        raw[::3, big // 32, 2 + big % 32] = 0
    ref = oracle.dequant_row(t, data, rows * cols).reshape(rows, cols).astype(np.float64)
    assert (ref[:, big] == 0).any()
    rng = np.random.default_rng(rows + cols + n)
    x = rng.standard_normal((n, cols)).astype(np.float32)
    for i, e in enumerate((18, 20, 22, 26, 30, 40, 60, 100)):
        x[1 + i, big] = np.float32(2.0 ** e)
    x[9, np.arange(cols) % 16 != 0] *= np.float32(2.0 ** -30)
    infs = {10: [(big, np.inf)], 11: [(1, -np.inf)], 12: [(big, np.inf), (5, np.inf)],
            13: [(big, np.inf), (5, -np.inf)], n - 1: [(cols - 1, np.inf)]}
    for r, at in infs.items():
        for k, v in at:
            x[r, k] = v
    x[14, 7] = np.nan
    w, y = K.Weight(t, rows, cols, data), K.DeviceArray((n, rows))
    K.matmul(w, K.DeviceArray.from_numpy(x), n, y)
    got = y.numpy()
    for r, at in infs.items():
        with np.errstate(invalid="ignore"):
            want = sum(v * ref[:, k] for k, v in at)
        assert np.array_equal(got[r], want.astype(np.float32), equal_nan=True), r
    assert np.isnan(got[14]).all()
    f = [r for r in range(n) if r not in infs and r != 14]
    want, scale = x[f].astype(np.float64) @ ref.T, np.abs(x[f]).astype(np.float64) @ np.abs(ref).T
    err = np.abs(got[f] - want) / (scale + 1e-300)
    mark = [i for i, r in enumerate(f) if 1 <= r <= 9]
    assert np.max(err[mark]) < (130 + cols / 128) * 2.0 ** -24
    assert np.max(np.delete(err, mark, 0)) < (cols / 32 + 40) * 2.0 ** -24


@pytest.mark.parametrize("h,heads,kv,inter,n,t,v", [
    (256, 4, 4, 2048, 133, synth.Q8_0, None), (1024, 16, 8, 512, 401, synth.Q4_K, synth.Q6_K),
    (2048, 32, 4, 512, 100, synth.Q6_K, None), (448, 7, 1, 2048, 130, synth.F16, None),
])
def test_prompt_rows_beyond_the_planes(h, heads, kv, inter, n, t, v):
    """Norm gains that leave one value in sixteen 2^30 above the others: the norm's planes do not hold
    it, and the products read the floats it writes beside them.  Within the model
    tests' 1e-3 of the oracle."""
    cfg = ModelConfig(h, inter, 2, heads, kv, 4096, 1e-5, 1e4)
    tensors = synth.synth_model(cfg, t, 5, tied=True, type_of=lambda _, p: v if v and p == "v_proj" else t)
    for x in tensors:
        if "norm" in x.name:
            g = x.data.view(np.float32)
            g[np.arange(g.size) % 16 != 0] *= np.float32(2.0 ** -30)
    eng, om = Engine.from_tensors(cfg, tensors), oracle.Model(cfg, tensors)
    toks = np.random.default_rng(h).integers(0, cfg.vocab_size, n).astype(np.uint32)
    s, s2, o = eng.session(n, kv_dtype="f32"), eng.session(n, kv_dtype="f32"), om.session(n)
    want = [o.forward(int(x), i) for i, x in enumerate(toks)]
    got = list(s.forward_batch(toks[:65], 0)) + [s2.prefill(toks)]
    for g, w in zip(got, want[:65] + want[-1:]):
        assert np.max(np.abs(g - w)) < 1e-3 * np.max(np.abs(w))
    for x in (s, s2, o, eng, om):
        x.close()


def test_matmul_smallest_normal_rows():
    """Rows down to the smallest normal numbers keep their 24 bits in the operand
    planes: weights of up to 2032, so that the results are normal too (a sum that
    cancels below that rounds at 2^-150)."""
    rows, cols, n = 6061, 64, 33
    rng = np.random.default_rng(2)
    q = rng.integers(-127, 128, (rows, cols // 32, 32)).astype(np.int8)
    blocks = np.empty((rows, cols // 32, 34), np.uint8)
    blocks[..., :2] = np.frombuffer(np.float16(16).tobytes(), np.uint8)
    blocks[..., 2:] = q.view(np.uint8)
    ref = 16.0 * q.reshape(rows, cols).astype(np.float64)
    x = ((1 + rng.random((n, cols))) * rng.choice([-1, 1], (n, cols)) * 2.0 ** -rng.integers(110, 127, (n, 1)))
    x = x.astype(np.float32)
    w, y = K.Weight(synth.Q8_0, rows, cols, blocks.reshape(-1)), K.DeviceArray((n, rows))
    K.matmul(w, K.DeviceArray.from_numpy(x), n, y)
    want, scale = x.astype(np.float64) @ ref.T, np.abs(x).astype(np.float64) @ np.abs(ref).T
    assert np.all(np.abs(y.numpy() - want) <= (cols / 32 + 40) * 2.0 ** -24 * scale + 2.0 ** -150)


@pytest.mark.parametrize("rows,n,ldy", [
    (32741, 64, 68_300_001),   # 64-row tiles: row 63 starts past 2^32 floats
    (6301, 32, 138_700_003),   # 32-row tiles: row 31 does
])
def test_matmul_output_rows_past_2_pow_32_floats(rows, n, ldy):
    """An output row stride at which the rows of one tile lie more than 2^32
    floats apart: every row is stored, and accumulated, in its own place."""
    cols = 64
    data = synth.gen_weight(synth.Q8_0, 11, f"w{rows}x{cols}", rows, cols).data
    w = K.Weight(synth.Q8_0, rows, cols, data)
    x = np.random.default_rng(n).standard_normal((n, cols)).astype(np.float32)
    xd, y, small = K.DeviceArray.from_numpy(x), K.DeviceArray(((n - 1) * ldy + rows,)), K.DeviceArray((n, rows))
    K.matmul(w, xd, n, small)
    K.matmul(w, xd, n, y, ldy=ldy)
    K.matmul(w, xd, n, y, accumulate=True, ldy=ldy)
    want = small.numpy()
    got = np.empty(rows, np.float32)
    for r in range(n):
        check(lib().lkhip_memcpy_dtoh(got.ctypes.data, y.ptr.value + 4 * r * ldy, got.nbytes))
        assert np.array_equal(got, 2 * want[r]), r
    y.free()


@pytest.mark.parametrize("h,heads,kv,inter,n,t,v", [
    (256, 4, 4, 512, 273, synth.Q8_0, None),          # one wave per row in the norm that writes the operand planes
    (448, 7, 1, 512, 353, synth.F16, None),           # a row that ends inside a 128-column chunk
    (1024, 16, 8, 512, 401, synth.Q4_K, synth.Q6_K),  # q / k / v of two types read the same planes
    (2048, 32, 4, 512, 100, synth.Q8_0, None),
    (4096, 64, 8, 512, 65, synth.Q4_K, None),         # the widest model the engine takes
    (1024, 16, 2, 4864, 24, synth.Q8_0, None),        # gate / up of few rows, 32 x 32 tiles
    (256, 4, 4, 4096, 31, synth.Q4_K, None),
    (448, 7, 1, 4000, 30, synth.F16, None),
    (512, 8, 2, 4352, 25, synth.Q6_K, None),
    (256, 4, 2, 16640, 17, synth.Q8_0, None),         # more of them than CUs
    (448, 7, 1, 4000, 40, synth.F16, None),           # F16 gate / up: four wave groups,
    (448, 7, 1, 4000, 150, synth.F16, None),          # one with more blocks than CUs,
    (448, 7, 1, 4000, 300, synth.F16, None),          # 64 x 64 tiles
    (512, 8, 2, 2048, 60, synth.Q6_K, None),          # Q6_K / Q5_K gate / up: two wave groups, K split over the grid,
    (512, 8, 2, 4352, 50, synth.Q5_K, None),          # not split,
    (512, 8, 2, 4352, 250, synth.Q6_K, None),         # 64 x 64 tiles
])
def test_prompt_through_planes_matches_oracle(h, heads, kv, inter, n, t, v):
    """A prompt, and every position's logits of its first 65, of a two-layer
    model, ragged row tiles included; within the model tests' 1e-3."""
    cfg = ModelConfig(h, inter, 2, heads, kv, 4096, 1e-5, 1e4)
    tensors = synth.synth_model(cfg, t, 5, tied=True, type_of=lambda _, p: v if v and p == "v_proj" else t)
    eng, om = Engine.from_tensors(cfg, tensors), oracle.Model(cfg, tensors)
    toks = np.random.default_rng(h).integers(0, cfg.vocab_size, n).astype(np.uint32)
    s, s2, o = eng.session(n, kv_dtype="f32"), eng.session(n, kv_dtype="f32"), om.session(n)
    want = [o.forward(int(x), i) for i, x in enumerate(toks)]
    got = list(s.forward_batch(toks[:65], 0)) + [s2.prefill(toks)]
    for g, w in zip(got, want[:65] + want[-1:]):
        assert np.max(np.abs(g - w)) < 1e-3 * np.max(np.abs(w))
    for x in (s, s2, o, eng, om):
        x.close()


@pytest.mark.parametrize("h,heads,kv,vocab,n,t", [
    (256, 4, 4, 16385, 17, synth.Q4_K),   # the fewest rows
    (512, 8, 2, 12001, 32, synth.Q8_0),   # below the rows of gemm16_wide_kernel
    (448, 7, 1, 11999, 29, synth.F16),
    (512, 8, 2, 12500, 24, synth.Q6_K),
])
def test_lm_head_of_few_rows_reads_the_norms_planes(h, heads, kv, vocab, n, t):
    """A vocabulary large enough that the lm_head over 17-32 rows multiplies the
    operand planes that the final norm writes: every position's logits within
    the model tests' 1e-3 of the oracle."""
    cfg = ModelConfig(h, 512, 2, heads, kv, vocab, 1e-5, 1e4)
    tensors = synth.synth_model(cfg, t, 5, tied=True)
    eng, om = Engine.from_tensors(cfg, tensors), oracle.Model(cfg, tensors)
    toks = np.random.default_rng(h).integers(0, vocab, n).astype(np.uint32)
    s, o = eng.session(n, kv_dtype="f32"), om.session(n)
    for i, g in enumerate(s.forward_batch(toks, 0)):
        w = o.forward(int(toks[i]), i)
        assert np.max(np.abs(g - w)) < 1e-3 * np.max(np.abs(w)), i
    for x in (s, o, eng, om):
        x.close()
