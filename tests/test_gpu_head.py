"""GPU parity of the streaming row-chain GEMVs and what uses them, against
the oracle on identical inputs, bit for bit:

* the vocabulary head, the reference's per-row fmaf chain
  (head_logits_block, src/dsv4/dsv4_model.c:7221-7255), at its full shape
  (129280 x 4096 BF16, about 1 GiB) for one token and for 3- and 64-token
  verify batches (head_logits_block_batch, :7257-7308), then the greedy token
  of every row (src/cli/dsv4_run.c:357-359, NaN and tie edges included);
* dsv4_gemv_bf16_batch at the batch sizes of each kernel instance;
* dsv4_gemv_fp8 / _tbl at the FP8 matvec benchmark's shape (2048 x 4096,
  fp32 absmax block scales, fp32 x);
* expert_forward (src/dsv4/dsv4_model.c:6289-6345) at the model's expert
  shape, with and without a route weight."""
import numpy as np
import pytest

from common import bf16_bits, bf16_input, expert_slot, make_layer, pyoracle, same_bits

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def env():
    import torch
    import dsv4_gpu
    return dict(torch=torch, lib=dsv4_gpu.lib(), orc=pyoracle.Oracle(),
                dev=torch.device("cuda:0"))


def T(env, a):
    a = np.ascontiguousarray(a)
    if a.dtype == np.uint16:
        a = a.view(np.int16)
    return env["torch"].from_numpy(a.copy()).to(env["dev"])


def H(t):
    return t.detach().cpu().numpy()


def cli_greedy(row):
    """src/cli/dsv4_run.c:357-359 restated: best = 0; v wins if strictly
    greater."""
    best = 0
    for v in range(1, row.shape[0]):
        if row[v] > row[best]:
            best = v
    return best


def cli_greedy_fast(row):
    """The same rule vectorised: 0 when row[0] is NaN, else the first index of
    the largest non-NaN value (pinned against cli_greedy below)."""
    if np.isnan(row[0]):
        return 0
    m = np.nanmax(row)
    return int(np.flatnonzero(row == m)[0])


def test_vocab_head_full_size_and_greedy(env):
    orc, lib, torch = env["orc"], env["lib"], env["torch"]
    vocab, hid = 129280, 4096
    rng = np.random.default_rng(2)
    W = bf16_bits(rng.standard_normal((vocab, hid), dtype=np.float32) * 0.02)
    h = bf16_input(rng, (3, hid))
    Wd, hd = T(env, W), T(env, h)
    one = H(lib.gemv_bf16(hd[0:1], Wd, hid, vocab, 0))[0]
    assert same_bits(one, orc.gemv_bf16(h[0], W, hid, vocab, 0))
    three = H(lib.gemv_bf16(hd, Wd, hid, vocab, 0))
    for t in range(3):
        assert same_bits(three[t], orc.gemv_bf16(h[t], W, hid, vocab, 0)), t
    idx = H(lib.argmax(torch.from_numpy(three).to(env["dev"])))
    for t in range(3):
        assert idx[t] == cli_greedy_fast(three[t]), t
    # 64 tokens (a verify batch; the batched row chains): every token equal to
    # its own one-token head, three of them to the oracle
    h64 = bf16_input(rng, (64, hid))
    h64d = T(env, h64)
    b64 = H(lib.gemv_bf16(h64d, Wd, hid, vocab, 0))
    for t in range(64):
        assert same_bits(b64[t], H(lib.gemv_bf16(h64d[t:t + 1], Wd, hid, vocab, 0))[0]), t
    for t in (0, 37, 63):
        assert same_bits(b64[t], orc.gemv_bf16(h64[t], W, hid, vocab, 0)), t
    del Wd


def test_greedy_edges(env):
    lib, torch = env["lib"], env["torch"]
    rng = np.random.default_rng(4)
    rows = [rng.standard_normal(1000).astype(np.float32) for _ in range(6)]
    rows[1][[17, 500, 999]] = 9.0                 # ties: the first wins
    rows[2][0] = np.nan                           # logits[0] NaN: 0
    rows[3][[3, 40]] = np.nan
    rows[3][41] = 50.0                            # NaNs never taken
    rows[4][:] = -np.inf
    rows[4][700] = -1e30                          # all -inf but one
    rows[5][:] = 0.0
    rows[5][::2] = -0.0                           # signed zeros compare equal
    L = np.stack(rows)
    for r in L:
        assert cli_greedy(r) == cli_greedy_fast(r)
    got = H(lib.argmax(torch.from_numpy(L).to(env["dev"])))
    assert [int(g) for g in got] == [cli_greedy(r) for r in L]


@pytest.mark.parametrize("rows,in_,batch", [(300, 1024, 5), (300, 1024, 9), (1000, 256, 33),
                                            (64, 4096, 2), (200, 4096, 5), (130, 4096, 71),
                                            (64, 2048, 40), (100, 1024, 20), (77, 4096, 3),
                                            (300, 1000, 3), (50, 2056, 9)])
def test_bf16_batch_instances(env, rows, in_, batch):
    """Every kernel form: for in a multiple of 64, the matrix unit's chains in
    runs of up to 64 tokens (71 = 64 + 7, ragged token and row tiles);
    for other in, the x-in-LDS row chains (x up to 64 KB) and the
    one-row-per-(row, token) fallback."""
    orc, lib = env["orc"], env["lib"]
    rng = np.random.default_rng(rows + batch)
    W = bf16_bits(rng.standard_normal((rows, in_), dtype=np.float32) * 0.05)
    x = rng.standard_normal((batch, in_)).astype(np.float32)
    for ro in (0, 1):
        y = H(lib.gemv_bf16(T(env, x), T(env, W), in_, rows, ro))
        for t in range(batch):
            assert same_bits(y[t], orc.gemv_bf16(x[t], W, in_, rows, ro)), (t, ro)


def test_fp8_matvec_benchmark_shape(env):
    """W N(0, 0.02) quantised per 128x128 block with fp32 absmax/448 scales,
    x fp32 N(0, 1): both float-scale chains, every row."""
    orc, lib = env["orc"], env["lib"]
    rng = np.random.default_rng(0)
    w = (rng.standard_normal((2048, 4096)) * 0.02).astype(np.float32)
    codes, scales = orc.quant_fp8_blocks_absmax(w)
    x = rng.standard_normal(4096).astype(np.float32)
    gx, gc, gs = T(env, x), T(env, codes), T(env, scales)
    assert same_bits(H(lib.gemv_fp8_float(gx, gc, gs, 4096, 2048, 128, 0)),
                     orc.gemv_fp8_legacy(x, codes, scales, 4096, 2048, 128))
    assert same_bits(H(lib.gemv_fp8_float(gx, gc, gs, 4096, 2048, 128, 1)),
                     orc.gemv_fp8_tbl(x, codes, scales, 4096, 2048, 128))


def test_expert_forward_full_size(env):
    orc, lib, torch = env["orc"], env["lib"], env["torch"]
    L = make_layer(orc, 4096, 2048, 2, 1, seed=12)
    scales, weights = expert_slot(L, 1)
    slot = np.concatenate([scales, weights])
    rng = np.random.default_rng(3)
    x = bf16_input(rng, (1, 4096))
    qx, qs = orc.quant_fp8_act(x)
    gslot = T(env, slot)
    gqx, gqs = T(env, qx[0]), T(env, qs[0])
    for w in (None, 0.3712):
        out = torch.empty(4096, dtype=torch.float32, device=env["dev"])
        gw = None if w is None else torch.tensor([w], dtype=torch.float32, device=env["dev"])
        lib.expert_forward(out, gqx, gqs, gslot, L["scale_run"], 4096, 2048, 10.0, gw)
        ref = orc.expert_forward(qx[0], qs[0], scales, weights, 4096, 2048, 10,
                                 1.0 if w is None else w)
        assert same_bits(H(out), ref), w


@pytest.mark.parametrize("hidden,inter", [(256, 128), (1024, 384), (2048, 4096)])
def test_expert_forward_shapes(env, hidden, inter):
    """The two-launch expert_forward (gate/up with the SwiGLU epilogue, then the
    down rows with the requant folded in) at other shapes: an inter that is not
    a multiple of 512 and the widest inter the fused path takes."""
    orc, lib, torch = env["orc"], env["lib"], env["torch"]
    L = make_layer(orc, hidden, inter, 2, 1, seed=hidden + inter)
    scales, weights = expert_slot(L, 0)
    slot = np.concatenate([scales, weights])
    rng = np.random.default_rng(inter)
    x = bf16_input(rng, (1, hidden))
    qx, qs = orc.quant_fp8_act(x)
    out = torch.empty(hidden, dtype=torch.float32, device=env["dev"])
    gw = torch.tensor([0.618], dtype=torch.float32, device=env["dev"])
    lib.expert_forward(out, T(env, qx[0]), T(env, qs[0]), T(env, slot), L["scale_run"], hidden,
                       inter, 10.0, gw)
    ref = orc.expert_forward(qx[0], qs[0], scales, weights, hidden, inter, 10, 0.618)
    assert same_bits(H(out), ref)


@pytest.mark.parametrize("vocab", [1, 2, 3, 4, 5, 7, 255, 256, 257, 1023, 1024, 1025, 4095, 4097,
                                   16383, 16384, 16385, 32767, 32768, 32769, 32771, 129280])
def test_greedy_row_lengths(env, vocab):
    """Rows around the 4-value loads, the sizes where more waves or loads begin
    (256, 1024, 16384) and the rounds of 4096 and 32768 values, rows that start
    at any float (stride = an odd vocab), the maximum at the first, the last
    and a clamped position, ties across the clamp, and rows of -inf and NaN."""
    lib, torch = env["lib"], env["torch"]
    rng = np.random.default_rng(vocab)
    L = np.round(rng.standard_normal((7, vocab)) * 4).astype(np.float32)  # many ties
    L[1, vocab - 1] = 99.0
    L[2, 0] = 99.0
    L[3, max(0, vocab - 3):] = 99.0
    L[4, :] = -np.inf
    L[5, :] = -np.inf
    L[5, vocab // 2:] = np.nan
    L[6, :] = np.nan
    got = H(lib.argmax(torch.from_numpy(L).to(env["dev"])))
    assert [int(g) for g in got] == [cli_greedy_fast(r) for r in L]


@pytest.mark.parametrize("kind", ["wide", "subnormal", "cancel"])
def test_f32_mfma_is_fma_chain(env, kind):
    """The batched rows run their chains on the fp32 matrix unit, four columns
    an instruction: the same bits as the host's fmaf chain where every step
    rounds (exponents over 2^-40..2^40), where terms and sums are subnormal,
    and where the sum cancels."""
    orc, lib = env["orc"], env["lib"]
    rng = np.random.default_rng(17)
    rows, in_, batch = 70, 192, 19
    W = rng.standard_normal((rows, in_)).astype(np.float32)
    x = rng.standard_normal((batch, in_)).astype(np.float32)
    if kind == "wide":
        W = np.ldexp(W, rng.integers(-20, 21, W.shape))
        x = np.ldexp(x, rng.integers(-20, 21, x.shape))
    elif kind == "subnormal":
        W = np.ldexp(W, rng.integers(-80, -60, W.shape))
        x = np.ldexp(x, rng.integers(-80, -60, x.shape))
    else:
        x[:, 1::2] = -x[:, ::2]
        W[:, 1::2] = W[:, ::2]
    W = bf16_bits(W.astype(np.float32))
    x = x.astype(np.float32)
    y = H(lib.gemv_bf16(T(env, x), T(env, W), in_, rows, 0))
    for t in range(batch):
        assert same_bits(y[t], orc.gemv_bf16(x[t], W, in_, rows, 0)), t


@pytest.mark.parametrize("rows,batch", [(16384, 64), (32768 + 5, 4), (65537, 49), (129280, 17),
                                        (129280, 48), (16384, 33), (130, 128), (1, 16),
                                        (114688, 2), (114689, 2), (114689, 65), (114689, 66)])
def test_bf16_batch_row_tiles(env, rows, batch, in_=192):
    """1, 2 and 4 row tiles per wave by the number of rows, 1 to 4 token tiles,
    ragged in both, runs of 64, an odd number of 64-column steps: every token
    equal to its one-token result, and the last row's to the host's chain.
    A few tokens of many rows take the tiled chains."""
    orc, lib, torch, dev = env["orc"], env["lib"], env["torch"], env["dev"]
    g = torch.Generator(device=dev)
    g.manual_seed(rows + batch)
    W = (torch.randn(rows, in_, generator=g, device=dev) * 0.05).to(torch.bfloat16) \
        .view(torch.int16).contiguous()
    x = torch.randn(batch, in_, generator=g, device=dev)
    y = lib.gemv_bf16(x, W, in_, rows, 0)
    for t in range(batch):
        one = lib.gemv_bf16(x[t:t + 1].contiguous(), W, in_, rows, 0)[0]
        assert torch.equal(y[t].view(torch.int32), one.view(torch.int32)), t
        last = orc.gemv_bf16(H(x[t]), H(W[-1:]).view(np.uint16), in_, 1, 0)
        assert same_bits(H(y[t, -1:]), last), t


@pytest.mark.parametrize("rows,in_,batch", [(17, 64, 4), (16384, 128, 1), (16384, 192, 1),
                                            (16385, 64, 8), (16385, 128, 3), (16385, 192, 3),
                                            (40000, 192, 4), (40000, 256, 68), (40000, 320, 2), (40000, 384, 2),
                                            (70000, 512, 1), (82000, 128, 8), (82000, 128, 7),
                                            (82000, 576, 65), (98305, 768, 3), (98305, 1024, 2)])
def test_bf16_narrow_rows(env, rows, in_, batch):
    """Both sides of the rule between the tiled chains (1, 2, 3, 4 or 8 tokens,
    whole batches and what a run of 64 leaves) and the matrix unit's, by the
    number of rows and their width."""
    test_bf16_batch_row_tiles(env, rows, batch, in_)


@pytest.mark.parametrize("rows,in_,block", [(1, 1024, 128), (5, 1040, 16), (130, 4096, 128),
                                            (67, 4080, 32), (33, 2064, 48), (16, 1008, 16),
                                            (12, 4112, 16), (2600, 1040, 128), (2700, 1040, 128),
                                            (3500, 1040, 16), (6600, 4096, 128), (6700, 4096, 128),
                                            (8300, 4064, 48)])
def test_fp8_split_rows(env, rows, in_, block):
    """The split product chains (rows of 1024 to 4096 columns, ragged last
    segments, groups and workgroups, small blocks), the widths just outside and
    the numbers of rows from which a lane takes a whole row."""
    orc, lib = env["orc"], env["lib"]
    rng = np.random.default_rng(rows + in_)
    codes = rng.integers(0, 256, (rows, in_)).astype(np.uint8)
    codes[(codes & 0x7F) == 0x7F] = 0
    scales = (rng.random(((rows + block - 1) // block, (in_ + block - 1) // block)) + 0.01) \
        .astype(np.float32)
    for x in (rng.standard_normal(in_).astype(np.float32),
              np.ldexp(rng.standard_normal(in_), rng.integers(-30, 30, in_)).astype(np.float32)):
        for mode, ref in ((0, orc.gemv_fp8_legacy), (1, orc.gemv_fp8_tbl)):
            y = H(lib.gemv_fp8_float(T(env, x), T(env, codes), T(env, scales), in_, rows, block,
                                     mode))
            assert same_bits(y, ref(x, codes, scales, in_, rows, block)), mode


@pytest.mark.parametrize("kind", ["zeros", "growing", "ones", "cancelling", "power_of_two",
                                  "subnormal", "huge", "steps", "ties", "sparse",
                                  "overflow", "infinite"])
def test_fp8_split_values(env, kind):
    """Sums whose segments do not follow from their guesses (as
    test_hc_pre_split_chain_values): every row bit-exact. "overflow": the first
    product, then terms below half a step that the chain loses and a guess
    counts, then one that takes the guess past the fp32 range and the chain
    just below it, in both signs; "infinite": sums that leave it."""
    orc, lib = env["orc"], env["lib"]
    rows, in_ = 12, 4096
    rng = np.random.default_rng(23)
    w = (rng.standard_normal((rows, in_)) * 0.02).astype(np.float32)
    x = rng.standard_normal(in_).astype(np.float32)
    k = np.arange(in_)
    if kind == "zeros":
        x[:] = 0
    elif kind == "growing":
        x, w = np.exp2(k / 200.0).astype(np.float32), np.abs(w)
    elif kind == "ones":
        x[:], w[:] = 1, 1
    elif kind == "cancelling":
        x[1::2], w[:, 1::2] = -x[::2], w[:, ::2]
    elif kind == "power_of_two":
        w[:] = 1
        x = (x * 1e-7).astype(np.float32)
        x[0] = 1
    elif kind == "subnormal":
        x = np.ldexp(x, -140).astype(np.float32)
    elif kind == "huge":
        x = np.ldexp(x, 125).astype(np.float32)
    elif kind == "steps":
        x[:] = np.where((k // 300) % 2 == 0, 1.0, -1.0)
        w = np.sign(w) * 0.25 + 0.5
    elif kind == "ties":  # half a step of the sum's grid at every column
        w[:] = 1
        x[:] = 2.0 ** -24
        x[0] = 1.0
        x[2000:] *= -1
    elif kind == "overflow":
        x[:] = 0
        x[0], x[1:600] = 1.5 * 2.0 ** 126, 0.4 * 2.0 ** 103
        x[in_ - 20] = 2.0 ** 127 + 2.0 ** 125 - 2.0 ** 110
    elif kind == "infinite":
        x[:] = np.where(k % 900 < 450, 2.0 ** 122, -2.0 ** 122)
        x[k > 3000] = 2.0 ** 126
    else:
        x[rng.random(in_) < 0.98] = 0
    codes, scales = orc.quant_fp8_blocks_absmax(w.astype(np.float32))
    if kind in ("power_of_two", "ties", "overflow", "infinite"):
        scales[:] = 1.0 / 448.0 * 448.0
        codes[:] = 0x38  # 1.0
    if kind == "overflow":
        codes[rows // 2:] = 0xB8  # -1.0
        assert np.isfinite(orc.gemv_fp8_legacy(x, codes, scales, in_, rows, 128)).all()
    for mode, ref in ((0, orc.gemv_fp8_legacy), (1, orc.gemv_fp8_tbl)):
        y = H(lib.gemv_fp8_float(T(env, x), T(env, codes), T(env, scales), in_, rows, 128, mode))
        assert same_bits(y, ref(x, codes, scales, in_, rows, 128)), mode
