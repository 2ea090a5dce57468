"""GPU parity of the caller step around the MoE layer: rmsnorm_bf16,
dsv4_hc_split, hc_pre (+ the fused RMSNorm), hc_post and the whole FFN half
of a decoder layer (dsv4g_ffn_step), all bit-exact against the oracle on the
same inputs, including the sums of squares that land exactly on a float
rounding midpoint (settled by the kernels' sequential fallback)."""
from __future__ import annotations

import os
import time

import numpy as np
import pytest

from common import ROOT, bf16_bits, bf16_input, bf16_values, make_layer, pyoracle, same_bits

pytestmark = pytest.mark.gpu

TINY = os.path.join(ROOT, "tests", "golden", "tiny_dsv4")


@pytest.fixture(scope="module")
def env():
    import torch
    import dsv4_gpu
    return dict(torch=torch, lib=dsv4_gpu.lib(), orc=pyoracle.Oracle(),
                dev=torch.device("cuda:0"), dg=dsv4_gpu)


def T(env, a):
    a = np.ascontiguousarray(a)
    if a.dtype == np.uint16:
        a = a.view(np.int16)
    return env["torch"].from_numpy(a.copy()).to(env["dev"])


def H(t):
    return t.detach().cpu().numpy()


def hc_inputs(rng, mult, hid, fn_sigma=0.01):
    mix_n = (2 + mult) * mult
    state = bf16_values(rng.standard_normal(mult * hid).astype(np.float32))
    fn = (rng.standard_normal((mix_n, mult * hid)) * fn_sigma).astype(np.float32)
    scale3 = (0.5 + rng.random(3)).astype(np.float32)
    base = (rng.standard_normal(mix_n) * 0.5).astype(np.float32)
    return state, fn, scale3, base


def midpoint_vec(n):
    """n = 2^k (k even) values whose sum of squares divided by n is exactly
    1 + 2^-24, a float midpoint."""
    k = int(np.log2(n))
    assert 2 ** k == n and k % 2 == 0
    s = np.zeros(n, np.float32)
    s[: n // 4] = 2.0
    s[n // 4] = np.float32(2.0 ** ((k - 24) // 2))
    return s


def test_rmsnorm_bit_exact(env):
    orc, lib = env["orc"], env["lib"]
    rng = np.random.default_rng(11)
    for n in (4096, 1024, 7168, 8, 4, 5):
        x = (rng.standard_normal((5, n)) * rng.random((5, 1)) * 3).astype(np.float32)
        x[1] = 0.0
        if n in (4096, 1024):
            x[2] = midpoint_vec(n)
        w = bf16_bits((1.0 + 0.1 * rng.standard_normal(n)).astype(np.float32))
        for gain in (w, None):
            for rnd in (0, 1):
                for eps in (1e-6, 0.0):
                    got = H(lib.rmsnorm_bf16(T(env, x), None if gain is None else T(env, gain),
                                             eps, rnd))
                    assert same_bits(got, orc.rmsnorm_bf16(x, gain, eps, rnd)), (n, rnd, eps)
    # in place
    x = bf16_input(rng, (3, 4096))
    w = bf16_bits((1.0 + 0.1 * rng.standard_normal(4096)).astype(np.float32))
    xt = T(env, x)
    lib.rmsnorm_bf16(xt, T(env, w), 1e-6, 1, out=xt)
    assert same_bits(H(xt), orc.rmsnorm_bf16(x, w, 1e-6, 1))


def test_hc_split_bit_exact(env):
    orc, lib = env["orc"], env["lib"]
    rng = np.random.default_rng(12)
    for mult in (1, 2, 3, 4, 7):
        mix_n = (2 + mult) * mult
        for iters in (1, 20):
            mixes = (rng.standard_normal((64, mix_n)) * 3).astype(np.float32)
            sc = (rng.random(3) * 2).astype(np.float32)
            base = rng.standard_normal(mix_n).astype(np.float32)
            pre, post, comb = (H(v) for v in lib.hc_split(T(env, mixes), T(env, sc),
                                                         T(env, base), mult, iters))
            for r in range(64):
                p, q, c = orc.hc_split(mixes[r], sc, base, mult, iters, 1e-6)
                assert same_bits(pre[r], p) and same_bits(post[r], q) and same_bits(comb[r], c), \
                    (mult, iters, r)


@pytest.mark.parametrize("mult,hid,n", [(4, 4096, 3), (4, 256, 2), (2, 8, 2), (1, 64, 1),
                                        (3, 100, 2), (7, 32, 2), (4, 4100, 1)])
def test_hc_pre_bit_exact(env, mult, hid, n):
    orc, lib = env["orc"], env["lib"]
    rng = np.random.default_rng(mult * 100 + hid)
    states, fn, sc, base = [], None, None, None
    for t in range(n):
        st, fn_t, sc_t, base_t = hc_inputs(rng, mult, hid)
        states.append(st)
        if fn is None:
            fn, sc, base = fn_t, sc_t, base_t
    S = np.stack(states)
    norm = bf16_bits((1.0 + 0.1 * rng.standard_normal(hid)).astype(np.float32))
    for w in (None, norm):
        b, p, c = (H(v) for v in lib.hc_pre(T(env, S), T(env, fn), T(env, sc), T(env, base), mult,
                                            None if w is None else T(env, w)))
        for t in range(n):
            ob, op, oc = orc.hc_pre(S[t], fn, sc, base, mult)
            if w is not None:
                ob = orc.rmsnorm_bf16(ob[None], w, 1e-6, 1)[0]
            assert same_bits(p[t], op) and same_bits(c[t], oc), (t, "post/comb")
            assert same_bits(b[t], ob), (t, "bin")


def test_hc_pre_midpoint_sum(env):
    """The state's sum of squares on a float midpoint (ss/n = 1 + 2^-24): the
    scale comes from the sequential fallback. (The RMSNorm's own midpoint
    case is in test_rmsnorm_bit_exact.)"""
    orc, lib = env["orc"], env["lib"]
    mult, hid = 4, 4096
    rng = np.random.default_rng(13)
    _, fn, sc, base = hc_inputs(rng, mult, hid)
    S = midpoint_vec(mult * hid)[None]
    norm = bf16_bits(np.ones(hid, np.float32))
    b, p, c = (H(v) for v in lib.hc_pre(T(env, S), T(env, fn), T(env, sc), T(env, base), mult,
                                        T(env, norm)))
    ob, op, oc = orc.hc_pre(S[0], fn, sc, base, mult)
    assert same_bits(p[0], op) and same_bits(c[0], oc)
    assert same_bits(b[0], orc.rmsnorm_bf16(ob[None], norm, 1e-6, 1)[0])


def test_hc_post_bit_exact(env):
    orc, lib = env["orc"], env["lib"]
    rng = np.random.default_rng(14)
    for mult, hid, n in ((4, 4096, 3), (2, 8, 1), (7, 300, 2)):
        S = bf16_values(rng.standard_normal((n, mult * hid)).astype(np.float32))
        br = bf16_values(rng.standard_normal((n, hid)).astype(np.float32))
        post = (rng.random((n, mult)) * 2).astype(np.float32)
        comb = rng.random((n, mult * mult)).astype(np.float32)
        st = T(env, S)
        lib.hc_post(st, T(env, br), T(env, post), T(env, comb), mult)
        got = H(st)
        for t in range(n):
            assert same_bits(got[t], orc.hc_post(S[t], br[t], post[t], comb[t], mult))


def test_tiny_checkpoint_hc_weights(env):
    """The reference's tiny checkpoint (hidden 8, hc_mult 2): hc_pre with its
    hc_ffn weights and ffn_norm, read through the checkpoint index."""
    orc, lib, dg = env["orc"], env["lib"], env["dg"]
    ck = dg.Checkpoint(TINY)
    rng = np.random.default_rng(15)
    for layer in range(4):
        pre = f"layers.{layer}."
        fn = ck.read_f32(pre + "hc_ffn_fn").reshape(8, 16)
        sc = ck.read_f32(pre + "hc_ffn_scale")
        base = ck.read_f32(pre + "hc_ffn_base")
        norm = np.frombuffer(ck.read(pre + "ffn_norm.weight"), np.uint16).copy()
        S = bf16_values(rng.standard_normal((2, 16)).astype(np.float32))
        b, p, c = (H(v) for v in lib.hc_pre(T(env, S), T(env, fn), T(env, sc), T(env, base), 2,
                                            T(env, norm)))
        for t in range(2):
            ob, op, oc = orc.hc_pre(S[t], fn, sc, base, 2)
            assert same_bits(p[t], op) and same_bits(c[t], oc)
            assert same_bits(b[t], orc.rmsnorm_bf16(ob[None], norm, 1e-6, 1)[0])


def run_ffn_step(env, L, mult, n, seed, token_ids=None, DL=None, workspace=None):
    orc, lib, dg, torch = env["orc"], env["lib"], env["dg"], env["torch"]
    rng = np.random.default_rng(seed)
    hid = L["hidden"]
    S = bf16_values((rng.standard_normal((n, mult * hid)) * 0.5).astype(np.float32))
    _, fn, sc, base = hc_inputs(rng, mult, hid, fn_sigma=0.005)
    norm = bf16_bits((1.0 + 0.1 * rng.standard_normal(hid)).astype(np.float32))
    DL = dg.DeviceLayer.from_host(L, env["dev"]) if DL is None else DL
    st = T(env, S)
    tok = None if token_ids is None else torch.from_numpy(token_ids).to(env["dev"])
    _, idx, wt = lib.ffn_step(st, T(env, fn), T(env, sc), T(env, base), T(env, norm), DL, mult,
                              token_ids=tok, workspace=workspace)
    got, idx, wt = H(st), H(idx), H(wt)
    for t in range(n):
        x, post, comb = orc.hc_pre(S[t], fn, sc, base, mult)
        x = orc.rmsnorm_bf16(x[None], norm, 1e-6, 1)[0]
        out, i, w = orc.moe_forward(L, x, 0 if token_ids is None else int(token_ids[t]))
        want = orc.hc_post(S[t], out, post, comb, mult)
        assert np.array_equal(idx[t], i) and same_bits(wt[t], w), t
        assert same_bits(got[t], want), t
    return st, (fn, sc, base, norm, DL)


def test_ffn_step_bit_exact(env):
    """hc_pre + RMSNorm -> decode MoE -> hc_post on device for 3 tokens of a
    synthetic layer, against the oracle's composition of the same steps."""
    L = make_layer(env["orc"], 256, 128, 16, 6, seed=31, bias=True)
    run_ffn_step(env, L, 4, 3, seed=32)


def test_ffn_step_workspace_reused_across_token_counts(env):
    """One workspace sized for 4 tokens serves steps of 4, 1, 3 and 4 tokens
    in a row, each bit-exact: a step with fewer tokens must not write its
    own buffers over the decode records and flags of the tokens it does not
    use (a later step with more tokens needs them zero)."""
    torch, lib, dg = env["torch"], env["lib"], env["dg"]
    L = make_layer(env["orc"], 256, 128, 16, 6, seed=37, bias=True)
    DL = dg.DeviceLayer.from_host(L, env["dev"])
    ws = torch.zeros(lib.ffn_step_workspace_bytes(DL, 4, 4), dtype=torch.uint8,
                     device=env["dev"])
    for i, n in enumerate((4, 1, 3, 4)):
        print(f"ffn_step on a 4-token workspace: {n} tokens", flush=True)
        run_ffn_step(env, L, 4, n, seed=38 + i, DL=DL, workspace=ws)


def test_ffn_step_hash_layer(env):
    L = make_layer(env["orc"], 256, 128, 16, 6, seed=33, hash_vocab=40)
    run_ffn_step(env, L, 4, 2, seed=34, token_ids=np.array([3, 39], np.int32))


def test_ffn_step_full_size(env):
    """hidden 4096 (state 4 x 4096, hc_fn 24 x 16384), inter 2048, 16
    experts, top-6; prints the hc_pre, hc_post and whole-step times."""
    torch, lib = env["torch"], env["lib"]
    L = make_layer(env["orc"], 4096, 2048, 16, 6, seed=35, bias=True)
    st, (fn, sc, base, norm, DL) = run_ffn_step(env, L, 4, 1, seed=36)
    fn_t, sc_t, base_t, norm_t = T(env, fn), T(env, sc), T(env, base), T(env, norm)
    ws = torch.zeros(lib.ffn_step_workspace_bytes(DL, 4, 1), dtype=torch.uint8,
                     device=env["dev"])

    def timed(fn_call, reps=50):
        fn_call()
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for _ in range(reps):
            fn_call()
        torch.cuda.synchronize()
        return (time.perf_counter() - t0) / reps * 1e6

    t_pre = timed(lambda: lib.hc_pre(st, fn_t, sc_t, base_t, 4, norm_t))
    b, p, c = lib.hc_pre(st, fn_t, sc_t, base_t, 4, norm_t)
    t_post = timed(lambda: lib.hc_post(st, b, p, c, 4))
    t_step = timed(lambda: lib.ffn_step(st, fn_t, sc_t, base_t, norm_t, DL, 4, workspace=ws,
                                        check=False))
    lib.check_decode_status(ws)
    print(f"\nhc_pre+norm {t_pre:.1f} us, hc_post {t_post:.1f} us, ffn_step {t_step:.1f} us "
          f"(1 token, host-timed launches)", flush=True)


@pytest.mark.parametrize("mult,hid,n", [(4, 4096, 1), (4, 4096, 40), (4, 4096, 41), (1, 2048, 2),
                                        (1, 16384, 1), (2, 1032, 1), (4, 516, 3), (7, 304, 2),
                                        (3, 5456, 1), (4, 508, 1), (4, 4096, 256), (4, 4096, 257),
                                        (4, 128, 300), (2, 256, 259), (7, 512, 273),
                                        (4, 132, 257), (4, 816, 1), (1, 3280, 40),
                                        (2, 2056, 5), (4, 1024, 21), (4, 1024, 22), (7, 512, 8),
                                        (7, 512, 9), (7, 2048, 12), (7, 2048, 18)])
def test_hc_pre_split_chains(env, mult, hid, n):
    """The chains split over segments (rows of 3264 to 16384 columns, 3 to 63
    mixes, ragged last segments, up to 40 tokens, both sides of the rounds of
    workgroups where that pays), on the fp32 matrix unit (from 257 tokens, ragged
    tiles of mixes and tokens), and the shapes just outside either."""
    orc, lib = env["orc"], env["lib"]
    rng = np.random.default_rng(mult * 1000 + hid + n)
    _, fn, sc, base = hc_inputs(rng, mult, hid)
    S = bf16_values(rng.standard_normal((n, mult * hid)).astype(np.float32))
    norm = bf16_bits((1.0 + 0.1 * rng.standard_normal(hid)).astype(np.float32))
    b, p, c = (H(v) for v in lib.hc_pre(T(env, S), T(env, fn), T(env, sc), T(env, base), mult,
                                        T(env, norm)))
    for t in sorted({*range(0, n, max(1, n // 8)), n - 1}):
        ob, op, oc = orc.hc_pre(S[t], fn, sc, base, mult)
        assert same_bits(p[t], op) and same_bits(c[t], oc), t
        assert same_bits(b[t], orc.rmsnorm_bf16(ob[None], norm, 1e-6, 1)[0]), t


def hc_split_scales(orc, S, fn, base):
    """Scales for mult 4 (powers of two) with which post's arguments are about
    -12, where the sigmoid passes a relative change on, and the others' about 3 in
    magnitude, so that a chain off by its last place shows in post or comb: checked
    here on at least half of the 20 mixes that those depend on. fn's post rows are
    negated where their sums are positive."""
    K = S.size
    acc = np.zeros(24, np.float32)
    for k in range(K):  # the chains, to a rare double rounding
        acc = (fn[:, k].astype(np.float64) * np.float64(S[k]) + acc).astype(np.float32)
    flip = np.flatnonzero(acc[4:8] > 0) + 4
    fn[flip] *= -1
    acc[flip] *= -1
    rs = np.float32(1 / np.sqrt(np.mean(S.astype(np.float64) ** 2) + 1e-6))
    mix = np.abs(acc.astype(np.float64) * rs)
    size = [float(np.median(mix[i])) for i in (slice(0, 4), slice(4, 8), slice(8, 24))]
    sc = np.array([2.0 ** np.clip(np.round(np.log2(t / m)), -126, 127) if m > 0 else 2.0 ** 120
                   for m, t in zip(size, (3, 12, 3))], np.float32)

    def outputs(a):
        _, post, comb = orc.hc_split((a * rs).astype(np.float32), sc, base, 4, 20, 1e-6)
        return post.tobytes() + comb.tobytes()
    was, seen = outputs(acc), 0
    for i in range(4, 24):
        a = acc.copy()
        a[i] = np.nextafter(a[i], np.float32(-np.inf)) if a[i] else np.float32(2.0 ** -126)
        seen += outputs(a) != was
    assert seen >= 10, seen
    return sc


@pytest.mark.parametrize("kind", ["zeros", "growing", "ones", "cancelling", "power_of_two",
                                  "tiny", "subnormal", "huge", "steps", "zero_crossings", "sparse",
                                  "overflow", "infinite"])
def test_hc_pre_split_chain_values(env, kind):
    """Sums whose segments do not follow from their guesses: exact zeros, sums
    that double from segment to segment, ties at every step, sums that return
    to zero, that stay at a power of two, subnormal, huge and infinite sums, and
    sums just inside the fp32 range whose guesses overflow (terms that the chain
    loses, then one that takes only the guess past it; both signs). The mixes
    reach the outputs through post and comb, with a scale at which one last
    place of a chain shows there (hc_split_scales)."""
    orc, lib = env["orc"], env["lib"]
    mult, hid = 4, 4096
    K, mix_n = mult * hid, 24
    rng = np.random.default_rng(5)
    _, fn, sc, base = hc_inputs(rng, mult, hid)
    S = bf16_values(rng.standard_normal(K).astype(np.float32))
    k = np.arange(K)
    if kind == "zeros":
        S[:] = 0
    elif kind == "growing":
        S = bf16_values(np.exp2(k / 1024.0).astype(np.float32))
        fn = np.abs(fn)
    elif kind == "ones":
        S[:] = 1
        fn = np.full_like(fn, 2.0 ** -12) * (1 + 2.0 ** -23 * rng.integers(0, 2, fn.shape))
    elif kind == "cancelling":
        S[1::2] = -S[::2]
        fn[:, 1::2] = fn[:, ::2]
    elif kind == "power_of_two":
        fn[:, 1:] *= 1e-6
        S[0] = 1
        fn[:, 0] = 1
    elif kind == "tiny":
        S *= 2.0 ** -60
        fn *= 2.0 ** -60
    elif kind == "subnormal":
        S *= 2.0 ** -70
        fn *= 2.0 ** -70
    elif kind == "huge":
        S *= 2.0 ** 60
        fn *= 2.0 ** 62
    elif kind == "steps":
        S[:] = np.where((k // 512) % 2 == 0, 1.0, -1.0)
        fn = np.round(fn * 64) / 64
    elif kind == "zero_crossings":
        S = bf16_values((np.sin(k / 100.0)).astype(np.float32))
        fn = np.abs(fn) * 0 + np.float32(0.01)
        fn += (rng.standard_normal(fn.shape) * 1e-4).astype(np.float32)
    elif kind == "overflow":
        S[:], fn[:] = 1, 0
        fn[:, 0], fn[:, 1:600] = 1.5 * 2.0 ** 126, 0.4 * 2.0 ** 103
        fn[:, K - 20] = 2.0 ** 127 + 2.0 ** 125 - 2.0 ** 110
        fn[::2] *= -1
    elif kind == "infinite":  # post's sums alone: comb's would be NaN
        fn[4:8] = 2.0 ** 125
    else:
        S[rng.random(K) < 0.99] = 0
    S, fn = S.astype(np.float32), fn.astype(np.float32)
    base = np.zeros(mix_n, np.float32)
    sc = hc_split_scales(orc, S, fn, base)
    b, p, c = (H(v) for v in lib.hc_pre(T(env, S[None]), T(env, fn), T(env, sc), T(env, base),
                                        mult))
    ob, op, oc = orc.hc_pre(S, fn, sc, base, mult)
    assert same_bits(p[0], op) and same_bits(c[0], oc)
    assert same_bits(b[0], ob)


@pytest.mark.parametrize("hid,off", [(4, 0), (260, 0), (4100, 0), (256, 1), (255, 0)])
def test_hc_post_four_columns(env, hid, off):
    """mult 4: four columns per thread (ragged last workgroups), and the one-column
    form for a state off 16-byte alignment or an odd width."""
    orc, lib, torch = env["orc"], env["lib"], env["torch"]
    rng = np.random.default_rng(hid)
    n = 3
    S = bf16_values(rng.standard_normal((n, 4 * hid)).astype(np.float32))
    br = bf16_values(rng.standard_normal((n, hid)).astype(np.float32))
    post = (rng.random((n, 4)) * 2).astype(np.float32)
    comb = rng.random((n, 16)).astype(np.float32)
    st = torch.zeros(n * 4 * hid + off, dtype=torch.float32, device=env["dev"])[off:]
    st = st.view(n, 4 * hid)
    st.copy_(T(env, S))
    lib.hc_post(st, T(env, br), T(env, post), T(env, comb), 4)
    got = H(st)
    for t in range(n):
        assert same_bits(got[t], orc.hc_post(S[t], br[t], post[t], comb[t], 4)), t
