"""Batched decode (fdm_moe_forward_batched): T tokens through one resident
R1-shape layer in one step with token -> expert dispatch, against the
oracle applied token by token -- routing bit-exact per token, outputs
within 1e-4 relative L2 of the float64 truth, and the distinct-expert count
equal to the number of distinct routed ids."""
import numpy as np
import pytest

from tests._helpers import empty_f32, rel_l2, say, to_dev, to_host

pytestmark = pytest.mark.gpu
TOL = 1e-3


@pytest.fixture(scope="module", params=[False, True], ids=["q4k_down", "q6k_down"])
def layer(request, fdm):
    from flash_deepseek_amd.synthetic import make_layer
    L = 11 if request.param else 10
    say(f"building layer L={L} down_q6={request.param}")
    lay = make_layer(2000 + L, down_q6=request.param)
    fdm.attach_layer(L, lay.experts, lay.expert_size, lay.Wg, lay.bias, lay.shared)
    yield L, lay
    fdm.release_layer(L)


@pytest.fixture(params=["dot4", "mfma"])
def batch_kernel(request, fdm):
    """Runs the test under each expert path behind moe_forward_batched: the
    per-token digit dot products and the grouped MFMA GEMMs (three fp16
    planes of the activations)."""
    mode = fdm.BATCH_DOT4 if request.param == "dot4" else fdm.BATCH_MFMA
    prev = fdm.set_batch_kernel(mode)
    yield request.param
    fdm.set_batch_kernel(prev)


def check_tokens(fdm, oracle, L, lay, T, K, seed, tokens_checked, tol=TOL):
    import torch
    X = np.stack([oracle.synth_normal(7168, 0.0, 1.0, seed + t) for t in range(T)])
    Hin = np.stack([oracle.synth_normal(7168, 0.0, 1.0, seed + 1000 + t) for t in range(T)])
    out = empty_f32(T * 7168)
    idx = torch.empty(T * K, dtype=torch.int32, device="cuda")
    w = empty_f32(T * K)
    nd = torch.zeros(1, dtype=torch.int32, device="cuda")
    say(f"moe_forward_batched L={L} T={T} K={K}")
    fdm.moe_forward_batched(L, to_dev(X.ravel()), to_dev(Hin.ravel()), T, K, out, idx, w, nd)
    got = to_host(out).reshape(T, 7168)
    gi = to_host(idx).reshape(T, K)
    gw = to_host(w).reshape(T, K)
    assert int(to_host(nd)[0]) == len(np.unique(gi))
    Wg, bias = to_host(lay.Wg), to_host(lay.bias)
    cache = {}

    def ffn(e):
        if e not in cache:
            cache[e] = oracle.expert_ffn(lay.expert_bytes(e), lay.down_q6, X_t)
        return cache[e]

    for t in tokens_checked:
        X_t = X[t]
        cache.clear()
        ri, rw = oracle.route(oracle.router_logits(Wg, X_t), bias, K=K)
        assert np.array_equal(gi[t], ri), t
        assert np.array_equal(gw[t].view(np.uint32), rw.view(np.uint32)), t
        moe = np.zeros(7168)
        for k in range(K):
            moe += np.float64(rw[k]) * ffn(int(ri[k]))
        want = Hin[t].astype(np.float64) + moe + ffn(-1)
        err = rel_l2(got[t], want)
        assert err <= tol, (t, err)
    # every token's routing is checked (cheap); outputs on the sampled tokens
    for t in range(T):
        ri, rw = oracle.route(oracle.router_logits(Wg, X[t]), bias, K=K)
        assert np.array_equal(gi[t], ri), t


@pytest.mark.parametrize("T,K", [(1, 8), (16, 8), (5, 3), (70, 8), (64, 8), (256, 8)])
def test_batched_matches_per_token_oracle(fdm, oracle, layer, batch_kernel, T, K):
    """T = 70: several tokens per expert and a shared expert spread over
    several items; T = 64 and 256: the batched-decode workloads (routing
    checked on every token, outputs on four of them)."""
    L, lay = layer
    checked = sorted({0, T // 3, (2 * T) // 3, T - 1})
    check_tokens(fdm, oracle, L, lay, T, K, 9000 + 17 * T, tokens_checked=checked, tol=1e-4)


def activations(kind, n, seed):
    """N(0,1); heavy-tailed (a product of normals, a few huge entries); or one
    outlier of +-1e3 in every 32-element sub-block among N(0,1) values (as
    the matvec fp32-grade test): the fp16 planes of the grouped GEMMs are
    scaled per token row, so an outlier pushes the rest of the row down."""
    rng = np.random.default_rng(seed)
    if kind == "normal":
        return rng.standard_normal(n).astype(np.float32)
    if kind == "heavy":
        x = rng.standard_normal(n) * rng.standard_normal(n) * 300
        x[::97] *= 50
        return x.astype(np.float32)
    x = rng.standard_normal(n)
    x[rng.integers(0, 32, n // 32) + 32 * np.arange(n // 32)] = 1e3 * rng.choice([-1.0, 1.0], n // 32)
    return x.astype(np.float32)


@pytest.mark.parametrize("kind", ["normal", "heavy", "outlier"])
@pytest.mark.parametrize("T", [16, 64, 256])
def test_batched_fp32_grade(fdm, oracle, layer, batch_kernel, T, kind):
    """Both expert paths keep every token at fp32 grade on hard inputs: for
    sampled tokens the relative L2 and the largest per-element error of the
    MoE part (sum_k w_k E_k + S) against float64 stay within 4x of the same
    sum in the reference's fp32 arithmetic; routing of every token is
    bit-exact."""
    import torch
    L, lay = layer
    K = 8
    X = activations(kind, T * 7168, 500 + T).reshape(T, 7168)
    out = empty_f32(T * 7168)
    idx = torch.empty(T * K, dtype=torch.int32, device="cuda")
    w = empty_f32(T * K)
    say(f"moe_forward_batched fp32 grade L={L} T={T} input={kind}")
    fdm.moe_forward_batched(L, to_dev(X.ravel()), None, T, K, out, idx, w)
    got = to_host(out).reshape(T, 7168)
    gi = to_host(idx).reshape(T, K)
    gw = to_host(w).reshape(T, K)
    Wg, bias = to_host(lay.Wg), to_host(lay.bias)
    for t in range(T):
        ri, rw = oracle.route(oracle.router_logits(Wg, X[t]), bias, K=K)
        assert np.array_equal(gi[t], ri), t
        assert np.array_equal(gw[t].view(np.uint32), rw.view(np.uint32)), t
    blobs = {}

    def blob(e):
        if e not in blobs:
            blobs[e] = lay.expert_bytes(e)
        return blobs[e]

    for t in sorted({0, T // 2, T - 1}):
        ri, rw = oracle.route(oracle.router_logits(Wg, X[t]), bias, K=K)
        want = oracle.expert_ffn(blob(-1), lay.down_q6, X[t]).astype(np.float64)
        f32 = oracle.expert_ffn_f32(blob(-1), lay.down_q6, X[t]).astype(np.float32)
        for k in range(K):
            e = int(ri[k])
            want += np.float64(rw[k]) * oracle.expert_ffn(blob(e), lay.down_q6, X[t])
            f32 += rw[k] * oracle.expert_ffn_f32(blob(e), lay.down_q6, X[t])
        g = got[t].astype(np.float64)
        e_got, e_f32 = rel_l2(g, want), rel_l2(f32, want)
        m_got, m_f32 = np.abs(g - want).max(), np.abs(f32.astype(np.float64) - want).max()
        print(f"T={T} {kind} token {t}: rel_l2 {e_got:.3e} (fp32 {e_f32:.3e}), max {m_got:.3e} (fp32 {m_f32:.3e})")
        assert e_got <= 4 * e_f32, (t, e_got, e_f32)
        assert m_got <= 4 * m_f32, (t, m_got, m_f32)


@pytest.mark.parametrize("q6", [False, True], ids=["q4k_down", "q6k_down"])
def test_grouped_gemms_no_further_off_than_dot4(fdm, oracle, q6):
    """Small steps run the grouped GEMMs by default, so these may be no further
    from float64 than the dot4 kernels, on weights around zero (the min term
    takes back most of what the quants sum to).  They carry more bits of the
    activations (33 against 24) and no sum of theirs is less exact, hence 0.9:
    the scatter of the ratio over 5 x 7168 outputs is a few percent."""
    import torch
    from flash_deepseek_amd.synthetic import make_layer
    L, T, K, gate = 16, 5, 8, 57344 * 144
    say(f"building layer L={L} around zero, down_q6={q6}")
    lay = make_layer(2050, down_q6=q6)
    g = torch.Generator(device="cuda").manual_seed(3)

    def scales(shape, unit):
        return ((torch.rand(shape, generator=g, device="cuda") + 0.5) * unit).half()

    for e in (lay.experts.view(256, -1), lay.shared.view(1, -1)):
        q4 = e[:, :(2 if q6 else 3) * gate].view(len(e), -1, 144)
        d = scales(q4.shape[:2], 8e-5)
        q4[..., :4] = torch.stack([d, (d.float() * 7.5).half()], -1).view(torch.uint8)
        if q6:
            down = e[:, 2 * gate:].view(len(e), -1, 210)
            down[..., 208:] = scales(down.shape[:2] + (1,), 1.5e-5).view(torch.uint8)
    fdm.attach_layer(L, lay.experts, lay.expert_size, lay.Wg, lay.bias, lay.shared)
    try:
        X = np.random.default_rng(21).standard_normal((T, 7168)).astype(np.float32)
        got, dX = {}, to_dev(X.ravel())
        idx, w = torch.empty(T * K, dtype=torch.int32, device="cuda"), empty_f32(T * K)
        for mode in (fdm.BATCH_DOT4, fdm.BATCH_MFMA):
            prev = fdm.set_batch_kernel(mode)
            out = empty_f32(T * 7168)
            say(f"moe_forward_batched L={L} T={T} mode {mode}")
            fdm.moe_forward_batched(L, dX, None, T, K, out, idx, w)
            fdm.set_batch_kernel(prev)
            got[mode] = to_host(out).reshape(T, 7168)
    finally:
        fdm.release_layer(L)
    gi, gw = to_host(idx).reshape(T, K), to_host(w).reshape(T, K)
    want = np.stack([np.float64(oracle.expert_ffn(lay.expert_bytes(-1), q6, X[t])) +
                     sum(np.float64(gw[t][k]) * oracle.expert_ffn(lay.expert_bytes(int(gi[t][k])), q6, X[t])
                         for k in range(K)) for t in range(T)])
    dot4, mfma = (rel_l2(got[m], want) for m in (fdm.BATCH_DOT4, fdm.BATCH_MFMA))
    print(f"q6={q6}: dot4 {dot4:.3e}, grouped GEMMs {mfma:.3e} of float64")
    assert mfma <= 0.9 * dot4


@pytest.mark.parametrize("n", [1, 5, 6, 10, 11, 16, 17, 22, 27, 32, 33])
def test_grouped_gemm_chunk_sizes(fdm, oracle, layer, n):
    """n tokens that all choose the same experts, so every chunk of the
    grouped GEMMs is n tokens (16 and a remainder above 16): the operand
    layouts change at 5 / 6 and 10 / 11 tokens.  The tokens are one routing
    vector plus noise too small to change a choice; every token is held to
    1e-5 of float64 (the fp32 grade tests pin the paths' own precision)."""
    import torch
    L, lay = layer
    K = 8
    Wg, bias = to_host(lay.Wg), to_host(lay.bias)
    rng = np.random.default_rng(n)
    base = oracle.synth_normal(7168, 0.0, 1.0, 77)
    X = (base + 1e-3 * rng.standard_normal((n, 7168))).astype(np.float32)
    out = empty_f32(n * 7168)
    idx = torch.empty(n * K, dtype=torch.int32, device="cuda")
    w = empty_f32(n * K)
    prev = fdm.set_batch_kernel(fdm.BATCH_MFMA)
    try:
        say(f"moe_forward_batched L={L} chunk of {n} tokens")
        fdm.moe_forward_batched(L, to_dev(X.ravel()), None, n, K, out, idx, w)
    finally:
        fdm.set_batch_kernel(prev)
    got, gi, gw = to_host(out).reshape(n, 7168), to_host(idx).reshape(n, K), to_host(w).reshape(n, K)
    assert len(np.unique(gi)) == K
    blobs = {e: lay.expert_bytes(e) for e in [-1] + [int(e) for e in gi[0]]}
    for t in range(n):
        ri, _ = oracle.route(oracle.router_logits(Wg, X[t]), bias, K=K)
        assert np.array_equal(gi[t], ri), t
    for t in sorted({0, n // 3, n // 2, n - 1}):
        want = np.float64(oracle.expert_ffn(blobs[-1], lay.down_q6, X[t]))
        for k in range(K):
            want = want + np.float64(gw[t][k]) * oracle.expert_ffn(blobs[int(gi[t][k])], lay.down_q6, X[t])
        assert rel_l2(got[t], want) <= 1e-5, t


def test_token_bits_do_not_depend_on_the_batch(fdm, layer, batch_kernel):
    """A token's output bits are the same whatever other tokens share its step,
    on either path.  Tokens of one routing put every chunk of the grouped GEMMs
    at n tokens (each operand layout and its edges; 33: 16, 16 and 1), tokens of
    their own routing mix chunk sizes."""
    from flash_deepseek_amd.synthetic import make_tokens
    import torch
    L, _ = layer
    K = 8

    def run(X):
        out = torch.empty_like(X)
        say(f"moe_forward_batched L={L} T={len(X)} {batch_kernel}")
        fdm.moe_forward_batched(L, X, None, len(X), K, out)
        return out

    g = torch.Generator(device="cuda").manual_seed(9)
    same = torch.randn(7168, generator=g, device="cuda") + \
        1e-3 * torch.randn(33, 7168, generator=g, device="cuda")
    mixed = make_tokens(300, 91).view(300, 7168)
    for X, sizes in ((same, (1, 2, 5, 6, 10, 11, 15, 16, 17)), (mixed, (1, 2, 5, 11, 16, 40, 128))):
        full = run(X)
        for n in sizes:
            assert torch.equal(run(X[:n].contiguous()), full[:n]), n
        assert torch.equal(run(X[7:29].contiguous()), full[7:29])  # other places in the step


@pytest.mark.parametrize("T,K", [(40, 8), (256, 8), (512, 16)])
def test_grouped_gemm_repeats_bit_exact(fdm, layer, T, K):
    """The same step gives the same bits every time: experts with more than
    one chunk get their tokens in the same order.  (512, 16) has more pairs
    than the dispatch holds in registers."""
    import torch
    from flash_deepseek_amd.synthetic import make_tokens
    L, _ = layer
    X = make_tokens(T, 6000 + T)
    prev = fdm.set_batch_kernel(fdm.BATCH_MFMA)
    try:
        outs = []
        for rep in range(4):
            out = empty_f32(T * 7168)
            say(f"moe_forward_batched L={L} T={T} K={K} pass {rep}")
            fdm.moe_forward_batched(L, X, None, T, K, out)
            outs.append(out)
    finally:
        fdm.set_batch_kernel(prev)
    torch.cuda.synchronize()
    assert all(torch.equal(o, outs[0]) for o in outs[1:])


def test_batched_paths_agree(fdm, layer):
    """The two expert paths on the same 96-token step: identical routing,
    outputs within 1e-4 of each other (both carry the activations at fp32
    grade)."""
    import torch
    from flash_deepseek_amd.synthetic import make_tokens
    L, _ = layer
    T, K = 96, 8
    X = make_tokens(T, 4321)
    outs = []
    for mode in (fdm.BATCH_DOT4, fdm.BATCH_MFMA):
        prev = fdm.set_batch_kernel(mode)
        try:
            out = empty_f32(T * 7168)
            idx = torch.empty(T * K, dtype=torch.int32, device="cuda")
            say(f"moe_forward_batched L={L} T={T} mode={mode}")
            fdm.moe_forward_batched(L, X, None, T, K, out, idx, None, None)
            outs.append((to_host(out).reshape(T, 7168), to_host(idx)))
        finally:
            fdm.set_batch_kernel(prev)
    assert np.array_equal(outs[0][1], outs[1][1])
    for t in range(T):
        assert rel_l2(outs[1][0][t], outs[0][0][t].astype(np.float64)) <= 1e-4, t


def test_batched_unaligned_residual_and_output(fdm, layer, batch_kernel):
    """h_in and hidden need no 16-byte alignment: the same step with both
    pointers 4 bytes past an aligned address (the combine's one-value-per-
    thread variant) gives the same bits as with aligned ones (its 16-byte
    vector variant)."""
    import torch
    from flash_deepseek_amd.synthetic import make_tokens
    L, _ = layer
    T, K = 24, 8
    X = make_tokens(T, 5150)
    Hin = make_tokens(T, 5151).reshape(-1)
    n = T * 7168
    out_a = empty_f32(n)
    say(f"moe_forward_batched L={L} T={T} aligned")
    fdm.moe_forward_batched(L, X, Hin, T, K, out_a)
    hbuf = torch.zeros(n + 4, dtype=torch.float32, device="cuda")
    hbuf[1:1 + n].copy_(Hin)
    obuf = torch.zeros(n + 4, dtype=torch.float32, device="cuda")
    h_off, o_off = hbuf[1:1 + n], obuf[1:1 + n]
    assert h_off.data_ptr() % 16 != 0 and o_off.data_ptr() % 16 != 0
    say(f"moe_forward_batched L={L} T={T} unaligned h_in / hidden")
    fdm.moe_forward_batched(L, X, h_off, T, K, o_off)
    assert np.array_equal(to_host(out_a).view(np.uint32), to_host(o_off).view(np.uint32))
    assert float(obuf[0]) == 0.0 and float(obuf[1 + n]) == 0.0  # nothing written outside


def test_batched_equals_single_token_layer(fdm, oracle, layer, batch_kernel):
    """Each token of a batch gets the same routing as fdm_moe_layer and an
    output within 1e-4 of it."""
    import torch
    L, lay = layer
    T, K = 12, 8
    X = np.stack([oracle.synth_normal(7168, 0.0, 1.0, 777 + t) for t in range(T)]).astype(np.float32)
    out = empty_f32(T * 7168)
    idx = torch.empty(T * K, dtype=torch.int32, device="cuda")
    fdm.moe_forward_batched(L, to_dev(X.ravel()), None, T, K, out, idx, None, None)
    got = to_host(out).reshape(T, 7168)
    gi = to_host(idx).reshape(T, K)
    for t in (0, 7, 11):
        one = empty_f32(7168)
        i1 = torch.empty(K, dtype=torch.int32, device="cuda")
        fdm.moe_layer(L, to_dev(X[t]), None, K, one, i1)
        assert np.array_equal(to_host(i1), gi[t])
        assert rel_l2(got[t], to_host(one).astype(np.float64)) <= 1e-4


def test_batched_errors(fdm, layer):
    L, _ = layer
    x = empty_f32(7168)
    with pytest.raises(fdm.FdmError):
        fdm.moe_forward_batched(L, x, None, 0, 8, empty_f32(7168))
    with pytest.raises(fdm.FdmError):
        fdm.moe_forward_batched(L, x, None, 513, 8, empty_f32(7168))
    with pytest.raises(fdm.FdmError):
        fdm.moe_forward_batched(L, x, None, 1, 17, empty_f32(7168))
    with pytest.raises(fdm.FdmError):
        fdm.set_batch_kernel(3)
