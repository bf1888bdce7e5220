"""GPU parity tests of the speculative-verification path: Gated DeltaNet over a speculated token tree
(csrc/k_deltanet_tree.hip <- cpu/kernel/gdn/tree_verify/*.rs) through the C ABI against the CPU oracle, and the engine's
verify_tree -> accept protocol (stream.rs:380-470, 556-628) against the oracle model and against plain decoding."""
import ctypes as C

import numpy as np
import pytest

from helpers import bf16, f32, ulp_diff_bf16
from oracle import oracle as O
from test_gpu_kernels import run
from test_oracle_tree_verify import linear_stream, logit_error_sigma, path_of, random_tree
from uzu_amd import _ffi
from uzu_amd import backend as B
from uzu_amd import desc as D
from uzu_amd import synthetic as S
from uzu_amd.engine import MODEL_BATCH, HipModel
from uzu_amd.trie import TrieNode

pytestmark = pytest.mark.gpu


def _set_exact(on):
    fn = _ffi.lib().uzu_hip_set_exact
    fn.restype, fn.argtypes = None, [C.c_int32]
    fn(1 if on else 0)


# ------------------------------------------------------------------------------------------ kernels, through the C ABI
@pytest.mark.parametrize("n,Hk,Hv", [(1, 16, 16), (16, 16, 16), (23, 2, 4), (32, 4, 8)])
def test_conv_tree_scan_and_tree_prep_bit_exact(hip_ctx, n, Hk, Hv):
    """ConvTreeScan (tree_verify/conv_scan.rs) and DeltaNetPrefillPrep's tree instantiation (prefill_prep.rs with QKT = T, log decays,
    compact V) -- Qwen3.5 shape first -- BIT-EXACT against the CPU kernels: same tap order, glibc-exact exp / log, and the l2 norms
    summed by one thread in the reference's order."""
    rng = np.random.default_rng(200 + n)
    D, ks = 128, 4
    key_dim, value_dim = Hk * D, Hv * D
    conv_dim = 2 * key_dim + value_dim
    total = conv_dim + value_dim + 2 * Hv
    _, parents = random_tree(n, rng)
    x = bf16(rng.normal(size=(n, total)))
    w = rng.uniform(-0.6, 0.6, size=(conv_dim, ks)).astype(np.float32)
    bias = rng.uniform(-0.1, 0.1, size=(conv_dim,)).astype(np.float32)
    base = rng.normal(size=(conv_dim, ks - 1)).astype(np.float32)
    a_log, dt_bias = rng.uniform(-1, 1, Hv).astype(np.float32), rng.uniform(-1, 1, Hv).astype(np.float32)
    # oracle
    w_out = np.zeros_like(x)
    w_states = np.zeros((n, conv_dim, ks - 1), np.float32)
    O.call("orc_conv_tree_scan", x, w, bias, base, parents, w_out, w_states, O.BF16, n, ks, total, conv_dim)
    w_q, w_k = np.zeros((n, key_dim), np.uint16), np.zeros((n, key_dim), np.uint16)
    w_v = np.zeros((n, value_dim), np.uint16)
    w_beta, w_ld = np.zeros((n, Hv), np.float32), np.zeros((n, Hv), np.float32)
    O.call("orc_delta_net_tree_prep", w_out, a_log, dt_bias, w_q, w_k, w_v, w_beta, w_ld, O.BF16, Hv, Hk, D, key_dim, value_dim, n)
    # HIP: the two kernels of the trait surface
    scan = B.ConvTreeScanKernel.new(hip_ctx, B.BF16, ks, 1)
    prep = B.DeltaNetPrefillPrepKernel.new(hip_ctx, B.BF16, B.BF16, 128, 1, 1)
    bx, bw, bb, bbase, bpar = (hip_ctx.buffer_from(z) for z in (x, w, bias, base, parents))
    bout, bst = hip_ctx.buffer_from(np.zeros_like(x)), hip_ctx.buffer_from(np.zeros_like(w_states))
    bq, bk, bv = (hip_ctx.buffer_from(np.zeros_like(z)) for z in (w_q, w_k, w_v))
    bbeta, bld = hip_ctx.buffer_from(np.zeros_like(w_beta)), hip_ctx.buffer_from(np.zeros_like(w_ld))
    ba, bdt = hip_ctx.buffer_from(a_log), hip_ctx.buffer_from(dt_bias)

    def encode(cb):
        scan.encode(bx, bw, bb, bbase, bpar, bout, bst, n, total, conv_dim, cb)
        prep.encode(bout, ba, bdt, bq, bk, bv, bbeta, bld, Hv, Hk, key_dim, value_dim, n, cb)
    run(hip_ctx, encode)
    assert np.array_equal(bout.download(np.uint16, x.size).reshape(x.shape), w_out)
    assert np.array_equal(bst.download(np.float32, w_states.size).reshape(w_states.shape), w_states)
    assert np.array_equal(bq.download(np.uint16, w_q.size).reshape(w_q.shape), w_q)
    assert np.array_equal(bk.download(np.uint16, w_k.size).reshape(w_k.shape), w_k)
    assert np.array_equal(bv.download(np.uint16, w_v.size).reshape(w_v.shape), w_v)
    assert np.array_equal(bbeta.download(np.float32, w_beta.size).reshape(w_beta.shape), w_beta)
    assert np.array_equal(bld.download(np.float32, w_ld.size).reshape(w_ld.shape), w_ld)


def tree_verify_inputs(rng, n, Hk, Hv):
    D = 128
    nodes, parents = random_tree(n, rng)
    q = bf16(rng.normal(size=(n, Hk, D)) / np.sqrt(D) / np.sqrt(D) * 8)
    k = rng.normal(size=(n, Hk, D))
    k = bf16(k / np.linalg.norm(k, axis=-1, keepdims=True))
    v = bf16(rng.normal(size=(n, Hv, D)))
    log_decay = -rng.uniform(0.01, 0.6, size=(n, Hv)).astype(np.float32)
    beta = rng.uniform(0.1, 0.9, size=(n, Hv)).astype(np.float32)
    h0 = (rng.normal(size=(Hv, D, D)) * 0.3).astype(np.float32)
    return nodes, parents, q, k, v, log_decay, beta, h0


def oracle_tree_verify(nodes, q, k, v, log_decay, beta, h0, n, Hk, Hv):
    D = 128
    nb = (n + 15) // 16
    ncp = (nb + 1) // 2
    h0_idx = np.zeros(1, np.int32)
    prefix = np.zeros((n, Hv), np.float32)
    a_packed = np.zeros((Hv, nb, ncp, 16, 32), np.float32)
    qkd = np.zeros((Hv, n, n), np.float32)
    a_inv = np.zeros((Hv, nb, 16, 16), np.float32)
    kh0 = np.zeros((n, Hv, D), np.float32)
    u = np.zeros((Hv, n, D), np.float32)
    out = np.zeros((n, Hv, D), np.uint16)
    O.call("orc_build_tree_prefix", nodes, log_decay, prefix, 1, n, Hv)
    O.call("orc_build_tree_gram", q, k, O.BF16, nodes, prefix, beta, h0, h0_idx, a_packed, qkd, a_inv, kh0, 1.0, 1, n, Hk, Hv, D, D)
    O.call("orc_tree_update_solve", kh0, v, O.BF16, prefix, beta, a_packed, a_inv, h0_idx, u, 1, n, Hv, D)
    O.call("orc_build_tree_out", q, O.BF16, prefix, qkd, u, h0, h0_idx, out, O.BF16, 1.0, 1, n, Hk, Hv, D, D)
    return out


@pytest.mark.parametrize("n,Hk,Hv", [(1, 16, 16), (4, 16, 16), (8, 16, 16), (16, 16, 16), (17, 2, 4), (32, 4, 8)])
def test_delta_net_tree_verify_bit_exact(hip_ctx, n, Hk, Hv):
    """DeltaNetTreeVerify (prefix -> Gram -> solve -> out as the Metal backend composes the CPU-tested kernels,
    metal/kernel/gdn/tree_verify.rs:92-187) as ONE kernel: every output element is computed by one thread walking the reference's loops in
    the reference's order -> BIT-IDENTICAL to the composition of the CPU kernels (tree_gram_test.rs / tree_update_solve_test.rs compare
    Metal with them at 2e-4 ... 5e-3)."""
    rng = np.random.default_rng(300 + n)
    nodes, _, q, k, v, log_decay, beta, h0 = tree_verify_inputs(rng, n, Hk, Hv)
    want = oracle_tree_verify(nodes, q, k, v, log_decay, beta, h0, n, Hk, Hv)
    kern = B.DeltaNetTreeVerify.new(hip_ctx, B.BF16, Hk, Hv, 128, 128)
    bufs = [hip_ctx.buffer_from(z) for z in (q, k, v, nodes, log_decay, beta, h0)]
    bo = hip_ctx.buffer_from(np.zeros_like(want))
    run(hip_ctx, lambda cb: kern.encode(*bufs, bo, n, cb))
    got = bo.download(np.uint16, want.size).reshape(want.shape)
    assert np.array_equal(got, want), f"{(got != want).sum()} of {got.size} outputs differ (max {ulp_diff_bf16(want, got).max():.2f} bf16 ulps)"


@pytest.mark.parametrize("exact", [False, True])
def test_state_advance(hip_ctx, exact):
    """StateAdvance (state_advance.rs) over an accepted path of 9 nodes, Qwen3.5 shape.  Production: a state row per half-wave (f32
    butterfly sums): <= 1e-5 against the CPU kernel; reference-order mode: bit-identical."""
    rng = np.random.default_rng(17)
    n, Hk, Hv, D = 16, 16, 16, 128
    _, parents, _, k, v, log_decay, beta, h0 = tree_verify_inputs(rng, n, Hk, Hv)
    node = n - 1
    path = []
    while node >= 0:
        path.append(node)
        node = int(parents[node])
    accepted = np.array(path[::-1], np.uint32)
    want = h0.copy()
    O.call("orc_state_advance", k, v, O.BF16, log_decay, beta, accepted, want, len(accepted), Hv, Hk, D)
    kern = B.StateAdvanceKernel.new(hip_ctx, B.BF16, 128, Hv, Hk)
    bufs = [hip_ctx.buffer_from(z) for z in (k, v, log_decay, beta, accepted)]
    bs = hip_ctx.buffer_from(h0)
    _set_exact(exact)
    try:
        run(hip_ctx, lambda cb: kern.encode(*bufs, bs, len(accepted), cb))
    finally:
        _set_exact(False)
    got = bs.download(np.float32, h0.size).reshape(h0.shape)
    if exact:
        assert np.array_equal(got, want)
    else:
        np.testing.assert_allclose(got, want, rtol=1e-5, atol=1e-5)


def test_kv_cache_update_with_dependent_copies_runs_in_the_reference_order(hip_ctx):
    """The accept compaction of a speculated path (state.rs:180-196): copy i moves row a_i down to row i, so a later copy's destination
    can be an earlier copy's source ([0, 2, 3] -> (2 -> 1), (3 -> 2)); the reference runs the copies sequentially per element column
    (kv_cache_update.rs:14-27)."""
    rng = np.random.default_rng(5)
    rows, dim = 12, 512
    keys, values = bf16(rng.normal(size=(rows, dim))), bf16(rng.normal(size=(rows, dim)))
    copies = [(6, 5), (7, 6), (9, 7), (10, 8)]  # accepted nodes [0, 2, 3, 5, 6] behind a context of 4 rows
    wk, wv = keys.copy(), values.copy()
    for s, d in copies:
        wk[d], wv[d] = wk[s], wv[s]
    kern = B.KVCacheUpdateKernel.new(hip_ctx, B.BF16)
    bk, bv = hip_ctx.buffer_from(keys), hip_ctx.buffer_from(values)
    run(hip_ctx, lambda cb: kern.encode(bk, bv, copies, len(copies), dim, cb))
    assert np.array_equal(bk.download(np.uint16, keys.size).reshape(keys.shape), wk)
    assert np.array_equal(bv.download(np.uint16, values.size).reshape(values.shape), wv)


# ------------------------------------------------------------------------------------------ the engine's verify -> accept
def speculative_tree(got_last, want, i, depth, vocab):
    """the true continuation want[i+1 .. i+depth] as a chain, a wrong sibling at every level, one of them with a child"""
    root = TrieNode(got_last)
    node = root
    for d in range(1, depth + 1):
        wrong = TrieNode((want[i + d] + 17 * d) % vocab)
        if d == 2:
            wrong.add(TrieNode((want[i + d] + 5) % vocab))
        node.add(wrong)
        true_child = TrieNode(want[i + d])
        node.add(true_child)
        node = true_child
    return root


@pytest.mark.parametrize("preset,mult", [("tiny-qwen", 81), ("tiny-qwen", 121), ("tiny-qwen", 151), ("tiny-llama", 191)])
def test_engine_verify_then_accept_matches_the_oracle_and_linear_decoding(hip_ctx, preset, mult):
    """uzu_hip_model_verify_tree / uzu_hip_model_accept against the oracle model's verify_tree / accept on the same trees (the prompts
    of tests/test_oracle_tree_verify.py): per round the logits of EVERY node -- right and wrong branches -- within 0.25 sigma
    (row-normalised) of the oracle's, the sampled tokens equal wherever the oracle's decision is not a near-tie, the accepted path the
    same; after three rounds plain (graph-replayed, fused) decoding carries on with the linear stream's tokens: the KV compaction, the
    DeltaNet conv state and the advanced SSM state are those of linear decoding."""
    cfg = S.PRESETS[preset]()
    bundle = S.build_model(cfg)
    row_mult = S.readout_row_multipliers(cfg)
    base = S.synthetic_prompt(37, cfg.vocab_size).astype(np.int64)
    prompt = ((base * mult + 11 * mult) % cfg.vocab_size).astype(np.uint32)
    om = O.OracleModel(bundle)
    depth, rounds = 4, 3
    want, _ = linear_stream(om, prompt, rounds * (depth + 1) + 6)
    om.reset()
    om.prefill(prompt)
    hm = HipModel(hip_ctx, bundle)
    got = [hm.prefill(prompt)]
    assert got[0] == want[0]
    worst = 0.0
    for rnd in range(rounds):
        i = len(got) - 1
        flat = speculative_tree(got[-1], want, i, depth, cfg.vocab_size).linearize()
        o_sampled, o_logits = om.verify_tree(flat.token_ids(), flat.nodes(), True)
        h_sampled = hm.verify_tree(flat.token_ids(), flat.nodes())
        h_logits = hm.read_tree_logits()
        for node in range(len(flat)):
            worst = max(worst, logit_error_sigma(o_logits[node], h_logits[node], row_mult))
            if int(h_sampled[node]) != int(o_sampled[node]):
                w = np.sort(f32(o_logits[node]).astype(np.float64))
                assert (w[-1] - w[-2]) / w.std() < 0.05, f"round {rnd} node {node}: oracle {o_sampled[node]}, hip {h_sampled[node]} without a near-tie"
        o_acc, h_acc = flat.accept(o_sampled), flat.accept(h_sampled)
        assert h_acc == o_acc and len(h_acc) == depth + 1
        om.accept([idx for idx, _, _ in o_acc])
        hm.accept([idx for idx, _, _ in h_acc])
        got.extend(int(s) for _, _, s in h_acc)
        assert hm.context_length == om.context_length
    assert worst <= 0.25, f"tree-pass logits {worst:.3f} sigma off the oracle's"
    assert got == want[:len(got)]
    toks, _ = hm.decode(len(want) - len(got))
    assert [int(t) for t in toks] == want[len(got):], "decoding after the accepts leaves the linear stream"
    assert [int(t) for t in hm.read_tokens(len(prompt), len(got) - 1)] == got[1:]  # the accepted tokens sit at their positions
    print(f"{preset} x{mult}: tree-pass logits within {worst:.3f} sigma of the oracle's")
    hm.close()
    om.close()


def test_engine_verify_and_accept_on_ring_kv_states(hip_ctx):
    """Sliding-window layers (AttentionStateType::Ring, state.rs:16-55, 200-219) under speculation: the tree's rows sit behind the ring
    during the pass (trie mask + window on positions), the accepted ones enter the ring slot by slot.  A window of 40 with a 37-token
    prompt wraps during the second round.  Against the oracle model round by round, then plain decoding continues identically."""
    cfg = S.tiny_llama(sliding_windows=[40, 0], sinks=True, seed=48)
    bundle = S.build_model(cfg)
    # the multiplier: of 200 tried on the CPU oracle, the one whose accepted path and the four decode steps behind it are decided by the widest
    # top-two gap (>= 0.46 sigma of the logit row, eleven distinct tokens) -- the production kernels sit 0.04-0.08 sigma off the oracle's logits,
    # and the first choice (191) had a 0.04-sigma decision on the path (tools/scratch/diag_ring.py on the GPU: every node within 0.08 sigma)
    prompt = ((S.synthetic_prompt(37, cfg.vocab_size).astype(np.int64) * 493 + 2101) % cfg.vocab_size).astype(np.uint32)
    om = O.OracleModel(bundle)
    want, _ = linear_stream(om, prompt, 20)
    om.reset()
    om.prefill(prompt)
    hm = HipModel(hip_ctx, bundle)
    got = [hm.prefill(prompt)]
    for rnd in range(3):
        flat = speculative_tree(got[-1], want, len(got) - 1, 4, cfg.vocab_size).linearize()
        o_sampled = om.verify_tree(flat.token_ids(), flat.nodes())
        h_sampled = hm.verify_tree(flat.token_ids(), flat.nodes())
        o_acc, h_acc = flat.accept(o_sampled), flat.accept(h_sampled)
        assert h_acc == o_acc, f"round {rnd}: oracle accepts {o_acc}, hip {h_acc}"
        om.accept([i for i, _, _ in o_acc])
        hm.accept([i for i, _, _ in h_acc])
        got.extend(int(s_) for _, _, s_ in h_acc)
    toks, _ = hm.decode(4)
    tok = got[-1]
    for t in toks:
        tok = om.forward([tok])
        assert int(t) == tok
    hm.close()
    om.close()


@pytest.mark.parametrize("n,groups,kernel", [(1, 2, 4), (2, 4, 3), (13, 1, 4), (16, 4, 2), (17, 2, 4), (31, 4, 4), (32, 2, 3)])
def test_engine_tree_passes_of_every_size_are_bit_identical_in_reference_order_mode(hip_ctx, n, groups, kernel):
    """The DeltaNet layers' pass over a tree in one launch (dn_tree_step): tree sizes around a block of 16 nodes, the smallest and the largest, key heads of one, two and four value
    heads (who files the keys), two to four taps; every node's logits, and after an accepted path (keys, values, decays and conv states that the launch filed) a decode step's."""
    rng = np.random.default_rng(n)
    cfg = S.tiny_qwen(dn_num_groups=groups, dn_kernel_size=kernel)
    bundle = S.build_model(cfg)
    prompt = ((S.synthetic_prompt(37, cfg.vocab_size).astype(np.int64) * 81 + 891) % cfg.vocab_size).astype(np.uint32)
    nodes, parents = random_tree(n, rng)
    om = O.OracleModel(bundle)
    _set_exact(True)
    try:
        hm = HipModel(hip_ctx, bundle)
        tok = om.prefill(prompt)
        assert hm.prefill(prompt) == tok
        tokens = np.concatenate([[tok], rng.integers(0, cfg.vocab_size, n - 1)]).astype(np.uint32)
        o_sampled, o_logits = om.verify_tree(tokens, nodes, True)
        h_sampled = hm.verify_tree(tokens, nodes)
        h_logits = hm.read_tree_logits()
        assert np.array_equal(h_logits, o_logits), f"{(h_logits != o_logits).sum()} of {o_logits.size} tree logits differ"
        path = path_of(parents, n - 1)
        om.accept(path)
        hm.accept(path)
        _, lg = om.forward([int(o_sampled[path[-1]])], True)
        hm.decode(1)
        assert np.array_equal(hm.read_logits(), lg)
        hm.close()
    finally:
        _set_exact(False)
        om.close()


def test_engine_accept_advances_the_states_of_more_layers_than_one_table_holds(hip_ctx):
    """65 DeltaNet layers: a table of 64 states and one of a single one (dn_states_advance).  Everything but the acceptance in reference order, so that what differs from the oracle is
    the advanced states' f32 sums (1e-5 of a state, test_state_advance): the logits behind the accepted path within the 0.25 sigma that the tests above give whole production passes."""
    cfg = S.tiny_qwen(layer_kinds=[D.MIXER_DELTA_NET] * 65 + [D.MIXER_ATTENTION], vocab_size=512)
    bundle = S.build_model(cfg)
    row_mult = S.readout_row_multipliers(cfg)
    prompt = S.synthetic_prompt(21, cfg.vocab_size)
    om = O.OracleModel(bundle)
    _set_exact(True)
    try:
        hm = HipModel(hip_ctx, bundle)
        tok = om.prefill(prompt)
        assert hm.prefill(prompt) == tok
        nodes, _ = random_tree(4, np.random.default_rng(1), branch=0.0)  # a chain
        tokens = np.array([tok, 3, 141, 59], np.uint32)
        o_sampled = om.verify_tree(tokens, nodes)
        assert np.array_equal(hm.verify_tree(tokens, nodes), o_sampled)
        om.accept([0, 1, 2, 3])
        _set_exact(False)
        hm.accept([0, 1, 2, 3])
        _set_exact(True)
        _, want = om.forward([int(o_sampled[3])], True)
        hm.decode(1)
        assert logit_error_sigma(want, hm.read_logits(), row_mult) <= 0.25
        hm.close()
    finally:
        _set_exact(False)
        om.close()


def test_engine_tree_pass_with_stochastic_sampling_uses_each_nodes_own_seed(hip_ctx):
    """SamplingMethod::Stochastic over a tree: node i draws with PRng::derive(context + height_i) (speculators/dflash_tfm.rs:267,304), i.e.
    exactly the seed plain decoding uses at that position -- checked per node against the CPU restatement of UnifiedSampling applied to
    the pass's own logits of that node."""
    cfg = S.tiny_qwen()
    bundle = S.build_model(cfg)
    prompt = S.synthetic_prompt(21, cfg.vocab_size)
    hm = HipModel(hip_ctx, bundle)
    seed = 0x1234567
    hm.set_sampling(seed=seed, temperature=25.0, top_k=40)
    tok = hm.prefill(prompt)
    root = TrieNode(tok)
    a, b = TrieNode(5), TrieNode(9)
    root.add(a), root.add(b)
    a.add(TrieNode(11)), b.add(TrieNode(13))
    flat = root.linearize()
    sampled = hm.verify_tree(flat.token_ids(), flat.nodes())
    logits = hm.read_tree_logits()
    from test_gpu_model import prng_derive
    ctx_len = len(prompt)
    for i, node in enumerate(flat.nodes()):
        want = np.zeros(1, np.uint32)
        seeds = np.array([prng_derive(seed, ctx_len + int(node[2]))], np.uint64)
        O.lib().orc_unified_sampling(O.p(np.ascontiguousarray(logits[i])), O.BF16, O.p(want), O.p(seeds), None, 1, C.c_float(25.0), 1, 40, 0, C.c_float(0.0), 0, C.c_float(0.0),
                                     cfg.vocab_size, 1)
        assert int(sampled[i]) == int(want[0]), f"node {i} (height {node[2]}): {sampled[i]} != {want[0]}"
    assert len(set(int(t) for t in sampled)) > 1
    hm.accept([0])
    hm.close()


@pytest.mark.parametrize("preset", ["tiny-qwen", "tiny-llama"])
def test_engine_tree_pass_is_bit_identical_to_the_oracle_in_reference_order_mode(hip_ctx, preset):
    """uzu_hip_set_exact(1): the whole tree pass -- trie-masked attention at positions context + height, ConvTreeScan, tree prep,
    DeltaNetTreeVerify, norm-gate, every node's read-out -- gives logits BIT-IDENTICAL to the oracle's for every node, and after the
    accept (reference-order StateAdvance) so do the logits of the decode steps that follow."""
    cfg = S.PRESETS[preset]()
    bundle = S.build_model(cfg)
    prompt = ((S.synthetic_prompt(37, cfg.vocab_size).astype(np.int64) * 81 + 891) % cfg.vocab_size).astype(np.uint32)
    om = O.OracleModel(bundle)
    want, _ = linear_stream(om, prompt, 12)
    om.reset()
    _set_exact(True)
    try:
        hm = HipModel(hip_ctx, bundle)
        assert hm.prefill(prompt) == om.prefill(prompt)
        flat = speculative_tree(want[0], want, 0, 5, cfg.vocab_size).linearize()
        o_sampled, o_logits = om.verify_tree(flat.token_ids(), flat.nodes(), True)
        h_sampled = hm.verify_tree(flat.token_ids(), flat.nodes())
        h_logits = hm.read_tree_logits()
        assert np.array_equal(h_logits, o_logits), f"{(h_logits != o_logits).sum()} of {o_logits.size} tree logits differ"
        assert np.array_equal(h_sampled, o_sampled)
        acc = [idx for idx, _, _ in flat.accept(o_sampled)]
        om.accept(acc)
        hm.accept(acc)
        tok = int(o_sampled[acc[-1]])
        for _ in range(3):
            tok, lg = om.forward([tok], True)
            t, _ = hm.decode(1)
            assert np.array_equal(hm.read_logits(), lg) and int(t[0]) == tok
        hm.close()
    finally:
        _set_exact(False)
    om.close()


def test_engine_verify_guards(hip_ctx):
    from uzu_amd._ffi import UzuHipError
    cfg = S.tiny_qwen()
    hm = HipModel(hip_ctx, S.build_model(cfg))
    with pytest.raises(UzuHipError):  # nothing to hang the tree off
        hm.verify_tree([1, 2], [[0, 1, 0], [1, 1, 1]])
    tok = hm.prefill(S.synthetic_prompt(9, cfg.vocab_size))
    with pytest.raises(UzuHipError):  # not DFS order: node 1 claims height 2 under a root of height 0
        hm.verify_tree([tok, 2], [[0, 1, 0], [1, 1, 2]])
    with pytest.raises(UzuHipError):  # nothing pending
        hm.accept([0])
    flat = TrieNode.flat([tok, 5, 6]).linearize()
    hm.verify_tree(flat.token_ids(), flat.nodes())
    with pytest.raises(UzuHipError):  # a second tree before the accept
        hm.verify_tree(flat.token_ids(), flat.nodes())
    with pytest.raises(UzuHipError):  # not a root path
        hm.accept([0, 2])
    hm.accept([0, 1])
    assert hm.context_length == 11
    hm.close()


def test_engine_tree_pass_takes_the_tries_own_seeds(hip_ctx):
    """stream.rs:690-695: under stochastic sampling the reference uploads the trie's token_seeds -- whatever the speculator put into its
    nodes -- as the per-node seeds of UnifiedSampling.  verify_tree(..., seeds) does the same; each node must draw exactly what the CPU
    restatement draws from the pass's own logits of that node with THAT seed, eagerly and in the captured graph of the second pass (a pass
    with host seeds and one with derived seeds are different graphs); without seeds the position-derived ones are back."""
    from test_gpu_model import prng_derive
    cfg = S.tiny_qwen()
    bundle = S.build_model(cfg)
    prompt = S.synthetic_prompt(21, cfg.vocab_size)
    hm = HipModel(hip_ctx, bundle)
    seed = 0x7654321
    hm.set_sampling(seed=seed, temperature=25.0, top_k=40)
    tok = hm.prefill(prompt)

    def draw(row, s_):
        want = np.zeros(1, np.uint32)
        seeds = np.array([s_], np.uint64)
        O.lib().orc_unified_sampling(O.p(np.ascontiguousarray(row)), O.BF16, O.p(want), O.p(seeds), None, 1, C.c_float(25.0), 1, 40, 0, C.c_float(0.0), 0, C.c_float(0.0),
                                     cfg.vocab_size, 1)
        return int(want[0])

    for rnd in range(3):
        root = TrieNode(tok, seed=0xA000 + rnd)
        a, b = TrieNode(5, seed=0xB111 * (rnd + 1)), TrieNode(9, seed=0xC222 + 7 * rnd)
        root.add(a), root.add(b)
        a.add(TrieNode(11, seed=0xD333 ^ rnd)), b.add(TrieNode(13, seed=(1 << 63) + rnd))
        flat = root.linearize()
        use_trie = rnd != 1
        sampled = hm.verify_tree(flat.token_ids(), flat.nodes(), flat.token_seeds() if use_trie else None)
        logits = hm.read_tree_logits()
        ctx_len = hm.context_length
        for i, node in enumerate(flat.nodes()):
            s_ = int(flat.token_seeds()[i]) if use_trie else prng_derive(seed, ctx_len + int(node[2]))
            assert int(sampled[i]) == draw(logits[i], s_), f"round {rnd} node {i}"
        hm.accept([0])
        tok = int(sampled[0])
    hm.close()


def test_a_pending_tree_is_void_once_the_sequence_moves_on_another_way(hip_ctx):
    """A verified tree that is never accepted must not survive a prefill / decode of the same sequence (a later
    accept would compact KV rows at the new context offsets and advance the DeltaNet states a second time from stale tree buffers)."""
    from uzu_amd._ffi import UzuHipError
    cfg = S.tiny_qwen()
    bundle = S.build_model(cfg)
    prompt = S.synthetic_prompt(15, cfg.vocab_size)
    hm = HipModel(hip_ctx, bundle)
    tok = hm.prefill(prompt)
    ref, _ = hm.decode(5)
    for mover in ("decode", "prefill"):
        hm.reset()
        assert hm.prefill(prompt) == tok
        flat = TrieNode.flat([tok, 5, 6]).linearize()
        hm.verify_tree(flat.token_ids(), flat.nodes())
        if mover == "decode":
            got, _ = hm.decode(5)  # the tree is dropped; the stream is the plain one
            assert np.array_equal(got, ref)
        else:
            hm.prefill(np.array([int(ref[0])], np.uint32))
        with pytest.raises(UzuHipError):  # nothing is pending any more
            hm.accept([0, 1])
        flat2 = TrieNode.flat([int(ref[-1]), 5]).linearize()
        hm.verify_tree(flat2.token_ids(), flat2.nodes())  # and a new tree can be verified (it was refused as "already pending" before)
        hm.accept([0])
    hm.close()


def test_a_pending_tree_survives_a_pass_over_another_sequence(hip_ctx):
    """One model, two sequence states: verify a tree on A, prefill B (and a batched prefill over B and C), bind A again, accept -- A's suffix rows and the
    tree buffers were not touched, so the accept goes through and the stream behind it is the one without the detour (the pending
    tree was dropped by ANY pass)."""
    cfg = S.tiny_qwen()
    bundle = S.build_model(cfg)
    prompt = S.synthetic_prompt(15, cfg.vocab_size)
    other = S.synthetic_prompt(9, cfg.vocab_size, variant=3)
    runs = []
    for detour in (False, True):
        hm = HipModel(hip_ctx, bundle, MODEL_BATCH(2))
        b, c = hm.new_state(), hm.new_state()
        tok = hm.prefill(prompt)
        flat = TrieNode.flat([tok, 5, 6]).linearize()
        sampled = hm.verify_tree(flat.token_ids(), flat.nodes())
        if detour:
            hm.bind(b)
            hm.prefill(other)
            hm.prefill_batch([b, c], np.stack([other[:4], other[4:8]]))
            hm.bind(None)
        hm.accept([0])
        nxt, _ = hm.decode(4)
        runs.append((list(sampled), [int(t) for t in nxt]))
        b.close(), c.close(), hm.close()
    assert runs[0] == runs[1]


@pytest.mark.parametrize("preset,kw", [("tiny-qwen", {"model_dim": 1024, "group_size": 128}), ("tiny-llama", {"model_dim": 1024, "group_size": 128, "method": 1}),
                                       ("tiny-qwen", {"model_dim": 1024, "group_size": 128, "norm_full_layer": False, "norm_scale_offset": 0.0})])
def test_few_rows_passes_run_the_normalization_in_the_linears_prologue(hip_ctx, preset, kw, monkeypatch):
    """Speculative verify passes and prefill tails of 2 or 3 rows: the pre-mixer Normalization rides in the prologue of the qkv / DeltaNet
    in-projection launch, the pre-MLP Normalization in the fused up | gate + GatedActMul launch (k_gemv_rows.hip, RowsNorm: every workgroup
    normalises the rows it stages, normalization_kernel's element mapping and reduction order; the residual rows ping-pong between two
    buffers).  Logits of every tree node, of a 3-row prefill tail and of the decode steps behind an accept must be BIT-IDENTICAL to the
    passes with separate Normalization launches (UZU_HIP_TUNE=rows_norm=0), with two launches per layer fewer.  (From four rows on the prologue
    costs more than the launch it saves -- every workgroup redoes every row -- and the engine keeps the separate kernel: engine_forward.hip::linear_normed.)"""
    cfg = S.PRESETS[preset](max_context_length=256, **kw)
    bundle = S.build_model(cfg)
    prompt = S.synthetic_prompt(50, cfg.vocab_size)
    runs = {}
    for mode in ("0", "1"):
        monkeypatch.setenv("UZU_HIP_TUNE", f"rows_norm={mode}")
        hm = HipModel(hip_ctx, bundle)
        hm.prefill(prompt[:47])
        tok = hm.prefill(prompt[47:])  # a 3-row tail
        tail_logits = hm.read_logits()
        root = TrieNode(tok)
        root.add(TrieNode(5)), root.add(TrieNode(9))
        flat = root.linearize()
        sampled = hm.verify_tree(flat.token_ids(), flat.nodes())
        tree_logits = hm.read_tree_logits()
        launches = hm.decode_launch_count
        acc = [i for i, _, _ in flat.accept(sampled)]
        hm.accept(acc)
        toks, _ = hm.decode(3)
        runs[mode] = (tok, tail_logits, [int(t) for t in sampled], tree_logits, [int(t) for t in toks], hm.read_logits(), launches)
        hm.close()
    a, b = runs["0"], runs["1"]
    assert a[0] == b[0] and np.array_equal(a[1], b[1]), "the 3-row prefill tail differs"
    assert a[2] == b[2] and np.array_equal(a[3], b[3]), "the tree pass differs"
    assert a[4] == b[4] and np.array_equal(a[5], b[5]), "the decode steps behind the accept differ"
    assert a[6] - b[6] == 2 * len(bundle.layers), f"launches of the tree pass: {a[6]} -> {b[6]} ({len(bundle.layers)} layers)"
