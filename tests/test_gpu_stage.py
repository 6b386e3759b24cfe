"""The HIP stage behind the xj_stage vtable and the device chain, against the
oracle's CPU stage with an fp16 KV cache, on identical seeded inputs.

Mirrors the reference's own GPU-vs-CPU check (src/xiaoju-pipe/tools/xjpipe-check.c:61-109):
prefill 12 tokens then 3 single tokens, head top-1, keep/rollback equal to
never having computed the rolled-back tokens; plus greedy token identity.
"""
import ctypes as C

import numpy as np
import pytest

import oracle as orc
import xjpipe as xp
from conftest import rel_l2
from helpers import in_child

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tiny(tiny_path):
    return xp.Model(tiny_path)


def embed(m, toks):
    return np.stack([orc.embed(m.ptr, int(t)) for t in toks]).astype(np.float32)


def prompt_ids(m, n, seed):
    return np.random.default_rng(seed).integers(0, m.hp.n_vocab, n).astype(np.int32)


def test_forward_and_head_match_oracle(tiny):
    m, L = tiny, tiny.hp.n_layer
    toks = prompt_ids(m, 15, 1)
    g = xp.HipStage(m, 0, L, 128, 16, True)
    c = orc.CpuStage(m.ptr, 0, L, 128, 16, True, kv_f16=True)
    pos = 0
    for T in (12, 1, 1, 1):
        x = embed(m, toks[pos:pos + T])
        xg, xc = g.forward(x.copy()), c.forward(x.copy())
        assert rel_l2(xg, xc) < 1e-3, T
        pos += T
    assert g.n_past == c.n_past == 15
    lg, lc = g.logits(xg[-1:]), c.logits(xc[-1:])
    assert rel_l2(lg, lc) < 1e-3
    assert int(np.argmax(lg)) == int(np.argmax(lc))
    g.destroy()
    c.destroy()


def test_two_stages_equal_one(tiny):
    m, L = tiny, tiny.hp.n_layer
    toks = prompt_ids(m, 10, 2)
    one = xp.HipStage(m, 0, L, 64, 8, True)
    a, b = xp.HipStage(m, 0, 4, 64, 8, False), xp.HipStage(m, 4, L, 64, 8, True)
    for T in (8, 2):
        x = embed(m, toks[:T]) if T == 8 else embed(m, toks[8:10])
        x1 = one.forward(x.copy())
        x2 = b.forward(a.forward(x.copy()))
        assert np.array_equal(x1, x2)
    for s in (one, a, b):
        s.destroy()


def test_keep_rollback_equals_never_computed(tiny):
    """forward 6, verify 4 with keep, roll back to 8, forward 2 others == forward the 10 kept tokens."""
    m, L = tiny, tiny.hp.n_layer
    toks = prompt_ids(m, 14, 3)
    g = xp.HipStage(m, 0, L, 64, 8, True)
    g.forward(embed(m, toks[:6]))
    g.set_keep(4)
    g.forward(embed(m, toks[6:10]))
    assert g.s.ck_start == 6 and g.s.ck_T == 4
    g.rollback(8)
    assert g.n_past == 8
    x_after = g.forward(embed(m, toks[12:14]))
    ref = xp.HipStage(m, 0, L, 64, 16, True)
    seq = np.concatenate([toks[:8], toks[12:14]])
    xr = ref.forward(embed(m, seq))
    assert rel_l2(x_after, xr[8:]) < 1e-6
    c = orc.CpuStage(m.ptr, 0, L, 64, 16, True, kv_f16=True)
    xc = c.forward(embed(m, seq))
    assert rel_l2(x_after, xc[8:]) < 1e-3
    for s in (g, ref, c):
        s.destroy()


def test_rollback_rules(tiny):
    m, L = tiny, tiny.hp.n_layer
    toks = prompt_ids(m, 8, 4)
    g = xp.HipStage(m, 0, L, 64, 8, True)
    g.forward(embed(m, toks[:4]))
    with pytest.raises(xp.XjError):       # no checkpoint window
        g.rollback(2)
    g.rollback(4)                          # unchanged position is a no-op
    g.set_keep(3)
    g.forward(embed(m, toks[4:7]))
    with pytest.raises(xp.XjError):       # outside [ck_start+1, ck_start+ck_T-1]
        g.rollback(4)
    g.rollback(6)
    # attention-only stage (layer 3 is full attention) truncates freely
    att = xp.HipStage(m, 3, 4, 64, 8, False)
    att.forward(embed(m, toks[:5]))
    att.rollback(2)
    assert att.n_past == 2
    with pytest.raises(xp.XjError):
        att.rollback(3)
    with pytest.raises(xp.XjError):       # T > max_batch
        g.forward(embed(m, np.zeros(9, np.int32)))
    g.destroy()
    att.destroy()


def test_reset_and_context_limit(tiny):
    m, L = tiny, tiny.hp.n_layer
    toks = prompt_ids(m, 8, 5)
    g = xp.HipStage(m, 0, L, 8, 8, True)
    x1 = g.forward(embed(m, toks))
    with pytest.raises(xp.XjError):
        g.forward(embed(m, toks[:1]))      # context full
    g.reset()
    assert g.n_past == 0
    x2 = g.forward(embed(m, toks))
    assert np.array_equal(x1, x2)
    g.destroy()


def test_chain_greedy_matches_oracle(tiny):
    m, L = tiny, tiny.hp.n_layer
    prompt = prompt_ids(m, 21, 6)
    g = xp.HipStage(m, 0, L, 256, 8, True)
    ch = xp.Chain([g])
    toks = np.concatenate([ch.eval(prompt), ch.decode(63)])
    c = orc.CpuStage(m.ptr, 0, L, 256, 8, True, kv_f16=True)
    want, margins = orc.greedy([c], prompt, 64)
    assert np.array_equal(toks, want), (toks, want, margins)
    ch.free()
    g.destroy()
    c.destroy()


def test_decode_never_reads_unwritten_cache(tiny):
    """The cache slots at and past the decode position hold whatever the memory held (here an fp16 NaN in
    every slot) until a step writes them; a single-token step writes its own slot inside the attention
    kernel, so it must not combine those bytes, not even with a zero weight (0 * NaN = NaN)."""
    m, L = tiny, tiny.hp.n_layer
    prompt = prompt_ids(m, 21, 6)
    g = xp.HipStage(m, 0, L, 256, 8, True)
    ch = xp.Chain([g])
    first = ch.eval(prompt)
    g.fill_kv(len(prompt), 0x7E00)
    toks = np.concatenate([first, ch.decode(40)])
    c = orc.CpuStage(m.ptr, 0, L, 256, 8, True, kv_f16=True)
    want, margins = orc.greedy([c], prompt, 41)
    assert np.array_equal(toks, want), (toks, want, margins)
    ch.free()
    g.destroy()
    c.destroy()


def test_chain_split_and_vtable_agree(tiny):
    """Two chained stages on the device give the same tokens as the host-driven vtable loop."""
    m, L = tiny, tiny.hp.n_layer
    prompt = prompt_ids(m, 9, 7)
    a, b = xp.HipStage(m, 0, 4, 128, 8, False), xp.HipStage(m, 4, L, 128, 8, True)
    ch = xp.Chain([a, b])
    toks = np.concatenate([ch.eval(prompt), ch.decode(31)])
    ch.free()
    a.destroy()
    b.destroy()
    g = xp.HipStage(m, 0, L, 128, 8, True)
    x = g.forward(embed(m, prompt[:8]))
    x = g.forward(embed(m, prompt[8:]))
    host = []
    for _ in range(32):
        t = int(np.argmax(g.logits(x[-1:])[0]))
        host.append(t)
        x = g.forward(embed(m, [t]))
    assert toks.tolist() == host
    g.destroy()


@pytest.mark.parametrize("cuts", [(0, 4, 8), (0, 2, 5, 8)])
def test_pipelined_chain_prefill_equals_one_stage(tiny, cuts):
    """A prompt beyond max_batch through a chain whose stages run on their own
    streams (xj_net.c:561-604), here as one piece handed from stage to stage:
    the logits of the last rows, the hidden rows left for the drivers and the
    tokens decoded after it equal those of one stage, bit for bit."""
    m, L = tiny, tiny.hp.n_layer
    assert cuts[-1] == L
    prompt = prompt_ids(m, 70, 29)            # max_batch 16: one piece of 70
    one = xp.HipStage(m, 0, L, 128, 16, True)
    c1 = xp.Chain([one])
    am1, lg1 = c1.eval(prompt, nlog=3, want_logits=True)
    t1 = c1.decode(12)
    sts = [xp.HipStage(m, cuts[i], cuts[i + 1], 128, 16, i + 2 == len(cuts)) for i in range(len(cuts) - 1)]
    c2 = xp.Chain(sts)
    am2, lg2 = c2.eval(prompt, nlog=3, want_logits=True)
    assert np.array_equal(lg1.view(np.uint32), lg2.view(np.uint32))
    assert am1.tolist() == am2.tolist()
    assert c2.decode(12).tolist() == t1.tolist()
    # again from a reset state: the device positions restart with the host's
    c2.reset()
    c1.reset()
    a1 = c1.eval(prompt[:37])
    a2 = c2.eval(prompt[:37])
    assert a1.tolist() == a2.tolist()
    for c in (c1, c2):
        c.free()
    for st in [one] + sts:
        st.destroy()


@pytest.mark.parametrize("cuts", [(0, 4, 8), (0, 2, 5, 8)])
def test_pipelined_pieces_equal_one_stage(tiny, cuts):
    """2600 tokens: pieces of 1024, 1024 and 552, piece k + 1 in stage i while
    piece k is in stage i + 1, so that a stage's buffer is overwritten only once
    the next stage has taken it: the logits of the last rows and the tokens
    decoded after them equal those of one stage, bit for bit, twice in a row."""
    m, L = tiny, tiny.hp.n_layer
    prompt = prompt_ids(m, 2600, 31)
    one = xp.HipStage(m, 0, L, 2688, 16, True)
    c1 = xp.Chain([one])
    am1, lg1 = c1.eval(prompt, nlog=8, want_logits=True)   # the last chunk of max_batch holds 8 rows
    t1 = c1.decode(12).tolist()
    sts = [xp.HipStage(m, cuts[i], cuts[i + 1], 2688, 16, i + 2 == len(cuts)) for i in range(len(cuts) - 1)]
    c2 = xp.Chain(sts)
    for _ in range(2):
        c2.reset()
        am2, lg2 = c2.eval(prompt, nlog=8, want_logits=True)
        assert np.array_equal(lg1.view(np.uint32), lg2.view(np.uint32))
        assert am1.tolist() == am2.tolist()
        assert c2.decode(12).tolist() == t1
    for c in (c1, c2):
        c.free()
    for st in [one] + sts:
        st.destroy()


@pytest.mark.parametrize("cuts", [(0, 4, 8), (0, 2, 5, 8)])
def test_pipelined_chunks_equal_one_stage(tiny_path, cuts):
    """The same in chunks of max_batch (XJ_PREFILL_GEMM=0: no pieces): 70 tokens
    in chunks of 16 x 4 + 6 through two and three stages, against one stage whose
    layers run undivided (XJ_STAGE_SPLIT=1), bit for bit."""
    in_child(f"""
        import numpy as np, xjpipe as xp
        m = xp.Model({tiny_path!r})
        L, cuts = m.hp.n_layer, {cuts!r}
        ids = np.random.default_rng(29).integers(0, m.hp.n_vocab, 70).astype(np.int32)
        one = xp.HipStage(m, 0, L, 128, 16, True)
        c1 = xp.Chain([one])
        am1, lg1 = c1.eval(ids, nlog=3, want_logits=True)
        t1 = c1.decode(12).tolist()
        sts = [xp.HipStage(m, cuts[i], cuts[i + 1], 128, 16, i + 2 == len(cuts)) for i in range(len(cuts) - 1)]
        c2 = xp.Chain(sts)
        for _ in range(2):
            c2.reset()
            am2, lg2 = c2.eval(ids, nlog=3, want_logits=True)
            assert np.array_equal(lg1.view(np.uint32), lg2.view(np.uint32))
            assert am1.tolist() == am2.tolist()
            assert c2.decode(12).tolist() == t1
        for o in (c1, c2):
            o.free()
        for o in [one] + sts:
            o.destroy()
        """, XJ_PREFILL_GEMM="0", XJ_STAGE_SPLIT="1")


def test_chain_verify_and_rollback(tiny):
    m, L = tiny, tiny.hp.n_layer
    prompt = prompt_ids(m, 16, 8)
    g = xp.HipStage(m, 0, L, 128, 8, True)
    ch = xp.Chain([g])
    ch.eval(prompt)
    greedy = ch.decode(5)                       # reference continuation
    g2 = xp.HipStage(m, 0, L, 128, 8, True)
    c2 = xp.Chain([g2])
    first = c2.eval(prompt)
    cand = np.concatenate([first, greedy[:4]])  # [t, d1..d4] all correct
    am = c2.eval(cand, nlog=5, keep=True)
    assert am.tolist() == greedy.tolist()
    c2.rollback(16 + 2)                          # keep t, d1
    nxt = c2.eval(greedy[1:2])
    assert int(nxt[0]) == int(greedy[2])
    for o in (ch, c2):
        o.free()
    g.destroy()
    g2.destroy()


def test_verify_pass_logits_equal_single_steps(tiny):
    """A 5-token verification pass gives, bit for bit, the logits of feeding
    the same tokens one at a time (the decode step's kernels)."""
    m, L = tiny, tiny.hp.n_layer
    prompt, cand = prompt_ids(m, 16, 8), prompt_ids(m, 5, 9)
    g1, g2 = xp.HipStage(m, 0, L, 128, 8, True), xp.HipStage(m, 0, L, 128, 8, True)
    c1, c2 = xp.Chain([g1]), xp.Chain([g2])
    c1.eval(prompt)
    c2.eval(prompt)
    _, lg5 = c1.eval(cand, nlog=5, keep=True, want_logits=True)
    lg1 = np.stack([c2.eval(cand[i:i + 1], nlog=1, want_logits=True)[1][0] for i in range(5)])
    assert np.array_equal(lg5.view(np.uint32), lg1.view(np.uint32))
    for o in (c1, c2):
        o.free()
    g1.destroy()
    g2.destroy()


@pytest.mark.parametrize("mode", ["draft", "oracle_all", "oracle_miss", "oracle_guess_miss"])
def test_spec_decode_equals_greedy(tiny, tiny_draft_path, mode):
    """Speculative generation equals plain greedy decoding. oracle_guess_miss:
    oracle drafts with wrong tokens at positions 15 and 31, where fully
    accepted rounds that overlap the next round's drafting with their
    verification guess the target's next token (the guess fails, the draft
    returns to its state after the round's last draft)."""
    m, L = tiny, tiny.hp.n_layer
    dm = xp.Model(tiny_draft_path)
    prompt = prompt_ids(m, 13, 9)
    n_gen = 40
    g = xp.HipStage(m, 0, L, 256, 8, True)
    ch = xp.Chain([g])
    plain = np.concatenate([ch.eval(prompt), ch.decode(n_gen - 1)])
    ch.free()
    g.destroy()
    t = xp.HipStage(m, 0, L, 256, 8, True)
    d = xp.HipStage(dm, 0, dm.hp.n_layer, 256, 8, True)
    tc, dc = xp.Chain([t]), xp.Chain([d])
    tc.eval(prompt)
    dc.eval(prompt)
    oracle = None if mode == "draft" else plain.copy()
    if mode == "oracle_guess_miss":
        V = int(m.hp.n_vocab)
        for gi in (15, 31):
            oracle[gi] = (oracle[gi] + 1) % V
    miss = 3 if mode == "oracle_miss" else 0
    out, st = xp.spec_generate(tc, dc, 4, n_gen, oracle=oracle, oracle_miss=miss)
    assert out.tolist() == plain.tolist()
    if mode == "oracle_all":
        assert st.n_accepted == st.n_drafted
        assert st.n_overlap_held == st.n_overlap > 0
    if mode == "oracle_guess_miss":
        assert 0 < st.n_overlap_held < st.n_overlap
    for o in (tc, dc):
        o.free()
    t.destroy()
    d.destroy()


def test_stage_over_a_layer_range_load(tiny, tiny_path, tmp_path):
    """A stage built from xj_model_load_layers on a file cut after its layers
    (a partial download, xj_model.c:214-233) computes bit for bit what the stage
    built from the whole file computes; a stage over layers outside the mapping
    is refused."""
    m, L = tiny, tiny.hp.n_layer
    part0 = xp.Model(tiny_path, layers=(0, L // 2))
    hi = part0.ranges(0, L // 2)[-1][1]
    part0.close()
    cut = str(tmp_path / "front.gguf")
    with open(tiny_path, "rb") as f, open(cut, "wb") as g:
        g.write(f.read(hi))
    part = xp.Model(cut, layers=(0, L // 2))
    toks = prompt_ids(m, 9, 5)
    x = embed(m, toks)
    a = xp.HipStage(part, 0, L // 2, 64, 16, False)
    b = xp.HipStage(m, 0, L // 2, 64, 16, False)
    xa, xb = a.forward(x[:8].copy()), b.forward(x[:8].copy())
    assert np.array_equal(xa, xb)
    xa, xb = a.forward(x[8:].copy()), b.forward(x[8:].copy())
    assert np.array_equal(xa, xb)
    a.destroy()
    b.destroy()
    with pytest.raises(xp.XjError, match="not mapped"):
        xp.HipStage(part, L // 2, L, 64, 16, False)
    with pytest.raises(xp.XjError, match="not mapped"):
        xp.HipStage(part, 0, L // 2, 64, 16, True)
    part.close()


class RefLoaded:
    """A model table built by the reference's own loader (xj_model_load,
    core/xj_model.c:204), seen through the boundary struct."""

    def __init__(self, path, mtp_from=None):
        err = orc.C.create_string_buffer(512)
        r = orc.rlib().ref_model_load(path.encode(), err, 512)
        assert r, err.value
        if mtp_from:
            assert orc.rlib().ref_model_attach_mtp(r, mtp_from.encode(), err, 512) == 0, err.value
        self.r = r
        self.ptr = orc.C.cast(r, orc.C.POINTER(xp.XjModel))

    @property
    def hp(self):
        return self.ptr.contents.hp

    def free(self):
        orc.rlib().ref_model_free(self.r)


@pytest.mark.skipif(not orc.ref_available(), reason="reference build (oracle/_ref) not present")
def test_hip_stages_over_the_reference_loader(model_dir, tiny_path):
    """The literal drop-in (core/xj_stage.h:46): xj_hip_stage_new over a model
    that the reference's own loader built, driven by the reference's own
    pipeline and greedy driver (split 0-3 | 3-8, as xjpipe-host runs it):
    the oracle's fp16-KV greedy tokens, and bit for bit the tokens of HIP
    stages over this library's loader. The MTP layer attached by the
    reference's xj_model_attach_mtp (core/xj_model.c:275-300) from a second
    file serves a HIP MTP stage whose drafts leave the output unchanged."""
    from conftest import synth_model
    rec_prompt = prompt_ids(xp.Model(tiny_path), 24, 41)
    mine = xp.Model(tiny_path)
    L = mine.hp.n_layer
    ref = RefLoaded(tiny_path, mtp_from=synth_model(model_dir, xp.TINY_MTP, "tiny_mtp"))
    n_gen = 32

    def drive(model, k):
        a, b = xp.HipStage(model, 0, 3, 256, 8, False), xp.HipStage(model, 3, L, 256, 8, True)
        mt = xp.HipStage(model, L, L + 1, 256, 8, True) if k else None
        out, st = orc.ref_spec_run(model.ptr, a.ptr, b.ptr, mt.ptr if mt else None, k, rec_prompt, n_gen)
        for s in (a, b, mt):
            if s:
                s.destroy()
        return out, st

    c = orc.CpuStage(mine.ptr, 0, L, 256, 8, True, kv_f16=True)
    want, _ = orc.greedy([c], rec_prompt, n_gen)
    c.destroy()
    got_ref, _ = drive(ref, 0)
    got_mine, _ = drive(mine, 0)
    assert got_ref.tolist() == got_mine.tolist() == want.tolist()
    spec, st = drive(ref, 3)
    assert spec.tolist() == want.tolist() and st[1] > 0
    ref.free()


@pytest.mark.parametrize("T", [16, 40, 64])
def test_prefill_chunk_matches_oracle(tiny, T):
    """A prefill chunk of at least 16 tokens takes the matrix-core path: GEMM
    projections (RMSNorm scale per token after the dot products), the conv +
    SiLU launch, the chunked delta rule over prepared q/k/v/decay/beta (GQA
    heads: key head hv % Hk), the gated RMSNorm as ssm_out's prep. Hidden states
    against the oracle, then decode steps continue from the chunk's recurrent
    and KV state."""
    m, L = tiny, tiny.hp.n_layer
    toks = prompt_ids(m, T + 3, 21 + T)
    g = xp.HipStage(m, 0, L, 128, 64, True)
    c = orc.CpuStage(m.ptr, 0, L, 128, 64, True, kv_f16=True)
    x = embed(m, toks[:T])
    xg, xc = g.forward(x.copy()), c.forward(x.copy())
    assert rel_l2(xg, xc) < 1e-3
    for t in range(T, T + 3):
        x1 = embed(m, toks[t:t + 1])
        yg, yc = g.forward(x1.copy()), c.forward(x1.copy())
        assert rel_l2(yg, yc) < 1e-3, t
    lg, lc = g.logits(yg), c.logits(yc)
    assert rel_l2(lg, lc) < 1e-3
    assert int(np.argmax(lg)) == int(np.argmax(lc))
    g.destroy()
    c.destroy()


def test_prefill_chunk_with_checkpoints_rolls_back(tiny):
    """A 20-token chunk with keep: GEMM projections, the conv launch writing
    its checkpoints, the recurrent rule writing the state checkpoints; rolled
    back into the chunk it continues as a fresh stage fed the kept prefix
    (which itself takes the chunked rule, 18 tokens without keep)."""
    m, L = tiny, tiny.hp.n_layer
    toks = prompt_ids(m, 40, 22)
    g = xp.HipStage(m, 0, L, 128, 64, True)
    g.forward(embed(m, toks[:8]))
    g.set_keep(20)
    g.forward(embed(m, toks[8:28]))
    g.rollback(14)
    assert g.n_past == 14
    x_after = g.forward(embed(m, toks[30:34]))
    ref = xp.HipStage(m, 0, L, 128, 64, True)
    xr = ref.forward(embed(m, np.concatenate([toks[:14], toks[30:34]])))
    assert rel_l2(x_after, xr[14:]) < 1e-4
    c = orc.CpuStage(m.ptr, 0, L, 128, 64, True, kv_f16=True)
    xc = c.forward(embed(m, np.concatenate([toks[:14], toks[30:34]])))
    assert rel_l2(x_after, xc[14:]) < 1e-3
    for s_ in (g, ref, c):
        s_.destroy()



@pytest.mark.parametrize("T", [11, 15])
def test_short_chunk_on_the_gemm(tiny, T):
    """Eleven to fifteen tokens take the GEMM with the decode's attention and
    DeltaNet kernels: hidden rows against the same tokens one at a time, and a
    step after them. Bound: products 1e-6
    apart (21- against 22-bit activations) round about 1e-6 / 2^-11 = 0.2% of
    the fp16 keys and values the other way, each by 2^-11 of itself: 2e-5 of an
    attention output, in two of the tiny model's eight layers, whose later
    layers' norms and gates add up to a factor of a few (measured 7e-5)."""
    m, L = tiny, tiny.hp.n_layer
    toks = prompt_ids(m, T + 1, 600 + T)
    a, b = xp.HipStage(m, 0, L, 64, 16, True), xp.HipStage(m, 0, L, 64, 16, True)
    ya = a.forward(embed(m, toks[:T]))
    yb = np.concatenate([b.forward(embed(m, toks[i:i + 1])) for i in range(T)])
    assert rel_l2(ya, yb) < 2e-4
    assert rel_l2(a.forward(embed(m, toks[T:])), b.forward(embed(m, toks[T:]))) < 2e-4
    for s in (a, b):
        s.destroy()


@pytest.mark.parametrize("T", [11, 15])
def test_short_chunk_with_checkpoints_keeps_the_steps_bits(tiny, T):
    """With checkpoints a chunk of eleven to fifteen tokens is a verification:
    its rows, and the step after a rollback into it, are those of the tokens
    fed one at a time, bit for bit."""
    m, L = tiny, tiny.hp.n_layer
    toks = prompt_ids(m, T + 2, 600 + T)
    a, b = xp.HipStage(m, 0, L, 64, 16, True), xp.HipStage(m, 0, L, 64, 16, True)
    a.set_keep(T)
    ya = a.forward(embed(m, toks[:T]))
    yb = np.concatenate([b.forward(embed(m, toks[i:i + 1])) for i in range(T - 1)])
    assert np.array_equal(ya[:-1].view(np.uint32), yb.view(np.uint32))
    a.rollback(T - 1)
    ya, yb = (s.forward(embed(m, toks[T:])[:1]) for s in (a, b))
    assert np.array_equal(ya.view(np.uint32), yb.view(np.uint32))
    for s in (a, b):
        s.destroy()


@pytest.mark.parametrize("T", [65, 96, 129, 200, 256])
def test_wide_chunk_equals_chunks_of_64(tiny, T):
    """A chunk beyond 64 tokens takes the narrow GEMM in slices of 64 (65: a
    slice of one token) or, for the tiny model's matrices from 193 tokens on,
    the wide one (256 x 128 tiles over every segment; 200 and 256: a ragged
    and a whole second token group); its hidden rows are those of the same
    tokens in chunks of 64, and the state it leaves serves a decode step. Both round only in fp32 sums: 1e-6 of a
    product, 6e-6 after four layers."""
    m, L = tiny, tiny.hp.n_layer
    toks = prompt_ids(m, T + 1, 300 + T)
    a = xp.HipStage(m, 0, L, 320, 256, True)
    b = xp.HipStage(m, 0, L, 320, 64, True)
    x = embed(m, toks[:T])
    ya = a.forward(x.copy())
    yb = np.concatenate([b.forward(x[i:i + 64].copy()) for i in range(0, T, 64)])
    assert rel_l2(ya, yb) < 5e-5
    x1 = embed(m, toks[T:])
    assert rel_l2(a.forward(x1.copy()), b.forward(x1.copy())) < 5e-5
    c = orc.CpuStage(m.ptr, 0, L, 320, 256, True, kv_f16=True)
    assert rel_l2(ya, c.forward(x.copy())) < 1e-3
    for s in (a, b, c):
        s.destroy()


@pytest.mark.parametrize("n,mb", [(40, 16), (200, 16), (16, 8), (17, 8), (1030, 64), (1601, 64)])
def test_chain_prompt_pieces(tiny, n, mb):
    """A prompt beyond max_batch goes through the layers in pieces of up to
    1024 tokens (1030: 512 + 518, so that the last piece holds max_batch
    rows; two chunks of 8 stay chunks): the logits of its
    last rows are those of the vtable's chunks, one chain of two stages gives
    them bit for bit, and decoding continues from its state."""
    m, L = tiny, tiny.hp.n_layer
    prompt = prompt_ids(m, n, 400 + n)
    one = xp.HipStage(m, 0, L, 2048, mb, True)
    c1 = xp.Chain([one])
    nl = min(3, n - (n - 1) // mb * mb)
    am1, lg1 = c1.eval(prompt, nlog=3, want_logits=True)
    ref = xp.HipStage(m, 0, L, 2048, mb, True)
    x = embed(m, prompt)
    y = np.concatenate([ref.forward(x[i:i + mb].copy()) for i in range(0, n, mb)])
    want = ref.logits(y[-nl:])
    assert rel_l2(lg1[:nl], want) < 2e-4
    sts = [xp.HipStage(m, 0, 3, 2048, mb, False), xp.HipStage(m, 3, L, 2048, mb, True)]
    c2 = xp.Chain(sts)
    am2, lg2 = c2.eval(prompt, nlog=3, want_logits=True)
    assert np.array_equal(lg1[:nl].view(np.uint32), lg2[:nl].view(np.uint32))
    assert c2.decode(6).tolist() == c1.decode(6).tolist()
    for c in (c1, c2):
        c.free()
    for s in [one, ref] + sts:
        s.destroy()


@pytest.mark.parametrize("H,Hkv,D", [(4, 4, 64), (8, 1, 64), (2, 1, 128), (4, 4, 128), (4, 1, 256), (8, 1, 256)])
@pytest.mark.parametrize("n_past,T", [(0, 16), (0, 130), (63, 17), (64, 64), (200, 33)])
def test_chunk_attention_equals_single_steps(model_dir, H, Hkv, D, n_past, T):
    """The matrix-core attention of chunks of 16 tokens and more (64 query
    rows per work-group over all group sizes, tiles of 64 positions cut by the
    prefix and the diagonal, splits merged) against the decode kernels: the
    same layers fed the same rows one at a time. Unwritten cache positions
    hold NaN. Both differ from float64 by fp32 sums and 21- to 22-bit
    activations: 6e-6 after four layers."""
    from conftest import synth_model
    cfg = xp.TINY.with_(n_layer=4, n_head=H, n_head_kv=Hkv, head_dim=D)
    m = xp.Model(synth_model(model_dir, cfg, "tiny_h%d_%d_%d" % (H, Hkv, D)))
    a, b = (xp.HipStage(m, 0, 4, 288, 144, False) for _ in range(2))
    rows = np.random.default_rng(T + n_past).standard_normal((n_past + T, cfg.n_embd)).astype(np.float32)
    for s in (a, b):
        s.fill_kv(0, 0x7E00)
        for i in range(0, n_past, 8):
            s.forward(rows[i:min(i + 8, n_past)].copy())
    ya = a.forward(rows[n_past:].copy())
    yb = np.concatenate([b.forward(rows[n_past + i:n_past + i + 1].copy()) for i in range(T)])
    assert rel_l2(ya, yb) < 5e-5
    for s in (a, b):
        s.destroy()


@pytest.mark.parametrize("conv_k,s_k,T", [(2, 64, 16), (3, 128, 23), (4, 128, 17), (8, 64, 65)])
def test_chunk_conv_equals_single_steps(model_dir, conv_k, s_k, T):
    """The conv + SiLU and L2 norms of a chunk in one launch (eight tokens per
    wavefront, inputs before the chunk from the conv state, two value heads
    per key head) and the state it leaves, over kernel sizes: hidden rows of a
    chunk after five tokens and of two steps after it, against the same rows
    fed one at a time."""
    from conftest import synth_model
    cfg = xp.TINY.with_(n_layer=4, conv_k=conv_k, s_k=s_k, h_k=2, h_v=4)
    m = xp.Model(synth_model(model_dir, cfg, "tiny_c%d_%d" % (conv_k, s_k)))
    a, b = (xp.HipStage(m, 0, 4, 128, 96, False) for _ in range(2))
    rows = np.random.default_rng(T).standard_normal((T + 7, cfg.n_embd)).astype(np.float32)
    a.forward(rows[:5].copy())
    ya = np.concatenate([a.forward(rows[5:5 + T].copy())] + [a.forward(rows[i:i + 1].copy()) for i in (T + 5, T + 6)])
    yb = np.concatenate([b.forward(rows[i:i + 1].copy()) for i in range(T + 7)])[5:]
    assert rel_l2(ya, yb) < 5e-5
    for s in (a, b):
        s.destroy()


@pytest.mark.parametrize("H,Hkv,D", [(8, 1, 64), (4, 1, 256)])
@pytest.mark.parametrize("n_past,T,bad", [(0, 16, 5), (63, 17, 10), (200, 33, 20), (0, 130, 100)])
def test_nan_token_leaves_earlier_rows_alone(model_dir, H, Hkv, D, n_past, T, bad):
    """A token whose row is NaN, in the middle of a chunk on the matrix cores
    (one split and several): the rows before it see neither its key nor its
    value, so they are those of the same chunk with a finite row there (the
    bound of two orders of the same fp32 sums, as against single steps); every
    row from it on is NaN."""
    from conftest import synth_model
    cfg = xp.TINY.with_(n_layer=4, n_head=H, n_head_kv=Hkv, head_dim=D)
    m = xp.Model(synth_model(model_dir, cfg, "tiny_h%d_%d_%d" % (H, Hkv, D)))
    s = xp.HipStage(m, 3, 4, 288, 144, False)   # the attention layer alone
    rows = np.random.default_rng(T + n_past).standard_normal((n_past + T, cfg.n_embd)).astype(np.float32)
    if n_past:
        for i in range(0, n_past, 100):
            s.forward(rows[i:min(i + 100, n_past)].copy())
    want = s.forward(rows[n_past:].copy())
    s.rollback(n_past)
    x = rows[n_past:].copy()
    x[bad] = np.nan
    got = s.forward(x)
    assert rel_l2(got[:bad], want[:bad]) < 5e-5
    assert np.isnan(got[bad:]).all()
    s.destroy()


def test_chunk_on_the_gemv_keeps_the_steps_bits(tiny_path):
    """Chunks kept on the GEMV's arithmetic (XJ_PREFILL_GEMM=0, read once per
    process) take the decode's attention too: 70 rows with checkpoints, and a
    step after a rollback into them, are those of the rows fed one at a time,
    bit for bit."""
    in_child(f"""
        import numpy as np, xjpipe as xp
        m = xp.Model({tiny_path!r})
        rows = np.random.default_rng(5).standard_normal((72, m.hp.n_embd)).astype(np.float32)
        a, b = (xp.HipStage(m, 0, m.hp.n_layer, 128, 96, False) for _ in range(2))
        a.set_keep(70)
        ya = a.forward(rows[:70].copy())
        yb = np.concatenate([b.forward(rows[i:i + 1].copy()) for i in range(33)])
        assert np.array_equal(ya[:33].view(np.uint32), yb.view(np.uint32))
        a.rollback(33)
        ya, yb = (s.forward(rows[70:71].copy()) for s in (a, b))
        assert np.array_equal(ya.view(np.uint32), yb.view(np.uint32))
        for s in (a, b):
            s.destroy()
        """, XJ_PREFILL_GEMM="0")


def test_short_prompt_takes_little_memory(tiny):
    """A prompt just beyond a small max_batch must not allocate the scratch of
    1024-token pieces (over 100 MB for this model, 1 GB for the 4B shape):
    only further sets of the stage's own scratch, of max_batch tokens."""
    m, L = tiny, tiny.hp.n_layer
    path = next(l.split()[-1] for l in open("/proc/self/maps") if "libamdhip64" in l)
    hip = C.CDLL(path)

    def free():
        f, t = C.c_size_t(), C.c_size_t()
        assert hip.hipMemGetInfo(C.byref(f), C.byref(t)) == 0
        return f.value

    g = xp.HipStage(m, 0, L, 2048, 8, True)
    ch = xp.Chain([g])
    before = free()
    ch.eval(prompt_ids(m, 9, 3))
    assert before - free() < 32 << 20
    ch.free()
    g.destroy()


@pytest.mark.parametrize("n,mb,split", [(70, 16, 3), (70, 16, 4), (9, 4, 2), (33, 32, 3)])
def test_layers_in_parts_equal_chunks_in_turn(tiny_path, n, mb, split):
    """A prompt that goes in chunks of max_batch through a single stage
    (XJ_PREFILL_GEMM=0: no pieces) runs its layers in parts on streams of
    their own, each part's buffer overwritten only once the next has taken it:
    the logits of the last rows and the tokens decoded after it are those of
    the same chunks one after the other, bit for bit, twice in a row."""
    in_child(f"""
        import numpy as np, xjpipe as xp
        m = xp.Model({tiny_path!r})
        L, n, mb = m.hp.n_layer, {n}, {mb}
        ids = np.random.default_rng(n).integers(0, m.hp.n_vocab, n).astype(np.int32)
        def tail():
            return n - (n - 1) // mb * mb
        a, b = xp.HipStage(m, 0, L, 128, mb, True), xp.HipStage(m, 0, L, 128, mb, True)
        ca, cb = xp.Chain([a]), xp.Chain([b])
        for i in range(0, n, mb):
            am, want = cb.eval(ids[i:i + mb], nlog=tail(), want_logits=True)
        toks = cb.decode(6).tolist()
        for _ in range(2):
            ca.reset()
            am2, got = ca.eval(ids, nlog=mb, want_logits=True)
            assert np.array_equal(got[:tail()].view(np.uint32), want.view(np.uint32))
            assert ca.decode(6).tolist() == toks
        for o in (ca, cb):
            o.free()
        for o in (a, b):
            o.destroy()
        """, XJ_PREFILL_GEMM="0", XJ_STAGE_SPLIT=str(split))
