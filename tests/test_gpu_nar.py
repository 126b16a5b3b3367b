"""Acoustic-model attention on the GPU (yuear_nar_attention, the drop-in for
nar_attention() and its Metal kernel lyra_nar_precise_attention,
nar_attention.cpp:63-270) against the oracle's restatement, at the
conditioning and acoustic-chunk shapes of the 3B / YuE2 layers and at the
edges (one query, one key, key counts off the 32-key blocks, causal), plus
the reference's ValueError checks (nar_attention.cpp:227-243)."""
import numpy as np
import pytest

from conftest import assert_close_bf16

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch as t
    t.cuda.init()
    return t


def bf(x):
    import cpu_ref
    return cpu_ref.f32_to_bf16(np.asarray(x, dtype=np.float32))


def dev(torch, a):
    return torch.from_numpy(np.ascontiguousarray(a).view(np.int16)).cuda().view(torch.bfloat16)


def host(torch, t):
    torch.cuda.synchronize()
    return t.view(torch.int16).cpu().numpy().view(np.uint16)


@pytest.mark.parametrize("B,Hq,Hkv,Lq,Lk,causal", [
    (1, 16, 8, 130, 700, False),   # YuE2 heads: acoustic chunk over cached AR keys + its own
    (1, 24, 8, 300, 1100, False),  # 3B heads
    (2, 4, 2, 9, 65, False),       # batch 2, short chunk, keys off the 32-key blocks
    (1, 4, 2, 1, 33, False),       # one query
    (1, 4, 4, 40, 1, False),       # one key
    (1, 16, 8, 257, 257, True),    # causal conditioning prefill
    (2, 6, 3, 64, 64, True),
    # whole 64-query tiles, one or two key blocks a step (ragged last tiles)
    (2, 24, 8, 1000, 1100, False),
    (1, 24, 8, 2050, 2050, True),
    (32, 24, 8, 64, 1, False),     # 768 workgroups of 64 queries over one key
    (16, 24, 8, 130, 130, True),   # 1152 workgroups, causal, 2-query last tiles
    # keys dealt over workgroups
    (1, 16, 8, 64, 2570, False),   # 16-query tiles, 81 key blocks
    (1, 24, 8, 512, 3512, False),  # the benchmarked acoustic chunk over conditioning keys
    (1, 16, 8, 4, 3100, False),    # 4 queries in one tile, 12-13 workgroups a tile
    (2, 16, 8, 100, 1500, False),  # batch 2, whole key-split tiles, ragged last one
])
def test_nar_attention_matches_oracle(torch, yuear_lib, oracle, B, Hq, Hkv, Lq, Lk, causal):
    print(f"[nar] B={B} Hq={Hq} Hkv={Hkv} Lq={Lq} Lk={Lk} causal={causal}", flush=True)
    rng = np.random.default_rng(Lq * 7 + Lk)
    q = bf(rng.normal(size=(B, Hq, Lq, 128)))
    k = bf(rng.normal(size=(B, Hkv, Lk, 128)))
    v = bf(rng.normal(size=(B, Hkv, Lk, 128)))
    ref = oracle.nar_attention(q, k, v, causal)
    got = yuear_lib.nar_attention(dev(torch, q), dev(torch, k), dev(torch, v), causal)
    assert_close_bf16(host(torch, got), ref, exact_frac=0.8)


@pytest.mark.parametrize("B,Hq,Hkv,Lq,Lk,causal", [
    # whole key-split tiles of 16 and 32 queries, 4 and 8 waves: fewer blocks
    # than waves, a partial last block, a last tile of one query
    (1, 1, 1, 1, 31, False), (2, 6, 3, 17, 289, False), (1, 1, 1, 1, 697, False),
    (1, 6, 3, 677, 919, False), (1, 24, 8, 300, 1100, False), (1, 24, 8, 250, 3600, False),
    (1, 24, 8, 1001, 1500, False), (1, 24, 8, 341, 1500, False),
    # dealt to all CUs: key-split tiles of 16 and 32 queries by 8 waves, steps
    # and blocks that do not divide, a ragged last tile
    (2, 16, 8, 1, 4001, False), (1, 16, 8, 53, 2000, False), (1, 24, 8, 53, 6500, False),
    (1, 6, 3, 274, 6000, False), (1, 16, 8, 100, 8001, False),
    # ... to fewer workgroups, as few keys or heads allow: 8, 56, 64, 104, 208, 24
    (1, 1, 1, 1, 20000, False), (1, 1, 1, 100, 2000, False), (1, 2, 1, 33, 8001, False),
    (1, 2, 2, 130, 1500, False), (1, 16, 8, 17, 12001, False), (1, 1, 1, 65, 1500, False),
    # ... 4 waves, 264 and 360 workgroups of 16 queries, 256 of 32; 64-query tiles, an
    # odd last block
    (1, 1, 1, 341, 3001, False), (1, 6, 2, 65, 3001, False), (1, 2, 1, 341, 6001, False),
    (1, 24, 8, 500, 3470, False),
    # 64-query tiles, one and two blocks a step, an odd last block; causal forms
    (1, 12, 4, 677, 31, False), (1, 24, 8, 1024, 400, False), (1, 48, 16, 1025, 97, False),
    (1, 24, 8, 1001, 289, False), (1, 24, 8, 100, 100, True),
    (1, 24, 8, 449, 449, True), (1, 48, 16, 850, 850, True), (2, 48, 16, 330, 330, True),
])
def test_nar_attention_tile_forms(torch, yuear_lib, oracle, B, Hq, Hkv, Lq, Lk, causal):
    test_nar_attention_matches_oracle(torch, yuear_lib, oracle, B, Hq, Hkv, Lq, Lk, causal)


@pytest.mark.parametrize("mag", [5e4, 1e9])
@pytest.mark.parametrize("Hq,Hkv,Lq,Lk,causal", [
    (2, 1, 9, 70, False), (2, 2, 3, 3000, False),      # whole and dealt key-split tiles
    (96, 1, 257, 31, False), (96, 8, 65, 65, True),     # 64-query tiles
])
def test_nar_attention_large_scores(torch, yuear_lib, mag, Hq, Hkv, Lq, Lk, causal):
    # every query's weight is all on one key (see test_attention_prefill_large_scores)
    from test_gpu_kernels import one_hot_scores
    rng = np.random.default_rng(int(mag) + Lk)
    q, k, v, want = one_hot_scores(rng, Hq, Hkv, Lq, Lk, mag, lambda t: t + 1 if causal else Lk)
    got = yuear_lib.nar_attention(*(dev(torch, x[None]) for x in (q, k, v)), causal)
    np.testing.assert_array_equal(host(torch, got)[0], want)


# (heads, kv heads, queries, keys), each with a last key block that is not full:
# key-split tiles of 16 and 32 queries by 4 and 8 waves, dealt, 64-query tiles by one
# and two blocks a step (an odd number of blocks)
@pytest.mark.parametrize("Hq,Hkv,Lq,Lk", [
    (2, 2, 9, 70), (2, 2, 1, 697), (16, 2, 257, 289), (6, 3, 677, 919), (2, 2, 100, 2001),
    (16, 8, 100, 8001), (24, 2, 341, 1505), (24, 8, 500, 3470), (96, 2, 257, 31),
    (24, 2, 1001, 289),
])
def test_nar_attention_reads_no_neighbouring_keys(torch, yuear_lib, oracle, Hq, Hkv, Lq, Lk):
    """The last key block of a kv head lies over the next head's first rows, and of the
    last head past the tensor: NaN and inf there (weights 0 times them would be NaN) must
    not reach the head's queries."""
    rng = np.random.default_rng(Lk)
    per = Hq // Hkv
    q = bf(rng.normal(size=(1, Hq, Lq, 128)))
    for good in (0, Hkv - 1):  # the one head with numbers in it
        k, v = (np.full(((Hkv + 1) * Lk * 128 + 4096,), 0x7FC0, np.uint16) for _ in range(2))
        v[::3] = 0x7F80
        kv = [bf(rng.normal(size=(1, 1, Lk, 128))) for _ in range(2)]
        at = 2048 + good * Lk * 128  # (rows before the first head are NaN too)
        k[at:at + Lk * 128], v[at:at + Lk * 128] = (t.reshape(-1) for t in kv)
        dk, dv = dev(torch, k), dev(torch, v)
        got = host(torch, yuear_lib.nar_attention(
            dev(torch, q), dk[2048:2048 + Hkv * Lk * 128].view(1, Hkv, Lk, 128),
            dv[2048:2048 + Hkv * Lk * 128].view(1, Hkv, Lk, 128)))
        mine = slice(good * per, good * per + per)
        ref = oracle.nar_attention(q[:, mine], *kv)
        assert_close_bf16(got[:, mine], ref, exact_frac=0.8)


def test_nar_attention_leaves_the_workspace(torch, yuear_lib, oracle):
    # V is read as given: the workspace is neither read (NaN) nor written
    rng = np.random.default_rng(1)
    q = bf(rng.normal(size=(1, 4, 20, 128)))
    k = bf(rng.normal(size=(1, 2, 50, 128)))
    v = bf(rng.normal(size=(1, 2, 50, 128)))
    nbytes = yuear_lib.lib.yuear_nar_attention_workspace_bytes(1, 2, 50)
    assert nbytes == 2 * 64 * 128 * 2
    ws = dev(torch, np.full(nbytes // 2, 0x7FC0, np.uint16))
    got = host(torch, yuear_lib.nar_attention(dev(torch, q), dev(torch, k), dev(torch, v),
                                              workspace=ws))
    assert_close_bf16(got, oracle.nar_attention(q, k, v), exact_frac=0.8)
    assert (host(torch, ws) == 0x7FC0).all()


def test_nar_attention_errors(torch, yuear_lib):
    x = dev(torch, np.zeros((1, 4, 8, 128), np.uint16))
    w = torch.empty(1 << 16, dtype=torch.uint8, device="cuda")
    lib = yuear_lib.lib
    import ctypes as C

    def call(heads, kv_heads, q_len, kv_len, head_dim=128, causal=0, chunk=64):
        err = C.c_void_p()
        st = lib.yuear_nar_attention(x.data_ptr(), x.data_ptr(), x.data_ptr(), 1, heads,
                                     kv_heads, q_len, kv_len, head_dim, causal, chunk,
                                     w.data_ptr(), x.data_ptr(), None, C.byref(err))
        msg = C.string_at(err.value).decode() if err.value else ""
        if err.value:
            lib.yuear_string_free(err)
        return st, msg

    st, msg = call(4, 3, 8, 8)
    assert st == 2 and "Invalid grouped-query head count" in msg
    assert "nonempty" in call(4, 2, 0, 8)[1]
    assert "equal query and key lengths" in call(4, 2, 8, 4, causal=1)[1]
    assert "query_chunk_size" in call(4, 2, 8, 8, chunk=0)[1]
    assert "head_dim 128" in call(4, 2, 8, 8, head_dim=64)[1]
    assert call(4, 2, 8, 8)[0] == 0


def test_nar_condition_is_the_prefill_cache(torch, yuear_lib, oracle):
    """CachedNAR's conditioning prefill (nar.cpp:139-190): the keys and values
    of the visible prefix equal the engine's prefill cache bit for bit and the
    oracle's within the prefill tolerance."""
    from conftest import TINY
    w = yuear_lib.random_weights(TINY, seed=8, norm_std=0.1)
    engine = yuear_lib.Engine(TINY, w)
    model = oracle.Model(TINY, w)
    ids = [5, 9, 14, 200, 33, 1, 511, 256, 3, 77, 12, 40, 41, 42]
    for visible_end in (0, 9, 100):
        print(f"[nar condition] visible_end={visible_end}", flush=True)
        k, v = engine.nar_condition(ids, visible_end)
        vis = min(visible_end, len(ids)) if visible_end else len(ids)
        assert tuple(k.shape) == (TINY["num_hidden_layers"], TINY["num_key_value_heads"], vis, 128)
        s = engine.session(1, 32)
        s.prefill(0, ids)
        cache = model.cache(32)
        model.hidden(ids, cache)
        kh, vh = host(torch, k), host(torch, v)
        for layer in range(TINY["num_hidden_layers"]):
            ks, vs = s.read_kv(layer, 0, len(ids))
            np.testing.assert_array_equal(kh[layer], ks[:, :vis])
            np.testing.assert_array_equal(vh[layer], vs[:, :vis])
            assert_close_bf16(kh[layer], cache.keys(layer)[:, :vis], exact_frac=0.8)
            assert_close_bf16(vh[layer], cache.values(layer)[:, :vis], exact_frac=0.8)
        s.close()
    with pytest.raises(ValueError, match="outside the model vocabulary"):
        engine.nar_condition([1, 2, 512])
    with pytest.raises(ValueError, match="nonnegative"):
        engine.nar_condition([1, 2], -1)
    engine.close()
    q = yuear_lib.Engine(TINY, seed=3, bits=4)
    with pytest.raises(ValueError, match="quantized AR cannot condition NAR"):
        q.nar_condition([1, 2, 3])
    q.close()


def merges(torch, call):
    """Merge kernels that `call` launches: a dealt launch has one."""
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        call()
        torch.cuda.synchronize()
    return sum(e.count for e in prof.key_averages() if "nar_merge_kernel" in e.key)


def nar_inputs(torch, rng, hq, hkv, lq, lk):
    return [bf(rng.normal(size=(1, h, n, 128))) for h, n in ((hq, lq), (hkv, lk), (hkv, lk))]


def test_nar_attention_graph_survives_a_larger_call(torch, yuear_lib):
    """The partials of a dealt launch come from a pool per (device, stream). A
    graph captured on a stream keeps the pool buffer it was captured with: a later
    call on that stream that needs a larger buffer allocates a new one and
    keeps the old one alive, so replays of the graph stay correct."""
    rng = np.random.default_rng(21)
    # 256 workgroups x 2 pieces of 16 and of 32 queries: 4.3 and 8.7 MB, over and
    # under the 8 MB that the pool's first buffer rounds up to
    small = [dev(torch, a) for a in nar_inputs(torch, rng, 16, 8, 64, 2570)]
    large = [dev(torch, a) for a in nar_inputs(torch, rng, 6, 3, 274, 6000)]
    for args in (small, large):
        assert merges(torch, lambda: yuear_lib.nar_attention(*args)) == 1
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        ws = torch.empty(yuear_lib.lib.yuear_nar_attention_workspace_bytes(1, 8, 6000) // 2,
                         dtype=torch.bfloat16, device="cuda")
        want = yuear_lib.nar_attention(*small, workspace=ws, stream=s.cuda_stream)
        want = host(torch, want)
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            out = yuear_lib.nar_attention(*small, workspace=ws, stream=s.cuda_stream)
        big = host(torch, yuear_lib.nar_attention(*large, workspace=ws, stream=s.cuda_stream))
        for replay in range(3):
            out.zero_()
            g.replay()
            np.testing.assert_array_equal(host(torch, out), want, err_msg=f"replay {replay}")
    again = host(torch, yuear_lib.nar_attention(*large, workspace=ws, stream=s.cuda_stream))
    np.testing.assert_array_equal(again, big)


@pytest.mark.parametrize("Hq,Hkv,Lq,Lk", [(16, 8, 64, 2570), (1, 1, 1, 20000), (24, 8, 500, 3470)])
def test_nar_attention_captured_before_its_pool(torch, yuear_lib, oracle, Hq, Hkv, Lq, Lk):
    """A dealt shape captured on a stream that has no pool buffer yet: the capture
    cannot allocate, so whole tiles run."""
    args = nar_inputs(torch, np.random.default_rng(Lk), Hq, Hkv, Lq, Lk)
    ref = oracle.nar_attention(*args)
    args = [dev(torch, a) for a in args]
    assert merges(torch, lambda: yuear_lib.nar_attention(*args)) == 1
    s = torch.cuda.Stream()
    ws = torch.empty(yuear_lib.lib.yuear_nar_attention_workspace_bytes(1, Hkv, Lk) // 2,
                     dtype=torch.bfloat16, device="cuda")
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        out = yuear_lib.nar_attention(*args, workspace=ws, stream=s.cuda_stream)
    for _ in range(3):
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert_close_bf16(host(torch, out), ref, exact_frac=0.8)
    assert merges(torch, g.replay) == 0


def test_nar_attention_threads_share_a_stream(torch, yuear_lib):
    """Dealt calls of two threads on one stream share its pool buffer: a call's
    attention and merge are enqueued as one, so that neither reads the other's
    partial sums."""
    import threading
    rng = np.random.default_rng(5)
    sets = [[dev(torch, bf(rng.normal(size=(1, h, n, 128)))) for h, n in ((16, 100), (8, 8001), (8, 8001))]
            for _ in range(2)]
    want = [yuear_lib.nar_attention(*s) for s in sets]
    torch.cuda.synchronize()
    got, errors = [[], []], []

    def work(i):
        try:
            got[i] += [yuear_lib.nar_attention(*sets[i]) for _ in range(60)]
        except Exception as e:  # noqa: BLE001
            errors.append(e)
    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not errors
    for i in range(2):
        for out in got[i]:
            assert torch.equal(out, want[i])


@pytest.mark.parametrize("which", ["q", "k", "v", "q shifted"])
@pytest.mark.parametrize("heads,n,lk", [(2, 64, 2100), (48, 300, 300)])
def test_nar_attention_output_over_an_input(torch, yuear_lib, which, heads, n, lk):
    """Output written over the queries, keys or values: workgroups that still read
    them must not see it. Dealt and whole tiles, against separate buffers."""
    import ctypes as C
    rng = np.random.default_rng(n)
    q, k, v = (dev(torch, bf(rng.normal(size=(1, heads, m, 128)))) for m in (n, lk, lk))
    want = host(torch, yuear_lib.nar_attention(q, k, v))
    room = torch.zeros(heads * n * 128 + 4096, dtype=torch.bfloat16, device="cuda")
    room[4096:] = q.view(-1)
    out = {"q": room[4096:], "q shifted": room, "k": k, "v": v}[which]
    ws = torch.empty(yuear_lib.lib.yuear_nar_attention_workspace_bytes(1, heads, lk) // 2,
                     dtype=torch.bfloat16, device="cuda")
    err = C.c_void_p()
    assert yuear_lib.lib.yuear_nar_attention(room.data_ptr() + 8192, k.data_ptr(), v.data_ptr(), 1, heads,
                                             heads, n, lk, 128, 0, 64, ws.data_ptr(), out.data_ptr(), None,
                                             C.byref(err)) == 0
    got = host(torch, out.view(-1)[:heads * n * 128]).reshape(want.shape)
    np.testing.assert_array_equal(got, want)
