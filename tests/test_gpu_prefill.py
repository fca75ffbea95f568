"""HIP parity for the prompt path (asdsl_decode_prefill): a prompt run in
chunks leaves what forward_token on each of its tokens leaves (the decode step
itself is checked against the oracle in test_gpu_decode*.py).  Tolerance: none.
The chunk repeats the step's arithmetic operation for operation, so every bit
of the K/V rows and the logits agrees."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _state(eng):
    names = ("k_cache", "v_cache") + (("k_scale", "v_scale") if eng.kv_int8 else ())
    return (eng.logits.clone(), eng.next_token(), int(eng.pos.item()), eng._host_pos, eng.get_kv_seq_len(),
            [L[n].clone() for L in eng.layers for n in names])


def _compare(cfg, plens, seed=5):
    import torch
    from asdsl.engine import DecodeEngine

    eng = DecodeEngine.synthetic(cfg, seed=seed, fatrelu_threshold=0.0)
    rng = np.random.default_rng(seed)
    prompt = [int(t) for t in rng.integers(0, cfg.vocab, max(plens))]
    for n in plens:
        eng.reset_session()
        eng.prefill(prompt[:n])
        got = _state(eng)
        eng.reset_session()
        for i, t in enumerate(prompt[:n]):
            eng.forward_token(t, i)
        want = _state(eng)
        assert got[1:5] == want[1:5] == (want[1], n, n, n), n
        for a, b in zip(got[5], want[5]):
            assert torch.equal(a, b), n
        assert torch.equal(got[0], want[0]), n


# 4: the smallest chunk; 16 and 17: one column block and the first of two; 64
# and 65: a workgroup's 4 blocks and a tile of positions, and one past; 512 and
# 530: the columns of an attention launch, and a second one; 1024 and 1030: a
# whole chunk, and two
@pytest.mark.parametrize("kv", ["fp16", "int8"])
def test_prompt_lengths(gpu, kv):
    from asdsl.engine import DecodeConfig

    _compare(DecodeConfig(n_layers=2, vocab=4096, max_seq=1088, kv_format=kv), (4, 16, 17, 64, 65, 197, 512, 530, 1024, 1030))


# group sizes in both places, query heads per KV head 1, 2 and 4, and in_features
# whose K split masks units (3712 = 29 groups of 128) or leaves a class of
# groups empty (1152: 9 groups of 128)
@pytest.mark.parametrize("heads,kv_heads,ffn,gs_attn,gs_ffn", [
    (8, 4, 3712, 32, 128), (8, 8, 1152, 128, 32), (16, 4, 8192, 32, 32), (9, 3, 2944, 128, 128)])
def test_shapes(gpu, heads, kv_heads, ffn, gs_attn, gs_ffn):
    from asdsl.engine import DecodeConfig

    _compare(DecodeConfig(hidden=128 * heads, n_heads=heads, n_kv_heads=kv_heads, ffn=ffn, vocab=1003, n_layers=3,
                          max_seq=160, gs_attn=gs_attn, gs_ffn=gs_ffn), (18, 77, 150))


# past 2048 positions a split holds two tiles, past 4096 three
@pytest.mark.parametrize("kv,kv_heads,plen", [("fp16", 4, 2130), ("int8", 4, 4101), ("int8", 2, 2070)])
def test_deep_positions(gpu, kv, kv_heads, plen):
    from asdsl.engine import DecodeConfig

    _compare(DecodeConfig(hidden=1024, n_heads=8, n_kv_heads=kv_heads, ffn=1536, vocab=2048, n_layers=2,
                          max_seq=plen + 3, kv_format=kv), (plen,))


# three query heads per KV head past 2048 positions, fp16 rows
def test_deep_positions_three_heads(gpu):
    from asdsl.engine import DecodeConfig

    _compare(DecodeConfig(hidden=768, n_heads=6, n_kv_heads=2, ffn=1536, vocab=2048, n_layers=2, max_seq=2100), (2085,))


# chunks of up to 16 tokens at positions past 0: the projections' 16-column form
# (every in_features of the first model has it) and the GEMM's split form
@pytest.mark.parametrize("hidden,heads,kv_heads,ffn", [(3072, 24, 8, 8192), (1024, 8, 4, 3712)])
def test_short_chunks(gpu, monkeypatch, hidden, heads, kv_heads, ffn):
    from asdsl.engine import DecodeConfig, DecodeEngine

    monkeypatch.setattr(DecodeEngine, "MAX_PREFILL_TOKENS", 16)
    _compare(DecodeConfig(hidden=hidden, n_heads=heads, n_kv_heads=kv_heads, ffn=ffn, vocab=1003, n_layers=2,
                          max_seq=64), (17, 40))


@pytest.mark.parametrize("switch", ["ASDSL_HIP_VERIFY_DOT4", "ASDSL_HIP_NORM_FACTORED"])
def test_prompts_under_the_switches(gpu, monkeypatch, switch):
    """Prompts that run as verify passes of up to 16 tokens (16 + a single
    step, 16 + 16 + 8) and single steps past position 2048, against
    forward_token under the same switch."""
    from asdsl.engine import DecodeConfig, DecodeEngine

    monkeypatch.setenv(switch, "1")
    monkeypatch.setattr(DecodeEngine, "_prefill_chunks", None)  # not called
    _compare(DecodeConfig(hidden=1024, n_heads=8, n_kv_heads=4, ffn=1536, vocab=2048, n_layers=2, max_seq=2112),
             (17, 40, 2051))


def test_refused_by_the_library(gpu, monkeypatch):
    """asdsl_decode_prefill's argument checks; nothing is queued."""
    import ctypes

    import torch
    from asdsl import _hip
    from asdsl.engine import DecodeConfig, DecodeEngine

    eng = DecodeEngine.synthetic(DecodeConfig(hidden=1024, n_heads=8, n_kv_heads=4, ffn=1536, vocab=2048, n_layers=1,
                                              max_seq=64), seed=1)
    eng.prefill([1, 2, 3, 4])
    lib, model, P = _hip.LIB, ctypes.byref(eng._model), _hip.ptr
    ids = torch.ones(64, dtype=torch.int32, device="cuda")

    def call(n=4, start=0, work=0, tokens=None, logits=None):
        return lib.asdsl_decode_prefill(model, P(ids) if tokens is None else tokens, n, start, P(eng.token),
                                        P(eng.pos), logits, P(eng._prefill_work) + work, _hip.stream_handle())

    bad = _hip.ASDSL_ERR_INVALID_ARGUMENT
    assert lib.asdsl_decode_prefill_work_bytes(model, 0) == lib.asdsl_decode_prefill_work_bytes(model, 1025) == 0
    assert lib.asdsl_decode_prefill_work_bytes(None, 4) == 0
    assert call(n=0) == call(n=1025) == call(start=-1) == call(start=61) == call(work=64) == call(tokens=0) == bad
    monkeypatch.setenv("ASDSL_HIP_NORM_FACTORED", "1")
    assert call() not in (bad, 0) and "factored" in _hip.last_error()
    assert int(eng.pos.item()) == 4


def test_refused(gpu):
    from asdsl.engine import DecodeConfig, DecodeEngine

    eng = DecodeEngine.synthetic(DecodeConfig(hidden=1024, n_heads=8, n_kv_heads=4, ffn=1536, vocab=2048, n_layers=1,
                                              max_seq=64), seed=1)
    with pytest.raises(ValueError, match="vocab"):
        eng.prefill([1, 2, 3, 4, 2048])
    with pytest.raises(ValueError, match="range"):
        eng.prefill([1] * 65)


# 3, 4: a pass and a chunk; 17: its last pass is the first 16 tokens; 40: the
# last 8; 2090: the pass that ends at position 2048
@pytest.mark.parametrize("plen", [3, 4, 17, 40, 2090])
def test_verify_next_tokens_after_a_prompt(gpu, monkeypatch, plen):
    """The tokens of the prompt's last pass as the passes themselves give them
    (ASDSL_HIP_VERIFY_DOT4, the pass's other form with the same bits, keeps
    prefill on them), whatever pass came before; the K/V rows, the position
    and the step after it as if they had not been asked for."""
    import torch
    from asdsl.engine import DecodeConfig, DecodeEngine

    eng = DecodeEngine.synthetic(DecodeConfig(hidden=1024, n_heads=8, n_kv_heads=4, ffn=1536, vocab=2048, n_layers=2,
                                              max_seq=2112), seed=3)
    toks = [int(t) for t in np.random.default_rng(plen).integers(0, 2048, plen)]
    monkeypatch.setenv("ASDSL_HIP_VERIFY_DOT4", "1")
    eng.prefill(toks)
    want = eng.verify_next_tokens()
    monkeypatch.delenv("ASDSL_HIP_VERIFY_DOT4")
    eng.reset_session()
    eng.forward_batch_all_logits([5, 6], 0)
    eng.prefill(toks)
    state = _state(eng)
    assert eng.verify_next_tokens() == want == eng.verify_next_tokens()
    again = _state(eng)
    assert state[1:5] == again[1:5] and torch.equal(state[0], again[0])
    assert all(torch.equal(a, b) for a, b in zip(state[5], again[5]))
    eng.reset_session()
    eng.prefill(toks)
    eng.forward_token(7, plen)  # rows after the prompt's leave it as it was
    assert eng.verify_next_tokens() == want and eng._host_pos == plen + 1 == int(eng.pos.item())


def test_verify_next_tokens_without_a_pass(gpu):
    from asdsl.engine import DecodeConfig, DecodeEngine

    eng = DecodeEngine.synthetic(DecodeConfig(hidden=1024, n_heads=8, n_kv_heads=4, ffn=1536, vocab=2048, n_layers=1,
                                              max_seq=64), seed=1)
    with pytest.raises(RuntimeError, match="no multi-token pass"):
        eng.verify_next_tokens()
    eng.prefill([1, 2, 3, 4, 5])
    eng.truncate_kv(4)
    with pytest.raises(RuntimeError, match="cut or overwritten"):
        eng.verify_next_tokens()
    eng.forward_batch_all_logits([3, 4, 5], 4)
    assert len(eng.verify_next_tokens()) == 3


def test_work_buffer_outlives_its_launches(gpu, monkeypatch):
    """A longer prompt replaces the engine's work buffer.  While a prompt
    queued on another stream still uses the old one, its memory is not handed
    out again on the stream that allocated it (here at the moment the longer
    prompt uploads its tokens, as another thread could)."""
    import torch
    from asdsl.engine import DecodeConfig, DecodeEngine

    eng = DecodeEngine.synthetic(DecodeConfig(hidden=1024, n_heads=8, n_kv_heads=4, ffn=1536, vocab=2048, n_layers=1,
                                              max_seq=256), seed=1)
    eng.prefill([1] * 64)
    torch.cuda.synchronize()
    old = eng._prefill_work.data_ptr()
    nbytes = eng._prefill_work.numel()
    main, side = torch.cuda.current_stream(), torch.cuda.Stream()
    seen = []
    upload = torch.tensor

    def tensor(*a, **k):
        with torch.cuda.stream(main):
            seen.append(torch.empty(nbytes, dtype=torch.uint8, device="cuda"))
        return upload(*a, **k)

    with torch.cuda.stream(side):
        eng.prefill([2] * 64)
        torch.cuda._sleep(200_000_000)  # the launches still queued
        monkeypatch.setattr(torch, "tensor", tensor)
        eng.prefill([3] * 200)
        monkeypatch.setattr(torch, "tensor", upload)
    assert len(seen) == 1 and seen[0].data_ptr() != old
    torch.cuda.synchronize()
