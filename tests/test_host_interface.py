"""Host-side mirror of the reference call surface: names, signature, and the
errors raised before any GPU work (runs without a GPU)."""
import inspect

import pytest
import torch

from longcat_video_amd.block_sparse_attention import bsa_interface as I


def test_reference_names_exist():
    for name in ("flash_attn_bsa_3d", "flash_attn_bsa", "rearrange_THW_to_3d_block", "rearrange_3d_block_to_THW",
                 "mean_pooling_compression", "cal_score", "get_select_indices", "get_select_indices_topk",
                 "get_select_indices_topk_from_score", "attn_fwd_bsa_varlen_triton"):
        assert callable(getattr(I, name))


def test_flash_attn_bsa_3d_signature_matches_the_reference():
    sig = inspect.signature(I.flash_attn_bsa_3d)
    names = list(sig.parameters)
    assert names[:9] == ["q", "k", "v", "latent_shape_q", "latent_shape_k", "sparsity", "cdf_threshold",
                         "chunk_3d_shape_q", "chunk_3d_shape_k"]
    assert sig.parameters["sparsity"].default == 0.875
    assert sig.parameters["cdf_threshold"].default is None
    assert sig.parameters["chunk_3d_shape_q"].default == [4, 4, 8]
    assert sig.parameters["chunk_3d_shape_k"].default == [4, 4, 8]


def qkv(S=256, D=128, H=2):
    return [torch.zeros(1, H, S, D, dtype=torch.bfloat16) for _ in range(3)]


def test_shape_violations_raise_assertion_error():
    q, k, v = qkv()
    prm = dict(chunk_3d_shape_q=[4, 4, 4], chunk_3d_shape_k=[4, 4, 4])
    with pytest.raises(AssertionError):
        I.flash_attn_bsa_3d(q, k, v, (4, 8, 9), (4, 8, 8), **prm)            # T*H*W != S
    with pytest.raises(AssertionError):
        I.flash_attn_bsa_3d(q, k[..., :64], v[..., :64], (4, 8, 8), (4, 8, 8), **prm)   # head dims differ
    with pytest.raises(AssertionError):
        I.flash_attn_bsa_3d(q, k, v, (4, 8, 8), (4, 8, 8), chunk_3d_shape_q=[4, 4, 3], chunk_3d_shape_k=[4, 4, 4],
                            allow_padding=False)                               # reference divisibility assert
    q96 = [t[..., :96] for t in (q, k, v)]
    with pytest.raises(AssertionError):
        I.flash_attn_bsa_3d(*q96, (4, 8, 8), (4, 8, 8), **prm)                # head dim outside {16..256}


def test_selection_mode_errors():
    q, k, v = qkv()
    with pytest.raises(ValueError):
        I.flash_attn_bsa_3d(q, k, v, (4, 8, 8), (4, 8, 8), sparsity=None, cdf_threshold=None)
    with pytest.raises(RuntimeError, match="GPU only"):          # the CDF rule is built: CPU tensors get as far as the engine
        I.flash_attn_bsa_3d(q, k, v, (4, 8, 8), (4, 8, 8), sparsity=None, cdf_threshold=0.9)
    with pytest.raises(ValueError):
        I.get_select_indices(q, k, None, None)
    with pytest.raises(ValueError):
        I.get_select_indices_from_score(q, None, None)


def test_no_cpu_fallback_with_or_without_gradients():
    q, k, v = qkv()
    with pytest.raises(RuntimeError, match="GPU only"):
        I.flash_attn_bsa_3d(q, k, v, (4, 8, 8), (4, 8, 8), chunk_3d_shape_q=[4, 4, 4], chunk_3d_shape_k=[4, 4, 4])
    with pytest.raises(RuntimeError, match="GPU only"):
        I.mean_pooling_compression(q, 64)
    q.requires_grad_(True)                       # the differentiable route runs on the GPU only as well
    with pytest.raises(RuntimeError, match="GPU only"):
        I.flash_attn_bsa_3d(q, k, v, (4, 8, 8), (4, 8, 8), chunk_3d_shape_q=[4, 4, 4], chunk_3d_shape_k=[4, 4, 4])
    with pytest.raises(NotImplementedError, match="bf16 and fp16"):
        I.flash_attn_bsa_3d(q.float().requires_grad_(True), k.float(), v.float(), (4, 8, 8), (4, 8, 8),
                            chunk_3d_shape_q=[4, 4, 4], chunk_3d_shape_k=[4, 4, 4])


def test_num_selected():
    assert I.num_selected(0.9375, 1440) == 90 and I.num_selected(0.9, 10) == 0


def test_module_caches_are_bounded():
    """The per-stream GEMM workspaces and the per-grid rotation tables forget their oldest entry beyond a limit."""
    from longcat_video_amd.modules import attention as A
    d = A._Bounded(3)
    for i in range(5):
        d[i] = i
    assert list(d) == [2, 3, 4]
    d[3] = 30                                    # rewriting a key evicts nothing
    assert list(d) == [2, 3, 4] and d[3] == 30
    assert isinstance(A._GEMM_WORKSPACES, A._Bounded) and isinstance(A._ROPE_TABLES, A._Bounded)


def _small_module(monkeypatch):
    from longcat_video_amd.modules.attention import Attention
    attn = Attention(256, 2, enable_bsa=True, bsa_params=dict(sparsity=0.5, chunk_3d_shape_q=[4, 4, 4], chunk_3d_shape_k=[4, 4, 4]))

    def launched(x):
        raise RuntimeError("GPU work was reached")

    monkeypatch.setattr(attn, "_project_qkv", launched)
    return attn


@pytest.mark.parametrize("k_shape,v_shape", [
    ((1, 2, 128, 128), (1, 2, 64, 128)),       # fewer values than keys
    ((1, 1, 128, 128), (1, 1, 128, 128)),      # a head share of the cache
    ((1, 2, 128, 128), (1, 1, 128, 128)),
    ((1, 2, 128, 64), (1, 2, 128, 64)),        # another head dim
    ((1, 2, 64, 128), (1, 2, 64, 128)),        # fewer frames than said
])
def test_a_cache_of_another_shape_is_refused_before_any_launch(monkeypatch, k_shape, v_shape):
    attn = _small_module(monkeypatch)
    x = torch.zeros(1, 256, 256, dtype=torch.bfloat16)
    caches = [torch.zeros(s, dtype=torch.bfloat16) for s in (k_shape, v_shape)]
    with pytest.raises(AssertionError):
        attn.forward_with_kv_cache(x, shape=(4, 8, 8), num_cond_latents=2, kv_cache=caches)
    good = [torch.zeros(1, 2, 128, 128, dtype=torch.bfloat16) for _ in range(2)]
    with pytest.raises(RuntimeError, match="was reached"):
        attn.forward_with_kv_cache(x, shape=(4, 8, 8), num_cond_latents=2, kv_cache=good)


def test_the_operators_cache_argument_is_held_against_q_and_k():
    t = lambda *s, dtype=torch.bfloat16: torch.zeros(*s, dtype=dtype)      # noqa: E731
    q, k = t(1, 2, 256, 128), t(1, 2, 256, 128)
    c = I._kv_cache_arg(q, k, 64, (t(1, 2, 128, 128), t(1, 2, 128, 128), 2), (t(1, 2, 256, 128), t(1, 2, 256, 128)))
    assert c.cached_frames == 2 and list(c.v_cache_strides) == [2 * 128 * 128, 128 * 128, 128]
    assert I._kv_cache_arg(q, k, 64, None, None) is None
    for cache in ((t(1, 2, 128, 128), t(1, 2, 64, 128), 2), (t(1, 1, 128, 128), t(1, 2, 128, 128), 2),
                  (t(1, 2, 128, 128), t(1, 2, 128, 128), 3), (t(1, 2, 128, 128), t(1, 2, 128, 128, dtype=torch.float16), 2)):
        with pytest.raises(AssertionError):
            I._kv_cache_arg(q, k, 64, cache, None)
    with pytest.raises(AssertionError):
        I._kv_cache_arg(q, k, 64, None, (t(1, 2, 256, 128), t(1, 2, 192, 128)))


@pytest.mark.parametrize("kw", [dict(num_cond_latents=1), dict(return_kv=True), dict()])
def test_tokens_that_do_not_fill_the_grid_are_refused(monkeypatch, kw):
    attn = _small_module(monkeypatch)
    for n in (250, 260):
        with pytest.raises(AssertionError):
            attn(torch.zeros(1, n, 256, dtype=torch.bfloat16), shape=(4, 8, 8), **kw)
    with pytest.raises(RuntimeError, match="was reached"):
        attn(torch.zeros(1, 256, 256, dtype=torch.bfloat16), shape=(4, 8, 8), **kw)


@pytest.mark.parametrize("name", ["forward", "forward_with_kv_cache", "__call__", "_linear"])
@pytest.mark.parametrize("where", ["class", "object"])
def test_a_replaced_attention_is_called_with_the_signature_it_had(monkeypatch, name, where):
    """The adaLN branch, with a method of Attention replaced on the class or on the object by one that knows no gate."""
    from longcat_video_amd.modules import attention as A
    if (name, where) == ("__call__", "object"):
        pytest.skip("looked up on the class alone")
    attn = A.Attention(256, 2, enable_bsa=True, bsa_params=dict(sparsity=0.5, chunk_3d_shape_q=[4, 4, 4], chunk_3d_shape_k=[4, 4, 4])).to(torch.bfloat16)
    calls = []

    def replaced(self, x, shape=None, num_cond_latents=None, return_kv=False):
        calls.append(name)
        return (x + 1, "cache") if return_kv else x + 1

    def replaced_cached(self, x, shape=None, num_cond_latents=None, kv_cache=None):
        calls.append(name)
        return x + 1

    def replaced_linear(self, x, layer, loras, residual=None):
        calls.append(layer)
        y = torch.nn.functional.linear(x, layer.weight, layer.bias)
        return y if residual is None else y + residual

    new = {"forward_with_kv_cache": replaced_cached, "_linear": replaced_linear}.get(name, replaced)
    if where == "class":
        monkeypatch.setattr(A.Attention, name, new)
    else:
        monkeypatch.setattr(attn, name, new.__get__(attn))
    monkeypatch.setattr(A, "layernorm_modulate", lambda x, shift, scale: x)
    monkeypatch.setattr(A, "gated_residual", lambda x, gate, y: ("gated", y))
    monkeypatch.setattr(A, "rope_table", lambda *a: None)
    monkeypatch.setattr(A.Attention, "_process_attn", lambda self, q, k, v, shape, out=None, **kw: out.zero_())
    x, mod = torch.zeros(1, 256, 256, dtype=torch.bfloat16), torch.zeros(1, 4, 1, 256)
    cache = [torch.zeros(1, 2, 128, 128, dtype=torch.bfloat16) for _ in range(2)]
    run = lambda **kw: A.dit_self_attention_branch(x, mod, mod, mod, attn, (4, 8, 8), **kw)      # noqa: E731
    with torch.no_grad():
        after = x + 1 if name != "_linear" else torch.nn.functional.linear(x, attn.proj.weight, attn.proj.bias)
    if name != "forward_with_kv_cache":
        for kw in (dict(), dict(num_cond_latents=1)):
            out = run(**kw)
            assert out[0] == "gated" and torch.equal(out[1], after)
        out, kept = run(return_kv=True)
        assert out[0] == "gated" and torch.equal(out[1], after) and (kept == "cache" or len(kept) == 2)
    if name in ("forward_with_kv_cache", "_linear"):
        out = run(num_cond_latents=2, kv_cache=cache)
        assert out[0] == "gated" and torch.equal(out[1], after)
    assert len(calls) > 0


def test_a_gate_without_its_residual_is_refused_before_any_launch(monkeypatch):
    attn = _small_module(monkeypatch)
    x, gate = torch.zeros(1, 256, 256, dtype=torch.bfloat16), torch.zeros(1, 4, 1, 256)
    cache = [torch.zeros(1, 2, 128, 128, dtype=torch.bfloat16) for _ in range(2)]
    with pytest.raises(ValueError, match="residual"):
        attn(x, shape=(4, 8, 8), gate=gate)
    with pytest.raises(ValueError, match="residual"):
        attn.forward_with_kv_cache(x, shape=(4, 8, 8), num_cond_latents=2, kv_cache=cache, gate=gate)
    with pytest.raises(AssertionError, match="gate"):
        attn(x, shape=(4, 8, 8), residual=x, gate=gate[..., :128])
    with pytest.raises(AssertionError, match="gate"):
        attn.forward_with_kv_cache(x, shape=(4, 8, 8), num_cond_latents=2, kv_cache=cache, residual=x, gate=gate.bfloat16())


def test_plans_are_kept_by_value():
    """Grids as tensor elements (what an int() of them would have read at each call), rules as tensors."""
    I._capi.load()
    grid = [torch.tensor(8), torch.tensor(8), torch.tensor(16)]
    rule = torch.tensor(0.5)
    plan = lambda: I._plan_of(1, 2, 128, 0, grid, grid, (4, 4, 4), [4, 4, 4], rule, None)      # noqa: E731
    assert (plan().nbq, plan().width) == (16, 8)
    grid[0].fill_(16)
    assert (plan().nbq, plan().width) == (32, 16)
    rule.fill_(0.75)
    assert plan().width == 8
    assert I._plan_of(1, 2, 128, 0, (16, 8, 16), (16, 8, 16), (4, 4, 4), (4, 4, 4), 0.75, None).width == 8


@pytest.mark.parametrize("free,unused,asked", [(2 << 30, 1 << 30, [1 << 20]), (2 << 30, 5 << 30, [6 << 30]), (7 << 30, 0, [6 << 30])])
def test_a_backward_does_not_ask_for_room_that_is_not_there(monkeypatch, free, unused, asked):
    """A request that fails makes torch's allocator give back all it holds, at every call."""
    made = []
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.setattr(torch.cuda, "mem_get_info", lambda d=None: (free, 288 << 30))
    monkeypatch.setattr(torch.cuda, "memory_reserved", lambda d=None: 20 << 30)
    monkeypatch.setattr(torch.cuda, "memory_allocated", lambda d=None: (20 << 30) - unused)

    def empty(n, **kw):
        made.append(n)
        if n > free + unused:
            raise torch.OutOfMemoryError("no room")
        return n
    monkeypatch.setattr(torch, "empty", empty)
    assert I._backward_workspace(6 << 30, 1 << 20, torch.device("cuda", 0)) == asked[-1]
    assert made == asked
