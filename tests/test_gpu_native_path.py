"""The native launch path (mica_amd._lib.FAST) against the Python path it stands in front of: every form of a call
gives the same bits, or the same refusal, with and without it."""
import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from mica_amd import _lib, fused_kernels, gdn, int8_kernels
from mica_amd.attention import causal_gqa_attention

BF, F32 = torch.bfloat16, torch.float32


class Sub(torch.Tensor):
    pass


def outcome(fn, fast):
    keep = _lib.FAST
    if not fast:
        _lib.FAST = _lib._NotLoaded()
    n0, misses = int8_kernels.STATS["launch"], dict(int8_kernels.STATS["fallback"])
    try:
        r = fn()
        err = None
    except Exception as e:  # noqa: BLE001  (the refusal itself is compared)
        r, err = None, (type(e), str(e))
    finally:
        _lib.FAST = keep
    new = {k: v - misses.get(k, 0) for k, v in int8_kernels.STATS["fallback"].items() if v != misses.get(k, 0)}
    return r, err, new, int8_kernels.STATS["launch"] - n0


def flat(r):
    if isinstance(r, torch.Tensor):
        return [r]
    return [x for v in r for x in flat(v)] if isinstance(r, (list, tuple)) else [r]


def forms(gpu):
    g = torch.Generator(device=gpu).manual_seed(3)
    rn = lambda *s, dt=BF: torch.randn(*s, generator=g, device=gpu).to(dt)  # noqa: E731
    x = rn(33, 2560)
    inv = torch.rand(2560, generator=g, device=gpu) + 0.5
    qx, sx = int8_kernels.act_quant(x)
    qw = torch.randint(-127, 128, (256, 2560), generator=g, device=gpu, dtype=torch.int8)
    sw = torch.rand(256, generator=g, device=gpu)
    w = rn(2560)
    aq, mm, nq = int8_kernels.act_quant, int8_kernels.mm_i8, fused_kernels.rms_norm_quant
    nm = fused_kernels.rms_norm_quant_multi
    q, kv = rn(2, 40, 16, 256), rn(2, 40, 8, 256)
    k, v = kv.split((4, 4), dim=2)
    pre = (rn(64, 4, 256), rn(64, 4, 256))
    cx, cw = rn(2, 70, 512), rn(512, 4)
    gq, gv = rn(2, 70, 2, 128) * 0.1, rn(2, 70, 4, 128)
    gg, beta = -torch.rand(2, 70, 4, generator=g, device=gpu), torch.rand(2, 70, 4, generator=g, device=gpu)
    ab = rn(33, 8)
    A, dt = torch.rand(4, generator=g, device=gpu), torch.rand(4, generator=g, device=gpu)
    z = rn(33, 1024)
    big = rn(33, 2560 * 2)
    out = {
        "quant": lambda: aq(x), "quant_smooth": lambda: aq(x, inv), "quant_away": lambda: aq(x, rounding="away"),
        "quant_fp32": lambda: aq(x.float()), "quant_fp16": lambda: aq(x.half()), "quant_strided": lambda: aq(big[:, :2560]),
        "quant_one_strided_row": lambda: aq(big[:1, :2560]), "quant_1d": lambda: aq(x[0]), "quant_t": lambda: aq(x.t()),
        "quant_misaligned": lambda: aq(big.view(-1)[1:2561].view(1, 2560)), "quant_empty": lambda: aq(x[:0]),
        "quant_int": lambda: aq(qx), "quant_bad_inv": lambda: aq(x, inv[:7]), "quant_bad_rounding": lambda: aq(x, rounding="up"),
        "quant_subclass": lambda: aq(x.as_subclass(Sub)), "quant_cpu": lambda: aq(x.cpu()),
        "quant_param": lambda: aq(torch.nn.Parameter(x)), "quant_none": lambda: aq(None),
        "mm": lambda: mm(qx, sx, qw, sw), "mm_bias_res": lambda: mm(qx, sx, qw, sw, sw, residual=x[:, :256].contiguous()),
        "mm_fp32": lambda: mm(qx, sx, qw, sw, out_dtype=F32), "mm_fp16": lambda: mm(qx, sx, qw, sw, out_dtype=torch.float16),
        "mm_silu": lambda: mm(qx, sx, qw, sw, epilogue="silu_mul"), "mm_silu_bias": lambda: mm(qx, sx, qw, sw, sw, epilogue="silu_mul"),
        "mm_split": lambda: mm(qx, sx, qw, sw, split=True), "mm_auto": lambda: mm(qx, sx, qw, sw, split="auto"),
        "mm_requant": lambda: mm(qx, sx, qw, sw, requant=True),
        "mm_out_int": lambda: mm(qx, sx, qw, sw, out_dtype=torch.int32), "mm_epi": lambda: mm(qx, sx, qw, sw, epilogue="gelu"),
        "mm_k": lambda: mm(qx[:, :40].contiguous(), sx, qw[:, :40].contiguous(), sw), "mm_scales": lambda: mm(qx, sw, qw, sw),
        "mm_res_strided": lambda: mm(qx, sx, qw, sw, residual=x[:, :256]), "mm_empty": lambda: mm(qx[:0], sx[:0], qw, sw),
        "mm_rows_view": lambda: mm(qx[1:9], sx[16:24], qw[16:32], sw[16:32]), "mm_scale_misaligned": lambda: mm(qx[1:9], sx[1:9], qw, sw),
        "norm": lambda: nq(x, w, 1e-6), "norm_res_y": lambda: nq(x, w, 1e-6, residual=x, return_normed=True),
        "norm_inv": lambda: nq(x, w, 1e-6, inv, offset=0.0), "norm_3d": lambda: nq(x.view(3, 11, 2560), w, 1e-6, return_normed=True),
        "norm_strided": lambda: nq(big[:, :2560], w, 1e-6), "norm_fp32_w": lambda: nq(x, w.float(), 1e-6),
        "norm_fp32": lambda: nq(x.float(), w, 1e-6), "norm_w_short": lambda: nq(x, w[:9], 1e-6), "norm_cpu": lambda: nq(x.cpu(), w, 1e-6),
        "norm_bad_res": lambda: nq(x, w, 1e-6, residual=x[:3]), "norm_only": lambda: fused_kernels.rms_norm(x, w, 1e-6, x),
        "multi": lambda: nm(x, w, 1e-6, [None, inv]), "multi_res": lambda: nm(x, w, 1e-6, [inv, inv, inv], residual=x),
        "multi_tuple": lambda: nm(x, w, 1e-6, (None, inv)), "multi_0": lambda: nm(x, w, 1e-6, []), "multi_bad": lambda: nm(x, w, 1e-6, [inv[:3]]),
        "attn": lambda: causal_gqa_attention(q, k, v), "attn_scale": lambda: causal_gqa_attention(q, k, v, 0.3),
        "attn_prefix": lambda: causal_gqa_attention(q, k, v, prefix=pre), "attn_prefix_4d": lambda: causal_gqa_attention(q, k, v, prefix=tuple(t[None] for t in pre)),
        "attn_prefix_33": lambda: causal_gqa_attention(q, k, v, prefix=tuple(t[:33] for t in pre)), "attn_tail": lambda: causal_gqa_attention(q[:, :7], k, v),
        "attn_bhsd": lambda: int8_kernels.attn_fwd(q.transpose(1, 2), k.transpose(1, 2), v.transpose(1, 2), 0.0625),
        "attn_heads": lambda: causal_gqa_attention(q[:, :, :8], k, v), "attn_fp32": lambda: causal_gqa_attention(q.float(), k, v),
        "attn_stride": lambda: causal_gqa_attention(rn(2, 40, 16, 512)[..., ::2], k, v),
        "conv": lambda: gdn.causal_conv1d_fn(cx.transpose(1, 2), cw, activation="silu", l2norm_heads=2),
        "conv_state": lambda: gdn.causal_conv1d_fn(cx.transpose(1, 2), cw.float(), initial_states=rn(2, 512, 3) * 0 + 1, return_final_states=True),
        "conv_state_fp32": lambda: gdn.causal_conv1d_fn(cx.transpose(1, 2), cw, initial_states=torch.ones(2, 512, 3, device=gpu)),
        "conv_bias": lambda: gdn.causal_conv1d_fn(cx.transpose(1, 2), cw, cw[:, 0].contiguous()), "conv_act": lambda: gdn.causal_conv1d_fn(cx.transpose(1, 2), cw, activation="relu"),
        "conv_rows": lambda: gdn.causal_conv1d_fn(cx, cw), "conv_w3": lambda: gdn.causal_conv1d_fn(cx.transpose(1, 2), cw.view(512, 1, 4)),
        "chunk": lambda: gdn.chunk_gated_delta_rule(gq, gq, gv, gg, beta), "chunk_state": lambda: gdn.chunk_gated_delta_rule(gq, gq, gv, gg, beta.to(BF), 0.5, torch.ones(2, 4, 128, 128, device=gpu), True),
        "chunk_bf16_g": lambda: gdn.chunk_gated_delta_rule(gq, gq, gv, gg.to(BF), beta.half()), "chunk_g": lambda: gdn.chunk_gated_delta_rule(gq, gq, gv, gg[:, :3], beta),
        "chunk_l2": lambda: gdn.chunk_gated_delta_rule(gq, gq, gv, gg, beta, use_qk_l2norm_in_kernel=True), "chunk_hv": lambda: gdn.chunk_gated_delta_rule(gq, gq, gv[:, :, :3], gg, beta),
        "gate": lambda: gdn.gdn_gate(ab[:, :4], ab[:, 4:], A, dt), "gate_3d": lambda: gdn.gdn_gate(ab.view(3, 11, 8)[..., :4], ab.view(3, 11, 8)[..., 4:], A, dt),
        "gate_bf16": lambda: gdn.gdn_gate(ab[:, :4], ab[:, 4:], A.to(BF), dt), "gate_hv": lambda: gdn.gdn_gate(ab[:, :4], ab[:, 4:], A[:3], dt),
        "gnorm": lambda: gdn.gated_rmsnorm_quant(z, z, rn(128) * 0 + 1), "gnorm_y": lambda: gdn.gated_rmsnorm_quant(big[:, :1024], z, z[0, :128].contiguous(), want_y=True),
        "gnorm_3d": lambda: gdn.gated_rmsnorm_quant(z.view(3, 11, 1024), z.view(3, 11, 1024), z[0, :128].contiguous()), "gnorm_w": lambda: gdn.gated_rmsnorm_quant(z, z, w),
    }
    return out


@pytest.mark.gpu
def test_native_path_equals_python_path(gpu, monkeypatch):
    monkeypatch.setattr(int8_kernels, "STRICT", False)
    fns = forms(gpu)
    for name, fn in fns.items():
        a, b = outcome(fn, True), outcome(fn, False)
        assert a[1:] == b[1:], (name, a[1:], b[1:])
        fa, fb = flat(a[0]), flat(b[0])
        assert len(fa) == len(fb), name
        for s, t in zip(fa, fb):
            if t is None:
                assert s is None, name
                continue
            assert (s.shape, s.dtype, s.stride()) == (t.shape, t.dtype, t.stride()), name
            assert torch.equal(s, t), name


@pytest.mark.gpu
def test_native_path_equals_python_path_on_a_side_stream(gpu, monkeypatch):
    """As above on a stream of its own, which the inputs were not made on: launches, outputs and the GEMM's workspace
    are that stream's."""
    monkeypatch.setattr(int8_kernels, "STRICT", False)
    fns = forms(gpu)
    side = torch.cuda.Stream(gpu)
    side.wait_stream(torch.cuda.current_stream(gpu))
    for name, fn in fns.items():
        with torch.cuda.stream(side):
            a, b = outcome(fn, True), outcome(fn, False)
        side.synchronize()
        assert a[1:] == b[1:], (name, a[1:], b[1:])
        for s, t in zip(flat(a[0]), flat(b[0])):
            assert (s is None and t is None) or torch.equal(s, t), name
    torch.cuda.current_stream(gpu).wait_stream(side)


@pytest.mark.gpu
def test_native_path_equals_python_path_in_a_captured_graph(gpu):
    """One graph of a chain of calls on the native path, one on the Python path: every replay, with eager work between,
    gives the eager bits, after the inputs changed in place too."""
    g = torch.Generator(device=gpu).manual_seed(11)
    x = torch.randn(40, 2560, generator=g, device=gpu).to(BF)
    w = torch.randn(2560, generator=g, device=gpu).to(BF)
    qw = torch.randint(-127, 128, (6144, 2560), generator=g, device=gpu, dtype=torch.int8)
    sw = torch.rand(6144, generator=g, device=gpu) * 1e-2
    dw = torch.randint(-127, 128, (2560, 9728), generator=g, device=gpu, dtype=torch.int8)
    ds = torch.rand(2560, generator=g, device=gpu) * 1e-2
    h = torch.randn(440, 9728, generator=g, device=gpu).to(BF)

    def chain():
        (q, s), = fused_kernels.rms_norm_quant_multi(x, w, 1e-6, [None])
        y = int8_kernels.mm_i8(q, s, qw, sw, split="auto").view(1, 40, 24, 256)
        o = causal_gqa_attention(*y.split((16, 4, 4), dim=2))
        # 440 rows: the split along K, through the capturing stream's workspace
        return o, int8_kernels.mm_i8(*int8_kernels.act_quant(h), dw, ds, split="auto")

    stream = torch.cuda.Stream(gpu)
    runs = []
    keep = _lib.FAST
    try:
        for fast in (True, False):
            _lib.FAST = keep if fast else _lib._NotLoaded()
            stream.wait_stream(torch.cuda.current_stream(gpu))
            with torch.cuda.stream(stream):
                chain()
                graph = torch.cuda.CUDAGraph()
                with torch.cuda.graph(graph, stream=stream):
                    out = chain()
            runs.append((graph, out))
    finally:
        _lib.FAST = keep
    for i in range(4):
        if i == 2:
            x.mul_(-0.5)
            h.mul_(0.25)
        want = chain()
        for graph, out in runs:
            graph.replay()
            torch.cuda.synchronize()
            for a, b in zip(out, want):
                assert torch.equal(a, b), i


@pytest.mark.gpu
def test_prefix_from_an_iterator_survives_a_declined_call(gpu):
    """The native path declines [1, P, heads, 256] prefix views; the Python path after it still finds them."""
    g = torch.Generator(device=gpu).manual_seed(5)
    qkv = torch.randn(2, 40, 24, 256, generator=g, device=gpu).to(BF)
    q, k, v = qkv.split((16, 4, 4), dim=2)
    pre = torch.randn(2, 64, 4, 256, generator=g, device=gpu).to(BF)
    want = causal_gqa_attention(q, k, v, prefix=(pre[0], pre[1]))
    assert torch.equal(causal_gqa_attention(q, k, v, prefix=iter((pre[:1], pre[1:]))), want)


@pytest.mark.gpu
def test_native_path_leaves_watched_calls_to_python(gpu):
    """A dispatch mode, vmap or a tensor subclass: the native path declines, whatever Python then does."""
    x = torch.ones(4, 512, device=gpu, dtype=BF)
    assert _lib.FAST.act_quant(x, None, 0) is not None

    class Watch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    with Watch():
        assert _lib.FAST.act_quant(x, None, 0) is None
    seen = []

    def one(r):
        seen.append(_lib.FAST.act_quant(r, None, 0))
        return r

    torch.vmap(one)(x.view(2, 2, 512))
    assert seen == [None]
    assert _lib.FAST.act_quant(x.as_subclass(Sub), None, 0) is None


def test_native_path_declines_cpu_tensors_and_other_objects():
    _lib.load()
    x = torch.ones(4, 512, dtype=BF)
    for bad in (x, None, 3, "x"):
        assert _lib.FAST.act_quant(bad, None, 0) is None
        assert _lib.FAST.mm_i8(bad, x, x, x, None, 0, None, 0, False) is None
        assert _lib.FAST.norm_multi(bad, x, 1e-6, [None], None, 1.0, 0) is None
    with pytest.raises(TypeError):
        _lib.FAST.act_quant(x)
