"""The shim's native host path under the parts of torch that have to see a call as one operation of its own: what an
autograd Function is given (a tracer's record, a refusal of forward-mode gradients, zeros for outputs without a
gradient, saved tensors as they were) holds for the C++ nodes too."""
import pytest
import torch

from oracle import rotary as orot
from tests.util import make_qkv

pytestmark = pytest.mark.gpu


def _attention_args(B, H, Lq, Lk, D, block, seed, dropout=False):
    q, k, v = (t.cuda() for t in make_qkv(B, H, Lq, Lk, D, seed=seed))
    g = torch.Generator().manual_seed(seed)
    factors = (torch.rand(B, H, Lk // block, Lq, generator=g) >= 0.5).float().mul(2.0).cuda() if dropout else None
    return q, k, v, factors


def _rotary_args(B, H, L, D, seed):
    q, k, _ = (t.cuda() for t in make_qkv(B, H, L, L, D, seed=seed))
    cos, sin = (t.cuda() for t in orot.rotary_tables(2 * L, D, torch.bfloat16))
    return q, k, cos, sin, torch.arange(3, 3 + L, device="cuda")[None]


@pytest.mark.parametrize("D,block,dropout", [(128, 32, False), (64, 51, False), (32, 64, False), (64, 51, True)])
def test_a_traced_attention_computes_on_the_inputs_of_each_call(D, block, dropout):
    from ltriton.flash_landmark_attention import fused_landmark_attention
    print(f"case trace attention D{D} bs{block} dropout{dropout}", flush=True)
    f = (lambda q, k, v, gs: fused_landmark_attention(q, k, v, None, block_size=block, group_scale=gs)) if dropout else \
        (lambda q, k, v: fused_landmark_attention(q, k, v, None, block_size=block))
    args = [[t for t in _attention_args(1, 2, L, L + n * block, D, block, seed, dropout) if t is not None]
            for seed, (L, n) in enumerate([(4 * block, 0), (4 * block, 0), (2 * block, 3)])]       # other lengths, a history
    traced = torch.jit.trace(f, args[0])
    for a in args:
        leaves = [t.detach().requires_grad_(i < 3) for i, t in enumerate(a)]
        want, got = f(*leaves), traced(*leaves)
        assert torch.equal(got, want)
        do = torch.ones_like(want)
        for x, y in zip(torch.autograd.grad(got, leaves[:3], do), torch.autograd.grad(want, leaves[:3], do)):
            assert torch.equal(x, y)


@pytest.mark.parametrize("shapes", ["q and k", "k alone", "fewer key heads"])
def test_a_traced_rotary_computes_on_the_inputs_of_each_call(shapes):
    from landmark_hip.rotary import apply_rotary_pos_emb
    print(f"case trace rotary {shapes}", flush=True)

    def f(q, k, cos, sin, pos):
        q_embed, k_embed = apply_rotary_pos_emb(None if shapes == "k alone" else q, k, cos, sin, pos)
        return k_embed if q_embed is None else (q_embed, k_embed)

    args = [list(_rotary_args(2, 4, L, 64, seed)) for seed, L in enumerate([40, 40, 23])]
    for a in args:
        a[1] = a[1][:, :2].contiguous() if shapes == "fewer key heads" else a[1]
    traced = torch.jit.trace(f, args[0])
    for a in args:
        leaves = [t.detach().requires_grad_(i < 2) for i, t in enumerate(a)]
        used = leaves[1:2] if shapes == "k alone" else leaves[:2]
        outs = [f(*leaves), traced(*leaves)]
        grads = []
        for out in outs:
            out = out if isinstance(out, tuple) else (out,)
            grads.append(torch.autograd.grad(out, used, [torch.sin(o.detach().float()).bfloat16() for o in out]) + out)
        assert all(torch.equal(x, y) for x, y in zip(*grads))


@pytest.mark.parametrize("which", ["q", "k", "v", "group factors", "none"])
def test_attention_refuses_forward_mode_gradients(which):
    import torch.autograd.forward_ad as fw
    from ltriton.flash_landmark_attention import fused_landmark_attention
    args = dict(zip(["q", "k", "v", "group factors"], _attention_args(1, 2, 96, 96, 64, 32, 5, dropout=which == "group factors")))
    call = lambda: fused_landmark_attention(args["q"], args["k"], args["v"], None, block_size=32, group_scale=args["group factors"])
    want = call()
    with fw.dual_level():
        if which == "none":                                   # a dual level by itself changes nothing
            assert torch.equal(call(), want)
            return
        args[which] = fw.make_dual(args[which], torch.ones_like(args[which]))
        with pytest.raises(NotImplementedError):
            call()


@pytest.mark.parametrize("which", [0, 1, 2, 3, None])
def test_rotary_refuses_forward_mode_gradients(which):
    import torch.autograd.forward_ad as fw
    from landmark_hip.rotary import apply_rotary_pos_emb
    args = list(_rotary_args(1, 2, 33, 64, 6))
    want = apply_rotary_pos_emb(*args)
    with fw.dual_level():
        if which is None:
            assert all(torch.equal(a, b) for a, b in zip(apply_rotary_pos_emb(*args), want))
            return
        args[which] = fw.make_dual(args[which], torch.ones_like(args[which]))
        with pytest.raises(NotImplementedError):
            apply_rotary_pos_emb(*args)
        if which == 1:
            with pytest.raises(NotImplementedError):
                apply_rotary_pos_emb(None, *args[1:])


class _NoGradient(torch.autograd.Function):
    """Hands its input on and no gradient back."""

    @staticmethod
    def forward(ctx, x):
        return x.clone()

    @staticmethod
    def backward(ctx, dy):
        return None


@pytest.mark.parametrize("D,block,dropout", [(128, 32, False), (64, 51, True)])
def test_an_output_that_no_gradient_reaches_gives_zero_gradients(D, block, dropout):
    # as the reference's Function does, whose backward is handed zeros (flash_landmark_attention.py:356-389)
    from ltriton.flash_landmark_attention import fused_landmark_attention
    q, k, v, factors = _attention_args(1, 2, 2 * block, 4 * block, D, block, 7, dropout)
    leaves = [t.requires_grad_(True) for t in (q, k, v)]
    out = fused_landmark_attention(*leaves, None, block_size=block, group_scale=factors)
    for x, g in zip(leaves, torch.autograd.grad(_NoGradient.apply(out).float().sum(), leaves)):
        assert g.shape == x.shape and g.dtype == x.dtype and not g.any()


def _unpacked_as(change):
    return torch.autograd.graph.saved_tensors_hooks(lambda t: t, change)


_LAYOUTS = {
    "contiguous copies": lambda t: t.clone(memory_format=torch.contiguous_format),
    "rows apart": lambda t: torch.cat((t, t), dim=-1)[..., : t.shape[-1]],
    "through the host": lambda t: t.cpu().cuda(),
}
_NOT_AS_SAVED = {
    "another type": lambda t: t.half(),
    "wider": lambda t: t.float(),
    "last dim not dense": lambda t: torch.stack((t, t), dim=-1)[..., 0],
    "fewer rows": lambda t: t[..., : t.shape[-2] - 1, :],
    "on the host": lambda t: t.cpu(),
}


@pytest.mark.parametrize("how", [*_LAYOUTS, *_NOT_AS_SAVED])
@pytest.mark.parametrize("what", ["attention", "attention with factors", "rotary"])
def test_what_saved_tensor_hooks_hand_back_is_used_or_refused(what, how):
    # the kernels take a pointer, a type and strides: a hook's tensor is used when it is what was saved, in any layout they
    # read, and refused on the host otherwise
    from landmark_hip.rotary import apply_rotary_pos_emb
    from ltriton.flash_landmark_attention import fused_landmark_attention
    print(f"case hooks {what}: {how}", flush=True)
    if what == "rotary":
        q, k, *tables = _rotary_args(2, 3, 40, 64, 8)
        leaves = [t.requires_grad_(True) for t in (q, k)]
        call = lambda: torch.stack(apply_rotary_pos_emb(*leaves, *tables))
    else:
        q, k, v, factors = _attention_args(2, 2, 102, 153, 64, 51, 8, what != "attention")
        leaves = [t.transpose(1, 2).contiguous().transpose(1, 2).requires_grad_(True) for t in (q, k, v)]
        call = lambda: fused_landmark_attention(*leaves, None, block_size=51, group_scale=factors)
    do = torch.randn(call().shape, generator=torch.Generator().manual_seed(1)).bfloat16().cuda()
    want = torch.autograd.grad(call(), leaves, do)
    with _unpacked_as((_LAYOUTS | _NOT_AS_SAVED)[how]):
        out = call()
    if how in _LAYOUTS:
        for x, y in zip(torch.autograd.grad(out, leaves, do), want):
            assert torch.equal(x, y)
    elif not (what == "rotary" and how == "last dim not dense"):          # tables and positions are laid out anew
        with pytest.raises(AssertionError):
            torch.autograd.grad(out, leaves, do)


@pytest.mark.parametrize("what,other", [("attention", "backward"), ("attention", "saved_tensors"), ("rotary", "backward")])
def test_threads_use_a_shared_node_one_after_the_other(what, other):
    # a backward pass unpacks and releases a node's saved tensors in the engine's thread, another thread looks at them
    # through the node's `saved_tensors`: they belong to one of them at a time
    import threading
    from landmark_hip.rotary import apply_rotary_pos_emb
    from ltriton.flash_landmark_attention import fused_landmark_attention
    inside, peak, changed = 0, 0, threading.Condition()

    def unpack(t):                                            # stays a moment for the other thread to come in
        nonlocal inside, peak
        with changed:
            inside += 1
            peak = max(peak, inside)
            changed.notify_all()
            changed.wait_for(lambda: peak > 1, timeout=0.1)
            inside -= 1
        return t

    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, unpack):
        if what == "attention":
            q, k, v, _ = _attention_args(1, 2, 64, 64, 64, 32, 9)
            leaves = [t.requires_grad_(True) for t in (q, k, v)]
            out = fused_landmark_attention(*leaves, None, block_size=32)
        else:
            _, k, *tables = _rotary_args(1, 2, 40, 64, 9)
            leaves = [k.requires_grad_(True)]
            out = apply_rotary_pos_emb(None, k, *tables)[1]
    loss = out.float().sum()
    start, errors = threading.Barrier(2), []

    def use(kind):
        try:
            start.wait(timeout=20)
            if kind == "backward":
                torch.autograd.grad(loss, leaves, retain_graph=True)
            else:
                assert torch.equal(out.grad_fn.saved_tensors[3], out)
        except Exception as e:
            errors.append(e)

    threads = [threading.Thread(target=use, args=(kind,)) for kind in ("backward", other)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(timeout=30)
    assert not errors and not any(t.is_alive() for t in threads) and peak == 1
