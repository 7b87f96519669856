"""The calls whose speed matters to a user of this package, as cases that a timing program can run.

A case is a dict of plain values; ``listed()`` names twelve of them, ``draw(rng)`` makes more of the same
ranges.  Four kinds, each through the package's Python entry points as GPT-NeoX calls them:

* ``softmax`` -- ``FusedScaleMaskSoftmax`` on attention scores ``[b, np, s, s]``, forward only (evaluation,
  prefill) or forward and backward (training): causal or general fusion, a causal, sliding-window or padding
  mask, optionally with the ALiBi bias or the attention dropout folded in.  The module's backward pass writes
  the scores' gradient over the gradient it is given, which a model's graph makes anew every time and which
  therefore is copied here for every pass.  From 32 MiB of scores on that copy would be much of what is
  measured, and the host's time is hidden behind the kernels in any case: training pairs of that size go
  through the C-ABI of ``include/neox_fused.h``, forward and backward, which leaves its inputs alone;
* ``decode`` -- one generated token of one layer: the rotary of the token's q and k at its position, and the
  softmax of its scores against the key/value cache ``[b, np, 1, sk]``;
* ``rotary`` -- the rotary embedding of one layer's q and k over a whole sequence, in the form of
  ``form``: ``layer`` (q and k as views into the fused QKV projection, sliced to the rotated dims; the
  gradients come back dense), ``inplace`` (the fused QKV projection rotated where it lies), ``fused`` (the
  rope_fusion functions, one call per tensor, angles evaluated in the kernel) and ``cached`` (the same with
  tables);
* sizes: those of the repository's benchmark and tests (125M, 20B and 7B shapes, 2048 and 8192 tokens, a padded
  batch of 1024), evaluation and generation at whatever length a prompt has, and small models.
"""
import math

import torch

from gpt_neox_amd import _lib
from gpt_neox_amd.fused_kernels import scaled_masked_softmax_cuda as masked_softmax
from gpt_neox_amd.fused_rope import fused_apply_rotary_pos_emb, fused_apply_rotary_pos_emb_cached
from gpt_neox_amd.fused_softmax import FusedScaleMaskSoftmax, SoftmaxFusionTypes
from gpt_neox_amd.positional_embeddings import AliBi, apply_rotary_pos_emb, apply_rotary_pos_emb_qkv_

_DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}


def _softmax(name, b, np, s, hn, dtype, mask="causal", fusion="causal", train=False, window=0, dropout=0.0, alibi=False):
    return {"name": name, "kind": "softmax", "b": b, "np": np, "s": s, "hn": hn, "dtype": dtype, "mask": mask,
            "fusion": fusion, "train": train, "window": window, "dropout": dropout, "alibi": alibi}


def _rotary(name, s, b, np, hn, rot, dtype, form, train):
    return {"name": name, "kind": "rotary", "s": s, "b": b, "np": np, "hn": hn, "rot": rot, "dtype": dtype,
            "form": form, "train": train}


def _decode(name, b, np, hn, rot, sk, dtype):
    return {"name": name, "kind": "decode", "b": b, "np": np, "hn": hn, "rot": rot, "sk": sk, "dtype": dtype}


def listed():
    return [
        # the smallest call there is: one token of a 125M model's layer, four sequences, mid-generation
        _decode("decode_token", 4, 12, 64, 16, 517, "fp16"),
        # a training step of a small model on a short sequence: the host's own time counts
        _softmax("train_small", 2, 8, 256, 64, "bf16", train=True),
        # evaluation: a batch of short prompts, padded to the longest of them
        _softmax("eval_short_prompts", 32, 12, 129, 64, "fp16"),
        # evaluation at an odd length, one document per row
        _softmax("eval_odd_length", 6, 16, 1001, 64, "fp16"),
        # 125M pre-training, one layer of one micro-batch
        _softmax("train_125m", 4, 12, 2048, 64, "bf16", train=True),
        # a padded batch of sequences of different lengths, general fusion
        _softmax("train_padded_batch", 8, 16, 1024, 64, "fp16", mask="padding", fusion="general", train=True),
        # 20B shape with attention dropout
        _softmax("train_20b_dropout", 1, 64, 2048, 96, "fp16", train=True, dropout=0.1),
        # long context, 7B shape: the largest
        _softmax("train_long_context", 1, 32, 8192, 128, "bf16", train=True),
        # sliding-window attention at half the context of its model
        _softmax("train_sliding_window", 1, 32, 4096, 128, "bf16", mask="window", window=1024, train=True),
        # partial rotary (a quarter of every head) of one layer's q and k, and its gradients
        _rotary("rotary_partial", 2048, 4, 32, 128, 32, "bf16", "layer", True),
        # full rotary in place on the long-context QKV projection (no gradient: evaluation, prefill)
        _rotary("rotary_in_place", 8192, 1, 32, 128, 128, "bf16", "inplace", False),
        # rope_fusion on the 20B heads
        _rotary("rotary_fused", 2048, 2, 64, 96, 24, "fp16", "fused", True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _largest(c):
    """Elements a drawn case works on, kept within a quarter of the largest listed case's."""
    return c["b"] * c["np"] * c["s"] * (c["s"] if c["kind"] == "softmax" else c["hn"])


def draw(rng):
    """One more case: any kind, its sizes spread over the logarithm of their range, odd lengths among them."""
    kind = rng.choice(["decode", "softmax", "softmax", "softmax", "softmax", "rotary", "rotary"])
    dtype = rng.choice(["fp16", "bf16"])
    hn = rng.choice([64, 80, 96, 128, 256])
    np = rng.choice([4, 8, 12, 16, 20, 32, 40, 64])
    rot = rng.choice([hn, hn // 4, hn // 2])
    if kind == "decode":
        c = _decode("", rng.choice([1, 2, 3, 4, 8, 16]), np, hn, rot, _log_int(rng, 33, 4096), dtype)
    elif kind == "rotary":
        form = rng.choice(["layer", "inplace", "fused", "cached"])
        s = _log_int(rng, 128, 8192)
        b = rng.choice([1, 2, 4])
        c = _rotary("", s, b, np, hn, rot, dtype, form, form != "inplace" and rng.random() < 0.6)
        while _largest(c) > 2**27 and c["b"] > 1:
            c["b"] //= 2
        while _largest(c) > 2**27:
            c["s"] = c["s"] // 2 + 1
    else:
        use = rng.choice(["eval", "train", "train", "train_padded", "train_window"])
        s = _log_int(rng, 48, 8192)
        if use != "eval" and rng.random() < 0.7:  # training lengths are mostly multiples of 64, evaluation is any length
            s = max(64, s // 64 * 64)
        c = _softmax("", rng.choice([1, 2, 4, 8, 16, 32]), np, s, hn, dtype, train=use != "eval")
        if use == "train":
            c["dropout"] = rng.choice([0.0, 0.0, 0.1])
            c["alibi"] = rng.random() < 0.2
        elif use == "train_padded":
            c["mask"], c["fusion"] = "padding", "general"
        elif use == "train_window" and s >= 640:
            # (the lengths the sliding-window entry points take: a multiple of 8)
            c["s"] = s // 8 * 8
            c["mask"], c["window"] = "window", rng.choice([s // 4, s // 2])
        elif use == "eval" and rng.random() < 0.3:
            c["mask"], c["fusion"] = "padding", "general"
        while _largest(c) > 2**29 and c["b"] > 1:
            c["b"] //= 2
        while _largest(c) > 2**29:
            c["np"] //= 2
    del c["name"]
    return c


def _mask_func(scores, mask):
    return scores.masked_fill_(mask, torch.finfo(scores.dtype).min)


def _causal_mask(n, device, window=0):
    hidden = torch.ones(n, n, dtype=torch.bool, device=device).triu_(1)
    if window:
        hidden |= torch.ones(n, n, dtype=torch.bool, device=device).tril_(-window - 1)
    return hidden.view(1, 1, n, n)


def _tables(rot, n, device):
    """fp32 angles, cos and sin ``[n, 1, 1, rot]``, base 10000."""
    freqs = torch.outer(torch.arange(n, dtype=torch.float32),
                        1.0 / (10000 ** (torch.arange(0, rot, 2, dtype=torch.float32) / rot)))
    angles = torch.cat((freqs, freqs), dim=-1)[:, None, None, :].to(device)
    return angles, angles.cos(), angles.sin()


def _module(case):
    half = case["dtype"] == "fp16"
    fusion = SoftmaxFusionTypes.general if case.get("fusion") == "general" else SoftmaxFusionTypes.upper_triang
    return FusedScaleMaskSoftmax(half, not half, fusion, _mask_func, True, 1.0 / math.sqrt(case["hn"]))


def prepare(case, seed):
    device = torch.device("cuda")
    gen = torch.Generator(device=device)
    gen.manual_seed(seed)
    dtype = _DTYPES[case["dtype"]]

    def normal(*shape, std=1.0):
        t = torch.empty(shape, dtype=dtype, device=device)
        return t.normal_(0.0, std, generator=gen)

    state = dict(case)
    if case["kind"] == "softmax":
        b, np, s = case["b"], case["np"], case["s"]
        # attention scores as they leave the q.k product: a standard deviation of 8 before the scale
        state["x"] = normal(b, np, s, s, std=8.0).requires_grad_(case["train"])
        if case["train"]:
            state["g"] = normal(b, np, s, s)
        if case["mask"] == "padding":
            # sequences of a quarter to all of the common length; the last one fills it
            lens = torch.randint(max(1, s // 4), s + 1, (b,), device=device, generator=gen)
            lens[-1] = s
            keys = torch.arange(s, device=device)
            state["mask_tensor"] = (keys[None, :] >= lens[:, None])[:, None, None, :].expand(b, 1, s, s).contiguous()
        else:
            state["mask_tensor"] = _causal_mask(s, device, case["window"])
        state["module"] = _module(case)
        if case["alibi"]:
            state["slopes"] = AliBi(np, mp_size=1, mp_rank=0).slopes.to(device)
        if _through_the_c_abi(case):
            state["x"] = state["x"].detach()
            state["philox_seed"] = seed
            if case["mask"] == "padding":
                state["row_end"] = masked_softmax.scan_mask(state["mask_tensor"])[1]
        torch.manual_seed(seed)  # the generator that the module's attention dropout draws from
    elif case["kind"] == "decode":
        b, np, hn, sk = case["b"], case["np"], case["hn"], case["sk"]
        state["qkv"] = normal(1, b, np, 3 * hn)
        state["x"] = normal(b, np, 1, sk, std=8.0)
        _, state["cos"], state["sin"] = _tables(case["rot"], 4096, device)
        state["mask_tensor"] = _causal_mask(4096, device)
        state["module"] = _module(case)
    else:
        s, b, np, hn, rot = case["s"], case["b"], case["np"], case["hn"], case["rot"]
        train = case["train"]
        angles, cos, sin = _tables(rot, s, device)
        state["angles"], state["cos"], state["sin"] = angles, cos, sin
        if case["form"] in ("layer", "inplace"):
            mixed = normal(s, b, np, 3 * hn)
            if case["form"] == "layer":
                state["q"] = mixed[..., :hn].detach().requires_grad_(train)
                state["k"] = mixed[..., hn : 2 * hn].detach().requires_grad_(train)
            state["mixed"] = mixed
        else:
            state["q"] = normal(s, b, np, hn).requires_grad_(train)
            state["k"] = normal(s, b, np, hn).requires_grad_(train)
        if train:
            width = rot if case["form"] == "layer" else hn
            state["gq"], state["gk"] = normal(s, b, np, width), normal(s, b, np, width)
    return state


def _through_the_c_abi(case):
    return case["train"] and 2 * case["b"] * case["np"] * case["s"] ** 2 >= 32 << 20


def _run_softmax(state):
    if _through_the_c_abi(state):
        return _run_softmax_c_abi(state)
    module, x, mask = state["module"], state["x"], state["mask_tensor"]
    slopes, p = state.get("slopes"), state["dropout"]
    if not state["train"]:
        with torch.no_grad():
            return module(x, mask, alibi_slopes=slopes)
    y = module(x, mask, alibi_slopes=slopes, dropout_p=p)
    (dx,) = torch.autograd.grad(y, x, state["g"].clone())
    return y.detach(), dx


def _run_softmax_c_abi(state):
    """The two entry points the module would use for this mask, into new tensors: the probabilities (and the
    dropped ones) and the scores' gradient."""
    lib, x, g = _lib.lib(), state["x"], state["g"]
    b, np, s, p = state["b"], state["np"], state["s"], state["dropout"]
    scale, seed = 1.0 / math.sqrt(state["hn"]), state["philox_seed"]
    slopes = state["slopes"].data_ptr() if state["alibi"] else None
    code, stream = _lib.dtype_code(x.dtype), torch.cuda.current_stream().cuda_stream
    y, dx = torch.empty_like(x), torch.empty_like(x)
    xp, yp, gp, dxp = x.data_ptr(), y.data_ptr(), g.data_ptr(), dx.data_ptr()
    if state["mask"] == "padding":
        ends = state["row_end"]
        _lib.check(lib.neox_masked_softmax_ends_fwd(
            None, yp, xp, state["mask_tensor"].data_ptr(), ends.data_ptr(), slopes, None, 0, scale, 0.0, 0, 0, None,
            b, np, s, s, b, code, stream))
        _lib.check(lib.neox_masked_softmax_ends_bwd(
            dxp, gp, yp, ends.data_ptr(), scale, 0, 0.0, 0, 0, None, b, np, s, s, b, code, stream))
    elif state["mask"] == "window":
        window = state["window"]
        _lib.check(lib.neox_sliding_window_softmax_fwd(yp, xp, scale, b * np, s, s, window, code, stream))
        _lib.check(lib.neox_sliding_window_softmax_bwd(dxp, gp, yp, scale, b * np, s, s, window, code, stream))
    elif p:
        dropped = torch.empty_like(x)
        _lib.check(lib.neox_causal_softmax_dropout_fwd(
            dropped.data_ptr(), yp, xp, slopes, None, 0, scale, p, seed, 0, None, b, np, s, s, code, stream))
        _lib.check(lib.neox_causal_softmax_dropout_bwd(
            dxp, gp, yp, scale, p, seed, 0, None, b * np, s, s, code, stream))
        return dropped, y, dx
    else:
        if slopes:
            _lib.check(lib.neox_causal_softmax_alibi_fwd(yp, xp, slopes, scale, b, np, s, s, code, stream))
        else:
            _lib.check(lib.neox_causal_softmax_fwd(yp, xp, scale, b * np, s, s, code, stream))
        _lib.check(lib.neox_causal_softmax_bwd(dxp, gp, yp, scale, b * np, s, s, code, stream))
    return y, dx


def _run_decode(state):
    hn, rot, at = state["hn"], state["rot"], state["sk"] - 1
    with torch.no_grad():
        mixed = state["qkv"]
        q, k = mixed[..., :hn], mixed[..., hn : 2 * hn]
        q, k = apply_rotary_pos_emb(q[..., :rot], k[..., :rot], state["cos"], state["sin"], offset=at)
        mask = state["mask_tensor"][..., at, : at + 1].unsqueeze(2)
        return q, k, state["module"](state["x"], mask)


def _run_rotary(state):
    form, rot, train = state["form"], state["rot"], state["train"]
    cos, sin = state["cos"], state["sin"]
    if form == "inplace":
        with torch.no_grad():
            apply_rotary_pos_emb_qkv_(state["mixed"], cos, sin, rotary_ndims=rot)
        return state["mixed"]
    with torch.set_grad_enabled(train):
        q, k = state["q"], state["k"]
        if form == "layer":
            q, k = q[..., :rot], k[..., :rot]  # as the layer slices them; the gradient of the slice is the layer's
            oq, ok = apply_rotary_pos_emb(q, k, cos, sin)
        elif form == "fused":
            oq, ok = (fused_apply_rotary_pos_emb(t, state["angles"]) for t in (q, k))
        else:
            oq, ok = (fused_apply_rotary_pos_emb_cached(t, cos, sin) for t in (q, k))
        if not train:
            return oq, ok
        dq, dk = torch.autograd.grad((oq, ok), (q, k), (state["gq"], state["gk"]))
        return oq.detach(), ok.detach(), dq, dk


def run(state):
    kind = state["kind"]
    if kind == "softmax":
        return _run_softmax(state)
    if kind == "decode":
        return _run_decode(state)
    return _run_rotary(state)


def work(case):
    """Bytes: each input read once, each output written once.  Scores, probabilities and gradients of hidden
    keys need not be read, but the outputs are dense.  Flops: about ten per visible score and pass, six per
    rotated element."""
    e = 2
    if case["kind"] == "softmax":
        b, np, s = case["b"], case["np"], case["s"]
        full = s * s
        seen = s * (s + 1) // 2
        if case["mask"] == "window" and case["window"]:
            w = min(case["window"], s - 1)
            seen = (w + 1) * (w + 2) // 2 + (s - 1 - w) * (w + 1)
        elif case["mask"] == "padding":
            seen = int(full * (5 * (b - 1) / 8 + 1) / b)  # mean length 5/8 of the common one, the last is full
        mask_bytes = b * full if case["mask"] == "padding" else 0
        bytes_ = b * np * e * (seen + full) + mask_bytes  # forward: scores in, probabilities out
        flops = 10 * b * np * seen
        if case["train"]:
            bytes_ += b * np * e * (2 * seen + full)  # backward: gradient and probabilities in, gradient out
            if case["dropout"]:
                bytes_ += b * np * e * full  # the dropped probabilities beside the kept ones
            flops *= 2
        return {"bytes": bytes_, "flops": flops}
    if case["kind"] == "decode":
        b, np, sk, rot = case["b"], case["np"], case["sk"], case["rot"]
        bytes_ = 2 * b * np * sk * e + sk + 4 * b * np * rot * e + 2 * rot * 4
        return {"bytes": bytes_, "flops": 10 * b * np * sk + 12 * b * np * rot}
    s, b, np, hn, rot = case["s"], case["b"], case["np"], case["hn"], case["rot"]
    passes = 2 if case["train"] else 1
    width = rot if case["form"] in ("layer", "inplace") else hn  # the fused forms return whole heads
    table = 2 * s * rot * 4
    bytes_ = passes * (2 * 2 * s * b * np * width * e + table)
    return {"bytes": bytes_, "flops": passes * 2 * s * b * np * rot * 6}


# Four times what the paths differ by from the same computation in 64 bits: rounding to the storage type is
# all there is to see -- of the outputs (2e-4 and 1.7e-3 in the 2-norm), and for the softmax's gradient of the
# probabilities it is formed from too (3.0e-4 and 2.3e-3, the largest of any case).
_TOLERANCE = {"fp16": 1.2e-3, "bf16": 9.2e-3}


def tolerance(case):
    return {"rel": _TOLERANCE[case["dtype"]]}
