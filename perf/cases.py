"""The calls whose speed this framework is held to, with the inputs a user's program has in
hand, the call itself, and the same results in float64 from plain torch.

Seven kinds of call, each through the package's public entry points:

* ``forward``  -- `mamba3_siso_layer` without gradients (prefill, evaluation);
* ``segment``  -- the same from a carried state (the next block of a long prompt);
* ``train``    -- the layer forward and backward: the output and every gradient;
* ``decode``   -- `mamba3_siso_decode_step`, one token for a batch of sequences;
* ``run``      -- `decode_scan`, a known-length run of decode steps (a prompt's remainder,
  the verification of drafted tokens);
* ``lm_train`` -- the byte LM's logits, loss and all gradients;
* ``lm_decode``-- one recorded decode step of the whole byte LM (`DecodeGraph`).
"""

from __future__ import annotations

import math

import torch
import torch.nn.functional as F

import __graft_entry__

m3 = __graft_entry__.load_package()

DEVICE = "cuda"
VOCAB = 256
F64_CHUNK = 64


def listed():
    layer = dict(d_model=1024, d_state=128, headdim=64, expand=2, policy="bf16")
    lm_layer = dict(layer, d_model=768)
    return [
        # prefill or evaluation over full-length documents at a serving batch: the largest forward
        dict(name="forward_b8_l8192", kind="forward", batch=8, seqlen=8192, chunk=128, **layer),
        # one user's prompt: few sequences, so few independent scans
        dict(name="forward_b1_l2048", kind="forward", batch=1, seqlen=2048, chunk=128, **layer),
        # a few prompts of uneven length, padded to the next whole chunk
        dict(name="forward_b3_l1920", kind="forward", batch=3, seqlen=1920, chunk=128, **lm_layer),
        # the next block of one long prompt, from the state that the last one left
        dict(name="segment_b1_l896", kind="segment", batch=1, seqlen=896, chunk=128, **lm_layer),
        # one layer of long-context pretraining
        dict(name="train_b8_l8192", kind="train", batch=8, seqlen=8192, chunk=128, **layer),
        # one layer of the byte LM's training step
        dict(name="train_b16_l2048", kind="train", batch=16, seqlen=2048, chunk=128, **lm_layer),
        # fine-tuning on single documents: batch one, a middling length
        dict(name="train_b1_l4096", kind="train", batch=1, seqlen=4096, chunk=128, **layer),
        # the float32 policy, which validates a port or a small model
        dict(name="train_f32_b1_l512", kind="train", batch=1, seqlen=512, chunk=64, d_model=64,
             d_state=16, headdim=16, expand=1, policy="f32"),
        # serving: one token for each of many sequences, bound by the states' traffic
        dict(name="decode_b256", kind="decode", batch=256, **layer),
        # a prompt's remainder for one user, in one launch
        dict(name="run_b1_t512", kind="run", batch=1, steps=512, **layer),
        # the byte LM's training step up to its gradients, at four layers of its stack
        dict(name="lm_train_b16_l2048", kind="lm_train", batch=16, seqlen=2048, n_layers=4,
             d_intermediate=1536, chunk=128, **lm_layer),
        # interactive generation, the smallest call: one token for one user, latency alone
        dict(name="lm_decode_b1", kind="lm_decode", batch=1, n_layers=8, d_intermediate=1536,
             chunk=128, **lm_layer),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["forward", "forward", "segment", "train", "train", "train_f32", "decode",
                       "decode", "run", "lm_train", "lm_decode"])
    if kind == "train_f32":
        return dict(kind="train", batch=rng.randint(1, 4), seqlen=64 * _log_int(rng, 1, 24),
                    chunk=64, d_model=16 * rng.randint(2, 8), d_state=rng.choice([16, 32]),
                    headdim=16, expand=rng.choice([1, 2]), policy="f32")
    shape = dict(d_model=64 * rng.randint(4, 16), d_state=rng.choice([128, 128, 128, 64]),
                 headdim=64, expand=2, policy="bf16")
    if kind in ("forward", "segment", "train"):
        if rng.random() < 0.15:
            shape.update(d_model=128 * rng.randint(2, 8), headdim=128)
        seqlen = 128 * _log_int(rng, 1, 64)
        limit = {"forward": 65536, "segment": 16384, "train": 65536}[kind]
        batch = min(_log_int(rng, 1, 16), max(1, limit // seqlen))
        return dict(kind=kind, batch=batch, seqlen=seqlen, chunk=128, **shape)
    if kind == "decode":
        return dict(kind=kind, batch=_log_int(rng, 1, 256), **shape)
    if kind == "run":
        steps = _log_int(rng, 2, 512)
        return dict(kind=kind, batch=min(_log_int(rng, 1, 256), max(1, 16384 // steps)),
                    steps=steps, **shape)
    shape.update(d_model=64 * rng.randint(6, 12), d_state=128)
    lm = dict(n_layers=rng.randint(2, 8 if kind == "lm_decode" else 5),
              d_intermediate=2 * shape["d_model"], chunk=128)
    if kind == "lm_decode":
        return dict(kind=kind, batch=_log_int(rng, 1, 64), **lm, **shape)
    seqlen = 128 * _log_int(rng, 1, 16)
    return dict(kind=kind, batch=min(_log_int(rng, 1, 16), 32768 // seqlen), seqlen=seqlen,
                **lm, **shape)


# ----------------------------------------------------------------------------------------
# inputs
# ----------------------------------------------------------------------------------------


def _config(case):
    return m3.SISOConfig(d_model=case["d_model"], d_state=case["d_state"],
                         headdim=case["headdim"], expand=case["expand"],
                         chunk=case.get("chunk", 128), policy_name=case["policy"])


def _lm_config(case):
    return m3.model.LMConfig(vocab_size=VOCAB, n_layers=case["n_layers"], siso=_config(case),
                             d_intermediate=case["d_intermediate"])


def _dtype(case):
    return torch.bfloat16 if case["policy"] == "bf16" else torch.float32


def _vary(params, gen):
    """Gains, biases and skips as training leaves them: not all the same value."""
    near = lambda t: t + 0.1 * torch.randn(t.shape, generator=gen, device=DEVICE)  # noqa: E731
    return params._replace(b_norm_weight=near(params.b_norm_weight),
                           c_norm_weight=near(params.c_norm_weight), b_bias=near(params.b_bias),
                           c_bias=near(params.c_bias), d_skip=near(params.d_skip))


def _carry(cfg, batch, gen):
    """A state as a prefill leaves it (float32; phi in [0, 2 pi))."""
    h, p, n, r = cfg.nheads, cfg.headdim, cfg.d_state, cfg.n_angles
    normal = lambda *s: torch.randn(*s, generator=gen, device=DEVICE)  # noqa: E731
    return m3.SISOState(
        ssm=0.1 * normal(batch, h, p, n), k=normal(batch, h, n), v=normal(batch, h, p),
        phi=2 * math.pi * torch.rand(batch, h, r, generator=gen, device=DEVICE))


def _inputs(case, seed):
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    kind, batch, dt = case["kind"], case["batch"], _dtype(case)
    normal = lambda *s: torch.randn(*s, generator=gen, device=DEVICE)  # noqa: E731
    cfg = _config(case)
    if kind in ("lm_train", "lm_decode"):
        lm = _lm_config(case)
        params = m3.model.init_lm(lm, seed, device=DEVICE)
        params = params._replace(blocks=[b._replace(siso=_vary(b.siso, gen))
                                         for b in params.blocks])
        ids = lambda *s: torch.randint(0, VOCAB, s, generator=gen, device=DEVICE)  # noqa: E731
        if kind == "lm_train":
            text = ids(batch, case["seqlen"] + 1)
            return dict(params=params, xs=text[:, :-1].contiguous(), ys=text[:, 1:].contiguous())
        return dict(params=params, token=ids(batch),
                    states=[_carry(cfg, batch, gen) for _ in range(case["n_layers"])])
    if kind == "run":
        h, p, n, r, steps = cfg.nheads, cfg.headdim, cfg.d_state, cfg.n_angles, case["steps"]
        uniform = lambda *s: torch.rand(*s, generator=gen, device=DEVICE)  # noqa: E731
        step = torch.exp(uniform(batch, h, steps) * math.log(100.0) + math.log(1e-3))
        return dict(q=normal(batch, steps, n).to(dt), k=normal(batch, steps, n).to(dt),
                    v=normal(batch, h, steps, p).to(dt), z=normal(batch, h, steps, p).to(dt),
                    adt=-step * (0.5 + uniform(batch, h, steps)), dt=step,
                    lam=uniform(batch, h, steps), angles=normal(batch, steps, r),
                    q_bias=1 + 0.1 * normal(h, n), k_bias=1 + 0.1 * normal(h, n),
                    d_skip=1 + 0.1 * normal(h), state=_carry(cfg, batch, gen))
    params = _vary(m3.init_params(cfg, seed, device=DEVICE), gen)
    if kind == "decode":
        return dict(params=params, u=normal(batch, cfg.d_model).to(dt),
                    state=_carry(cfg, batch, gen))
    out = dict(params=params, u=normal(batch, case["seqlen"], cfg.d_model).to(dt))
    if kind == "segment":
        out["state"] = _carry(cfg, batch, gen)
    if kind == "train":
        out["dy"] = normal(batch, case["seqlen"], cfg.d_model).to(dt)
    return out


def prepare(case, seed):
    state = _inputs(case, seed)
    state["kind"] = case["kind"]
    if case["kind"] in ("lm_train", "lm_decode"):
        state["cfg"] = _lm_config(case)
    else:
        state["cfg"] = _config(case)
    if case["kind"] in ("forward", "segment", "decode"):   # inference keeps its weights in bf16
        p, dt = state["params"], _dtype(case)
        state["params"] = p._replace(in_proj=p.in_proj.to(dt), out_proj=p.out_proj.to(dt))
    elif case["kind"] == "train":
        state["params"] = m3.SISOParams(*(t.requires_grad_(True) for t in state["params"]))
        state["u"].requires_grad_(True)
    elif case["kind"] == "lm_train":
        state["params"] = m3.train.train_params(state["params"])
    elif case["kind"] == "lm_decode":
        params = m3.model.decode_params(state["params"], state["cfg"])
        state["graph"] = m3.train.DecodeGraph(params, state["cfg"], batch=case["batch"])
        state["graph"].load_states(state["states"])
    return state


# ----------------------------------------------------------------------------------------
# the call
# ----------------------------------------------------------------------------------------


def run(state):
    kind, cfg = state["kind"], state["cfg"]
    if kind in ("forward", "segment"):
        with torch.no_grad():
            out, carry = m3.mamba3_siso_layer(state["params"], state["u"], cfg,
                                              state=state.get("state"))
        return dict(out=out, **carry._asdict())
    if kind == "train":
        out, _ = m3.mamba3_siso_layer(state["params"], state["u"], cfg)
        grads = torch.autograd.grad(out, (state["u"], *state["params"]), state["dy"])
        return dict(out=out.detach(), du=grads[0],
                    **{"d_" + f: g for f, g in zip(m3.SISOParams._fields, grads[1:])})
    if kind == "decode":
        with torch.no_grad():
            out, state["state"] = m3.mamba3_siso_decode_step(state["params"], state["u"], cfg,
                                                             state["state"])
        return dict(out=out, **state["state"]._asdict())
    if kind == "run":
        with torch.no_grad():
            y, state["state"] = m3.decode_scan(
                state["q"], state["k"], state["v"], state["adt"], state["dt"], state["lam"],
                state["angles"], state["q_bias"], state["k_bias"], state["state"],
                d_skip=state["d_skip"], z=state["z"], dtype_policy=cfg.policy_name)
        return dict(y=y, **state["state"]._asdict())
    if kind == "lm_train":
        logits = m3.model.lm_forward(state["params"], state["xs"], cfg)
        loss = F.cross_entropy(logits.reshape(-1, VOCAB), state["ys"].reshape(-1))
        grads = torch.autograd.grad(loss, m3.model.lm_leaves(state["params"]))
        return dict(logits=logits.detach(), loss=loss.detach(), grads=list(grads))
    logits = state["graph"].step(state["token"])
    return dict(logits=logits, states=[tuple(s) for s in state["graph"].states])


# ----------------------------------------------------------------------------------------
# what a pass cannot do without
# ----------------------------------------------------------------------------------------


def _shape(case):
    dm, n, p = case["d_model"], case["d_state"], case["headdim"]
    d_inner = case["expand"] * dm
    h, r = d_inner // p, n // 4
    return dm, n, p, d_inner, h, r, 2 * d_inner + 2 * n + 3 * h + r


def _scan_flops(case, tokens, backward=False):
    """A chunk's causal half of the score products, and the state's update and readout."""
    _, n, p, _, h, _, _ = _shape(case)
    c = case["chunk"]
    one = 2 * (2 * n * p + c * (n + p) / 2)
    if backward:
        one += c * (3 * n + 2 * p) + 8 * n * p
    return tokens * h * one


def work(case):
    dm, n, p, d_inner, h, r, d_in = _shape(case)
    kind, batch = case["kind"], case["batch"]
    size = 2 if case["policy"] == "bf16" else 4
    state = 4 * batch * h * (n * p + n + p + r)
    weights = dm * d_in + d_inner * dm
    vectors = 4 * (h * (2 * n + 2) + 2 * n)
    if kind == "run":
        rows = batch * case["steps"]
        nbytes = (2 * state + size * rows * (2 * n + 3 * h * p) + 4 * rows * (3 * h + r) + vectors)
        return {"bytes": nbytes, "flops": rows * h * 8 * n * p}
    if kind in ("decode", "lm_decode"):
        one_bytes = 2 * state + size * weights + vectors
        one_flops = batch * (2 * weights + h * 8 * n * p)
        if kind == "decode":
            return {"bytes": one_bytes + 2 * size * batch * dm, "flops": one_flops}
        di, layers = case["d_intermediate"], case["n_layers"]
        return {"bytes": layers * (one_bytes + size * 3 * dm * di + 8 * dm)
                + 4 * VOCAB * (dm + batch),
                "flops": layers * (one_flops + 6 * batch * dm * di) + 2 * batch * dm * VOCAB}
    tokens = batch * case["seqlen"]
    if kind in ("forward", "segment"):
        states = state if kind == "forward" else 2 * state
        return {"bytes": 2 * size * tokens * dm + size * weights + vectors + states,
                "flops": 2 * tokens * weights + _scan_flops(case, tokens)}
    if kind == "train":
        # u and dy in, the output and du out; the weights in and their gradients out
        return {"bytes": 4 * size * tokens * dm + 8 * weights + 2 * vectors,
                "flops": 6 * tokens * weights + _scan_flops(case, tokens, backward=True)}
    di, layers = case["d_intermediate"], case["n_layers"]
    params = layers * (weights + 3 * dm * di + vectors // 4 + 2 * dm) + VOCAB * dm
    return {"bytes": 8 * params + 16 * tokens + 4 * tokens * VOCAB,
            "flops": layers * (6 * tokens * (weights + 3 * dm * di)
                               + _scan_flops(case, tokens, backward=True))
            + 6 * tokens * dm * VOCAB}


def tolerance(case):
    # measured: chunks of 64 against chunks of 128 (the sums in another order) differ by 2.3e-3
    # in a layer's bf16 output, 2.9e-3 in its gradients and 2.4e-2 in the gradients of an
    # eight-layer model; one decoded token is 3.9e-3 from float64 through a layer and 2.7e-2
    # through eight, a run's y 1.8e-3, the float32 policy's gradients 7.8e-7. About four times each.
    if case["policy"] == "f32":
        return {"rel": 5e-6}
    return {"rel": {"forward": 1e-2, "segment": 1e-2, "train": 1.2e-2, "decode": 1e-2, "run": 7e-3,
                    "lm_train": 1e-1, "lm_decode": 1e-1}[case["kind"]]}


# ----------------------------------------------------------------------------------------
# the same in float64
# ----------------------------------------------------------------------------------------


def _wrap(phi):
    return phi - 2 * math.pi * torch.floor(phi / (2 * math.pi))


def _rotate(x, phi):
    """Rotate pairs (j, j + N/2) of the last axis by phi_j; pairs beyond phi's are left."""
    half, r = x.shape[-1] // 2, phi.shape[-1]
    lo, hi = x[..., :half], x[..., half:]
    cos, sin = torch.cos(phi), torch.sin(phi)
    a, b = lo[..., :r], hi[..., :r]
    return torch.cat([a * cos - b * sin, lo[..., r:], a * sin + b * cos, hi[..., r:]], dim=-1)


def _decay(a_raw, floor):
    tail = a_raw.clamp(min=0) + 1 / (1 - a_raw.clamp(max=0))
    return (-tail).clamp(max=-floor)


def _rms(x, gain, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * gain


def _split(proj, cfg):
    h, p, n = cfg.nheads, cfg.headdim, cfg.d_state
    z, x, b, c, dt, a, trap, ang = torch.split(
        proj, (cfg.d_inner, cfg.d_inner, n, n, h, h, h, cfg.n_angles), dim=-1)
    heads = lambda t: t.unflatten(-1, (h, p))  # noqa: E731
    return heads(z), heads(x), b, c, dt, a, trap, ang


def _scan(q, k, v, dt, adt, lam, theta, q_bias, k_bias, d_skip, z, carry):
    """q, k (B, L, N); v, z (B, H, L, P); dt, adt, lam (B, H, L); theta (B, L, Nr): the
    trapezoidal recurrence S_t = e^{adt} S + (1 - lam) dt e^{adt} v k'(t-1) + lam dt v k'(t)
    in chunks: a pair (t, s < t) meets with dt_s lam_s plus its successor's share."""
    seqlen = q.shape[1]
    phi = torch.cumsum(theta[:, None] * dt[..., None], dim=2)
    if carry is not None:
        phi = phi + carry[3][:, :, None]
    phi = _wrap(phi)
    u, w = q[:, None] + q_bias[:, None], k[:, None] + k_bias[:, None]
    qr, kr = _rotate(u, phi), _rotate(w, phi)
    own, late = dt * lam, dt * (1 - lam)
    kh = kr * (own + F.pad(late[..., 1:], (0, 1)))[..., None]
    here = own * (u * w).sum(-1) + d_skip[:, None]
    if carry is None:
        ssm = v.new_zeros(*v.shape[:2], v.shape[3], q.shape[-1])
    else:
        ssm = carry[0] + (late[..., :1] * carry[2])[..., None] * carry[1][:, :, None]
    ys = []
    for s in range(0, seqlen, F64_CHUNK):
        e = min(s + F64_CHUNK, seqlen)
        log_a = torch.cumsum(adt[..., s:e], dim=-1)
        gap = log_a[..., :, None] - log_a[..., None, :]
        mask = torch.ones(e - s, e - s, dtype=torch.bool, device=q.device).tril(-1)
        scores = (qr[:, :, s:e] @ kh[:, :, s:e].transpose(-1, -2)) * torch.exp(
            gap.masked_fill(~mask, -math.inf))
        y = scores @ v[:, :, s:e] + here[..., s:e, None] * v[:, :, s:e]
        y = y + (qr[:, :, s:e] @ ssm.transpose(-1, -2)) * torch.exp(log_a)[..., None]
        ys.append(y)
        keep = torch.exp(log_a[..., -1:] - log_a)
        ssm = ssm * torch.exp(log_a[..., -1])[..., None, None] + (
            (v[:, :, s:e] * keep[..., None]).transpose(-1, -2) @ kh[:, :, s:e])
    y = torch.cat(ys, dim=2) * F.silu(z)
    return y, (ssm, kr[:, :, -1], v[:, :, -1], phi[:, :, -1])


def _layer(p, u, cfg, carry=None):
    z, x, b, c, dt_raw, a_raw, trap, ang = _split(u @ p.in_proj, cfg)
    rows = lambda t: t.transpose(1, 2)  # noqa: E731
    dt = rows(F.softplus(dt_raw + p.dt_bias))
    y, carry = _scan(_rms(c, p.c_norm_weight, cfg.norm_eps), _rms(b, p.b_norm_weight, cfg.norm_eps),
                     rows(x), dt, rows(_decay(a_raw, cfg.a_floor)) * dt, rows(torch.sigmoid(trap)),
                     torch.tanh(ang) * math.pi, p.c_bias, p.b_bias, p.d_skip, rows(z), carry)
    return rows(y).flatten(2) @ p.out_proj, carry


def _step(q, k, v, adt, dt, lam, theta, q_bias, k_bias, d_skip, z, carry):
    """One token: q, k (B, N); v, z (B, H, P); adt, dt, lam (B, H); theta (B, Nr)."""
    ssm, k_prev, v_prev, phi = carry
    phi = _wrap(phi + theta[:, None] * dt[..., None])
    qr, kr = _rotate(q[:, None] + q_bias, phi), _rotate(k[:, None] + k_bias, phi)
    alpha = torch.exp(adt)
    ssm = (alpha[..., None, None] * ssm
           + (alpha * dt * (1 - lam))[..., None, None] * v_prev[..., None] * k_prev[:, :, None]
           + (dt * lam)[..., None, None] * v[..., None] * kr[:, :, None])
    y = (ssm @ qr[..., None])[..., 0] + d_skip[:, None] * v
    return y * F.silu(z), (ssm, kr, v, phi)


def _layer_step(p, u, cfg, carry):
    z, x, b, c, dt_raw, a_raw, trap, ang = _split(u @ p.in_proj, cfg)
    dt = F.softplus(dt_raw + p.dt_bias)
    y, carry = _step(_rms(c, p.c_norm_weight, cfg.norm_eps), _rms(b, p.b_norm_weight, cfg.norm_eps),
                     x, _decay(a_raw, cfg.a_floor) * dt, dt, torch.sigmoid(trap),
                     torch.tanh(ang) * math.pi, p.c_bias, p.b_bias, p.d_skip, z, carry)
    return y.flatten(1) @ p.out_proj, carry


def _lm(params, x, cfg, mixer):
    """The residual stack around ``mixer(i, siso params, normalised rows)``."""
    eps = cfg.siso.norm_eps
    for i, b in enumerate(params.blocks):
        x = x + mixer(i, b.siso, _rms(x, b.norm_gain, eps))
        value, gate = (_rms(x, b.mlp_norm_gain, eps) @ b.mlp.fc1).chunk(2, dim=-1)
        x = x + (value * F.silu(gate)) @ b.mlp.fc2
    return _rms(x, params.final_norm, eps) @ params.embed.t()


def _wide(params):
    return type(params)(*(t.detach().double() for t in params))


def _wide_lm(params):
    blocks = [b._replace(norm_gain=b.norm_gain.double(), siso=_wide(b.siso),
                         mlp_norm_gain=b.mlp_norm_gain.double(), mlp=_wide(b.mlp))
              for b in params.blocks]
    return params._replace(embed=params.embed.double(), blocks=blocks,
                           final_norm=params.final_norm.double())


def _lm_leaves(params):
    out = [params.embed]
    for b in params.blocks:
        out += [b.norm_gain, *b.siso, b.mlp_norm_gain, *b.mlp]
    return out + [params.final_norm]


def exact(case, seed):
    inp = _inputs(case, seed)
    kind, cfg = case["kind"], _config(case)
    if kind in ("forward", "segment"):
        p, parts = _wide(inp["params"]), []
        if case["policy"] == "bf16":   # the weights the call is given
            p = p._replace(in_proj=inp["params"].in_proj.bfloat16().double(),
                           out_proj=inp["params"].out_proj.bfloat16().double())
        carry = inp.get("state")
        with torch.no_grad():
            for i in range(case["batch"]):
                c = None if carry is None else tuple(t[i:i + 1].double() for t in carry)
                out, c = _layer(p, inp["u"][i:i + 1].double(), cfg, c)
                parts.append((out, *c))
        return dict(zip(("out", "ssm", "k", "v", "phi"), (torch.cat(t) for t in zip(*parts))))
    if kind == "train":
        p = type(inp["params"])(*(t.requires_grad_(True) for t in _wide(inp["params"])))
        outs, dus, sums = [], [], None
        for i in range(case["batch"]):
            u = inp["u"][i:i + 1].double().requires_grad_(True)
            out, _ = _layer(p, u, cfg)
            g = torch.autograd.grad(out, (u, *p), inp["dy"][i:i + 1].double())
            outs.append(out.detach())
            dus.append(g[0])
            sums = g[1:] if sums is None else [a + b for a, b in zip(sums, g[1:])]
        return dict(out=torch.cat(outs), du=torch.cat(dus),
                    **{"d_" + f: g for f, g in zip(p._fields, sums)})
    if kind == "decode":
        p = _wide(inp["params"])
        if case["policy"] == "bf16":
            p = p._replace(in_proj=inp["params"].in_proj.bfloat16().double(),
                           out_proj=inp["params"].out_proj.bfloat16().double())
        with torch.no_grad():
            out, c = _layer_step(p, inp["u"].double(), cfg, tuple(t.double() for t in inp["state"]))
        return dict(zip(("out", "ssm", "k", "v", "phi"), (out, *c)))
    if kind == "run":
        x = {k: v.double() for k, v in inp.items() if k != "state"}
        carry, ys = tuple(t.double() for t in inp["state"]), []
        for t in range(case["steps"]):
            y, carry = _step(x["q"][:, t], x["k"][:, t], x["v"][:, :, t], x["adt"][:, :, t],
                             x["dt"][:, :, t], x["lam"][:, :, t],
                             torch.tanh(x["angles"][:, t]) * math.pi, x["q_bias"], x["k_bias"],
                             x["d_skip"], x["z"][:, :, t], carry)
            ys.append(y)
        return dict(zip(("y", "ssm", "k", "v", "phi"), (torch.stack(ys, dim=2), *carry)))
    lm, p = _lm_config(case), _wide_lm(inp["params"])
    if kind == "lm_decode":
        states = [None] * case["n_layers"]

        def token_mixer(i, siso, h):
            y, states[i] = _layer_step(siso, h, cfg, tuple(t.double() for t in inp["states"][i]))
            return y

        with torch.no_grad():
            logits = _lm(p, p.embed[inp["token"]], lm, token_mixer)
        return dict(logits=logits, states=states)
    leaves = [t.requires_grad_(True) for t in _lm_leaves(p)]
    logits, loss, sums = [], 0.0, None
    for i in range(case["batch"]):
        out = _lm(p, F.embedding(inp["xs"][i:i + 1], p.embed), lm,
                  lambda _, siso, h: _layer(siso, h, cfg)[0])
        part = F.cross_entropy(out[0], inp["ys"][i]) / case["batch"]
        g = torch.autograd.grad(part, leaves)
        logits.append(out.detach())
        loss = loss + part.detach()
        sums = list(g) if sums is None else [a + b for a, b in zip(sums, g)]
    return dict(logits=torch.cat(logits), loss=loss, grads=sums)
