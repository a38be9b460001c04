"""The workloads whose time and results this repository holds itself to.

A user of this framework does four things with it: steps lockstep streams of a backbone
through the plugin ABI (host buffers, as the compressor's host does, or device buffers, as a
serving loop does), decodes archives of the CPU path on the reference-order tiers, turns
logits into the coder's CDFs on the device, and compresses and decompresses whole files with
the lockstep driver.  `listed()` holds one or more of each, from one stream to 1,024; `draw()`
gives more of the same kinds over the same ranges.

Weights are seeded random weights of the two architectures the framework ships (Mamba-130M
and RWKV-7 0.1B); token ids are Zipf for the BPE vocabulary and uniform bytes for RWKV-7.
One backend is open at a time, as the ABI has it, and each state owns slots of its pool.
"""
import os
import tempfile

import numpy as np
import torch

from redukt_amd import ffi, lockstep, rbin, rwkv, synth

MAMBA = rbin.MambaDims(vocab=50280, d_model=768, n_layer=24)
RWKV = rwkv.RWKV7_0_1B
F32, Q8_G64, Q8_ROW = ffi.PROFILE_F32, ffi.PROFILE_Q8_G64, ffi.PROFILE_Q8_ROW
Q8_ALL = Q8_ROW | ffi.PROFILE_Q8_SMALL          # x_proj and dt_proj int8 as well
REF_F32 = ffi.PROFILE_EXACT                     # numeric contract 1, F32
REF_G64 = Q8_G64 | ffi.PROFILE_EXACT | ffi.PROFILE_FMA   # numeric contract 2, int8 groups of 64
HISTORY = 3                                     # tokens each stream has seen before the pass
MAX_POOL = 4096                                 # the ABI's cap on streams


def listed():
    def step(name, arch, profile, n, host=False, probs=False):
        return {"name": name, "kind": "step", "arch": arch, "profile": profile, "n": n, "host": host, "probs": probs}

    return [
        # one interactive stream through the reference's host ABI: latency and launches only
        step("mamba_q8_1_host", "mamba", Q8_ALL, 1, host=True),
        # a small lockstep batch through the same ABI, logits into host memory
        step("mamba_q8_32_host", "mamba", Q8_ALL, 32, host=True),
        # the ordinary serving batch, device resident (the benchmark's workload)
        step("mamba_q8_128", "mamba", Q8_ALL, 128),
        # the large batch: every projection a 1,024-column product, 5.8 GB of state traffic
        step("mamba_q8_1024", "mamba", Q8_ALL, 1024),
        # unquantized weights, probabilities handed back instead of logits
        step("mamba_f32_128_probs", "mamba", F32, 128, probs=True),
        # the reference's own quantisation (groups of 64), a ragged batch
        step("mamba_g64_45", "mamba", Q8_G64, 45),
        # decoding archives of the CPU path: logits bit-identical to it (fma contract, int8)
        step("mamba_ref_g64_32", "mamba", REF_G64, 32),
        # the same for F32 archives (contract 1), a ragged larger batch
        step("mamba_ref_f32_100", "mamba", REF_F32, 100),
        # the second backbone, int8, its usual batch
        step("rwkv_q8_64", "rwkv", Q8_ROW, 64),
        # the second backbone decoding archives of the CPU path
        step("rwkv_ref_f32_64", "rwkv", REF_F32, 64),
        # logits a program already holds, turned into the range coder's CDFs
        {"name": "cdf_128", "kind": "cdf", "rows": 128, "vocab": 50280},
        # whole files through the driver, both directions
        {"name": "files_128", "kind": "files", "slots": 128, "files": 128, "tokens": 24},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    kind = rng.choice(["step"] * 8 + ["cdf", "cdf", "files"])
    if kind == "cdf":
        return {"kind": "cdf", "rows": _log_int(rng, 1, 512), "vocab": rng.choice([256, 50280, 65536, _log_int(rng, 300, 65536)])}
    if kind == "files":
        slots = _log_int(rng, 2, 128)
        return {"kind": "files", "slots": slots, "files": slots + rng.randrange(0, 8), "tokens": rng.randrange(8, 24)}
    arch, profile, most = rng.choice([("mamba", Q8_ALL, 1024), ("mamba", Q8_ALL, 1024), ("mamba", F32, 256),
                                      ("mamba", Q8_G64, 256), ("mamba", REF_G64, 144), ("mamba", REF_F32, 144),
                                      ("rwkv", Q8_ROW, 256), ("rwkv", REF_F32, 96)])
    n = _log_int(rng, 1, most)
    host = n <= 64 and rng.random() < 0.3
    return {"kind": "step", "arch": arch, "profile": profile, "n": n, "host": host,
            "probs": profile == F32 and rng.random() < 0.5}


# ---- weights and the open backend ----

_weights = {}     # arch -> {name: array}


def _tensors(arch):
    if arch not in _weights:
        _weights[arch] = dict(synth.mamba_tensors(MAMBA, 0)) if arch == "mamba" else rwkv.synthetic(RWKV, 0)
    return _weights[arch]


def _with_weight_file(arch, use):
    """use(path) with the architecture's weight file, which it has read when it returns."""
    with tempfile.TemporaryDirectory() as d:
        path = os.path.join(d, "model.rbin")
        if arch == "mamba":
            rbin.write_rbin(path, MAMBA, _tensors(arch).items())
        else:
            rwkv.write_rwkv(path, RWKV, _tensors(arch))
        return use(path)


class _Session:
    """The backend (or lockstep driver) that is open, and its free slots."""

    def __init__(self):
        self.key, self.be, self.cap, self.free = None, None, 0, []

    def _switch(self, key, arch, open_):
        if self.key == key:
            return False
        if self.be is not None:
            self.be.close()
        self.key, self.be, self.cap = None, None, 0
        self.be = _with_weight_file(arch, open_)
        self.key = key
        return True

    def backend(self, arch, profile, cap=0):
        self._switch((arch, profile), arch, lambda p: ffi.PluginBackend(p, 0, profile))
        if cap and self.cap != cap:
            self.be.batch_init(cap)
            self.cap, self.free = cap, list(range(cap))
        return self.be

    def driver(self, slots):
        self._switch(("files", slots), "mamba", lambda p: lockstep.Lockstep(p, profile=Q8_ALL, slots=slots))
        return self.be


_session = _Session()


class _Slots:
    """n slots of the open pool, given back when the state that holds them goes."""

    def __init__(self, n):
        self.owner, self.cap = (_session.key, _session.cap), _session.cap
        self.ids = [_session.free.pop(0) for _ in range(n)]

    def __del__(self):
        if (_session.key, _session.cap) == self.owner:
            _session.free.extend(self.ids)


def _tokens(case, seed):
    """[HISTORY + 1, n] token ids of the case's streams."""
    rng = np.random.default_rng([seed, case["n"]])
    shape = (HISTORY + 1, case["n"])
    return synth.zipf_tokens(rng, MAMBA.vocab, shape) if case["arch"] == "mamba" else synth.uniform_tokens(rng, 256, shape)


def _logit_rows(case, seed):
    """Logits as a language model gives them: most of the mass on few symbols in some rows, flat in others."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(case["rows"], case["vocab"], generator=g, device="cuda")
    return x * (1.0 + 3.0 * torch.rand(case["rows"], 1, generator=g, device="cuda"))


def _lengths(case):
    """The files' lengths: ragged, so that streams end and others take their slots."""
    return [case["tokens"] - k % 4 for k in range(case["files"])]


def prepare(case, seed):
    if case["kind"] == "cdf":
        be = _session.backend("mamba", Q8_ALL)
        cdf = torch.zeros(case["rows"], case["vocab"] + 1, dtype=torch.int32, device="cuda")
        state = {"case": case, "be": be, "logits": _logit_rows(case, seed), "cdf": cdf}
        torch.cuda.synchronize()
        return state
    if case["kind"] == "files":
        rng = np.random.default_rng([seed, case["slots"]])
        lens = _lengths(case)
        return {"case": case, "driver": _session.driver(case["slots"]),
                "files": [synth.zipf_tokens(rng, MAMBA.vocab, k) for k in lens], "lens": lens}
    n = case["n"]
    be = _session.backend(case["arch"], case["profile"], min(MAX_POOL, 4 * n))
    slots = _Slots(n)
    toks = _tokens(case, seed)
    out = np.empty((n, be.vocab), np.float32)
    be.batch_reset(slots.ids)
    for t in range(HISTORY):
        be.forward_batch(slots.ids, toks[t], out)
    state = {"case": case, "be": be, "slots": slots}
    if case["host"]:
        return {**state, "tokens": toks[HISTORY].tolist(), "out": out}
    state["d_slots"] = torch.tensor(slots.ids, dtype=torch.int32, device="cuda")
    state["d_tokens"] = torch.from_numpy(toks[HISTORY].astype(np.int32)).cuda()
    state["out"] = torch.zeros(n, be.vocab, device="cuda")
    torch.cuda.synchronize()
    return state


def run(state):
    case = state["case"]
    if case["kind"] == "cdf":
        res = state["be"].cdf_from_logits_device(state["logits"].data_ptr(), case["rows"], case["vocab"],
                                                 state["cdf"].data_ptr())
        if res != ffi.BackendResult.OK:
            raise ffi.BackendError(res, "cdf_from_logits_device")
        return state["cdf"]
    if case["kind"] == "files":
        coded, _ = state["driver"].compress(state["files"])
        back, _ = state["driver"].decompress(coded, state["lens"])
        rows = np.zeros((case["files"], lockstep.stream_bound(case["tokens"])), np.uint8)   # each file's bytes, then zeros
        for row, c in zip(rows, coded):
            row[:len(c)] = np.frombuffer(c, np.uint8)
        return {"coded": rows, "sizes": np.array([len(c) for c in coded]), "tokens": np.concatenate(back).astype(np.int64)}
    be = state["be"]
    if case["host"]:
        be.forward_batch(state["slots"].ids, state["tokens"], state["out"], probs=case["probs"])
    else:
        be.forward_batch_device(case["n"], state["d_slots"].data_ptr(), state["d_tokens"].data_ptr(),
                                state["out"].data_ptr(), probs=case["probs"])
    return state["out"]


# ---- what a pass cannot do without ----

def _matrices(arch):
    """(rows, cols, int8 in the quantized profiles) of every matrix a step multiplies by."""
    if arch == "mamba":
        d, di, dr, xr = MAMBA.d_model, MAMBA.d_inner, MAMBA.dt_rank, MAMBA.xr
        return [(2 * di, d, 1), (xr, di, 0), (di, dr, 0), (d, di, 1)] * MAMBA.n_layer + [(MAMBA.vocab, d, 1)]
    d, f = RWKV.d_model, RWKV.d_ffn
    lora = [m for r in (RWKV.lora_w, RWKV.lora_a, RWKV.lora_v, RWKV.lora_g) for m in ((r, d, 0), (d, r, 0))]
    return ([(d, d, 1)] * 4 + [(f, d, 1), (d, f, 1)] + lora) * RWKV.n_layer + [(RWKV.vocab, d, 1)]


def _step_work(arch, profile, n):
    weights = macs = 0
    for rows, cols, big in _matrices(arch):
        q = profile & 3 and (big or profile & ffi.PROFILE_Q8_SMALL)
        group = cols if profile & 3 == Q8_ROW or cols % 64 else 64
        weights += rows * cols + rows * (cols // group) * 4 if q else rows * cols * 4
        macs += rows * cols
    if arch == "mamba":
        state = 2 * 4 * MAMBA.n_layer * MAMBA.d_inner * (MAMBA.d_conv - 1 + MAMBA.d_state)
        vocab, row = MAMBA.vocab, MAMBA.d_model
    else:
        state = 2 * 4 * RWKV.n_layer * (2 * RWKV.d_model + RWKV.n_head * RWKV.head_size ** 2)
        vocab, row = RWKV.vocab, RWKV.d_model
    return {"bytes": weights + n * (state + 4 * vocab + 4 * row), "flops": 2 * macs * n}


def work(case):
    if case["kind"] == "cdf":      # logits in, cumulative frequencies out
        return {"bytes": case["rows"] * (8 * case["vocab"] + 4), "flops": 0}
    if case["kind"] == "files":
        # In each direction a step for every token but a file's first, as many streams at once
        # as there are slots; logits are written and their CDFs need not leave the device.
        tokens = sum(k - 1 for k in _lengths(case))
        one, two = _step_work("mamba", Q8_ALL, 1), _step_work("mamba", Q8_ALL, 2)
        stream = two["bytes"] - one["bytes"]
        steps = -(-tokens // case["slots"])
        return {"bytes": 2 * (steps * (one["bytes"] - stream) + tokens * stream), "flops": 2 * tokens * one["flops"]}
    return _step_work(case["arch"], case["profile"], case["n"])


def tolerance(case):
    # CDFs and coded bytes are whole numbers, and the reference-order tiers promise every bit.
    if case["kind"] != "step" or case["profile"] & (ffi.PROFILE_EXACT | ffi.PROFILE_FMA):
        return "exact"
    # f32 activations and sums through 24 (12) layers: the steps are 4e-7 to 1.4e-6 from the
    # 64-bit result, the tiers with another order of sums included.
    return {"rel": 4e-6}


# ---- 64-bit results ----

def _quantized(w, group):
    """The int8 recipe's weights: scale = max|w| / 127, its inverse and the scaled weights
    each rounded to f32 (divided in 64 bits first, which rounds as an f32 division does),
    round half away, at most 127."""
    g = torch.from_numpy(np.array(w)).cuda().reshape(w.shape[0], -1, group)
    scale = (g.abs().amax(-1, keepdim=True).double() / 127.0).float()
    scale = torch.where(scale > 0, scale, torch.ones_like(scale))
    r = g * (1.0 / scale.double()).float()
    q = torch.sign(r) * torch.floor(r.abs().double() + 0.5).clamp(max=127.0)
    return (q.double() * scale.double()).reshape(w.shape)


class _Exact64:
    def __init__(self, case):
        self.case = case
        self.t = _tensors(case["arch"])

    def small(self, name):
        return torch.from_numpy(np.array(self.t[name])).cuda().double()

    def mat(self, name, big=True):
        w, p = self.t[name], self.case["profile"]
        if not p & 3 or not (big or p & ffi.PROFILE_Q8_SMALL):
            return self.small(name)
        cols = w.shape[1]
        return _quantized(w, cols if p & 3 == Q8_ROW or cols % 64 else 64)

    def mamba(self, toks):
        d, L = MAMBA, MAMBA.n_layer
        n, di, ds, dr = toks.shape[1], MAMBA.d_inner, MAMBA.d_state, MAMBA.dt_rank
        emb = self.mat("emb")
        xs = emb[torch.from_numpy(toks.astype(np.int64)).cuda()]          # [steps, n, d]: layer by layer over all steps
        rms = lambda x, w: x * torch.rsqrt((x * x).mean(-1, keepdim=True) + 1e-5) * w  # noqa: E731
        for i in range(L):
            p = "layers.%d." % i
            w_in, w_x, w_dt, w_out = self.mat(p + "in_proj"), self.mat(p + "x_proj", False), self.mat(p + "dt_proj_w", False), self.mat(p + "out_proj")
            conv_w, conv_b, dt_b = self.small(p + "conv_w"), self.small(p + "conv_b"), self.small(p + "dt_proj_b")
            a, skip, nw = self.small(p + "A_log").exp(), self.small(p + "D"), self.small(p + "norm_w")
            hist = torch.zeros(n, di, d.d_conv - 1, dtype=torch.float64, device="cuda")
            ssm = torch.zeros(n, di, ds, dtype=torch.float64, device="cuda")
            for s in range(len(xs)):
                xz = rms(xs[s], nw) @ w_in.T
                window = torch.cat([hist, xz[:, :di, None]], -1)
                hist = window[:, :, 1:]
                u = (window * conv_w).sum(-1) + conv_b
                u = u * torch.sigmoid(u)
                z = u @ w_x.T
                dt = torch.nn.functional.softplus(z[:, :dr] @ w_dt.T + dt_b, threshold=20.0)
                b, c = z[:, None, dr:dr + ds], z[:, dr + ds:, None]
                ssm = torch.exp(-dt[:, :, None] * a) * ssm + (dt * u)[:, :, None] * b
                y = (ssm @ c)[:, :, 0] + skip * u
                g = xz[:, di:]
                xs[s] += (y * g * torch.sigmoid(g)) @ w_out.T
        return rms(xs[-1], self.small("norm_f_w")) @ emb.T

    def rwkv(self, toks):
        n, H, N, d = toks.shape[1], RWKV.n_head, RWKV.head_size, RWKV.d_model
        zeros = lambda *s: torch.zeros(*s, dtype=torch.float64, device="cuda")  # noqa: E731
        norm = lambda x, eps: (x - x.mean(-1, keepdim=True)) * torch.rsqrt(x.var(-1, unbiased=False, keepdim=True) + eps)  # noqa: E731
        xs = self.small("emb")[torch.from_numpy(toks.astype(np.int64)).cuda()]
        first = [None] * len(xs)
        for i in range(RWKV.n_layer):
            v = {k[len("blocks.%d." % i):]: k for k in self.t if k.startswith("blocks.%d." % i)}
            quantized = ("receptance", "key", "value", "output", "ffn_key", "ffn_value")
            w = {k: self.mat(f) if k in quantized else self.small(f) for k, f in v.items()}
            pa, pf, S = zeros(n, d), zeros(n, d), zeros(n, H, N, N)
            for s in range(len(xs)):
                x = norm(xs[s], 1e-5) * w["ln1_w"] + w["ln1_b"]
                m = {c: x + (pa - x) * w["x_" + c] for c in "rwkvag"}
                pa = x
                r, k, val = m["r"] @ w["receptance"].T, m["k"] @ w["key"].T, m["v"] @ w["value"].T
                decay = torch.exp(-0.606531 * torch.sigmoid(w["w0"] + torch.tanh(m["w"] @ w["w1"].T) @ w["w2"].T))
                a = torch.sigmoid(w["a0"] + m["a"] @ w["a1"].T @ w["a2"].T)
                gate = torch.sigmoid(m["g"] @ w["g1"].T) @ w["g2"].T
                if i == 0:
                    first[s] = val
                else:
                    val = val + (first[s] - val) * torch.sigmoid(w["v0"] + m["v"] @ w["v1"].T @ w["v2"].T)
                kk = torch.nn.functional.normalize((k * w["k_k"]).view(n, H, N), dim=-1)
                km = (k * (1.0 + (a - 1.0) * w["k_a"])).view(n, H, N)
                r, val = r.view(n, H, N), val.view(n, H, N)
                sa = (S @ -kk[..., None]) @ (kk * a.view(n, H, N))[:, :, None, :]
                S = S * decay.view(n, H, 1, N) + sa + val[..., None] @ km[:, :, None, :]
                o = norm((S @ r[..., None])[..., 0], 64e-5).reshape(n, d) * w["ln_x_w"] + w["ln_x_b"]
                kb = km if RWKV.g1k else k.view(n, H, N)
                o = o + ((r * kb * w["r_k"].view(H, N)).sum(-1, keepdim=True) * val).reshape(n, d)
                x2 = xs[s] + (o * gate) @ w["output"].T
                y = norm(x2, 1e-5) * w["ln2_w"] + w["ln2_b"]
                h = torch.relu((y + (pf - y) * w["ffn_x_k"]) @ w["ffn_key"].T) ** 2
                pf = y
                xs[s] = x2 + h @ w["ffn_value"].T
        return (norm(xs[-1], 1e-5) * self.small("ln_out_w") + self.small("ln_out_b")) @ self.mat("head").T


def exact(case, seed):
    if case["kind"] != "step":
        return None                # whole numbers: compared exactly instead
    e = _Exact64(case)
    logits = getattr(e, case["arch"])(_tokens(case, seed))
    logits = torch.softmax(logits, -1) if case["probs"] else logits
    return logits.cpu().numpy() if case["host"] else logits
