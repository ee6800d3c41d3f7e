"""The work whose time is measured: what a user of this engine has it do, in twelve listed cases and
as many drawn ones as are asked for.

Eleven of the listed cases are generation with the tokens known beforehand (a conversation's turn
replayed): prompts of unlike lengths are fed in portions under a token budget, beside the tokens of
requests that decode already, and every request then brings its tokens one a step until it ends.
That is the schedule of the engine's own step loop, and every step goes through
``ModelRunner.step``, the function that the loop, the trace runner and the replay of traces call.
The tokens are given rather than drawn so that another correct rounding of a logit cannot turn the
rest of the text; the logits of every prompt's end and of every decoded token come back whole.  The
twelfth case is the choice of the next tokens from a step's logits.

Shapes are this repository's presets with fewer layers (the benchmark measures them so), weights are
random with the spreads that the tests use, and ``exact`` computes the same logits from the designs'
equations in 64 bits with plain torch.
"""

from __future__ import annotations

import dataclasses
import math
import random
import zlib

import torch

DEVICE = "cuda:0"
PAGE = 16


# ---------------------------------------------------------------------------------------------
# the cases
def _case(name, model, layers, requests, shortest, longest, new, budget=2048, dtype="bfloat16"):
    return {"name": name, "model": model, "layers": layers, "dtype": dtype, "requests": requests, "shortest": shortest,
            "longest": longest, "new": new, "budget": budget}


def listed():
    return [
        # one user at a small model: a prompt, then an answer token by token (the smallest steps there are)
        _case("one chat", "qwen3-0.6b", 28, 1, 512, 512, 32),
        # a handful of users at a model of ordinary size, prompts of a few hundred tokens
        _case("eight chats", "qwen3-8b", 12, 8, 160, 1500, 32),
        # a server under load: as many requests as a recorded step takes, short prompts, mixed steps while they arrive
        _case("sixty-four requests", "qwen3-4b", 9, 64, 24, 700, 24),
        # a document to be read: one long prompt, cut at the step's budget (the first portion is the
        # benchmark's prompt of 2,048 tokens), and a short answer
        _case("document", "qwen3-8b", 6, 1, 7777, 7777, 4),
        # the true 32-bit path, as used to check a model's numbers
        _case("float32", "qwen3-1.7b", 6, 4, 33, 600, 12, dtype="float32"),
        # each further design at what it is for: recurrent and windowed mixers over longer prompts,
        # latent and differential attention and mixtures of experts at small and middling batches
        _case("rorosun", "rorosun-8b", 4, 3, 300, 3100, 16),
        _case("gubanex", "gubanex-8b", 4, 8, 90, 1800, 16),
        _case("supinex", "supinex-8b", 4, 1, 2500, 2500, 32),
        _case("mepupel", "mepupel-0.6b", 12, 16, 50, 600, 24),
        _case("korazen", "korazen-8b", 4, 5, 200, 2100, 24),
        _case("dopirax", "dopirax-0.6b", 12, 24, 20, 900, 24, budget=1024),
        # the next tokens of a step of forty requests, most of them with the usual thresholds
        {"name": "next tokens", "model": "sampler", "rows": 40, "vocab": 151936},
    ]


_LAYERS = {"qwen3-0.6b": (8, 28), "qwen3-1.7b": (6, 16), "qwen3-4b": (4, 9), "qwen3-8b": (4, 8), "qwen3-14b": (3, 6),
           "rorosun-0.6b": (4, 10), "rorosun-8b": (2, 4), "gubanex-0.6b": (4, 8), "gubanex-8b": (2, 4),
           "supinex-0.6b": (4, 8), "supinex-8b": (2, 4), "mepupel-0.6b": (6, 12), "mepupel-8b": (6, 6),
           "korazen-0.6b": (4, 8), "korazen-8b": (4, 4), "dopirax-0.6b": (4, 12), "dopirax-8b": (3, 4)}


def draw(rng):
    """One more case: half of them the dense design at some width, the others any of the further designs; now and
    then the 32-bit path or the choice of tokens."""
    kind = rng.random()
    if kind < 0.08:
        return {"model": "sampler", "rows": rng.randint(1, 64), "vocab": rng.choice([151936, 151936, 32003, 4096])}
    names = sorted(_LAYERS)
    dense = [n for n in names if n.startswith("qwen3")]
    model = rng.choice(dense) if kind < 0.54 else rng.choice([n for n in names if n not in dense])
    dtype = "float32" if rng.random() < 0.1 and model.endswith(("0.6b", "1.7b")) else "bfloat16"
    while True:
        low, high = _LAYERS[model]
        requests = round(2.0 ** rng.uniform(0.0, 6.0))
        longest = round(2.0 ** rng.uniform(4.0, 12.5 if dtype == "bfloat16" else 10.0))
        shortest = max(1, round(longest * rng.uniform(0.05, 1.0)))
        case = _case(None, model, rng.randint(low, high), requests, shortest, longest, rng.randint(4, 32),
                     rng.choice([512, 1024, 2048, 2048]), dtype)
        del case["name"]
        if sum(_lengths(case)) <= (9000 if dtype == "bfloat16" else 1500):
            need = work(case)
            if need["bytes"] / 6e12 + need["flops"] / 1.2e15 < 0.045:       # (the listed ones reach 0.05)
                return case


def _lengths(case):
    """Prompt lengths from the longest down to the shortest, even in their logarithm, in no order."""
    low, high = case["shortest"], case["longest"]
    return [round(high * (low / high) ** (i * 0.6180339887 % 1.0)) for i in range(case["requests"])]


def _schedule(case):
    """Steps as lists of (request, first position, tokens, whether its last token's logits are wanted): requests that
    decode bring their token, the others portions of their prompts in order of arrival while the budget lasts."""
    lengths, new = _lengths(case), case["new"]
    at = [0] * len(lengths)
    steps = []
    while True:
        step, room = [], case["budget"]
        for r, n in enumerate(lengths):
            if n <= at[r] < n + new:
                step.append((r, at[r], 1, True))
                room -= 1
        for r, n in enumerate(lengths):
            if at[r] < n and room > 0:
                take = min(room, n - at[r])
                step.append((r, at[r], take, at[r] + take == n))
                room -= take
        if not step:
            return steps
        for r, _, count, _ in step:
            at[r] += count
        steps.append(step)


def _tokens(case, seed, vocab):
    """Every request's prompt and answer; token ids uniform, as the benchmark draws them."""
    gen = torch.Generator().manual_seed(seed * 7919 + 17)
    return [torch.randint(0, vocab, (n + case["new"],), generator=gen).tolist() for n in _lengths(case)]


# ---------------------------------------------------------------------------------------------
# weights
def _config(case):
    from tokamak_amd.config import find_preset

    arch, cfg = find_preset(case["model"])
    cfg = arch.shorten(cfg, case["layers"])
    return arch, dataclasses.replace(cfg, max_position_embeddings=40960) if hasattr(cfg, "num_layers") else cfg


_ROUTED = ("gubanex", "supinex", "mepupel", "dopirax")     # designs with mixtures of experts
_TOPICS = 16


class Weights:
    """A checkpoint made from the seed alone, every tensor from a generator of its own: ``names`` and ``fetch`` as
    the engine asks a model folder.  Matrices are wide as their inputs ask (unit rows in, unit rows out, or the
    spread 0.02 of the dense design), gains lie around one, and the mechanisms' own constants where the tests have
    them (decays between about a half and one, biases of a third).  Routers choose as trained ones do, by what a
    token is about (drawn at random alone they would hardly prefer one expert to the next, and rounding would choose)."""

    def __init__(self, case, seed):
        from tokamak_amd.weights.random_init import expected_tensors_of

        arch, cfg = _config(case)
        self.family = case["model"].split("-")[0]
        self.dtype = torch.float32 if case["dtype"] == "float32" else torch.bfloat16
        self.specs = {n: s for n, s in expected_tensors_of(arch.plan(cfg)).items() if not s.ignored}
        self.seed = seed
        self.json = arch.to_json(cfg)

    def names(self):
        return {n: (tuple(s.shape), self._dtype(s)) for n, s in self.specs.items()}

    def _dtype(self, spec):
        return torch.float32 if spec.role == "vector" or spec.held == "float32" else self.dtype

    def fetch(self, name):
        spec = self.specs[name]
        shape, last, family = tuple(spec.shape), name.rsplit(".", 1)[-1], self.family
        gen = torch.Generator(device=DEVICE)
        gen.manual_seed((self.seed * 1000003 + zlib.crc32(name.encode())) % 2**62)
        x = torch.randn(shape, generator=gen, dtype=self._dtype(spec), device=DEVICE)
        if family == "qwen3":
            return x.mul_(0.1).add_(1.0) if spec.role == "vector" else x.mul_(0.02)
        if name == "embed":
            if family in _ROUTED:
                x.view(-1, shape[1]).add_(self.topics(shape[1]).to(x.dtype)[torch.arange(shape[0], device=DEVICE) % _TOPICS], alpha=5.0)
            return x.mul_({"gubanex": shape[1] ** -0.5, "dopirax": 0.125, "korazen": 3.0}.get(family, 1.0))
        if last == "router":
            return self.router(x, gen)
        if last in ("norm1", "norm2", "norm", "out", "ls1", "ls2"):
            around_zero = last != "norm" and family in ("gubanex", "dopirax") or name == "final.norm" and family in ("gubanex", "dopirax")
            return x.mul_(0.2).add_(0.0 if around_zero else 1.0)
        own = {"sink": (1.0, 1.0), "vmix": (0.1, 0.5), "correction": (0.03, 0.0), "b": (0.3, 0.0), "dt_bias": (1.0, -2.0),
               "A_log": (0.5, -0.5), "D": (0.5, 0.5), "conv": (0.5, 0.0), "w0": (0.8, -2.0), "u": (0.5, 0.0)}
        if name.endswith("a2.b"):
            return x.mul_(2.0).add_(2.0)
        if ".mu." in name:
            return x.mul_(0.2).add_(0.5).clamp_(0.0, 1.0)
        if last == "talk":
            return x.mul_(0.1).add_(torch.eye(shape[0], dtype=x.dtype, device=DEVICE))
        if last in ("lq1", "lk1", "lq2", "lk2"):
            return x.mul_(0.4 * shape[0] ** -0.25)
        if last in own and not (last == "b" and len(shape) == 2):
            scale, mean = own[last]
            return x.mul_(scale).add_(mean)
        x.mul_({"gate": 2.0, "up": 2.0, "a2": 2.0}.get(last, 1.0) * shape[1] ** -0.5)
        if family == "gubanex" and last == "q" and name[:-1] + "a1" in self.specs:
            x.add_(self.fetch(name[:-1] + "k"), alpha=2.0)      # queries that find their own keys
        return x

    def topics(self, width):
        """A direction for each of the topics that token ids belong to, as long as a row of unit numbers."""
        gen = torch.Generator(device=DEVICE).manual_seed(self.seed * 613 + 11)
        return torch.randn((_TOPICS, width), generator=gen, device=DEVICE)

    def router(self, noise, gen):
        """Rows of a trained router: a token's topic speaks for one expert, somewhat less for a second, and the rest of
        the stream says little; which experts, each layer has its own mind."""
        experts, width = noise.shape
        first = torch.randperm(_TOPICS, generator=gen, device=DEVICE) % experts
        second = (first + 1 + torch.randint(0, experts - 1, (_TOPICS,), generator=gen, device=DEVICE)) % experts
        votes = torch.zeros((experts, _TOPICS), device=DEVICE)
        at = torch.arange(_TOPICS, device=DEVICE)
        votes[first, at], votes[second, at] = 1.0, 0.8
        return noise.mul_(0.1 * width ** -0.5).add_(votes @ self.topics(width), alpha=8.0 / width)


# ---------------------------------------------------------------------------------------------
# what a program has in hand, and one pass
def prepare(case, seed):
    if case["model"] == "sampler":
        return _prepare_sampler(case, seed)
    from tokamak_amd.engine.runner import ModelRunner

    arch, cfg = _config(case)
    plan = arch.plan(cfg)
    lengths = _lengths(case)
    runner = ModelRunner(plan, Weights(case, seed), dtype=case["dtype"], page_size=PAGE, device=DEVICE,
                         kv_pool_tokens=sum(-(-(n + case["new"]) // PAGE) * PAGE for n in lengths),
                         max_requests=len(lengths), max_step_tokens=case["budget"])
    texts = _tokens(case, seed, plan.vocab_size)
    ends = [n + case["new"] for n in lengths]
    steps = [([(r, texts[r][at:at + n], [n - 1] if want else []) for r, at, n, want in step],
              sum(want for *_, want in step), [r for r, at, n, _ in step if at + n == ends[r]]) for step in _schedule(case)]
    rows = sum(wanted for _, wanted, _ in steps)
    return {"runner": runner, "steps": steps,
            "logits": torch.empty((rows, plan.vocab_size), dtype=torch.float32, device=DEVICE)}


def run(state):
    if "params" in state:
        from tokamak_amd.sampling.sampler import sample_tokens

        return sample_tokens(state["logits"], state["params"], state["seeds"], state["draws"])
    from tokamak_amd.engine.runner import StepEntry

    runner, out, row = state["runner"], state["logits"], 0
    for entries, wanted, ended in state["steps"]:
        logits = runner.step([StepEntry(*entry) for entry in entries])
        if wanted:
            out[row:row + wanted].copy_(logits)     # (a step may write over the logits of the one before)
            row += wanted
        for request in ended:
            runner.end(request)
    return out


def _prepare_sampler(case, seed):
    """Logits as a language model's are spread (a normal body, a short list of likely tokens well above it), and the
    parameters of a mixed lot of requests: greedy, plain temperature, top-k, top-p, both."""
    from tokamak_amd.sampling.params import SamplingParams

    rows, vocab = case["rows"], case["vocab"]
    gen = torch.Generator(device=DEVICE).manual_seed(seed * 31 + 7)
    logits = torch.randn((rows, vocab), generator=gen, device=DEVICE).mul_(2.0)
    likely = torch.randint(0, vocab, (rows, 40), generator=gen, device=DEVICE)
    logits.scatter_add_(1, likely, 6.0 + 2.0 * torch.randn((rows, 40), generator=gen, device=DEVICE))
    kinds = [SamplingParams(temperature=0.6, top_k=20, top_p=0.95), SamplingParams(temperature=0.8, top_p=0.9),
             SamplingParams(temperature=0.0), SamplingParams(temperature=1.0), SamplingParams(temperature=0.7, top_k=50)]
    rng = random.Random(seed)
    return {"logits": logits, "params": [kinds[i % len(kinds)] for i in range(rows)],
            "seeds": [rng.getrandbits(62) for _ in range(rows)], "draws": [rng.randrange(500) for _ in range(rows)]}


# ---------------------------------------------------------------------------------------------
# what a pass cannot do without, and how far two correct passes may lie apart
def work(case):
    """Per step: the matrices its tokens meet (of experts the share that so many tokens choose), the pages its
    tokens look at, the recurrent states in and out, and the wanted logits; the products and the attention's pairs."""
    if case["model"] == "sampler":
        return {"bytes": 4.0 * case["rows"] * case["vocab"], "flops": 2.0 * case["rows"] * case["vocab"]}
    from tokamak_amd.engine.model import LayeredModel

    arch, cfg = _config(case)
    plan = arch.plan(cfg)
    dtype = torch.float32 if case["dtype"] == "float32" else torch.bfloat16
    model = LayeredModel(plan, dtype=dtype, device="meta")
    head = plan.vocab_size * plan.hidden_size
    matrices = []
    for prefix, part in model._named_parts():
        if part is not model.embedding and part is not model.head:
            matrices.append((part, sum(math.prod(s.shape) for s in part.expected_tensors(prefix).values() if len(s.shape) == 2)))
    layouts = model.cache_layout()[1]
    mixers = [(mixer, layouts[slot].request.bytes_per_token(dtype) if slot in layouts else 0, mixer.pair_flops())
              for call in plan.order for mixer, slot in model._mixers_of(call)]
    state = sum(math.prod(a.shape) * a.dtype.itemsize for arrays in model.state_requests().values() for a in arrays.values())
    total_bytes = total_flops = 0.0
    for step in _schedule(case):
        tokens = sum(n for _, _, n, _ in step)
        wanted = sum(want for *_, want in step)
        for part, count in matrices:
            of_token, of_step = part.matrix_share(tokens)
            total_bytes += count * of_step * dtype.itemsize
            total_flops += 2.0 * count * of_token * tokens
        total_bytes += 2.0 * state * len(step) + tokens * plan.hidden_size * dtype.itemsize
        if wanted:
            total_bytes += head * dtype.itemsize + 4.0 * wanted * plan.vocab_size
            total_flops += 2.0 * head * wanted
        for mixer, per_token, pair in mixers:
            for _, at, n, _ in step:
                total_bytes += per_token * (mixer.visible_keys(at + n - 1) + n)
                if pair:
                    total_flops += pair * n * (mixer.visible_keys(at) + mixer.visible_keys(at + n - 1)) / 2
    return {"bytes": total_bytes, "flops": total_flops}


def tolerance(case):
    if case["model"] == "sampler":
        return {"rel": 0.0, "differ": 0.01}     # (a draw that falls on the edge of a token's share of the mass)
    # (measured between prompts cut at 2,048 tokens and at 333, which other kernels run: the dense design 1.6e-2 and
    # single logits 0.13, the others 3e-3 to 9e-3; in float32 1.7e-6 and 1e-5, and 5e-6 from the 64-bit result)
    if case["dtype"] == "float32":
        return {"rel": 2e-5, "max": 4e-4}
    return {"rel": {"supinex": 0.02, "gubanex": 0.025, "korazen": 0.025}.get(case["model"].split("-")[0], 0.03), "max": 0.5}


# ---------------------------------------------------------------------------------------------
# the same logits in 64 bits, from the designs' equations
def exact(case, seed):
    if case["model"] == "sampler":
        return None             # (tokens)
    weights = Weights(case, seed)
    model = _Reference(weights, _tokens(case, seed, weights.json.get("vocab") or weights.json["vocab_size"]))
    starts = [0]
    for text in model.texts:
        starts.append(starts[-1] + len(text))
    rows = [starts[r] + at + n - 1 for step in _schedule(case) for r, at, n, want in step if want]
    with torch.inference_mode():
        return model.logits(torch.tensor(rows, device=DEVICE))


def _rms(x, eps, gain=None):
    y = x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)
    return y if gain is None else y * gain


def _silu(x):
    return x * torch.sigmoid(x)


def _softplus(x):
    return torch.nn.functional.softplus(x, threshold=40.0)


def _angles(rot):
    """(frequencies, amplitude) of a rotation: plain, rescaled by wavelength, or stretched."""
    dims, base = int(rot["dims"]), float(rot["base"])
    f, amplitude, s = [base ** (-2.0 * i / dims) for i in range(dims // 2)], 1.0, rot.get("scaling")
    if s and "low" in s:
        for i, g in enumerate(f):
            wave = 2.0 * math.pi / g
            if wave > s["original"] / s["low"]:
                f[i] = g / s["factor"]
            elif wave >= s["original"] / s["high"]:
                t = (s["original"] / wave - s["low"]) / (s["high"] - s["low"])
                f[i] = (1.0 - t) * g / s["factor"] + t * g
    elif s:
        def turn(n):
            return dims * math.log(s["original"] / (2.0 * math.pi * n)) / (2.0 * math.log(base))

        lo, hi = max(math.floor(turn(s["fast"])), 0), min(math.ceil(turn(s["slow"])), dims - 1)
        for i, g in enumerate(f):
            r = min(max((i - lo) / max(hi - lo, 0.001), 0.0), 1.0)
            f[i] = g / s["factor"] * r + g * (1.0 - r)
        amplitude = 0.1 * math.log(s["factor"]) + 1.0
    return torch.tensor(f, dtype=torch.float64, device=DEVICE), amplitude


def _rotate(x, rot, interleaved=False):
    """x [T, heads, dim] at positions 0 .. T-1, its first ``dims`` dimensions rotated in pairs."""
    if not rot or not rot.get("dims"):
        return x
    f, amplitude = _angles(rot)
    half = f.numel()
    angle = torch.arange(x.shape[0], dtype=torch.float64, device=DEVICE)[:, None] * f
    cos, sin = (angle.cos() * amplitude)[:, None], (angle.sin() * amplitude)[:, None]
    first, second = (slice(0, 2 * half, 2), slice(1, 2 * half, 2)) if interleaved else (slice(0, half), slice(half, 2 * half))
    u, v, out = x[..., first], x[..., second], x.clone()
    out[..., first], out[..., second] = u * cos - v * sin, v * cos + u * sin
    return out


def _attend(q, k, v, scale, visible=None, sink=None, cap=None):
    """q [T, H, d], k [T, G, d], v [T, G, e] -> [T, H, e]: head a reads kv head a // (H / G) under the mask
    ``visible(i, j)`` (besides j <= i), 512 queries at a time."""
    t, heads, kv = q.shape[0], q.shape[1], k.shape[1]
    per, out = heads // kv, q.new_zeros(q.shape[0], heads, v.shape[-1])
    for first in range(0, t, 512):
        i = torch.arange(first, min(t, first + 512), device=DEVICE)[:, None]
        j = torch.arange(int(i[-1]) + 1, device=DEVICE)[None, :]
        mask = j <= i if visible is None else (j <= i) & visible(i, j)
        for g in range(kv):
            s = torch.matmul(q[i[:, 0], g * per:(g + 1) * per].transpose(0, 1).contiguous(), k[:j.numel(), g].T.contiguous()) * scale
            if cap is not None:
                s = cap * torch.tanh(s / cap)
            s = s.masked_fill(~mask, -math.inf)
            if sink is not None:
                s = torch.cat([s, sink[g * per:(g + 1) * per, None, None].expand(per, s.shape[1], 1)], dim=-1)
            p = torch.softmax(s, dim=-1)[..., :j.numel()]
            out[i[:, 0], g * per:(g + 1) * per] = torch.matmul(p, v[:j.numel(), g].contiguous()).transpose(0, 1)
    return out


def _window(mask):
    return None if not mask else lambda i, j: (i - j < int(mask["size"])) | (j < int(mask.get("keep_first", 0)))


def _chunk(mask):
    return None if not mask else lambda i, j: i // int(mask["size"]) == j // int(mask["size"])


class _Reference:
    """One design's whole sequences, layer by layer: products over the tokens of all requests at once, mixers a
    request at a time.  The equations are those of the tests' plain implementations."""

    def __init__(self, weights, texts):
        self.weights, self.cfg, self.texts = weights, weights.json, texts
        self.ids = torch.tensor([t for text in texts for t in text], device=DEVICE)
        self.eps = float(self.cfg["norm"]["eps"]) if "norm" in self.cfg else float(self.cfg["rms_norm_eps"])
        self.kept = {}

    def w(self, name):
        return self.weights.fetch(name).double()

    def mul(self, h, name):
        return h @ self.w(name).T

    def each(self, mixer, *rows):
        """``mixer`` on every request's own rows."""
        out, at = [], 0
        for text in self.texts:
            out.append(mixer(*(x[at:at + len(text)] for x in rows)))
            at += len(text)
        return torch.cat(out)

    def gated(self, h, p, act=_silu):
        return self.mul(act(self.mul(h, p + "gate")) * self.mul(h, p + "up"), p + "down")

    def logits(self, rows):
        family = self.weights.family
        if family == "qwen3":
            return self.qwen3(rows)
        c, x = self.cfg, self.w("embed")[self.ids]
        x = x * float(c.get("embedding", {}).get("scale", 1.0))
        if family == "korazen":
            x = _rms(x, self.eps, self.w("embed.norm"))
        for i, layer in enumerate(c["layers"]):
            x = getattr(self, family)(x, f"l{i}.", layer, i)
        gain, x = self.w("final.norm"), x[rows]
        if family == "supinex":
            h = self.layer_norm(x, gain)
        else:
            h = _rms(x, self.eps, gain + 1.0 if family in ("gubanex", "dopirax") else gain)
        out = self.mul(h, "head") * float(c.get("logit_scale") or 1.0)
        cap = c.get("logit_softcap")
        return out if cap is None else float(cap) * torch.tanh(out / float(cap))

    def layer_norm(self, x, gain):
        d = x - x.mean(-1, keepdim=True)
        return d / torch.sqrt((d * d).mean(-1, keepdim=True) + self.eps) * gain

    # -- the dense design -----------------------------------------------------------------------
    def qwen3(self, rows):
        c, eps = self.cfg, self.eps
        heads, kv, dim = c["num_attention_heads"], c["num_key_value_heads"], c["head_dim"]
        rot = {"base": c["rope_theta"], "dims": dim}
        embed = self.w("model.embed_tokens.weight")
        x = embed[self.ids]
        for i in range(c["num_hidden_layers"]):
            p = f"model.layers.{i}."
            h = _rms(x, eps, self.w(p + "input_layernorm.weight"))
            a = p + "self_attn."
            gq, gk = self.w(a + "q_norm.weight"), self.w(a + "k_norm.weight")
            o = self.each(lambda q, k, v: _attend(_rotate(_rms(q.view(-1, heads, dim), eps, gq), rot),
                                                  _rotate(_rms(k.view(-1, kv, dim), eps, gk), rot),
                                                  v.view(-1, kv, dim), dim ** -0.5).flatten(1),
                          *(self.mul(h, a + n + "_proj.weight") for n in "qkv"))
            x = x + self.mul(o, a + "o_proj.weight")
            h, m = _rms(x, eps, self.w(p + "post_attention_layernorm.weight")), p + "mlp."
            x = x + self.mul(_silu(self.mul(h, m + "gate_proj.weight")) * self.mul(h, m + "up_proj.weight"), m + "down_proj.weight")
        h = _rms(x[rows], eps, self.w("model.norm.weight"))
        return h @ (embed if c["tie_word_embeddings"] else self.w("lm_head.weight")).T

    # -- pooled window attention beside a time mix ----------------------------------------------
    def rorosun(self, x, p, layer, _):
        m = layer["mixer"]
        h = _rms(x, self.eps) * self.w(p + "norm1")
        left, right = self.pooled(h, p + "mix.left.", m["left"]), self.time_mix(h, p + "mix.right.", m["right"])
        x = x + (m["left_scale"] * left + m["right_scale"] * right) * self.w(p + "ls1")
        if layer.get("mlp") is None:
            return x
        return x + self.gated(_rms(x, self.eps) * self.w(p + "norm2"), p + "mlp.") * self.w(p + "ls2")

    def pooled(self, h, p, m):
        heads, kv, dim, vdim = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
        size, pool, scale, per, talk = m["mask"]["size"], m["mask"]["pool"], m["scale"], m["heads"] // m["kv_heads"], self.w(p + "talk")
        q, k, v = (self.mul(h, p + n) + self.w(p + n + ".b") for n in "qkv")
        q, k = _rms(q, self.eps, self.w(p + "q.norm")), _rms(k, self.eps, self.w(p + "k.norm"))

        def one(q, k, v):
            t = q.shape[0]
            q, k, v = q.view(t, heads, dim), k.view(t, kv, dim), v.view(t, kv, vdim)
            blocks = t // pool
            keys = torch.cat([k, k[:blocks * pool].view(blocks, pool, kv, dim).mean(1)])
            values = torch.cat([v, v[:blocks * pool].view(blocks, pool, kv, vdim).mean(1)])
            j, b = torch.arange(t, device=DEVICE)[None], torch.arange(blocks, device=DEVICE)[None]
            out = q.new_zeros(t, heads, vdim)
            for first in range(0, t, 512):
                i = torch.arange(first, min(t, first + 512), device=DEVICE)[:, None]
                seen = torch.cat([(j <= i) & (i - j < size), b * pool + pool - 1 <= i - size], dim=1)
                weights = []
                for a in range(heads):
                    s = (q[i[:, 0], a].contiguous() @ keys[:, a // per].T.contiguous()) * scale
                    weights.append(torch.softmax(s.masked_fill(~seen, -math.inf), dim=-1))
                mixed = (talk @ torch.stack(weights).flatten(1)).view(heads, i.shape[0], -1)
                for a in range(heads):
                    out[i[:, 0], a] = mixed[a] @ values[:, a // per].contiguous()
            return out.flatten(1)

        return self.mul(self.each(one, q, k, v), p + "o")

    def time_mix(self, h, p, m):
        heads, dim = m["heads"], m["dim"]
        prev = self.each(lambda rows: torch.cat([torch.zeros_like(rows[:1]), rows[:-1]]), h)

        def mixed(n):
            return h + (prev - h) * self.w(p + "mu." + n)

        r, k, v, g = (self.mul(mixed(n), p + n) for n in "rkvg")
        low = self.mul(torch.tanh(self.mul(mixed("w"), p + "w1")), p + "w2")
        decay, bonus = torch.exp(-torch.exp(low + self.w(p + "w0"))), self.w(p + "u")[:, :, None]

        def one(r, k, v, decay):
            r, k, v, decay = (a.reshape(-1, heads, dim) for a in (r, k, v, decay))
            state, out = r.new_zeros(heads, dim, dim), torch.empty_like(v)
            for i in range(r.shape[0]):
                kv = k[i, :, :, None] * v[i, :, None, :]
                out[i] = torch.baddbmm(r.new_zeros(1), r[i, :, None, :], state + bonus * kv, beta=0)[:, 0]
                state = decay[i, :, :, None] * state + kv
            return _rms(out, self.eps).flatten(1)

        return self.mul(self.each(one, r, k, v, decay) * self.w(p + "norm") * _silu(g), p + "o")

    # -- gated linear attention, chunked attention, experts weighed at their input ---------------
    def gubanex(self, x, p, layer, _):
        m = layer["mixer"]
        h = _rms(x, self.eps, 1.0 + self.w(p + "norm1"))
        x = x + (self.gated_linear(h, p + "mix.", m) if layer["type"] == "gla" else self.unit_attention(h, p + "mix.", m))
        if layer.get("mlp") is None:
            return x
        h = _rms(x, self.eps, 1.0 + self.w(p + "norm2"))
        return x + self.experts(h, p + "mlp.", layer["mlp"], torch.sigmoid(self.mul(h, p + "mlp.router")), at_input=True)

    def gated_linear(self, h, p, m):
        heads, dim, vdim = m["heads"], m["dim"], m["vdim"]
        q, k, v = (self.mul(h, p + n) for n in "qkv")
        z = self.mul(self.mul(h, p + "a1"), p + "a2") + self.w(p + "a2.b")
        gain = self.w(p + "norm")
        o = self.each(lambda *a: _rms(self.scan(*a, heads, dim, vdim), self.eps, gain).flatten(1),
                      q * dim ** -0.5, k, v, torch.sigmoid(z) ** (1.0 / float(m["tau"])))
        return self.mul(o * _silu(self.mul(h, p + "g")), p + "o")

    def scan(self, q, k, v, decay, heads, dim, vdim):
        """S <- decay S + k v^T, o = S^T q, a token after the other; decays a channel [T, heads dim] or a head [heads]."""
        q, k, v = q.reshape(-1, heads, dim), k.reshape(-1, heads, dim), v.reshape(-1, heads, vdim)
        decay = decay.reshape(-1, heads, dim, 1) if decay.dim() == 2 else decay.reshape(1, heads, 1, 1)
        state, out = q.new_zeros(heads, dim, vdim), torch.empty_like(v)
        for i in range(q.shape[0]):
            state = torch.baddbmm(decay[i if decay.shape[0] > 1 else 0] * state, k[i, :, :, None], v[i, :, None, :])
            out[i] = torch.bmm(q[i, :, None, :], state)[:, 0]
        return out

    def unit_attention(self, h, p, m):
        heads, kv, dim, vdim, rot = m["heads"], m["kv_heads"], m["dim"], m["vdim"], m.get("rot")
        o = self.each(lambda q, k, v: _attend(_rms(_rotate(q.reshape(-1, heads, dim), rot), self.eps), _rms(_rotate(k.reshape(-1, kv, dim), rot), self.eps),
                                              v.reshape(-1, kv, vdim), m["scale"], _chunk(m.get("mask"))).flatten(1),
                      *(self.mul(h, p + n) for n in "qkv"))
        return self.mul(o, p + "o")

    def experts(self, h, p, mlp, scores, chosen=None, weight=None, at_input=False):
        """The ``top`` experts of largest score, weighed by it (or by ``weight``) at their input or output."""
        if chosen is None:
            weight, chosen = scores.topk(mlp["router"]["top"], dim=-1)
        out = torch.zeros_like(h)
        for e in range(mlp["router"]["experts"]):
            token, place = (chosen == e).nonzero(as_tuple=True)
            if token.numel():
                g = weight[token, place][:, None]
                y = self.gated(h[token] * g, f"{p}e{e}.") if at_input else self.gated(h[token], f"{p}e{e}.") * g
                out.index_add_(0, token, y)
        return out

    # -- parallel sub-layers, sinks, latent attention ---------------------------------------------
    def supinex(self, x, p, layer, i):
        h = self.layer_norm(x, self.w(p + "norm1"))
        m, mlp = layer["mixer"], layer.get("mlp")
        mixed = (self.sink_attention if layer["type"] == "attention" else self.rotated_latent)(h, p + "mix.", m, i)
        if mlp is None:
            return x + mixed
        if mlp["kind"] == "dense":
            return x + mixed + self.gated(h, p + "mlp.", lambda z: torch.nn.functional.gelu(z, approximate="tanh"))
        return x + mixed + self.experts(h, p + "mlp.", mlp, torch.softmax(self.mul(h, p + "mlp.router"), dim=-1))

    def sink_attention(self, h, p, m, i):
        heads, kv, dim, vdim, rot, sink = m["heads"], m["kv_heads"], m["dim"], m["vdim"], m.get("rot"), self.w(p + "sink")
        v = self.mul(h, p + "v")
        if m.get("v_mix"):
            if "values" in self.kept:
                share = self.w(p + "vmix")
                v = (1.0 - share) * v + share * self.kept["values"]
            else:
                self.kept["values"] = v
        o = self.each(lambda q, k, v: _attend(_rotate(q.reshape(-1, heads, dim), rot, True), _rotate(k.reshape(-1, kv, dim), rot, True),
                                              v.reshape(-1, kv, vdim), m["scale"], _window(m.get("mask")), sink).flatten(1),
                      self.mul(h, p + "q"), self.mul(h, p + "k"), v)
        return self.mul(o, p + "o")

    def rotated_latent(self, h, p, m, i):
        heads, dim, rdim, vdim, rank = m["heads"], m["dim"], m["rot_dim"], m["vdim"], m["kv_rank"]
        down, sink = self.mul(h, p + "dkv"), self.w(p + "sink")
        c = _rms(down[:, :rank], self.eps, self.w(p + "dkv.norm"))

        def one(q, keys, values, turned):
            q = q.reshape(-1, heads, dim + rdim)
            q = torch.cat([q[..., :dim], _rotate(q[..., dim:], m.get("rot"), True)], dim=-1)
            turned = _rotate(turned[:, None], m.get("rot"), True).expand(-1, heads, -1)
            return _attend(q, torch.cat([keys.reshape(-1, heads, dim), turned], dim=-1), values.reshape(-1, heads, vdim), m["scale"],
                           _window(m.get("mask")), sink).flatten(1)

        return self.mul(self.each(one, self.mul(h, p + "q"), self.mul(c, p + "uk"), self.mul(c, p + "uv"), down[:, rank:]), p + "o")

    # -- state space, window attention with kept first positions, shared latents ------------------
    def mepupel(self, x, p, layer, i):
        m, mlp, h = layer["mixer"], layer.get("mlp"), _rms(x, self.eps, self.w(p + "norm1"))
        if layer["type"] == "mamba2":
            mixed = self.state_space(h, p + "mix.", m)
        elif layer["type"] == "attention":
            heads, kv, dim, vdim, rot = m["heads"], m["kv_heads"], m["dim"], m["vdim"], m.get("rot")
            o = self.each(lambda q, k, v: _attend(_rotate(q.reshape(-1, heads, dim), rot), _rotate(k.reshape(-1, kv, dim), rot),
                                                  v.reshape(-1, kv, vdim), m["scale"], _window(m.get("mask"))).flatten(1),
                          *(self.mul(h, p + "mix." + n) for n in "qkv"))
            mixed = self.mul(o, p + "mix.o")
        else:
            if m.get("kv_from") is None:
                self.kept[i] = _rms(self.mul(h, p + "mix.dkv"), self.eps, self.w(p + "mix.dkv.norm"))
            c = self.kept[i if m.get("kv_from") is None else int(m["kv_from"])]
            heads, dim, vdim = m["heads"], m["dim"], m["vdim"]
            q = self.mul(_rms(self.mul(h, p + "mix.dq"), self.eps, self.w(p + "mix.dq.norm")), p + "mix.uq")
            o = self.each(lambda q, k, v: _attend(q.reshape(-1, heads, dim), k.reshape(-1, heads, dim), v.reshape(-1, heads, vdim), m["scale"]).flatten(1),
                          q, self.mul(c, p + "mix.uk"), self.mul(c, p + "mix.uv"))
            mixed = self.mul(o, p + "mix.o")
        if mlp is not None:
            g = _rms(x, self.eps, self.w(p + "norm2"))
            mixed = mixed + (self.biased(g, p + "mlp.") if mlp["kind"] == "dense" else self.grouped_experts(g, p + "mlp.", mlp))
        return x + float(self.cfg.get("residual_mult", 1.0)) * mixed

    def biased(self, h, p):
        y = _silu(self.mul(h, p + "gate") + self.w(p + "gate.b")) * (self.mul(h, p + "up") + self.w(p + "up.b"))
        return self.mul(y, p + "down") + self.w(p + "down.b")

    def grouped_experts(self, h, p, mlp):
        router = mlp["router"]
        s = torch.sigmoid(self.mul(h, p + "router"))
        choice, groups = s + self.w(p + "correction"), router.get("groups")
        if groups:
            size = router["experts"] // groups["count"]
            score = choice.view(-1, groups["count"], size).topk(min(2, size), dim=-1).values.sum(-1)
            kept = torch.zeros_like(score, dtype=torch.bool).scatter_(1, score.topk(groups["keep"], dim=-1).indices, True)
            choice = choice.masked_fill(~kept[:, :, None].expand(-1, -1, size).reshape(choice.shape), -math.inf)
        chosen = choice.topk(router["top"], dim=-1).indices
        weight = s.gather(1, chosen)
        weight = weight / (weight.sum(-1, keepdim=True) + 1e-20) * float(router.get("scale", 1.0))
        out = self.experts(h, p, mlp, None, chosen, weight)
        return out + self.gated(h, p + "shared.") if mlp.get("shared") else out

    def conv(self, x, weight, bias=None):
        taps, out = weight.shape[1], torch.zeros_like(x)
        padded = torch.cat([x.new_zeros(taps - 1, x.shape[1]), x])
        for j in range(taps):
            out = out + padded[j:j + x.shape[0]] * weight[:, j]
        return out if bias is None else out + bias

    def state_space(self, h, p, m):
        heads, vdim, n, groups, parts = m["heads"], m["vdim"], m["state"], m["groups"], int(m.get("norm_groups", 1))
        inner, per = heads * vdim, heads // groups
        weight, bias, dt_bias, skip = self.w(p + "conv"), self.w(p + "conv.b"), self.w(p + "dt_bias"), self.w(p + "D")
        rate, gain = -torch.exp(self.w(p + "A_log")), self.w(p + "norm")

        def one(proj):
            z, dt = proj[:, :inner], _softplus(proj[:, 2 * inner + 2 * groups * n:] + dt_bias)
            mixed = _silu(self.conv(proj[:, inner:2 * inner + 2 * groups * n], weight, bias))
            x = mixed[:, :inner].reshape(-1, heads, vdim)
            b, c = (a.reshape(-1, groups, n).repeat_interleave(per, dim=1) for a in mixed[:, inner:].split(groups * n, dim=1))
            decay, b = torch.exp(rate * dt)[:, :, None, None], b * dt[:, :, None]
            state, y = x.new_zeros(heads, n, vdim), torch.empty_like(x)
            for i in range(x.shape[0]):
                state = torch.baddbmm(decay[i] * state, b[i, :, :, None], x[i, :, None, :])
                y[i] = torch.bmm(c[i, :, None, :], state)[:, 0]
            y = ((y + skip[:, None] * x).flatten(1) * _silu(z)).reshape(-1, parts, inner // parts)
            return _rms(y, self.eps).flatten(1) * gain

        return self.mul(self.each(one, self.mul(h, p + "in")), p + "o")

    # -- delta rule, chunked attention beside fixed decays, norms behind the sub-layers -----------
    def korazen(self, x, p, layer, _):
        m, q = layer["mixer"], p + "mix."
        mixed = self.delta(x, q, m) if layer["type"] == "channel_delta" else self.both(x, q, m)
        x = x + _rms(mixed, self.eps, self.w(p + "norm1"))
        mlp = layer.get("mlp")
        if mlp is None:
            return x
        limit = float(mlp["limit"])
        g, u = self.mul(x, p + "mlp.gate").clamp(max=limit), self.mul(x, p + "mlp.up").clamp(-limit, limit)
        return x + _rms(self.mul(g * torch.sigmoid(1.702 * g) * (u + 1.0), p + "mlp.down"), self.eps, self.w(p + "norm2"))

    def delta(self, h, p, m):
        heads, kv, dim, vdim = m["heads"], m.get("kv_heads") or m["heads"], m["dim"], m["vdim"]
        taps = {n: self.w(p + n + ".conv") for n in "qkv"}
        step = _softplus(self.mul(self.mul(h, p + "a1"), p + "a2") + self.w(p + "dt_bias")).view(-1, heads, dim)
        decay = torch.exp(-torch.exp(self.w(p + "A_log"))[None, :, None] * step)

        def unit(a):
            a = a.reshape(-1, kv, dim)
            return (a / torch.sqrt((a * a).sum(-1, keepdim=True) + 1e-6)).repeat_interleave(heads // kv, dim=1)

        def one(q, k, v, beta, decay):
            q, k, v = (_silu(self.conv(a, taps[n])) for a, n in ((q, "q"), (k, "k"), (v, "v")))
            q, k, v, decay = unit(q) * dim ** -0.5, unit(k), v.reshape(-1, heads, vdim), decay[..., None]
            state, out = q.new_zeros(heads, dim, vdim), torch.empty_like(v)
            for i in range(q.shape[0]):
                state = decay[i] * state
                u = beta[i, :, None] * (v[i] - torch.bmm(k[i, :, None, :], state)[:, 0])
                state = torch.baddbmm(state, k[i, :, :, None], u[:, None, :])
                out[i] = torch.bmm(q[i, :, None, :], state)[:, 0]
            return out

        o = self.each(one, *(self.mul(h, p + n) for n in "qkv"), torch.sigmoid(self.mul(h, p + "b")), decay)
        gate = torch.sigmoid(self.mul(self.mul(h, p + "g1"), p + "g2"))
        return self.mul(_rms(o, self.eps, self.w(p + "norm")).flatten(1) * gate, p + "o")

    def both(self, h, p, m):
        a, r = m["left"], m["right"]
        heads, kv, dim, vdim, rot = a["heads"], a.get("kv_heads") or a["heads"], a["dim"], a["vdim"], a.get("rot")
        gq, gk = self.w(p + "left.q.norm"), self.w(p + "left.k.norm")
        o = self.each(lambda q, k, v: _attend(_rotate(_rms(q.reshape(-1, heads, dim), self.eps, gq), rot), _rotate(_rms(k.reshape(-1, kv, dim), self.eps, gk), rot),
                                              v.reshape(-1, kv, vdim), a["scale"], _chunk(a.get("mask"))).flatten(1),
                      *(self.mul(h, p + "left." + n) + self.w(p + "left." + n + ".b") for n in "qkv"))
        left = self.mul(o * torch.sigmoid(self.mul(h, p + "left.g")), p + "left.o") + self.w(p + "left.o.b")
        decay = torch.tensor([float(d) for d in r["decay"]], dtype=torch.float64, device=DEVICE)
        q, k, v = (_silu(self.mul(h, p + "right." + n)) for n in "qkv")
        o = self.each(lambda q, k, v: self.scan(q, k, v, decay, r["heads"], r["dim"], r["vdim"]).flatten(1), q, k, v)
        right = self.mul(_rms(o, self.eps, self.w(p + "right.norm")) * torch.sigmoid(self.mul(h, p + "right.g")), p + "right.o")
        return 0.5 * (_rms(left, self.eps, self.w(p + "left.out")) + _rms(right, self.eps, self.w(p + "right.out")))

    # -- differential attention, capped attention over values that are keys -----------------------
    def dopirax(self, x, p, layer, i):
        m, mlp, h = layer["mixer"], layer.get("mlp"), _rms(x, self.eps, 1.0 + self.w(p + "norm1"))
        mixed = self.capped(h, p + "mix.", m) if layer["type"] == "attention" else self.differential(h, p + "mix.", m, i)
        if mlp is None:
            return x + mixed
        if mlp["kind"] == "dense":
            return x + mixed + self.mul(self.mul(h, p + "mlp.up").clamp(min=0.0) ** 2, p + "mlp.down")
        weight, chosen = (self.mul(h, p + "mlp.router") + self.w(p + "mlp.router.b")).topk(mlp["router"]["top"], dim=-1)
        out = self.experts(h, p + "mlp.", mlp, None, chosen, torch.softmax(weight, dim=-1))
        if mlp.get("shared"):
            out = out + torch.sigmoid(self.mul(h, p + "mlp.shared.sg")) * self.gated(h, p + "mlp.shared.")
        return x + mixed + out

    def capped(self, h, p, m):
        heads, kv, dim, rot = m["heads"], m.get("kv_heads") or m["heads"], m["dim"], m.get("rot")
        zero = torch.zeros(heads, dtype=torch.float64, device=DEVICE)
        q, v = self.mul(h, p + "q") + self.w(p + "q.b"), self.mul(h, p + "k") + self.w(p + "k.b")
        o = self.each(lambda q, v: _attend(_rotate(q.reshape(-1, heads, dim), rot), _rotate(v.reshape(-1, kv, dim), rot), v.reshape(-1, kv, dim),
                                           m["scale"], None, zero, m.get("softcap")), q, v)
        return self.mul((o * torch.sigmoid(self.mul(h, p + "g"))[..., None]).flatten(1), p + "o") + self.w(p + "o.b")

    def differential(self, h, p, m, i):
        heads, dim, vdim, rot, eps = m["heads"], m["dim"], m["vdim"], m.get("rot"), self.eps
        kv = m.get("kv_heads") or heads
        if m.get("kv_from") is None:
            gain = self.w(p + "k.norm")
            k = self.each(lambda k: _rotate(_rms(k.reshape(-1, kv * 2, dim), eps, gain), rot, True), self.mul(h, p + "k"))
            self.kept[i] = (k, self.mul(h, p + "v").view(-1, kv, vdim))
        k, v = self.kept[i if m.get("kv_from") is None else int(m["kv_from"])]
        gain = self.w(p + "q.norm")
        lam = torch.exp((self.w(p + "lq1") * self.w(p + "lk1")).sum()) - torch.exp((self.w(p + "lq2") * self.w(p + "lk2")).sum()) + float(m["diff"])

        def one(q, k, v):
            q = _rotate(_rms(q.reshape(-1, heads * 2, dim), eps, gain), rot, True)
            maps = [_attend(q[:, s::2], k[:, s::2], v, m["scale"]) for s in (0, 1)]
            return (_rms(maps[0] - lam * maps[1], eps) * (1.0 - float(m["diff"]))).flatten(1)

        return self.mul(self.each(one, self.mul(h, p + "q"), k, v), p + "o")
