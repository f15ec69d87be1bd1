"""What is timed when this framework is made faster: the work its users have it do, through its public entry points.

Twelve listed cases cover the sampling step (one sequence to a thousand), configurations per row, speculative verification,
decode loops, the fused head, prompt scoring and the classifiers at the reference's own scale.  `draw` gives more cases of the
same ranges.  Everything lives on the device; host work is what the entry points do themselves.
"""
import math

import torch

from born_amd import backend as BK
from born_amd import linear as L
from born_amd import loss as LS
from born_amd import sampler as S

DEV = "cuda"


def _case(name=None, **kw):
    return {"name": name, **kw} if name else kw


def _sample(name=None, *, batch, vocab, top_k, top_p, rep, temperature, history, shape):
    return _case(name, path="sample", batch=batch, vocab=vocab, top_k=top_k, top_p=top_p, rep=rep, temperature=temperature,
                 history=history, shape=shape)


def listed():
    return [
        # one sequence being decoded: a chat turn on an otherwise idle card, where the launch is what is felt
        _sample("sample_b1", batch=1, vocab=32000, top_k=40, top_p=0.95, rep=1.1, temperature=0.8, history=64, shape="normal"),
        # the headline: a full serving batch at a large vocabulary, the usual chat settings
        _sample("sample_b256", batch=256, vocab=128256, top_k=50, top_p=0.9, rep=1.15, temperature=0.7, history=512, shape="spikes"),
        # offline generation: a very large batch, nucleus sampling alone on flat rows, long histories
        _sample("sample_topp_b1024", batch=1024, vocab=152064, top_k=0, top_p=0.99, rep=1.05, temperature=1.2, history=2048,
                shape="flat"),
        # evaluation of a model's distribution: the greedy token, a draw from the whole distribution, and its log-probabilities
        _case("distribution_b64", path="distribution", batch=64, vocab=32000),
        # continuous batching: every request brings its own settings; an odd vocabulary, so rows start unaligned
        _case("rows_b96", path="rows", batch=96, vocab=100003, history=256),
        # speculative decoding: five draft tokens per sequence verified, with the bonus token
        _case("verify_b64", path="verify", batch=64, gamma=5, vocab=32000),
        # a decode loop for one sequence: embedding, LM head, sampling, history, bound by reading the weights
        _case("decode_b1", path="decode", batch=1, hidden=4096, vocab=32000, steps=16),
        # the same loop for a serving batch
        _case("decode_b64", path="decode", batch=64, hidden=4096, vocab=32000, steps=8),
        # head and sampling step in one call, at the headline's batch and vocabulary
        _case("head_sample_b256", path="head_sample", batch=256, hidden=4096, vocab=128256),
        # scoring a prompt (prefill): logits of every position and the log-probability of the token that follows
        _case("score_b1024", path="score", batch=1024, hidden=3584, vocab=152064),
        # an MNIST classifier's evaluation step: three linear layers, loss and predictions; the smallest products
        _case("mlp_b64", path="mlp", batch=64, n0=784, n1=512, n2=128, n3=10),
        # an MNIST convolutional network's forward pass through the tensor backend
        _case("cnn_b64", path="cnn", batch=64, size=28, c1=32, c2=64, n1=128),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


#: a drawn case's most: elements of logits, multiply-adds of a head
_MOST_LOGITS, _MOST_HEAD = 1024 * 152064, 1024 * 3584 * 152064


def draw(rng):
    path = rng.choice(["sample", "sample", "sample", "distribution", "rows", "verify", "decode", "decode", "head_sample", "score",
                       "mlp", "cnn"])
    while True:
        batch = _log(rng, 1, 1024)
        vocab = _log(rng, 1000, 152064)
        if rng.random() < 0.5:
            vocab -= vocab % 8                                  # half of the vocabularies keep rows aligned, as most models' do
        hidden = 32 * _log(rng, 8, 128)
        if path == "sample":
            c = _sample(batch=batch, vocab=vocab, top_k=rng.choice([0, 1, _log(rng, 2, 128), _log(rng, 2, 128), _log(rng, 128, 512)]),
                        top_p=rng.choice([1.0, 0.9, 0.95, round(rng.uniform(0.7, 0.99), 2)]),
                        rep=rng.choice([1.0, 1.1, round(rng.uniform(1.02, 1.3), 2)]), temperature=round(rng.uniform(0.6, 1.3), 2),
                        history=rng.choice([0, _log(rng, 16, 2048)]), shape=rng.choice(["normal", "spikes", "flat"]))
        elif path == "distribution":
            c = _case(path=path, batch=min(batch, 512), vocab=vocab)
        elif path == "rows":
            c = _case(path=path, batch=min(batch, 512), vocab=vocab, history=_log(rng, 16, 1024))
        elif path == "verify":
            c = _case(path=path, batch=min(batch, 256), gamma=rng.randint(1, 8), vocab=vocab)
        elif path == "decode":
            c = _case(path=path, batch=min(batch, 256), hidden=hidden, vocab=vocab, steps=rng.randint(4, 16))
        elif path == "head_sample":
            c = _case(path=path, batch=min(batch, 512), hidden=hidden, vocab=max(vocab, 4000))
        elif path == "score":
            c = _case(path=path, batch=max(batch, 16), hidden=hidden, vocab=vocab)
        elif path == "mlp":
            c = _case(path=path, batch=_log(rng, 1, 4096), n0=_log(rng, 16, 2048), n1=_log(rng, 16, 1024), n2=_log(rng, 16, 512),
                      n3=_log(rng, 2, 100))
        else:
            c = _case(path=path, batch=_log(rng, 1, 256), size=rng.randint(20, 64), c1=_log(rng, 4, 32), c2=_log(rng, 8, 64),
                      n1=_log(rng, 16, 256))
        logits = c["batch"] * c.get("vocab", 1) * (2 * c.get("gamma", 0) + 1)
        head = c["batch"] * c.get("vocab", 1) * c.get("hidden", 1) * c.get("steps", 1)
        if logits <= _MOST_LOGITS and head <= _MOST_HEAD:
            return c


# ---- inputs ------------------------------------------------------------------------------------


def _rand(g, *shape):
    return torch.rand(*shape, device=DEV, generator=g)


def _randn(g, *shape):
    return torch.randn(*shape, device=DEV, generator=g)


def _ints(g, hi, *shape):
    return torch.randint(0, hi, shape, device=DEV, generator=g, dtype=torch.int32)


def _zipf(g, vocab, *shape):
    """Token ids of running text: a few are frequent, most are rare (an exponent of about one)."""
    return (torch.exp(_rand(g, *shape) * math.log(vocab)) - 1).clamp_(0, vocab - 1).to(torch.int32)


def _logits(g, batch, vocab, shape):
    x = _randn(g, batch, vocab)
    if shape == "normal":
        x *= 2.0
    elif shape == "spikes":                                     # a trained model's rows: a bulk and about twenty likely tokens
        x *= 1.5
        x.scatter_add_(1, torch.randint(0, vocab, (batch, 20), device=DEV, generator=g), 6 + 6 * _rand(g, batch, 20))
    return x


def _uniforms(g, batch):
    return _rand(g, batch).clamp_(max=1 - 2.0 ** -24)


def _head(g, hidden, vocab):
    return L.Linear(hidden, vocab, _randn(g, vocab, hidden) * (2.0 / hidden ** 0.5), 0.1 * _randn(g, vocab))


def _layer(g, n_in, n_out):
    bound = (6.0 / (n_in + n_out)) ** 0.5
    return L.Linear(n_in, n_out, (2 * _rand(g, n_out, n_in) - 1) * bound, 0.1 * _randn(g, n_out))


def _out_size(size, pools=2):
    for _ in range(pools):
        size = (size - 4 - 2) // 2 + 1                          # a 5 x 5 convolution, then a 2 x 2 pool
    return size


def prepare(case, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    p, B = case["path"], case["batch"]
    s = {"case": case}
    i32 = lambda *shape: torch.zeros(*shape, device=DEV, dtype=torch.int32)  # noqa: E731
    f32 = lambda *shape: torch.zeros(*shape, device=DEV)  # noqa: E731
    if p in ("sample", "rows", "distribution"):
        V, H = case["vocab"], case.get("history", 0)
        s["logits"] = _logits(g, B, V, case.get("shape", "normal"))
        s["uniforms"], s["tokens"], s["probs"] = _uniforms(g, B), i32(B), f32(B)
        s["history"] = (_zipf(g, V, B, H) if p == "rows" or case["shape"] == "spikes" else _ints(g, V, B, H)) if H else None
        cfg = S.SamplerConfig()
        if p == "sample":
            cfg = S.SamplerConfig(Temperature=case["temperature"], TopK=case["top_k"], TopP=case["top_p"], RepetitionPenalty=case["rep"])
        elif p == "rows":
            pick = _rand(g, B)
            s["hist_len"] = _ints(g, H + 1, B)
            s["temperatures"] = 0.6 + 0.7 * _rand(g, B)
            # half of the requests bring a small top-k, the rest rely on top-p alone
            s["topKs"] = torch.where(pick < 0.5, 1 + _ints(g, min(100, V - 1), B), i32(B))
            s["topPs"] = torch.where(_rand(g, B) < 0.3, torch.ones(B, device=DEV), 0.8 + 0.19 * _rand(g, B))
            s["penalties"] = torch.where(_rand(g, B) < 0.5, torch.ones(B, device=DEV), 1 + 0.25 * _rand(g, B))
        else:
            s["greedy"], s["logprobs"] = i32(B), f32(B, V)
        s["sampler"] = S.NewSampler(cfg, max_batch=B, max_vocab=V)
    elif p == "verify":
        G, V = case["gamma"], case["vocab"]
        s["target"] = _randn(g, B, G + 1, V)
        s["draft"] = s["target"][:, :G] + 0.5 * _randn(g, B, G, V)
        # drawn from the draft model: the largest of the logits with Gumbel noise
        noise = -torch.log(-torch.log(_rand(g, B, G, V).clamp_(1e-30, 1 - 2.0 ** -24)))
        s["draft_tokens"] = (s["draft"] + noise).argmax(-1).to(torch.int32)
        s["u_accept"], s["u_residual"] = _uniforms(g, B * G).view(B, G), _uniforms(g, B)
        s["n_accepted"], s["next"] = i32(B), i32(B)
        s["sampler"] = S.NewSampler(S.SamplerConfig(), max_batch=B, max_vocab=V)
    elif p in ("decode", "head_sample"):
        K, V = case["hidden"], case["vocab"]
        s["head"] = _head(g, K, V)
        s["sampler"] = S.NewSampler(S.SamplerConfig(Temperature=0.7, TopK=min(50, V), TopP=0.9, RepetitionPenalty=1.15, Seed=seed),
                                    max_batch=B, max_vocab=V)
        s["tokens"], s["probs"] = i32(B), f32(B)
        if p == "decode":
            s["embedding"] = _randn(g, V, K)
            s["prompt_len"] = 16 + _ints(g, 48, B)
            s["len"] = 64 + case["steps"]
            s["history"] = _zipf(g, V, B, s["len"])
            s["prompt_last"] = s["history"].gather(1, (s["prompt_len"] - 1).long().view(B, 1)).view(B).contiguous()
            s["hist_len"], s["hidden"], s["logits"] = i32(B), f32(B, K), f32(B, V)
        else:
            s["x"], s["uniforms"], s["history"] = _randn(g, B, K), _uniforms(g, B), _zipf(g, V, B, 512)
    elif p == "score":
        K, V = case["hidden"], case["vocab"]
        s["head"], s["x"], s["targets"] = _head(g, K, V), _randn(g, B, K), _zipf(g, V, B)
        s["logits"], s["logprobs"] = f32(B, V), f32(B)
        s["sampler"] = S.NewSampler(S.SamplerConfig(), max_batch=B, max_vocab=V)
    elif p == "mlp":
        n = [case["n%d" % i] for i in range(4)]
        s["layers"] = [_layer(g, n[i], n[i + 1]) for i in range(3)]
        s["x"], s["targets"] = _rand(g, B, n[0]), _ints(g, n[3], B)
        s["outs"], s["predictions"] = [f32(B, m) for m in n[1:]], i32(B)
        s["sampler"] = S.NewSampler(S.SamplerConfig(), max_batch=B, max_vocab=n[3])
        s["loss"] = LS.CrossEntropyLoss(B, n[3])
    else:
        dt = lambda t: BK.DeviceTensor.from_numpy(t.cpu().numpy())  # noqa: E731
        c1, c2, n1, flat = case["c1"], case["c2"], case["n1"], case["c2"] * _out_size(case["size"]) ** 2
        s["flat"] = flat
        s["x"] = dt(_rand(g, B, 1, case["size"], case["size"]))
        s["k1"], s["b1"] = dt(0.2 * _randn(g, c1, 1, 5, 5)), dt(0.1 * _randn(g, 1, c1, 1, 1))
        s["k2"], s["b2"] = dt(_randn(g, c2, c1, 5, 5) * (25 * c1) ** -0.5), dt(0.1 * _randn(g, 1, c2, 1, 1))
        s["w3"], s["b3"] = dt(_randn(g, flat, n1) * flat ** -0.5), dt(0.1 * _randn(g, n1))
        s["w4"], s["b4"] = dt(_randn(g, n1, 10) * n1 ** -0.5), dt(0.1 * _randn(g, 10))
        s["backend"] = BK.New()
    return s


# ---- one pass -----------------------------------------------------------------------------------


def run(s):
    c = s["case"]
    p, B, V = c["path"], c["batch"], c.get("vocab")
    if p == "sample":
        s["sampler"].Sample(s["logits"], B, V, s["history"], None, s["uniforms"], s["tokens"], s["probs"], hist_stride=c["history"])
        return s["tokens"], s["probs"]
    if p == "distribution":
        s["sampler"].Argmax(s["logits"], B, V, s["greedy"])
        s["sampler"].Sample(s["logits"], B, V, None, None, s["uniforms"], s["tokens"], s["probs"])
        s["sampler"].Softmax(s["logits"], B, V, s["logprobs"], log=True)
        return s["greedy"], s["tokens"], s["probs"], s["logprobs"]
    if p == "rows":
        s["sampler"].SampleRows(s["logits"], B, V, s["history"], s["hist_len"], s["uniforms"], s["temperatures"], s["topKs"], s["topPs"],
                                s["penalties"], s["tokens"], s["probs"], hist_stride=c["history"])
        return s["tokens"], s["probs"]
    if p == "verify":
        G, t = c["gamma"], s["target"].data_ptr()
        s["sampler"].VerifyBonus(s["target"], (G + 1) * V, s["draft"], G * V, t + 4 * G * V, (G + 1) * V, B, G, V, s["draft_tokens"],
                                 s["u_accept"], s["u_residual"], s["n_accepted"], s["next"])
        return s["n_accepted"], s["next"]
    if p == "decode":
        smp, K = s["sampler"], c["hidden"]
        s["hist_len"].copy_(s["prompt_len"])                    # every pass decodes from the prompts
        s["tokens"].copy_(s["prompt_last"])
        smp.SetStep(0)
        for _ in range(c["steps"]):
            smp.GatherRows(s["embedding"], V, K, s["tokens"], B, s["hidden"])
            s["head"].Forward(s["hidden"], (B, K), s["logits"])
            smp.Sample(s["logits"], B, V, s["history"], s["hist_len"], None, s["tokens"], s["probs"], hist_stride=s["len"])
            smp.HistoryAppend(s["history"], s["hist_len"], s["len"], s["tokens"], B, V)
        return s["history"], s["hist_len"], s["logits"]
    if p == "head_sample":
        L.ForwardSample(s["sampler"], s["head"], s["x"], (B, c["hidden"]), s["history"], None, s["uniforms"], s["tokens"], s["probs"],
                        hist_stride=512)
        return s["tokens"], s["probs"]
    if p == "score":
        s["head"].Forward(s["x"], (B, c["hidden"]), s["logits"])
        s["sampler"].TokenLogprobs(s["logits"], B, V, None, None, s["targets"], s["logprobs"])
        return s["logits"], s["logprobs"]
    if p == "mlp":
        x, n = s["x"], c["n0"]
        for layer, out in zip(s["layers"], s["outs"]):
            layer.Forward(x, (B, n), out)
            x, n = out, layer.OutFeatures()
        s["sampler"].Argmax(x, B, n, s["predictions"])
        return x, s["predictions"], s["loss"].Forward(x, (B, n), s["targets"])
    b = s["backend"]
    y = b.MaxPool2D(b.Add(b.Conv2D(s["x"], s["k1"], 1, 0), s["b1"]), 2, 2)
    y = b.MaxPool2D(b.Add(b.Conv2D(y, s["k2"], 1, 0), s["b2"]), 2, 2)
    y = b.Reshape(y, (B, s["flat"]))
    y = b.Add(b.MatMul(y, s["w3"]), s["b3"])
    y = b.Add(b.MatMul(y, s["w4"]), s["b4"])
    return y.numpy()                                            # the class scores, read by the program


# ---- what a pass cannot do without -----------------------------------------------------------------


def work(case):
    p, B, V, K = case["path"], case["batch"], case.get("vocab", 0), case.get("hidden", 0)
    if p in ("sample", "rows"):                                 # logits and histories once; a maximum, a mass and a sum per logit
        return {"bytes": 4 * B * (V + case["history"] + 3 + (4 if p == "rows" else 0)), "flops": 4 * B * V}
    if p == "distribution":
        return {"bytes": 4 * B * (2 * V + 4), "flops": 6 * B * V}
    if p == "verify":
        G = case["gamma"]
        return {"bytes": 4 * B * ((2 * G + 1) * V + 2 * G + 3), "flops": 4 * B * (2 * G + 1) * V}
    if p == "decode":
        n = case["steps"]
        return {"bytes": n * 4 * (V * K + V + B * (V + K + 64)), "flops": n * (2 * B * V * K + 4 * B * V)}
    if p == "head_sample":
        return {"bytes": 4 * (V * K + V + B * (K + 512 + 3)), "flops": 2 * B * V * K + 4 * B * V}
    if p == "score":
        return {"bytes": 4 * (V * K + V + B * (V + K + 2)), "flops": 2 * B * V * K + 4 * B * V}
    if p == "mlp":
        n = [case["n%d" % i] for i in range(4)]
        w = sum(n[i] * n[i + 1] for i in range(3))
        return {"bytes": 4 * (w + B * (n[0] + n[3] + 2)), "flops": 2 * B * w}
    c1, c2, n1, size = case["c1"], case["c2"], case["n1"], case["size"]
    o1, o2, flat = size - 4, (size - 4) // 2 - 4, c2 * _out_size(size) ** 2
    w = 25 * c1 + 25 * c1 * c2 + flat * n1 + 10 * n1
    return {"bytes": 4 * (B * size * size + w + 10 * B), "flops": 2 * B * (25 * c1 * o1 * o1 + 25 * c1 * c2 * o2 * o2 + flat * n1 + 10 * n1)}


def tolerance(case):
    p = case["path"]
    if p in ("sample", "rows", "verify"):                       # tokens and probabilities are specified to the bit
        return "exact"
    # the rest: about four times what the path differs by from itself in 64 bits
    if p == "distribution":                                     # the tokens are exact; a log-probability is rounded once
        return {"rel": 1e-7, "max": 4e-7}
    if p in ("mlp", "cnn"):                                     # products over at most a few thousand terms
        return {"rel": 2.5e-6, "max": 1e-5, "differ": 0.01}
    if p == "head_sample":                                      # a probability feels its logits' absolute error over the temperature
        return {"rel": 3e-5, "max": 1e-4, "differ": 0.01}
    # a head's 32-bit sums in any order; a draw that lies within their rounding may fall on the other side
    return {"rel": 4e-6, "max": 4e-5, "differ": 0.01}
