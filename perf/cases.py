"""What a program built on this framework asks of it, as cases that can be timed.

Every case goes through the entry points such a program calls: `llm_api.LLM` for the token loop
(prompts, replies, turns of a held conversation, batched and speculative decoding), `sample_api.Sampler`
for drawn tokens and `hip_api.Context` for a single operation.  The model is the synthetic
Qwen3-Next-shape one the benchmark runs (512 experts, top 10, Q4_K); 16 of its 48 layers (four periods of
three DeltaNet layers and one attention layer) keep the preparation of a case under a second, one case
takes all 48.

The vocabulary projection is tied to the embedding table with its rows moved on by a stride: the token
that follows t is t + stride, by a wide margin, as a trained model's next token mostly is.  Over random
weights the two best logits are nearly level, and which of them wins is a matter of rounding.  The routers
are peaked, as trained ones are: over the synthetic ones a token's ten experts weigh about the same, and a
near tie between the tenth and the eleventh, which rounding decides, moves its row by a hundredth.
"""
import ctypes
import importlib
import math

import numpy as np
import torch

pkg = importlib.import_module("strix-halo-vulkan_amd")
hip_api = importlib.import_module(pkg.__name__ + ".hip_api")
llm_api = importlib.import_module(pkg.__name__ + ".llm_api")
sample_api = importlib.import_module(pkg.__name__ + ".sample_api")

LAYERS = 16
VOCAB, EMBD = 151936, 2048
Q6_K, Q6_K_BYTES = 14, 210  # ggml's type number and the bytes of a block of 256
Q8_0, Q8_0_BYTES = 8, 34    # ... of a block of 32


def listed():
    return [
        # the shortest exchange: a command of a few words, an answer of a few tokens
        dict(name="reply_short", kind="reply", layers=LAYERS, prompt=9, tokens=8),
        # a reply of the whole model, one sequence, greedy: the decode loop of the benchmark
        dict(name="reply_full_model", kind="reply", layers=48, prompt=64, tokens=96),
        # the next turn of a conversation: back to its checkpoint, the user's words, a greedy answer
        dict(name="turn_at_3k", kind="turn", layers=LAYERS, context=3000, turn=37, tokens=32),
        # the same behind a long document
        dict(name="turn_at_32k", kind="turn", layers=LAYERS, context=32768, turn=121, tokens=32),
        # tokens drawn by the host's sampler (temperature, top-k, top-p): logits leave the device every step
        dict(name="sampled_turn", kind="sampled", layers=LAYERS, context=700, tokens=24),
        # time to the first token: a paragraph, a few pages, a long document's next full chunk
        dict(name="prompt_150", kind="prompt", layers=LAYERS, context=0, rows=150),
        dict(name="prompt_1531", kind="prompt", layers=LAYERS, context=0, rows=1531),
        dict(name="prompt_4096_at_4096", kind="prompt", layers=LAYERS, context=4096, rows=4096),
        # a server's load: conversations that arrive together and are decoded in shared passes
        dict(name="batch_3", kind="batch", layers=LAYERS, slots=3, prompt=40, tokens=32),
        dict(name="batch_12", kind="batch", layers=LAYERS, slots=12, prompt=40, tokens=32),
        # speculative decoding at depth 2 where about two drafts of three are right
        dict(name="speculate", kind="speculate", layers=LAYERS, prompt=100, rounds=24),
        # the vocabulary projection of a mixed checkpoint, whose converter keeps it wider than the rest
        dict(name="head_q6_k", kind="head", type=Q6_K, rows=1),
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(("reply", "turn", "sampled", "prompt", "prompt", "batch", "speculate", "head"))
    if kind == "reply":
        return dict(kind=kind, layers=LAYERS, prompt=log(2, 400), tokens=log(4, 96))
    if kind == "turn":
        return dict(kind=kind, layers=LAYERS, context=log(100, 32768), turn=log(1, 300), tokens=log(4, 64))
    if kind == "sampled":
        return dict(kind=kind, layers=LAYERS, context=log(40, 4000), tokens=log(4, 32))
    if kind == "prompt":
        return dict(kind=kind, layers=LAYERS, context=rng.choice((0, 0, log(64, 4096))), rows=log(2, 4096))
    if kind == "batch":
        return dict(kind=kind, layers=LAYERS, slots=rng.randint(2, 12), prompt=log(4, 40), tokens=log(8, 32))
    if kind == "speculate":
        return dict(kind=kind, layers=LAYERS, prompt=log(8, 1000), rounds=log(6, 32))
    return dict(kind=kind, type=rng.choice((Q6_K, Q8_0)), rows=rng.randint(1, 14))


class State:
    """What a program keeps between calls; the model's memory goes back when this does."""
    llm = sampler = checkpoint = ctx = None

    def __init__(self, case):
        self.case = case

    def __del__(self):
        if self.llm is not None:
            if self.checkpoint is not None:
                self.llm.checkpoint_free(self.checkpoint)
            self.llm.close()
        if self.sampler is not None:
            self.sampler.close()
        if self.ctx is not None:
            self.ctx.destroy()


def _as_trained(m, seed, stride):
    """output.weight[(t + stride) % vocab] = 0.02 token_embd[t], in their own formats, and routers whose
    tenth choice weighs a few hundredths of the first."""
    t = {x[0]: x for x in m.tensors()}
    n = VOCAB * EMBD
    H, ctx = m.H, m.ctx
    stage = ctypes.c_void_p()
    hip_api.check(H.shv_alloc(ctx, n * 4, ctypes.byref(stage)))
    embd, out = t["token_embd.weight"][1], t["output.weight"][1]
    for dst, std, half in ((embd, 1.0, 1), (stage.value, 0.02, 0)):
        hip_api.check(H.shv_fill_normal(ctx, ctypes.byref(hip_api.FillNormalArgs(dst, n, seed + 1, 0.0, std, half))))
    row = EMBD // hip_api.Q4K_BLOCK * hip_api.Q4K_BYTES
    for src, dst, rows in ((0, stride, VOCAB - stride), (VOCAB - stride, 0, stride)):
        a = hip_api.QuantizeQ4KArgs(stage.value + src * EMBD * 4, out + dst * row, rows, EMBD)
        hip_api.check(H.shv_quantize_q4k(ctx, ctypes.byref(a)))
    hip_api.check(H.shv_free(ctx, stage))
    for i, name in enumerate(sorted(x for x in t if x.endswith("ffn_gate_inp.weight"))):
        a = hip_api.FillNormalArgs(t[name][1], t[name][4] * t[name][5], seed * 1009 + i, 0.0, 0.08, 0)
        hip_api.check(H.shv_fill_normal(ctx, ctypes.byref(a)))


def prepare(case, seed):
    s = State(case)
    rng = np.random.default_rng([seed, 77])
    kind = case["kind"]
    if kind == "head":
        return _prepare_head(s, case, seed)
    cells = {"reply": lambda: case["prompt"] + case["tokens"], "turn": lambda: case["context"] + case["turn"] + case["tokens"],
             "sampled": lambda: case["context"] + case["tokens"], "prompt": lambda: case["context"] + case["rows"],
             "batch": lambda: case["prompt"] + case["tokens"], "speculate": lambda: case["prompt"] + 3 * case["rounds"] + 4}[kind]()
    slots = case.get("slots", 1)
    spec = kind == "speculate"
    cfg = llm_api.Config(n_layer=case["layers"], nkv=max(4096, (cells + 8 + 127) // 128 * 128), max_tokens=4096 if kind == "prompt" else 2048,
                         slots=slots, head_rows=max(slots, 3 if spec else 1), speculative=int(spec), spec_rows=3, nextn=int(spec))
    m = s.llm = llm_api.LLM(cfg)
    m.init_synthetic(seed)
    s.stride = int(rng.integers(1000, 100000)) | 1
    _as_trained(m, seed, s.stride)
    m.stage()
    ids = lambda n: rng.integers(0, VOCAB, size=n).astype(np.int32)
    if case.get("context"):
        m.extend(ids(case["context"]), want_logits=False)
        s.checkpoint = m.checkpoint()
    if kind == "batch":
        s.prompts = [ids(case["prompt"]) for _ in range(slots)]
        s.slots = np.arange(slots, dtype=np.int32)
    else:
        s.prompt = ids({"turn": case.get("turn"), "prompt": case.get("rows"), "sampled": 1}.get(kind, case.get("prompt")))
    if kind == "sampled":
        s.sampler = sample_api.Sampler(0.8, 40, 0.95, seed)
    if spec:
        m.mtp_stage(max_tok=4, vocab_prefix=65536)
        m.spec_open(2)
    return s


def _prepare_head(s, case, seed):
    dev = torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(seed)
    blocks = VOCAB * EMBD // (256 if case["type"] == Q6_K else 32)
    width = Q6_K_BYTES if case["type"] == Q6_K else Q8_0_BYTES
    w = torch.randint(0, 256, (blocks, width), dtype=torch.uint8, device=dev, generator=g)
    # the blocks' float16 scales: of the size that gives weights of about 0.02
    d = (torch.rand(blocks, device=dev, generator=g) * 2e-5 + 1e-5 if case["type"] == Q6_K else
         torch.rand(blocks, device=dev, generator=g) * 2e-4 + 1e-4).half().view(torch.uint8).view(blocks, 2)
    at = width - 2 if case["type"] == Q6_K else 0
    w[:, at:at + 2] = d
    s.w = w
    s.x = torch.randn(case["rows"], EMBD, device=dev, generator=g)
    s.gamma = 1 + 0.1 * torch.randn(EMBD, device=dev, generator=g)
    s.y = torch.empty(case["rows"], VOCAB, device=dev)
    s.ctx = hip_api.Context()
    torch.cuda.synchronize()
    return s


def run(s):
    case, m = s.case, s.llm
    kind = case["kind"]
    if kind == "head":
        s.ctx.gemv(case["type"], s.w.data_ptr(), s.x.data_ptr(), s.y.data_ptr(), VOCAB, EMBD, n_tok=case["rows"],
                   gamma=s.gamma.data_ptr(), eps=1e-6)
        return s.y
    if kind == "batch":
        firsts = []
        for slot, prompt in zip(s.slots, s.prompts):
            m.use_slot(int(slot))
            m.reset()
            m.extend(prompt, want_logits=False)
            firsts.append(m.generate(1)[0][0])
        toks = [np.array(firsts, np.int32)]
        for _ in range(case["tokens"] - 1):
            toks.append(m.decode_rows(s.slots, toks[-1])[0])
        best, logits = m.decode_rows(s.slots, toks[-1], want_logits=True)
        return {"tokens": np.stack(toks + [best]), "logits": logits}
    if kind == "speculate":
        toks = [m.spec_start(s.prompt)]
        for i in range(case["rounds"]):
            # the drafts: the continuation, the second of every other round a miss
            drafts = [(int(toks[-1]) + s.stride) % VOCAB, (int(toks[-1]) + (2 if i % 2 else 3) * s.stride) % VOCAB]
            toks += [int(t) for t in m.spec_round(drafts)]
        logits, hidden = m.extend(toks[-1:], want_hidden=True)
        return {"tokens": np.array(toks, np.int32), "logits": logits, "hidden": hidden}
    if s.checkpoint is not None:
        m.restore(s.checkpoint)
    else:
        m.reset()
    if kind == "sampled":
        toks, logits = [int(s.prompt[0])], None
        for _ in range(case["tokens"]):
            logits, _ = m.extend(toks[-1:])
            toks.append(s.sampler.sample(logits))
        return {"tokens": np.array(toks, np.int32), "logits": logits}
    if kind == "prompt":
        logits, hidden = m.extend(s.prompt, want_hidden=True)
        return {"logits": logits, "hidden": hidden}
    m.extend(s.prompt, want_logits=False)
    toks, _ = m.generate(case["tokens"])
    logits, hidden = m.extend(toks[-1:], want_hidden=True)
    return {"tokens": toks, "logits": logits, "hidden": hidden}


# ---- what a pass cannot do without: each weight, state and cache byte once a pass over the model ----

def _pass(layers, rows, cells, seqs=1, heads=1):
    """(bytes, flops) of one pass of `rows` rows that end at `cells` cells, of `seqs` sequences, `heads` of them
    through the vocabulary projection."""
    E, U, F, HEADS, KV, D = 512, 10, 512, 16, 2, 256
    q4 = lambda n: n * 9 / 16
    dense_dn, dense_at, expert = 12352 * EMBD + EMBD * 4096, 9216 * EMBD + EMBD * 4096, 3 * F * EMBD
    n_at = layers // 4
    n_dn = layers - n_at
    distinct = E * (1 - (1 - U / E) ** rows) + 1
    nbytes = n_dn * (q4(dense_dn) + seqs * 2 * 32 * 128 * 128 * 4) + n_at * (q4(dense_at) + seqs * cells * KV * D * 4)
    nbytes += layers * (E * EMBD * 4 + distinct * q4(expert)) + q4(VOCAB * EMBD) + rows * EMBD * 2 + heads * VOCAB * 4
    per_row = n_dn * (2 * dense_dn + 6 * 32 * 128 * 128) + n_at * 2 * dense_at + layers * 2 * (E * EMBD + (U + 1) * expert)
    seen = max(1.0, cells - (rows / seqs - 1) / 2)  # cells a row attends to, on average
    flops = rows * (per_row + n_at * 4 * HEADS * D * seen) + heads * 2 * VOCAB * EMBD
    return nbytes, flops


def work(case):
    kind = case["kind"]
    if kind == "head":
        width = 256 / Q6_K_BYTES if case["type"] == Q6_K else 32 / Q8_0_BYTES
        n = VOCAB * EMBD
        return {"bytes": n / width + case["rows"] * (EMBD + VOCAB) * 4 + EMBD * 4, "flops": 2 * n * case["rows"]}
    L = case["layers"]
    passes = []
    if kind == "prompt":
        passes.append(_pass(L, case["rows"], case["context"] + case["rows"]))
    elif kind in ("reply", "turn"):
        at, n = case.get("context", 0), case["prompt" if kind == "reply" else "turn"]
        passes.append(_pass(L, n, at + n))
        passes += [_pass(L, 1, at + n + i + 1) for i in range(case["tokens"])]
    elif kind == "sampled":
        passes += [_pass(L, 1, case["context"] + i + 1) for i in range(case["tokens"])]
    elif kind == "batch":
        B, n = case["slots"], case["prompt"]
        passes += [_pass(L, n, n)] * B
        passes += [_pass(L, B, n + i + 1, B, B) for i in range(case["tokens"])]
    else:
        passes.append(_pass(L, case["prompt"], case["prompt"]))
        passes += [_pass(L, 3, case["prompt"] + i * 5 // 2 + 3, 1, 3) for i in range(case["rounds"])]
    return {"bytes": sum(p[0] for p in passes), "flops": sum(p[1] for p in passes)}


def tolerance(case):
    # one float32 operation: sums of 2048 products
    if case["kind"] == "head":
        return {"rel": 1e-5, "max": 1e-4}
    # Float32 activations through 16 (48) layers, keys and values of a quarter of them rounded to binary16: two
    # correct orders of summation part by 2e-5 after them, and by up to 7e-4 where rounding decides between a
    # token's tenth and eleventh expert, or which binary16 a key becomes.  Tokens are decided by wide margins.
    return {"rel": 2e-3, "max": 2e-2, "differ": 0.0}
