"""Performance cases of the MoE expert layer: what a serving or training program calls, over the sizes it calls it at.

A case is one layer (a family below: the shape, the weight format and the activation format of a named configuration) and
one batch: `tokens` rows of bf16 activations.  `mode` is

  "eager"  one `RoutedMoE` / `RoutedAndSharedMoE` call under no_grad, router included: prefill, and decode without a graph;
  "graph"  the same call captured once with `GraphedLayer` and replayed on each step's input: a serving loop's decode step;
  "train"  one call with bf16 weights that require gradients and its backward pass: the gradients of the input, the router
           and the three expert tensors.  `quant` is "none" (bf16 products) or "fp8_full" (e4m3 forward, e5m2 gradients).

Families come from the configurations of `maxtext_amd.synthetic`; tokens run from one decode step of one request to the
prefill batches those configurations are benchmarked with.
"""

import dataclasses
import math

import torch

from maxtext_amd import moe, synthetic
from maxtext_amd.graph import GraphedLayer

#: family -> (configuration, most tokens of one call).  Several formats of one model appear because each is served:
#: int8 x int8 and fp8 x fp8 with row and channel scales, fp8 in 128-wide blocks with a shared expert, int8 weights under
#: bf16 activations with few popular experts, and the two 4-bit weight formats.
SERVE = {
    "mixtral-int8": ("c2", 8192),
    "mixtral-fp8": ("c2f8", 8192),
    "deepseek-fp8": ("c3", 4099),
    "qwen3-int8w": ("c4", 16384),
    "gptoss-int4": ("c5", 4096),
    "gptoss-mxfp4": ("c5mx", 4096),
}
#: training runs the Mixtral shape with bf16 master weights; small batches are a gradient-accumulation microbatch
TRAIN = ("c2", 512, 8192)
#: largest decode batch that a serving loop keeps a captured graph for
MOST_GRAPHED = 256

_WEIGHT_BYTES = {"int8": 1.0, "fp8": 1.0, "fp8c": 1.0, "int4": 0.5, "mxfp4": 0.5}


def _serve(name, family, tokens, mode="eager"):
  return {"name": name, "family": family, "tokens": tokens, "mode": mode, "quant": "stored"}


def _train(name, quant, tokens):
  return {"name": name, "family": "mixtral-train", "tokens": tokens, "mode": "train", "quant": quant}


def listed():
  return [
      # one token of one request: nothing but launches, host work and the four experts it hits
      _serve("gptoss-int4-decode-1", "gptoss-int4", 1),
      # a small serving batch on checkpoint-format weights, replayed as a graph
      _serve("gptoss-mxfp4-graph-32", "gptoss-mxfp4", 32, "graph"),
      # decode of a model with many small experts, weight-only int8, popular experts drawn again and again
      _serve("qwen3-int8w-decode-48", "qwen3-int8w", 48),
      # a small batch on large 8-bit experts: every step streams all of them
      _serve("mixtral-int8-decode-16", "mixtral-int8", 16),
      # the large decode batch of a model with 256 experts and a shared one, block-scaled fp8
      _serve("deepseek-fp8-decode-256", "deepseek-fp8", 256),
      # a short prompt, or decode of several hundred requests: between streaming weights and filling the matrix cores
      _serve("mixtral-fp8-mixed-509", "mixtral-fp8", 509),
      # one prompt of moderate length on 4-bit weights
      _serve("gptoss-int4-prefill-1023", "gptoss-int4", 1023),
      # prefill batches: the benchmark's own sizes, and an odd one
      _serve("mixtral-int8-prefill-8192", "mixtral-int8", 8192),
      _serve("qwen3-int8w-prefill-16384", "qwen3-int8w", 16384),
      _serve("deepseek-fp8-prefill-4099", "deepseek-fp8", 4099),
      # a full training batch in bf16, and a ragged microbatch of the quantised recipe
      _train("train-bf16-8192", "none", 8192),
      _train("train-fp8_full-2999", "fp8_full", 2999),
  ]


def draw(rng):
  """One more case: a family, and tokens spread over the logarithm of its range (odd counts as likely as even ones)."""
  if rng.random() < 0.2:
    lo, hi = TRAIN[1], TRAIN[2]
    return {"family": "mixtral-train", "tokens": _log_uniform(rng, lo, hi), "mode": "train", "quant": rng.choice(["none", "fp8_full"])}
  family = rng.choice(sorted(SERVE))
  tokens = _log_uniform(rng, 1, SERVE[family][1])
  mode = "graph" if tokens <= MOST_GRAPHED and rng.random() < 0.4 else "eager"
  return {"family": family, "tokens": tokens, "mode": mode, "quant": "stored"}


def _log_uniform(rng, lo, hi):
  return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _workload(case):
  name = TRAIN[0] if case["mode"] == "train" else SERVE[case["family"]][0]
  return synthetic.workload(name, case["tokens"])


def _gate_bias(wl, gen, device):
  """Router bias: Zipf popularity where the configuration has it, DeepSeek's small correction bias, otherwise none."""
  e = wl.cfg.num_experts
  if wl.zipf_s > 0:
    return -2.0 * wl.zipf_s * torch.log(torch.arange(1, e + 1, device=device, dtype=torch.float32))
  if wl.cfg.is_deepseek:
    return torch.randn((e,), generator=gen, device=device) * 0.01
  return None


def prepare(case, seed):
  wl = _workload(case)
  gen = torch.Generator(device="cuda").manual_seed(seed)
  t, d, f, e = wl.tokens, wl.cfg.emb_dim, wl.cfg.moe_mlp_dim, wl.cfg.num_experts
  gate = torch.randn((d, e), generator=gen, device="cuda") * 0.02
  bias = _gate_bias(wl, gen, "cuda")
  if case["mode"] == "train":
    cfg = dataclasses.replace(wl.cfg, act_quant=None)
    if case["quant"] == "fp8_full":
      cfg = dataclasses.replace(cfg, quantization="fp8_full", use_qwix_quantization=True)
    weight = lambda n, k: torch.empty((e, n, k), device="cuda", dtype=torch.bfloat16).normal_(0.0, 0.02, generator=gen).requires_grad_()
    x = torch.randn((1, t, d), generator=gen, device="cuda").to(torch.bfloat16).requires_grad_()
    dout = torch.randn((1, t, d), generator=gen, device="cuda").to(torch.bfloat16)
    block = moe.RoutedMoE(cfg, weight(f, d), weight(f, d), weight(d, f), gate.requires_grad_(), bias)
    return {"mode": "train", "block": block, "x": x, "dout": dout}
  layer = synthetic.make_layer(dataclasses.replace(wl, seed=seed), device="cuda")
  kind = moe.RoutedAndSharedMoE if wl.cfg.shared_experts else moe.RoutedMoE
  block = kind(wl.cfg, layer["wi_0"], layer["wi_1"], layer["wo"], gate, bias)
  state = {"mode": case["mode"], "block": block, "x": layer["x"]}
  if case["mode"] == "graph":
    state["graphed"] = GraphedLayer(block, layer["x"])
  return state


def run(state):
  x, block = state["x"], state["block"]
  if state["mode"] == "graph":
    return {"out": state["graphed"](x)}
  if state["mode"] == "eager":
    with torch.no_grad():
      return {"out": block(x)[0]}
  out = block(x)[0]
  leaves = {"x": x, "gate_kernel": block.gate_kernel, "wi_0": block.wi_0, "wi_1": block.wi_1, "wo": block.wo}
  grads = torch.autograd.grad(out, list(leaves.values()), state["dout"])
  return {"out": out.detach(), **dict(zip(leaves, grads))}


def _experts_hit(wl):
  """Experts that a batch of this size selects, from one draw of router logits of the same distribution."""
  cfg = wl.cfg
  gen = torch.Generator().manual_seed(0)
  logits = torch.randn((wl.tokens, cfg.num_experts), generator=gen) * 0.02 * math.sqrt(cfg.emb_dim)
  if wl.zipf_s > 0:
    logits += _gate_bias(wl, gen, "cpu")
  return int(torch.topk(logits, cfg.num_experts_per_tok).indices.unique().numel())


def work(case):
  wl = _workload(case)
  cfg = wl.cfg
  t, d, f, e, shared = wl.tokens, cfg.emb_dim, cfg.moe_mlp_dim, cfg.num_experts, cfg.shared_experts
  products = 6.0 * t * (cfg.num_experts_per_tok + shared) * d * f
  router = 2.0 * t * d * e
  if case["mode"] == "train":
    # x, the output's gradient in; the output and x's gradient out; each weight read and its gradient written
    return {"bytes": 4.0 * t * d * 2 + 2.0 * 3 * e * d * f * 2 + 2.0 * d * e * 4, "flops": 3 * (products + router)}
  experts = _experts_hit(wl) + shared
  values = 3.0 * d * f
  scales = {"int8": (2 * f + d) * 4.0, "fp8c": (2 * f + d) * 4.0, "fp8": values / 128 / 128 * 4, "int4": values / 128 * 2, "mxfp4": values / 32}
  weights = experts * (values * _WEIGHT_BYTES[wl.weight_quant] + scales[wl.weight_quant])
  return {"bytes": 2.0 * t * d * 2 + weights + d * e * 4.0, "flops": products + router}


def tolerance(case):
  # bf16 results of f32 sums; the e5m2 gradients of the quantised recipe keep two bits, and one flipped rounding upstream
  # moves a value by a quarter
  return {"rel": 2e-2} if case["quant"] == "fp8_full" else {"rel": 1e-2}
