"""A layer through one library call (moe_layer) against the same layer through the single calls, bit for bit.

The single calls are what the layer runs when its stages are to be timed (profile_events set).
"""

import dataclasses

import pytest
import torch

from maxtext_amd import moe, synthetic

pytestmark = pytest.mark.gpu


def _block(name, tokens, groups=-1, **cfg):
  wl = synthetic.workload(name, tokens)
  small = dict(emb_dim=512, moe_mlp_dim=768, num_experts=min(wl.cfg.num_experts, 32), **cfg)
  if groups > 0:
    small.update(n_routing_groups=groups, topk_routing_group=2)
  wl = dataclasses.replace(wl, cfg=dataclasses.replace(wl.cfg, **small))
  layer = synthetic.make_layer(wl, device="cuda")
  gen = torch.Generator(device="cuda").manual_seed(tokens)
  gate = torch.randn((512, wl.cfg.num_experts), generator=gen, device="cuda") * 0.05
  bias = torch.randn((wl.cfg.num_experts,), generator=gen, device="cuda") * 0.1
  for key in ("wi_0", "wi_1", "wo"):  # (the generator makes one shared expert: the others are copies)
    missing = wl.cfg.num_experts + wl.cfg.shared_experts - layer[key].qvalue.shape[0]
    if missing:
      more = lambda t: torch.cat([t.view(torch.uint8)] + [t[-1:].view(torch.uint8)] * missing).view(t.dtype)
      layer[key] = dataclasses.replace(layer[key], qvalue=more(layer[key].qvalue), scale=more(layer[key].scale))
  kind = moe.RoutedAndSharedMoE if wl.cfg.shared_experts else moe.RoutedMoE
  return kind(wl.cfg, layer["wi_0"], layer["wi_1"], layer["wo"], gate, bias), layer["x"], gen


def _both(block, *args, **kw):
  routed = getattr(block, "routed", block)
  with torch.no_grad():
    got = block(*args, **kw)
    routed.profile_events = []
    want = block(*args, **kw)
    assert routed.profile_events  # the single calls ran
    routed.profile_events = None
  return got, want


@pytest.mark.parametrize("name", ["c2", "c2f8", "c3", "c4", "c5", "c5mx"])
# (one block routes and sorts up to 4 and up to 16 tokens; 65 rows and more: the sort's larger variants, with tile lists of 16 to 128
# rows; past 4096 rows and on the prefill kernels no tile list is handed on)
@pytest.mark.parametrize("tokens", [1, 4, 5, 16, 17, 60, 130, 300, 700, 2100])
def test_layer_call_equals_the_single_calls(name, tokens):
  block, x, _ = _block(name, tokens)
  got, want = _both(block, x)
  assert torch.equal(got[0], want[0]) and got[1:] == want[1:] == (None, None)


@pytest.mark.parametrize("tokens", [3, 40])
def test_layer_call_with_router_inputs_groups_and_two_shared_experts(tokens):
  block, x, gen = _block("c3", tokens, groups=4, shared_experts=2)
  other = torch.randn(x.shape, generator=gen, device="cuda").to(torch.bfloat16)
  got, want = _both(block, x, gate_inputs=other)
  assert torch.equal(got[0], want[0])
  assert not torch.equal(got[0], _both(block, x)[0][0])


def test_layer_call_leaves_to_the_single_calls_what_it_does_not_know():
  from maxtext_amd import kernels

  block, x, _ = _block("c2", 8)
  calls = []
  real = kernels.layer
  kernels.layer = lambda *a, **k: calls.append(1) or real(*a, **k)
  try:
    with torch.no_grad():
      block(x)
      assert len(calls) == 1
      out, loss, _ = moe.RoutedMoE(dataclasses.replace(block.config, load_balance_loss_weight=0.1), block.wi_0, block.wi_1, block.wo, block.gate_kernel)(x)
      assert loss is not None and torch.isfinite(loss)
      block.per_expert_scale = torch.ones(block.num_experts, device="cuda")
      block(x)
      block.per_expert_scale = None
      wide = torch.cat([block.wi_0.qvalue, block.wi_0.qvalue], 2)
      block.wi_0 = dataclasses.replace(block.wi_0, qvalue=wide[:, :, : x.shape[-1]])  # not contiguous: refused as it was
      with pytest.raises(ValueError):
        block(x)
    assert len(calls) == 1
  finally:
    kernels.layer = real
