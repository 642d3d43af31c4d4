"""Cases that time the framework's work through its public entry points.

Each case is one call that a structure-prediction program makes again and again: a module
forward of the trunk (triangle attention, triangle multiplication, transitions, single update),
of the diffusion transformer (token attention, transition) or of the atom transformer (windowed
attention), and two chains of them (a pairformer block, a super-block of the diffusion
transformer).  Channel counts, head counts and sample counts are the model's; token and atom
counts run from a peptide to the largest configuration of the benchmark, odd sizes included.

Parameters and inputs come from the seed alone; parameters are bf16-representable, as a bf16
checkpoint's are, and linear weights have variance 1 / fan_in, so that the updates are as large
as the residuals they are added to.
"""
from __future__ import annotations

import math

import torch

from sparsefold_amd import backends
from sparsefold_amd import modules as M
from sparsefold_amd.runtime import config

SAMPLES = 5            # diffusion samples of one prediction
HEADS_TRI, HEADS_SINGLE = 4, 16
C_PAIR, C_TEMPLATE, C_SINGLE, C_TOKEN, C_ATOM = 128, 64, 384, 768, 128
BLOCKS = 4             # attention + transition blocks of one diffusion super-block


# ---------------------------------------------------------------------------------------
# Cases
# ---------------------------------------------------------------------------------------

def listed():
  return [
      # a 20-residue peptide with float32 activations: nothing but launches and host work
      {"name": "triangle_start_20_f32", "op": "triangle", "n": 20, "c": C_PAIR, "end": False, "padded": False, "f32": True},
      # a small protein, its last tokens padding; the ending node walks columns
      {"name": "triangle_end_107_padded", "op": "triangle", "n": 107, "c": C_PAIR, "end": True, "padded": True, "f32": False},
      # the benchmark's headline call
      {"name": "triangle_start_768", "op": "triangle", "n": 768, "c": C_PAIR, "end": False, "padded": False, "f32": False},
      # the template stack's narrower triangle attention
      {"name": "triangle_template_384", "op": "triangle", "n": 384, "c": C_TEMPLATE, "end": False, "padded": True, "f32": False},
      # the triangle multiplicative update of a large complex
      {"name": "trimul_outgoing_768", "op": "trimul", "n": 768, "incoming": False, "padded": False},
      # the trunk's pair transition: one row per pair of tokens
      {"name": "pair_transition_384", "op": "pair_transition", "n": 384},
      # the trunk's single update: pair logits of all pairs, attention with pair bias, transition
      {"name": "single_update_740", "op": "single", "n": 740, "padded": True},
      # token attention and transition of the diffusion transformer, conditioned per call
      {"name": "diffusion_attention_5x1024", "op": "diffusion_attention", "n": 1024, "samples": SAMPLES, "padded": False},
      {"name": "diffusion_transition_5x1024", "op": "diffusion_transition", "n": 1024, "samples": SAMPLES},
      # windowed atom attention, the keys gathered from the queries (per-atom conditioning)
      {"name": "window_5x8192", "op": "window", "windows": 256, "samples": SAMPLES, "indexed": True},
      # whole calls: one pairformer block, and one diffusion super-block conditioned once
      {"name": "pairformer_block_436", "op": "pairformer", "n": 436},
      {"name": "diffusion_superblock_5x740", "op": "superblock", "n": 740, "samples": SAMPLES},
  ]


def _log_int(rng, lo, hi):
  return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
  op = rng.choice(["triangle", "triangle", "triangle", "trimul", "trimul", "pair_transition", "single",
                   "diffusion_attention", "diffusion_transition", "window", "pairformer", "superblock"])
  case = {"op": op}
  if op == "triangle":
    case.update(n=_log_int(rng, 16, 768), c=rng.choice([C_PAIR, C_PAIR, C_PAIR, C_TEMPLATE]), end=rng.random() < 0.5,
                padded=rng.random() < 0.4, f32=rng.random() < 0.25)
  elif op == "trimul":
    case.update(n=_log_int(rng, 16, 768), incoming=rng.random() < 0.5, padded=rng.random() < 0.4)
  elif op == "pair_transition":
    case.update(n=_log_int(rng, 16, 512))
  elif op == "single":
    case.update(n=_log_int(rng, 16, 1024), padded=rng.random() < 0.4)
  elif op == "diffusion_attention":
    case.update(n=_log_int(rng, 16, 1024), samples=rng.choice([1, 3, SAMPLES]), padded=rng.random() < 0.4)
  elif op == "diffusion_transition":
    case.update(n=_log_int(rng, 16, 1024), samples=rng.choice([1, 3, SAMPLES]))
  elif op == "window":
    case.update(windows=_log_int(rng, 4, 256), samples=rng.choice([1, 3, SAMPLES]), indexed=rng.random() < 0.5)
  elif op == "pairformer":
    case.update(n=_log_int(rng, 16, 436))
  else:
    case.update(n=_log_int(rng, 16, 740), samples=rng.choice([1, 3, SAMPLES]))
  return case


# ---------------------------------------------------------------------------------------
# Parameters: (name, shape, fan_in) with fan_in 0 for a norm's weight and -1 for an offset
# ---------------------------------------------------------------------------------------

def _triangle_spec(c):
  h, d = HEADS_TRI, c // HEADS_TRI
  return [("q_projection.weight", (h, d, c), c), ("k_projection.weight", (h, d, c), c),
          ("v_projection.weight", (c, h, d), c), ("gating_query.weight", (c, c), c),
          ("output_projection.weight", (c, c), c), ("act_norm.weight", (c,), 0),
          ("pair_bias_projection.weight", (c, h), c)]


def _trimul_spec(c=C_PAIR):
  return [("left_norm_input.weight", (c,), 0), ("left_norm_input.bias", (c,), -1),
          ("projection.weight", (c, 2 * c), c), ("gate_projection.weight", (c, 2 * c), c),
          ("center_norm.weight", (c,), 0), ("center_norm.bias", (c,), -1),
          ("output_projection.weight", (c, c), c), ("gating_linear.weight", (c, c), c)]


def _transition_spec(c, factor=4):
  i = c * factor
  return [("input_layer_norm.weight", (c,), 0), ("input_layer_norm.bias", (c,), -1),
          ("transition1.weight", (c, 2 * i), c), ("transition2.weight", (i, c), i)]


def _adaln_spec(prefix, c, cs):
  if cs is None:
    return [(prefix + "layer_norm.weight", (c,), 0), (prefix + "layer_norm.bias", (c,), -1)]
  return [(prefix + "single_cond_layer_norm.weight", (cs,), 0), (prefix + "single_cond_scale.weight", (cs, c), cs),
          (prefix + "single_cond_scale.bias", (c,), -1), (prefix + "single_cond_bias.weight", (cs, c), cs)]


def _zero_init_spec(prefix, hidden, c, cs):
  spec = [(prefix + "transition2.weight", (hidden, c), hidden)]
  if cs is not None:
    spec += [(prefix + "adaptive_zero_cond.weight", (cs, c), cs), (prefix + "adaptive_zero_cond.bias", (c,), -1)]
  return spec


def _attention_spec(c, h, cs):
  d = c // h
  return (_adaln_spec("layer_norm.", c, cs)
          + [("q_projection.weight", (c, h, d), c), ("q_projection.bias", (h, d), -1),
             ("k_projection.weight", (c, h, d), c), ("v_projection.weight", (c, h, d), c),
             ("gating_query.weight", (c, c), c)] + _zero_init_spec("zero_init.", c, c, cs))


def _cross_spec(c=C_ATOM, h=HEADS_TRI):
  d = c // h
  return (_adaln_spec("q_layernorm.", c, c) + _adaln_spec("k_layernorm.", c, c)
          + [("q_projection.weight", (c, h, d), c), ("q_projection.bias", (h, d), -1),
             ("k_projection.weight", (c, h, d), c), ("v_projection.weight", (c, h, d), c),
             ("gating_query.weight", (c, c), c)] + _zero_init_spec("zero_init.", c, c, c))


def _diffusion_transition_spec(c=C_TOKEN, cs=C_SINGLE, factor=2):
  i = c * factor
  return (_adaln_spec("layer_norm.", c, cs) + [("transition.weight", (c, 2 * i), c)]
          + _zero_init_spec("zero_init.", i, c, cs))


def _single_spec():
  return ([("single_pair_logits_norm.weight", (C_PAIR,), 0), ("single_pair_logits_norm.bias", (C_PAIR,), -1),
           ("single_pair_logits_projection.weight", (C_PAIR, HEADS_SINGLE), C_PAIR)]
          + _under("single_attention.", _attention_spec(C_SINGLE, HEADS_SINGLE, None))
          + _under("single_transition.", _transition_spec(C_SINGLE)))


def _superblock_spec():
  spec = [("pair_input_layer_norm.weight", (C_PAIR,), 0),
          ("pair_logits_projection.0.weight", (C_PAIR, BLOCKS, HEADS_SINGLE), C_PAIR)]
  for b in range(BLOCKS):
    spec += _under(f"self_attention.0.{b}.", _attention_spec(C_TOKEN, HEADS_SINGLE, C_SINGLE))
    spec += _under(f"transition_block.0.{b}.", _diffusion_transition_spec())
  return spec


def _under(prefix, spec):
  return [(prefix + name, shape, fan) for name, shape, fan in spec]


def _pairformer_specs():
  return {"outgoing": _trimul_spec(), "incoming": _trimul_spec(), "start": _triangle_spec(C_PAIR),
          "end": _triangle_spec(C_PAIR), "pair": _transition_spec(C_PAIR), "single": _single_spec()}


class _Draws:
  """Seeded normal draws on the GPU."""

  def __init__(self, seed):
    self.g = torch.Generator(device="cuda").manual_seed(int(seed))

  def normal(self, *shape):
    return torch.randn(*shape, generator=self.g, device="cuda", dtype=torch.float32)

  def act(self, *shape):
    return self.normal(*shape).to(torch.bfloat16)

  def weights(self, spec):
    out = {}
    for name, shape, fan in spec:
      r = self.normal(*shape)
      r = 1.0 + 0.1 * r if fan == 0 else 0.1 * r if fan < 0 else r / math.sqrt(fan)
      out[name] = r.to(torch.bfloat16).float()
    return out


def _mask(n, padded):
  mask = torch.ones(n, dtype=torch.bool, device="cuda")
  if padded:
    mask[n - max(1, n // 10):] = False
  return mask


def _window_layout(u):
  """32 queries per window, the 128 keys around them; indices off either end are masked."""
  atoms = 32 * u
  idx = torch.arange(u, device="cuda")[:, None] * 32 - 48 + torch.arange(128, device="cuda")[None]
  inside = (idx >= 0) & (idx < atoms)
  present = torch.ones(atoms, dtype=torch.bool, device="cuda")
  present[atoms - 17:] = False                       # the last window is only partly filled
  idx = idx.clamp(0, atoms - 1)
  return idx.to(torch.int32), inside, present.view(u, 32), inside & present[idx]


def _inputs(case, seed):
  """Weights and input tensors of a case, from the seed alone."""
  g = _Draws(seed)
  op = case["op"]
  if op == "window":
    u, s = case["windows"], case["samples"]
    idx, inside, qmask, kmask = _window_layout(u)
    cond = g.act(u, 32, C_ATOM)
    flat = cond.reshape(-1, C_ATOM)[idx.long()]
    return {"w": g.weights(_cross_spec()), "act": g.act(s, u, 32, C_ATOM), "cond": cond, "idx": idx, "inside": inside,
            "qmask": qmask, "kmask": kmask, "kcond": torch.where(inside[..., None], flat, torch.zeros_like(flat)),
            "bias": g.act(u, HEADS_TRI, 32, 128)}
  n = case["n"]
  if op == "triangle":
    z = g.act(n, n, case["c"])
    return {"w": g.weights(_triangle_spec(case["c"])), "z": z.float() if case["f32"] else z, "mask": _mask(n, case["padded"])}
  if op == "trimul":
    return {"w": g.weights(_trimul_spec()), "z": g.act(n, n, C_PAIR), "mask": _mask(n, case["padded"])}
  if op == "pair_transition":
    return {"w": g.weights(_transition_spec(C_PAIR)), "z": g.act(n, n, C_PAIR)}
  if op == "single":
    return {"w": g.weights(_single_spec()), "z": g.act(n, n, C_PAIR), "s": g.act(n, C_SINGLE), "mask": _mask(n, case["padded"])}
  if op == "pairformer":
    return {"w": {k: g.weights(spec) for k, spec in _pairformer_specs().items()}, "z": g.act(n, n, C_PAIR),
            "s": g.act(n, C_SINGLE), "mask": _mask(n, True)}
  s = case["samples"]
  x, cond = g.act(s, n, C_TOKEN), g.act(n, C_SINGLE)
  if op == "diffusion_attention":
    return {"w": g.weights(_attention_spec(C_TOKEN, HEADS_SINGLE, C_SINGLE)), "x": x, "cond": cond,
            "bias": g.act(HEADS_SINGLE, n, n), "mask": _mask(n, case["padded"])}
  if op == "diffusion_transition":
    return {"w": g.weights(_diffusion_transition_spec()), "x": x, "cond": cond}
  return {"w": g.weights(_superblock_spec()), "x": x, "cond": cond, "pair": g.act(n, n, C_PAIR), "mask": _mask(n, True)}


# ---------------------------------------------------------------------------------------
# The calls
# ---------------------------------------------------------------------------------------

def _ready(module, weights):
  module.load_state_dict(weights, strict=True)
  module = module.to("cuda")
  backends.prepare(module)
  return module


def _triangle(c, end):
  return M.GridSelfAttention(M.GridSelfAttention.Config(num_head=HEADS_TRI), M.GlobalConfig(), end, num_channels=c,
                             name="triangle_attention")


def _trimul(incoming):
  eq = M.TriangleMultiplication.EQUATIONS[int(incoming)]
  return M.TriangleMultiplication(M.TriangleMultiplication.Config(equation=eq), M.GlobalConfig(), num_channels=C_PAIR,
                                  name="triangle_multiplication")


def _transition(c):
  return M.TransitionBlock(M.TransitionBlock.Config(), M.GlobalConfig(), num_channels=c, name="transition")


def _single():
  return M.SingleActUpdate(M.GlobalConfig(), C_PAIR, C_SINGLE, M.SelfAttention.Config(num_head=HEADS_SINGLE),
                           M.TransitionBlock.Config())


def _token_attention():
  return M.SelfAttention(M.SelfAttention.Config(num_head=HEADS_SINGLE), M.GlobalConfig(), num_channels=C_TOKEN,
                         single_cond_size=C_SINGLE, name="token_attention")


def _token_transition():
  return M.DiffusionTransitionBlock(M.GlobalConfig(), num_channels=C_TOKEN, num_intermediate_factor=2,
                                    single_cond_size=C_SINGLE, name="token_transition")


class _PackInHand:
  """The Transformer's value cache once the example's pair-logit pack has been made."""

  def __init__(self):
    self.pack = None

  def get(self, *args, name=None, factory=None):
    return self.pack


def _superblock():
  """A Transformer of one super-block on the selected backend's class (its pair-logit half and
  its block loop), with the block stacks an integrating program's own class brings."""
  class Transformer(M.TransformerPairLogits):
    def __init__(self):
      super().__init__(num_blocks=BLOCKS, super_block_size=BLOCKS, num_head=HEADS_SINGLE, pair_cond_size=C_PAIR,
                       dtype=torch.bfloat16)
      stack = lambda make: torch.nn.ModuleList([torch.nn.ModuleList([make() for _ in range(BLOCKS)])])
      self.self_attention, self.transition_block = stack(_token_attention), stack(_token_transition)
      self._cache = _PackInHand()

  return Transformer()


def prepare(case, seed):
  config.configure_runtime(backend="hip", sdpa_implementation="hip", device="cuda")
  backends.init()
  state = _inputs(case, seed)
  state["case"] = case
  op, w = case["op"], state.pop("w")
  if op == "triangle":
    state["module"] = _ready(_triangle(case["c"], case["end"]), w)
  elif op == "trimul":
    state["module"] = _ready(_trimul(case["incoming"]), w)
  elif op == "pair_transition":
    state["module"] = _ready(_transition(C_PAIR), w)
  elif op == "single":
    state["module"] = _ready(_single(), w)
  elif op == "diffusion_attention":
    state["module"] = _ready(_token_attention(), w)
  elif op == "diffusion_transition":
    state["module"] = _ready(_token_transition(), w)
  elif op == "window":
    state["module"] = _ready(M.CrossAttention(M.CrossAttention.Config(num_head=HEADS_TRI, key_dim=C_ATOM, value_dim=C_ATOM),
                                              M.GlobalConfig(), num_channels=C_ATOM, name="atom_attention"), w)
    if not case["indexed"]:                            # the program gathers the keys itself
      flat = state["act"].reshape(case["samples"], -1, C_ATOM)[:, state["idx"].long()]
      state["keys"] = torch.where(state["inside"][..., None], flat, torch.zeros_like(flat))
  elif op == "pairformer":
    make = {"outgoing": _trimul(False), "incoming": _trimul(True), "start": _triangle(C_PAIR, False),
            "end": _triangle(C_PAIR, True), "pair": _transition(C_PAIR), "single": _single()}
    state["module"] = {k: _ready(m, w[k]) for k, m in make.items()}
  else:
    module = _ready(_superblock(), w)
    module._cache.pack = module.pair_logits_pack(state["pair"])       # made once per example
    state["module"] = module
  return state


def run(state):
  case, m = state["case"], state["module"]
  op = case["op"]
  if op in ("triangle", "trimul"):
    return m(state["z"], state["mask"])
  if op == "pair_transition":
    return m(state["z"])
  if op == "single":
    return m(state["z"], state["s"], state["mask"])
  if op == "diffusion_attention":
    return m(state["x"], state["mask"], pair_logits=state["bias"], single_cond=state["cond"])
  if op == "diffusion_transition":
    return m(state["x"], single_cond=state["cond"])
  if op == "window":
    if case["indexed"]:
      return m.forward_indexed(state["act"], state["qmask"], state["idx"], state["inside"], state["kmask"], state["cond"],
                               None, state["bias"])
    return m(state["act"], state["keys"], state["qmask"], state["kmask"], state["bias"], state["cond"], state["kcond"])
  if op == "pairformer":
    z, mask = state["z"], state["mask"]
    z = m["outgoing"](z, mask)
    z = m["incoming"](z, mask)
    z = m["start"](z, mask)
    z = m["end"](z, mask)
    z = m["pair"](z)
    return {"pair": z, "single": m["single"](z, state["s"], mask)}
  return m(state["x"], state["mask"], state["cond"], state["pair"])


# ---------------------------------------------------------------------------------------
# Work and tolerance
# ---------------------------------------------------------------------------------------

def _elements(spec):
  return sum(math.prod(shape) for _, shape, _ in spec)


def _triangle_flops(n, c):
  return 2 * n * n * c * (4 * c + HEADS_TRI) + 4 * c * n ** 3 + 2 * n * n * c * c


def _trimul_flops(n, c=C_PAIR):
  return 2 * n * n * c * 4 * c + 2 * c * n ** 3 + 2 * n * n * c * 2 * c


def _single_flops(n):
  c = C_SINGLE
  return 2 * n * n * C_PAIR * HEADS_SINGLE + 2 * n * c * 4 * c + 4 * c * n * n + 2 * n * c * c + 2 * n * c * 12 * c


def work(case):
  op = case["op"]
  if op == "window":
    u, s, c = case["windows"], case["samples"], C_ATOM
    atoms = 32 * u
    flops = 2 * s * atoms * c * 5 * c + 4 * s * u * 32 * 128 * c
    moved = 2 * (2 * s * atoms * c + u * HEADS_TRI * 32 * 128) + 5 * u * 160
    if case["indexed"]:
      moved += 2 * atoms * c * 5                       # the atoms' conditioning terms
    else:
      flops += 2 * s * u * 128 * c * 2 * c - 2 * s * atoms * c * 2 * c + 2 * u * c * c * (32 * 3 + 128 * 2)
      moved += 2 * (s * u * 128 * c + u * 160 * c)
    return {"bytes": moved + 2 * _elements(_cross_spec()), "flops": flops}
  n = case["n"]
  if op == "triangle":
    c = case["c"]
    return {"bytes": 2 * n * n * c * (4 if case["f32"] else 2) + 2 * _elements(_triangle_spec(c)), "flops": _triangle_flops(n, c)}
  if op == "trimul":
    return {"bytes": 4 * n * n * C_PAIR + 2 * _elements(_trimul_spec()), "flops": _trimul_flops(n)}
  if op == "pair_transition":
    return {"bytes": 4 * n * n * C_PAIR + 2 * _elements(_transition_spec(C_PAIR)), "flops": 2 * n * n * 12 * C_PAIR * C_PAIR}
  if op == "single":
    return {"bytes": 2 * n * n * C_PAIR + 4 * n * C_SINGLE + 2 * _elements(_single_spec()), "flops": _single_flops(n)}
  if op == "pairformer":
    # the pair activations are read and written once per module of the chain
    specs = _pairformer_specs()
    flops = 2 * _trimul_flops(n) + 2 * _triangle_flops(n, C_PAIR) + 24 * n * n * C_PAIR * C_PAIR + _single_flops(n)
    return {"bytes": 5 * 4 * n * n * C_PAIR + 2 * n * n * C_PAIR + 2 * sum(_elements(s) for s in specs.values()), "flops": flops}
  s, c, cs = case["samples"], C_TOKEN, C_SINGLE
  act = 4 * s * n * c
  att = 2 * s * n * c * 5 * c + 4 * c * n * n * s
  cond = 2 * n * cs * 3 * c
  if op == "diffusion_attention":
    return {"bytes": act + 2 * n * cs + 2 * HEADS_SINGLE * n * n + 2 * _elements(_attention_spec(c, HEADS_SINGLE, cs)),
            "flops": att + cond}
  if op == "diffusion_transition":
    return {"bytes": act + 2 * n * cs + 2 * _elements(_diffusion_transition_spec()), "flops": 12 * s * n * c * c + cond}
  # the activations are read and written once per module of the super-block
  return {"bytes": 2 * BLOCKS * act + 2 * n * cs + 2 * BLOCKS * HEADS_SINGLE * n * n + 2 * _elements(_superblock_spec()),
          "flops": BLOCKS * (att + 12 * s * n * c * c + 2 * cond)}


def tolerance(case):
  """bf16 operands with fp32 sums and a bf16 result: about four times the distance to the 64-bit
  result that was measured (0.002 for one attention, 0.003 where a bf16 intermediate follows a
  gated product, 0.006 for a chain of six modules)."""
  return {"rel": {"triangle": 8e-3, "trimul": 1.2e-2, "pair_transition": 1e-2, "single": 1.2e-2,
                  "diffusion_attention": 8e-3, "diffusion_transition": 1e-2, "window": 8e-3,
                  "pairformer": 2.5e-2, "superblock": 2.5e-2}[case["op"]]}


# ---------------------------------------------------------------------------------------
# 64-bit results
# ---------------------------------------------------------------------------------------

def _ln(x, w=None, b=None):
  x = x - x.mean(-1, keepdim=True)
  x = x / torch.sqrt(x.square().mean(-1, keepdim=True) + 1e-5)
  x = x if w is None else x * w
  return x if b is None else x + b


def _masked_softmax(logits, mask):
  """Masked keys weigh nothing; a row without a valid key weighs every key alike."""
  return torch.softmax(logits.masked_fill(~mask, -1e30), -1)


def _exact_triangle(z, mask, w, end):
  n, c = z.shape[0], z.shape[-1]
  h, d = HEADS_TRI, c // HEADS_TRI
  x = _ln(z, w["act_norm.weight"])
  bias = (x @ w["pair_bias_projection.weight"]).permute(2, 0, 1)
  x = x.transpose(0, 1).contiguous() if end else x
  pair = mask[:, None] & mask[None, :]
  wq, wk = (w[k].reshape(c, c).t().contiguous() for k in ("q_projection.weight", "k_projection.weight"))
  wv, wg = w["v_projection.weight"].reshape(c, c), w["gating_query.weight"].t().contiguous()
  out = torch.empty_like(x)
  step = max(1, (1 << 27) // (h * n * n))
  for r in range(0, n, step):
    xr = x[r:r + step]
    q, k, v = ((xr @ m).unflatten(-1, (h, d)).transpose(1, 2).contiguous() for m in (wq, wk, wv))
    logits = q @ k.transpose(-1, -2).contiguous() / math.sqrt(d) + bias
    o = _masked_softmax(logits, pair[r:r + step, None, None]) @ v
    o = o.transpose(1, 2).reshape(xr.shape) * torch.sigmoid(xr @ wg)
    out[r:r + step] = o @ w["output_projection.weight"]
  return z + (out.transpose(0, 1) if end else out)


def _exact_trimul(z, mask, w, incoming):
  pair = (mask[:, None] & mask[None, :])[..., None]
  x = _ln(z, w["left_norm_input.weight"], w["left_norm_input.bias"])
  ab = torch.sigmoid(x @ w["gate_projection.weight"]) * (x @ w["projection.weight"])
  ab = ab.masked_fill(~pair, 0.0).permute(2, 0, 1)
  a, b = ab[0::2].contiguous(), ab[1::2].contiguous()
  del ab
  t = b.transpose(1, 2).contiguous() @ a if incoming else a @ b.transpose(1, 2).contiguous()
  # outgoing: t[i, j] = sum_k a[i, k] b[j, k]; incoming: t[i, j] = sum_k a[k, j] b[k, i]
  t = _ln(t.permute(1, 2, 0), w["center_norm.weight"], w["center_norm.bias"])
  return z + (t @ w["output_projection.weight"]) * torch.sigmoid(x @ w["gating_linear.weight"])


def _swiglu(x, w1):
  a, b = (x @ w1).chunk(2, -1)
  return a * torch.sigmoid(a) * b


def _exact_transition(z, w):
  x = _ln(z, w["input_layer_norm.weight"], w["input_layer_norm.bias"])
  return z + _swiglu(x, w["transition1.weight"]) @ w["transition2.weight"]


def _sub(w, prefix):
  return {k[len(prefix):]: v for k, v in w.items() if k.startswith(prefix)}


def _exact_adaln(x, cond, w):
  if cond is None:
    return _ln(x, w["layer_norm.weight"], w["layer_norm.bias"])
  c = _ln(cond, w["single_cond_layer_norm.weight"])
  return torch.sigmoid(c @ w["single_cond_scale.weight"] + w["single_cond_scale.bias"]) * _ln(x) + c @ w["single_cond_bias.weight"]


def _exact_zero_init(y, cond, w):
  y = y @ w["transition2.weight"]
  return y if cond is None else y * torch.sigmoid(cond @ w["adaptive_zero_cond.weight"] + w["adaptive_zero_cond.bias"])


def _exact_attention(xq, xk, mask, bias, w, h, gate_x):
  """Attention of normalised queries xq on keys xk, gated by the queries; [..., L, C]."""
  c = xq.shape[-1]
  split = lambda y: y.unflatten(-1, (h, c // h)).transpose(-2, -3).contiguous()
  q = split(xq @ w["q_projection.weight"].reshape(c, c) + w["q_projection.bias"].reshape(c))
  k, v = (split(xk @ w[n].reshape(c, c)) for n in ("k_projection.weight", "v_projection.weight"))
  logits = q @ k.transpose(-1, -2).contiguous() / math.sqrt(c // h) + bias
  o = (_masked_softmax(logits, mask) @ v).transpose(-2, -3).flatten(-2)
  return o * torch.sigmoid(gate_x @ w["gating_query.weight"])


def _exact_self(x, mask, bias, cond, w):
  hn = _exact_adaln(x, cond, _sub(w, "layer_norm."))
  o = _exact_attention(hn, hn, mask, bias, w, HEADS_SINGLE, hn)
  return x + _exact_zero_init(o, cond, _sub(w, "zero_init."))


def _exact_token_transition(x, cond, w):
  hn = _exact_adaln(x, cond, _sub(w, "layer_norm."))
  return x + _exact_zero_init(_swiglu(hn, w["transition.weight"]), cond, _sub(w, "zero_init."))


def _exact_single(z, s, mask, w):
  pl = _ln(z, w["single_pair_logits_norm.weight"], w["single_pair_logits_norm.bias"])
  bias = (pl @ w["single_pair_logits_projection.weight"]).permute(2, 0, 1)
  s = _exact_self(s, mask, bias, None, _sub(w, "single_attention."))
  return _exact_transition(s, _sub(w, "single_transition."))


def _exact_window(i, w, samples):
  c = C_ATOM
  x = i["act"]
  keys = x.reshape(samples, -1, c)[:, i["idx"].long()].masked_fill(~i["inside"][..., None], 0.0)
  hq = _exact_adaln(x, i["cond"], _sub(w, "q_layernorm."))
  hk = _exact_adaln(keys, i["kcond"], _sub(w, "k_layernorm."))
  mask = i["qmask"][:, None, :, None] & i["kmask"][:, None, None, :]
  o = _exact_attention(hq, hk, mask, i["bias"], w, HEADS_TRI, hq)
  return x + _exact_zero_init(o, i["cond"], _sub(w, "zero_init."))


def exact(case, seed):
  def wide(v):
    if isinstance(v, dict):
      return {k: wide(x) for k, x in v.items()}
    return v.double() if v.is_floating_point() else v

  i = wide(_inputs(case, seed))
  op, w = case["op"], i["w"]
  if op == "triangle":
    return _exact_triangle(i["z"], i["mask"], w, case["end"])
  if op == "trimul":
    return _exact_trimul(i["z"], i["mask"], w, case["incoming"])
  if op == "pair_transition":
    return _exact_transition(i["z"], w)
  if op == "single":
    return _exact_single(i["z"], i["s"], i["mask"], w)
  if op == "diffusion_attention":
    return _exact_self(i["x"], i["mask"], i["bias"], i["cond"], w)
  if op == "diffusion_transition":
    return _exact_token_transition(i["x"], i["cond"], w)
  if op == "window":
    return _exact_window(i, w, case["samples"])
  if op == "pairformer":
    z, mask = i["z"], i["mask"]
    z = _exact_trimul(z, mask, w["outgoing"], False)
    z = _exact_trimul(z, mask, w["incoming"], True)
    z = _exact_triangle(z, mask, w["start"], False)
    z = _exact_triangle(z, mask, w["end"], True)
    z = _exact_transition(z, w["pair"])
    return {"pair": z, "single": _exact_single(z, i["s"], mask, w["single"])}
  x = i["x"]
  pl = _ln(i["pair"], w["pair_input_layer_norm.weight"])
  proj = w["pair_logits_projection.0.weight"]
  for b in range(BLOCKS):
    bias = (pl @ proj[:, b]).permute(2, 0, 1)
    x = _exact_self(x, i["mask"], bias, i["cond"], _sub(w, f"self_attention.0.{b}."))
    x = _exact_token_transition(x, i["cond"], _sub(w, f"transition_block.0.{b}."))
  return x
