"""What is timed of this framework: the work that a serving program has it do.

Every case is a dict of plain values with a ``kind``:

* ``decode``   one talker decode step (the step's plan, then per layer one ``decode_step``)
               over the slot arena, in one captured graph as ``SlotGraph`` keeps it;
* ``graph``    the same through the modules: ``SlotGraph.run`` of a talker whose attention is
               ``PackedAttention`` (projections and norms by torch);
* ``chain``    the code predictor's 15 steps over its 16-row cache, one ``decode_step`` a layer;
* ``prefill``  packed prompts through ``prefill_step``, layer by layer;
* ``padded``   a padded prompt batch under an explicit key-valid and causal mask through the
               drop-in ``attention``;
* ``gqa``      the drop-in ``attention`` for one query a request under the full-arena mask
               (the reference's operator call);
* ``fp32``     the step of a float32 module: ``rope_tables``, ``rotary``, ``write`` and
               ``attention``, each a call of its own;
* ``arena``    admission and upkeep of the packed arena: prompt loads, compaction moves and a
               capacity growth, called eagerly as the scheduler does.

Shapes are the talker's (28 layers, 16 query heads over 8 KV heads of 128, bf16) and the code
predictor's (5 layers, the same heads).  Cases of very large arenas run four layers instead of
28: every layer is the same work, and three whole arenas would fill the card.
"""
from __future__ import annotations

import math
from types import SimpleNamespace

import torch

import __graft_entry__

amd = __graft_entry__.import_package()

HQ, HKV, D, LAYERS = 16, 8, 128, 28
THETA = 1_000_000.0
HIDDEN = 2048
PREDICTOR_LAYERS, PREDICTOR_STEPS, PREDICTOR_ROWS = 5, 15, 16
DEVICE = 'cuda'
BF16, F32, F64 = torch.bfloat16, torch.float32, torch.float64


def listed():
    return [
        # the flagship: 64 concurrent requests somewhere between 64 and 1023 tokens into speech
        dict(name='talker_64', kind='decode', batch=64, capacity=1024, low=64, high=1023, masked=False, layers=28),
        # one user alone on the server: latency of the launches
        dict(name='talker_1', kind='decode', batch=1, capacity=512, low=200, high=400, masked=False, layers=28),
        # a full 128-slot server deep into long speech, each layer handed the step's mask as the
        # reference's graph does
        dict(name='talker_128_long_masked', kind='decode', batch=128, capacity=2048, low=100, high=2047, masked=True, layers=4),
        # a 21-request step through the modules, as a user of SlotGraph runs it
        dict(name='slot_graph_21', kind='graph', batch=21, capacity=512, low=30, high=511, layers=28),
        # the codes of one frame for 64 requests
        dict(name='predictor_64', kind='chain', batch=64),
        # an admission burst of 16 prompts
        dict(name='prefill_16', kind='prefill', prompts=16, low=32, high=512, layers=28),
        # one short prompt: time to first audio
        dict(name='prefill_1', kind='prefill', prompts=1, low=45, high=45, layers=28),
        # long reference texts: the matrix cores
        dict(name='prefill_long', kind='prefill', prompts=8, low=1024, high=2048, layers=4),
        # a padded batch with its mask, through the drop-in
        dict(name='padded_8', kind='padded', batch=8, length=256, layers=28),
        # the drop-in decode call over a 512-row arena under the full mask
        dict(name='gqa_masked_64', kind='gqa', batch=64, capacity=512, low=1, high=511, mask='bool', layers=28),
        # a float32 model, one request a KV slot of 16
        dict(name='step_fp32_16', kind='fp32', batch=16, capacity=512, low=20, high=511, layers=8),
        # the arena of a 32-slot server: eight prompts admitted, two slots compacted, capacity doubled
        dict(name='arena_32', kind='arena', slots=32, capacity=512, loads=8, longest=400),
    ]


def _log_int(rng, low, high):
    return min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def draw(rng):
    kind = rng.choice(['decode', 'decode', 'graph', 'chain', 'prefill', 'prefill', 'padded', 'gqa', 'fp32', 'arena'])
    if kind == 'decode':
        batch = _log_int(rng, 1, 128)
        capacity = _log_int(rng, 256, min(4096, 128 * 2048 // batch))
        low = rng.randrange(1, capacity // 2)
        return dict(kind=kind, batch=batch, capacity=capacity, low=low, high=rng.randrange(low, capacity),
                    masked=rng.random() < 0.4, layers=28 if batch * capacity <= 64 * 1024 else 4)
    if kind == 'graph':
        capacity = _log_int(rng, 128, 1024)
        return dict(kind=kind, batch=_log_int(rng, 1, 32), capacity=capacity, low=rng.randrange(1, capacity // 2),
                    high=capacity - 1, layers=28)
    if kind == 'chain':
        return dict(kind=kind, batch=_log_int(rng, 1, 128))
    if kind == 'prefill':
        prompts = _log_int(rng, 1, 32)
        high = _log_int(rng, 16, min(2048, 16384 // prompts))
        return dict(kind=kind, prompts=prompts, low=rng.randrange(1, high), high=high, layers=28 if prompts * high <= 8192 else 4)
    if kind == 'padded':
        batch = _log_int(rng, 1, 16)
        return dict(kind=kind, batch=batch, length=8 * _log_int(rng, 2, min(128, 512 // batch)), layers=28)
    if kind == 'gqa':
        batch = _log_int(rng, 1, 96)
        capacity = _log_int(rng, 64, min(2048, 64 * 1024 // batch))
        low = rng.randrange(1, capacity // 2)
        return dict(kind=kind, batch=batch, capacity=capacity, low=low, high=capacity - 1,
                    mask=rng.choice(['bool', 'bf16', 'positions']), layers=28)
    if kind == 'fp32':
        batch = _log_int(rng, 1, 48)
        capacity = _log_int(rng, 64, 1024)
        return dict(kind=kind, batch=batch, capacity=capacity, low=rng.randrange(1, capacity // 2), high=capacity - 1, layers=8)
    slots = 1 << rng.randrange(1, 6)
    capacity = rng.choice([64, 128, 256, 512])
    return dict(kind=kind, slots=slots, capacity=capacity, loads=rng.randrange(1, min(slots, 8) + 1),
                longest=rng.randrange(1, capacity))


# ---- inputs -------------------------------------------------------------------------------

def _generators(seed):
    return torch.Generator().manual_seed(seed), torch.Generator(device=DEVICE).manual_seed(seed)


def _normal(gen, *shape, dtype=BF16):
    return torch.randn(*shape, generator=gen, device=DEVICE, dtype=dtype)


def _contexts(case, gen):
    return torch.randint(case['low'], case['high'] + 1, (case['batch'],), generator=gen)


def _inverse_frequencies():
    return (1.0 / (THETA ** (torch.arange(0, D, 2, dtype=F32) / D))).to(DEVICE)


def _tables(positions, dtype=BF16, inv=None):
    """cos/sin rows of integer positions, as the talker's rotary module gives them."""
    inv = _inverse_frequencies() if inv is None else inv
    angle = positions[..., None].float() * inv
    angle = torch.cat((angle, angle), -1)
    return angle.cos().to(dtype), angle.sin().to(dtype)


def _split(rows):
    """Query, key and value views of fused projection rows (..., Hq + 2 Hkv, D)."""
    return rows[..., :HQ, :], rows[..., HQ:HQ + HKV, :], rows[..., HQ + HKV:, :]


def _capture(step):
    """One eager pass, then the captured graph of ``step``."""
    step()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step()
    return graph


def _decode_inputs(case, seed):
    host, gen = _generators(seed)
    layers, batch, capacity = case['layers'], case['batch'], case['capacity']
    contexts = _contexts(case, host)
    s = SimpleNamespace(contexts=contexts.tolist(), positions=contexts.to(DEVICE))
    s.arena = _normal(gen, 2 * layers, batch, HKV, capacity, D)
    s.rows = _normal(gen, layers, batch, 1, HQ + 2 * HKV, D)
    s.cos, s.sin = _tables(s.positions)
    return s


def _chain_inputs(case, seed):
    _, gen = _generators(seed)
    s = SimpleNamespace()
    s.rows = _normal(gen, PREDICTOR_STEPS, PREDICTOR_LAYERS, case['batch'], 2, HQ + 2 * HKV, D)
    # a cache of an earlier frame: rows past a step's position are stale
    s.arena = _normal(gen, 2 * PREDICTOR_LAYERS, case['batch'], HKV, PREDICTOR_ROWS, D)
    s.positions = [torch.full((case['batch'],), max(step + 1, 1), device=DEVICE) for step in range(PREDICTOR_STEPS)]
    s.tables = [_tables(p) for p in s.positions]
    s.tables[0] = _tables(torch.arange(2, device=DEVICE).expand(case['batch'], 2))
    return s


def _lengths(case):
    return torch.randint(case['low'], case['high'] + 1, (case['prompts'],), generator=torch.Generator().manual_seed(0))


def _prefill_inputs(case, seed):
    host, gen = _generators(seed)
    layers, prompts = case['layers'], case['prompts']
    # the burst's lengths are the case's own; the order in which they are packed is the seed's
    lengths = _lengths(case)[torch.randperm(prompts, generator=host)]
    total = int(lengths.sum())
    s = SimpleNamespace(lengths=lengths.tolist(), longest=int(lengths.max()))
    s.cu = torch.cat([torch.zeros(1, dtype=torch.long), lengths.cumsum(0)]).to(device=DEVICE, dtype=torch.int32)
    capacity = max(512, 1 << (case['high'] - 1).bit_length())
    s.slots = torch.randperm(prompts, generator=host)
    s.kv_slots = s.slots.to(DEVICE)
    s.arena = torch.zeros(2 * layers, prompts, HKV, capacity, D, device=DEVICE, dtype=BF16)
    s.rows = _normal(gen, layers, total, HQ + 2 * HKV, D)
    s.cos, s.sin = _tables(torch.cat([torch.arange(n) for n in s.lengths]).to(DEVICE))
    return s


def _padded_inputs(case, seed):
    host, gen = _generators(seed)
    layers, batch, length = case['layers'], case['batch'], case['length']
    s = SimpleNamespace()
    s.rows = _normal(gen, layers, batch, length, HQ + 2 * HKV, D)
    valid = torch.randint(max(1, length // 4), length + 1, (batch,), generator=host)
    valid[0] = length
    keys = torch.arange(length)
    visible = (keys[None, :] <= keys[:, None])[None] & (keys[None, :] < valid[:, None])[:, None]
    s.visible = visible[:, None].to(DEVICE)
    s.mask = torch.zeros(batch, 1, length, length, device=DEVICE, dtype=BF16).masked_fill(~s.visible, torch.finfo(BF16).min)
    return s


def _gqa_inputs(case, seed):
    host, gen = _generators(seed)
    layers, batch, capacity = case['layers'], case['batch'], case['capacity']
    contexts = _contexts(case, host)
    s = SimpleNamespace(contexts=contexts.tolist(), positions=contexts.to(DEVICE))
    s.query = _normal(gen, layers, batch, HQ, 1, D)
    s.arena = _normal(gen, 2 * layers, batch, HKV, capacity, D)
    visible = (torch.arange(capacity, device=DEVICE)[None, :] <= s.positions[:, None])[:, None, None, :]
    s.mask = None
    if case['mask'] == 'bool':
        s.mask = visible
    elif case['mask'] == 'bf16':
        s.mask = torch.zeros(visible.shape, device=DEVICE, dtype=BF16).masked_fill(~visible, torch.finfo(BF16).min)
    return s


def _fp32_inputs(case, seed):
    host, gen = _generators(seed)
    layers, batch, capacity = case['layers'], case['batch'], case['capacity']
    contexts = _contexts(case, host)
    s = SimpleNamespace(contexts=contexts.tolist(), positions=contexts.to(DEVICE))
    s.query = _normal(gen, layers, batch, 1, HQ, D, dtype=F32)
    s.key, s.value = (_normal(gen, layers, batch, 1, HKV, D, dtype=F32) for _ in range(2))
    s.arena = _normal(gen, 2 * layers, batch, HKV, capacity, D, dtype=F32)
    return s


def _reference():
    """What SlotArena reads of a talker."""
    weight = torch.empty(1, device=DEVICE, dtype=BF16)
    return SimpleNamespace(parameters=lambda: iter([weight]), layers=[None] * LAYERS,
                           config=SimpleNamespace(num_key_value_heads=HKV, head_dim=D, num_attention_heads=HQ))


def _arena_inputs(case, seed):
    host, gen = _generators(seed)
    s = SimpleNamespace(case=case)
    s.content = _normal(gen, 2 * LAYERS, case['slots'], HKV, case['capacity'], D)
    s.lengths = torch.randint(1, case['longest'] + 1, (case['loads'],), generator=host).tolist()
    s.lengths[0] = case['longest']
    s.cache = _normal(gen, 2 * LAYERS, case['loads'], HKV, case['longest'], D)
    s.slots = torch.randperm(case['slots'], generator=host)[:case['loads']].tolist()
    # compaction: a quarter of the slots' worth of moves between distinct slots
    count = max(1, case['loads'] // 4)
    order = torch.randperm(case['slots'], generator=host).tolist()
    s.moves = [(order[i], order[-1 - i]) for i in range(count) if order[i] != order[-1 - i]]
    s.moved = torch.randint(1, case['capacity'] + 1, (len(s.moves),), generator=host).tolist()
    return s


# ---- the modules of the whole call ----------------------------------------------------------

class RMSNorm(torch.nn.Module):
    def __init__(self, width, scale):
        super().__init__()
        self.weight = torch.nn.Parameter(torch.full((width,), scale, device=DEVICE, dtype=BF16), requires_grad=False)
        self.eps = 1e-6

    def forward(self, x):
        y = x.float()
        y = y * torch.rsqrt(y.pow(2).mean(-1, keepdim=True) + self.eps)
        return self.weight * y.to(x.dtype)


def _linear(gen, inputs, outputs):
    module = torch.nn.utils.skip_init(torch.nn.Linear, inputs, outputs, bias=False, device=DEVICE, dtype=BF16)
    module.weight.requires_grad_(False)
    module.weight.copy_(_normal(gen, outputs, inputs) * inputs ** -0.5)
    return module


class Qwen3TTSTalkerAttention(torch.nn.Module):
    """The attributes that PackedAttention reads of a talker's attention."""

    def __init__(self, layer_idx, gen):
        super().__init__()
        self.head_dim, self.layer_idx, self.scaling = D, layer_idx, D ** -0.5
        self.sliding_window, self.attention_dropout, self.is_causal = None, 0.0, True
        self.q_proj, self.k_proj, self.v_proj = _linear(gen, HIDDEN, HQ * D), _linear(gen, HIDDEN, HKV * D), _linear(gen, HIDDEN, HKV * D)
        self.o_proj = _linear(gen, HQ * D, HIDDEN)
        self.q_norm, self.k_norm = RMSNorm(D, 1.25), RMSNorm(D, 1.25)


class Layer(torch.nn.Module):
    def __init__(self, layer_idx, gen):
        super().__init__()
        self.input_layernorm = RMSNorm(HIDDEN, 1.0)
        self.self_attn = Qwen3TTSTalkerAttention(layer_idx, gen)

    def forward(self, hidden_states, attention_mask=None, past_key_values=None, cache_position=None,
                position_embeddings=None, **_):
        attended, _ = self.self_attn(hidden_states=self.input_layernorm(hidden_states), attention_mask=attention_mask,
                                     position_embeddings=position_embeddings, past_key_values=past_key_values,
                                     cache_position=cache_position)
        return (hidden_states + attended,)


class Talker(torch.nn.Module):
    def __init__(self, layers, gen):
        super().__init__()
        self.config = SimpleNamespace(hidden_size=HIDDEN, num_key_value_heads=HKV, num_attention_heads=HQ, head_dim=D)
        self.layers = torch.nn.ModuleList(Layer(i, gen) for i in range(layers))
        self.norm = RMSNorm(HIDDEN, 1.0)
        self.inv = _inverse_frequencies()

    def rotary_emb(self, hidden, position_ids):
        return _tables(position_ids, inv=self.inv)


def _graph_inputs(case, seed):
    host, gen = _generators(seed)
    s = SimpleNamespace(talker=Talker(case['layers'], gen).eval())
    contexts = _contexts(case, host)
    s.contexts, s.positions = contexts.tolist(), contexts.to(DEVICE)
    s.rotary = s.positions.view(1, -1, 1).expand(3, -1, 1)
    s.hidden = _normal(gen, case['batch'], 1, HIDDEN)
    s.content = _normal(gen, 2 * case['layers'], case['batch'], HKV, case['capacity'], D)
    return s


# ---- states -------------------------------------------------------------------------------

def prepare(case, seed):
    with torch.inference_mode():
        s = {'decode': _prepare_decode, 'graph': _prepare_graph, 'chain': _prepare_chain, 'prefill': _prepare_prefill,
             'padded': _prepare_padded, 'gqa': _prepare_gqa, 'fp32': _prepare_fp32, 'arena': _prepare_arena}[case['kind']](case, seed)
    s.kind = case['kind']
    return s


def _prepare_decode(case, seed):
    s = _decode_inputs(case, seed)
    layers, batch, capacity = case['layers'], case['batch'], case['capacity']
    masked = case['masked']
    mask = None
    if masked:
        visible = (torch.arange(capacity, device=DEVICE)[None, :] <= s.positions[:, None])[:, None, None, :]
        mask = torch.zeros(visible.shape, device=DEVICE, dtype=BF16).masked_fill(~visible, torch.finfo(BF16).min)
    # SlotCache.prepare plans a step whose launches take the bundled grid
    planned = amd.decode_grid_for(batch, 1, HQ, HKV, D, capacity, masked=masked) == 'bundled'
    plan = torch.empty(amd.plan_shape(batch, HQ, HKV), device=DEVICE, dtype=torch.int32) if planned else None
    out = torch.empty(layers, batch, 1, HQ, D, device=DEVICE, dtype=BF16)

    def step():
        if planned:
            amd.decode_plan(s.positions, capacity, HQ, HKV, out=plan)
        for layer in range(layers):
            q, k, v = _split(s.rows[layer])
            amd.decode_step(q, k, v, s.arena[layer], s.arena[layers + layer], s.positions, s.cos, s.sin,
                            out=out[layer], mask=mask, plan=plan)

    s.outputs = {'out': out, 'arena': s.arena}
    s.graph = _capture(step)
    s.keep = (mask, plan)
    return s


def _prepare_graph(case, seed):
    s = _graph_inputs(case, seed)
    amd.install_packed_attention(s.talker, native_gqa=True, text_only_rope=True, triton_talker_rope=True)
    s.arena = amd.SlotArena(s.talker, case['batch'], case['capacity'], packed_kv=True)
    s.arena.packed.copy_(s.content)
    del s.content
    s.graph = amd.SlotGraph(s.arena, case['batch'])
    s.graph.capture()
    return s


def _prepare_chain(case, seed):
    s = _chain_inputs(case, seed)
    batch, layers = case['batch'], PREDICTOR_LAYERS
    first = torch.empty(layers, batch, 2, HQ, D, device=DEVICE, dtype=BF16)
    later = torch.empty(PREDICTOR_STEPS - 1, layers, batch, 1, HQ, D, device=DEVICE, dtype=BF16)

    def chain():
        for step in range(PREDICTOR_STEPS):
            tokens = 2 if step == 0 else 1
            for layer in range(layers):
                q, k, v = _split(s.rows[step, layer, :, :tokens])
                amd.decode_step(q, k, v, s.arena[layer], s.arena[layers + layer], s.positions[step], *s.tables[step],
                                out=first[layer] if step == 0 else later[step - 1, layer])

    s.outputs = {'first': first, 'later': later, 'arena': s.arena}
    s.graph = _capture(chain)
    return s


def _prepare_prefill(case, seed):
    s = _prefill_inputs(case, seed)
    layers = case['layers']
    out = torch.empty(layers, s.rows.shape[1], HQ, D, device=DEVICE, dtype=BF16)

    def step():
        for layer in range(layers):
            q, k, v = _split(s.rows[layer])
            amd.prefill_step(q, k, v, s.cos, s.sin, s.cu, s.longest, s.arena[layer], s.arena[layers + layer],
                             kv_slots=s.kv_slots, out=out[layer])

    s.outputs = {'out': out, 'arena': s.arena}
    s.graph = _capture(step)
    return s


_MODULE = SimpleNamespace(training=False, is_causal=True, sliding_window=None)


def _prepare_padded(case, seed):
    s = _padded_inputs(case, seed)
    outputs = [None] * case['layers']
    # the cache holds keys and values head by head, as attention receives them
    caches = [tuple(t.transpose(1, 2).contiguous() for t in _split(s.rows[layer])[1:]) for layer in range(case['layers'])]

    def step():
        for layer in range(case['layers']):
            query = s.rows[layer, :, :, :HQ].transpose(1, 2)
            outputs[layer] = amd.attention(_MODULE, query, *caches[layer], s.mask, scaling=D ** -0.5)[0]

    s.graph = _capture(step)
    s.outputs = outputs
    s.keep = caches
    return s


def _prepare_gqa(case, seed):
    s = _gqa_inputs(case, seed)
    layers = case['layers']
    outputs = [None] * layers
    more = {'kv_positions': s.positions} if case['mask'] == 'positions' else {}

    def step():
        for layer in range(layers):
            outputs[layer] = amd.attention(_MODULE, s.query[layer], s.arena[layer], s.arena[layers + layer], s.mask,
                                           scaling=D ** -0.5, **more)[0]

    s.graph = _capture(step)
    s.outputs = outputs
    return s


def _prepare_fp32(case, seed):
    s = _fp32_inputs(case, seed)
    layers = case['layers']
    outputs = [None] * layers

    def step():
        cos, sin = amd.rope_tables(s.positions[:, None], D, theta=THETA, dtype=F32)
        for layer in range(layers):
            query = amd.rotary(s.query[layer], cos, sin).transpose(1, 2)
            key = amd.rotary(s.key[layer], cos, sin).transpose(1, 2)
            keys, values = s.arena[layer], s.arena[layers + layer]
            amd.write(key, s.value[layer].transpose(1, 2), keys, values, s.positions)
            outputs[layer] = amd.attention(_MODULE, query, keys, values, None, scaling=D ** -0.5, kv_positions=s.positions)[0]

    s.graph = _capture(step)
    s.outputs = {'out': outputs, 'arena': s.arena}
    return s


def _prepare_arena(case, seed):
    s = _arena_inputs(case, seed)
    s.arena = amd.SlotArena(_reference(), case['slots'], case['capacity'], packed_kv=True)
    s.arena.packed.copy_(s.content)
    del s.content
    return s


def run(s):
    with torch.inference_mode():
        if s.kind == 'arena':
            for row, (slot, length) in enumerate(zip(s.slots, s.lengths)):
                s.arena.load_packed(slot, s.cache, row=row, length=length)
            for (source, destination), length in zip(s.moves, s.moved):
                s.arena.move(source, destination, length=length)
            return amd.grow_arena(s.arena, s.arena.capacity).packed
        if s.kind == 'graph':
            hidden = s.graph.run(s.hidden, s.positions, s.rotary)
            return {'hidden': hidden, 'arena': s.arena.packed}
        s.graph.replay()
        return s.outputs


# ---- what a pass cannot do without --------------------------------------------------------

def _mean_tokens(case):
    return case['batch'] * ((case['low'] + case['high']) / 2 + 1)


def work(case):
    kind, row = case['kind'], D * 2
    if kind in ('decode', 'graph', 'gqa', 'fp32'):
        element = 2 if kind == 'fp32' else 1
        tokens, batch = _mean_tokens(case), case['batch']
        keys = tokens * HKV * row * 2                              # every visible key and value row
        step = batch * row * (2 * HQ + (0 if kind == 'gqa' else 4 * HKV))  # q, out; new rows in and out
        mask = 0
        if kind == 'gqa':
            mask = {'bool': 1, 'bf16': 2, 'positions': 0}[case['mask']] * batch * case['capacity']
        elif case.get('masked'):
            mask = 2 * tokens
        per_layer = (keys + step) * element + mask
        flops = 4 * D * HQ * tokens
        if kind == 'graph':
            weights = HIDDEN * (2 * HQ + 2 * HKV) * D
            per_layer += weights * 2 + 2 * batch * HIDDEN * 2
            flops += 2 * weights * batch
        return {'bytes': case['layers'] * per_layer, 'flops': case['layers'] * flops}
    if kind == 'chain':
        rows = sum(3 if step == 0 else step + 2 for step in range(PREDICTOR_STEPS))
        steps = PREDICTOR_STEPS + 1  # query tokens
        per_layer = case['batch'] * row * (rows * HKV * 2 + steps * (2 * HQ + 4 * HKV))
        return {'bytes': PREDICTOR_LAYERS * per_layer, 'flops': PREDICTOR_LAYERS * case['batch'] * rows * 4 * D * HQ}
    if kind == 'prefill':
        lengths = _lengths(case)
        # projection rows in (q, k, v), output and arena rows out
        return {'bytes': case['layers'] * int(lengths.sum()) * row * (2 * HQ + 4 * HKV),
                'flops': case['layers'] * int((lengths * (lengths + 1)).sum()) * 2 * D * HQ}
    if kind == 'padded':
        tokens = case['batch'] * case['length']
        return {'bytes': case['layers'] * (tokens * row * (2 * HQ + 2 * HKV) + tokens * case['length'] * 2),
                'flops': case['layers'] * tokens * (case['length'] + 1) / 2 * 4 * D * HQ}
    planes = 2 * LAYERS * HKV * row
    copied = case['loads'] * case['longest'] / 2 + max(1, case['loads'] // 4) * case['capacity'] / 2
    # loads and moves read and written; the growth reads every row and writes twice as many
    return {'bytes': planes * (2 * copied + 3 * case['slots'] * case['capacity']), 'flops': 0}


def tolerance(case):
    kind = case['kind']
    if kind == 'arena':
        return 'exact'
    if kind == 'fp32':
        return {'rel': 2e-6, 'max': 1e-4}
    if kind == 'graph':
        # 28 layers of bf16 rounding
        return {'rel': 2e-2, 'max': 0.2}
    return {'rel': 1e-2, 'max': 0.1}


# ---- the same in 64 bits --------------------------------------------------------------------

def _rotate(x, cos, sin):
    half = x.shape[-1] // 2
    turned = torch.cat((-x[..., half:], x[..., :half]), -1)
    return x * cos + turned * sin


def _attend(query, keys, values, visible=None):
    """query (H, S, D) over keys/values (Hkv, N, D), all float64; visible (S, N)."""
    group = query.shape[0] // keys.shape[0]
    keys, values = keys.repeat_interleave(group, 0), values.repeat_interleave(group, 0)
    scores = torch.bmm(query, keys.transpose(1, 2).contiguous()) * D ** -0.5
    if visible is not None:
        scores = scores.masked_fill(~visible, float('-inf'))
    return torch.bmm(scores.softmax(-1), values)


def exact(case, seed):
    with torch.inference_mode():
        return {'decode': _exact_decode, 'graph': _exact_graph, 'chain': _exact_chain, 'prefill': _exact_prefill,
                'padded': _exact_padded, 'gqa': _exact_gqa, 'fp32': _exact_fp32, 'arena': lambda c, s: None}[case['kind']](case, seed)


def _exact_step(q, k, v, keys, values, contexts, cos, sin):
    """One token a request: the write into keys/values (float64, in place), the attention."""
    out = torch.empty(q.shape, device=DEVICE, dtype=F64)
    for b, position in enumerate(contexts):
        keys[b, :, position] = _rotate(k[b, 0].double(), cos[b], sin[b])
        values[b, :, position] = v[b, 0].double()
        query = _rotate(q[b, 0].double(), cos[b], sin[b])[:, None]
        out[b, 0] = _attend(query, keys[b, :, :position + 1], values[b, :, :position + 1])[:, 0]
    return out


def _exact_decode(case, seed):
    s = _decode_inputs(case, seed)
    arena, layers = s.arena.double(), case['layers']
    cos, sin = s.cos.double(), s.sin.double()
    out = [_exact_step(*_split(s.rows[layer]), arena[layer], arena[layers + layer], s.contexts, cos, sin) for layer in range(layers)]
    return {'out': torch.stack(out), 'arena': arena}


def _exact_norm(x, weight):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + 1e-6) * weight.double()


def _exact_graph(case, seed):
    s = _graph_inputs(case, seed)
    arena, layers, batch = s.content.double(), case['layers'], case['batch']
    cos, sin = (t.double() for t in _tables(s.positions))
    hidden = s.hidden.double()
    for index, layer in enumerate(s.talker.layers):
        attn = layer.self_attn
        x = _exact_norm(hidden, layer.input_layernorm.weight)
        q, k, v = ((x @ p.weight.double().T).view(batch, 1, -1, D) for p in (attn.q_proj, attn.k_proj, attn.v_proj))
        out = _exact_step(_exact_norm(q, attn.q_norm.weight), _exact_norm(k, attn.k_norm.weight), v,
                          arena[index], arena[layers + index], s.contexts, cos, sin)
        hidden = hidden + out.reshape(batch, 1, -1) @ attn.o_proj.weight.double().T
    return {'hidden': _exact_norm(hidden, s.talker.norm.weight), 'arena': arena}


def _exact_chain(case, seed):
    s = _chain_inputs(case, seed)
    arena, layers = s.arena.double(), PREDICTOR_LAYERS
    first, later = [], []
    for step in range(PREDICTOR_STEPS):
        tokens = 2 if step == 0 else 1
        cos, sin = (t.double().view(case['batch'], tokens, 1, D) for t in s.tables[step])
        start = 0 if step == 0 else step + 1
        end = start + tokens
        causal = torch.ones(tokens, end, device=DEVICE, dtype=torch.bool).tril(start)
        for layer in range(layers):
            q, k, v = (x.double() for x in _split(s.rows[step, layer, :, :tokens]))
            q, k = _rotate(q, cos, sin), _rotate(k, cos, sin)
            arena[layer, :, :, start:end] = k.transpose(1, 2)
            arena[layers + layer, :, :, start:end] = v.transpose(1, 2)
            keys, values = (arena[i, :, :, :end].repeat_interleave(HQ // HKV, 1) for i in (layer, layers + layer))
            scores = torch.einsum('bshd,bhnd->bhsn', q, keys) * D ** -0.5
            weights = scores.masked_fill(~causal, float('-inf')).softmax(-1)
            out = torch.einsum('bhsn,bhnd->bshd', weights, values)
            (first if step == 0 else later).append(out)
    return {'first': torch.stack(first), 'later': torch.stack(later).view(PREDICTOR_STEPS - 1, layers, *later[0].shape), 'arena': arena}


def _exact_prefill(case, seed):
    s = _prefill_inputs(case, seed)
    arena, layers = s.arena.double(), case['layers']
    cos, sin = s.cos.double()[:, None], s.sin.double()[:, None]
    out = torch.empty(layers, s.rows.shape[1], HQ, D, device=DEVICE, dtype=F64)
    for layer in range(layers):
        q, k, v = (x.double() for x in _split(s.rows[layer]))
        q, k = _rotate(q, cos, sin), _rotate(k, cos, sin)
        at = 0
        for slot, n in zip(s.slots.tolist(), s.lengths):
            qb, kb, vb = (x[at:at + n].transpose(0, 1).contiguous() for x in (q, k, v))
            arena[layer, slot, :, :n], arena[layers + layer, slot, :, :n] = kb, vb
            visible = torch.ones(n, n, device=DEVICE, dtype=torch.bool).tril()
            out[layer, at:at + n] = _attend(qb, kb, vb, visible).transpose(0, 1)
            at += n
    return {'out': out, 'arena': arena}


def _exact_padded(case, seed):
    s = _padded_inputs(case, seed)
    out = []
    for layer in range(case['layers']):
        q, k, v = (x.double().transpose(1, 2).contiguous() for x in _split(s.rows[layer]))
        out.append(torch.stack([_attend(q[b], k[b], v[b], s.visible[b, 0]).transpose(0, 1) for b in range(case['batch'])]))
    return out


def _exact_gqa(case, seed):
    s = _gqa_inputs(case, seed)
    out, layers = [], case['layers']
    for layer in range(layers):
        out.append(torch.stack([
            _attend(s.query[layer, b].double(), s.arena[layer, b, :, :n + 1].double(),
                    s.arena[layers + layer, b, :, :n + 1].double()).transpose(0, 1) for b, n in enumerate(s.contexts)]))
    return out


def _exact_fp32(case, seed):
    s = _fp32_inputs(case, seed)
    arena, layers = s.arena.double(), case['layers']
    # the angle is a float32 product, as the rotary module's is; its cosine in 64 bits
    angle = (s.positions[:, None].float() * _inverse_frequencies()).double()
    angle = torch.cat((angle, angle), -1)
    cos, sin = angle.cos(), angle.sin()
    out = [_exact_step(s.query[i], s.key[i], s.value[i], arena[i], arena[layers + i], s.contexts, cos, sin) for i in range(layers)]
    return {'out': out, 'arena': arena}
