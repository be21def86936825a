"""The calls whose time this framework is judged by: what a multi-scene video run has it do on one GPU, through its
public entry points, with the sizes of the repository's own workloads (HunyuanVideo-1.5 480p, Wan2.2 704x1280, the
16-scene Wan step, the uneven scene sweep, the CPU-plumbing layout) and ragged ones between them.

listed() names the cases, draw(rng) gives more of the same ranges; prepare / run make the inputs and one pass, exact
restates a pass in float64 torch, work and tolerance say what a pass cannot do without and how far apart two correct
implementations are. A case is a dict of plain values; lists of frames and counts are comma-separated text.
"""
from __future__ import annotations

import math

import torch
import torch.nn.functional as F

DEV = 'cuda'


def listed():
    hunyuan = dict(heads=16, dim=128)
    return [
        # the smallest layer anyone runs (previews, smoke runs, unit-sized models): all launches and latency
        dict(name='scene-tiny', kind='scene', lengths='3,3', grid='8x8', counts='16,16', pad=0, reps='0,5',
             halo=0, sides='adj', position='adjacent', rotated=False, heads=2, dim=64),
        # the headline layer: HunyuanVideo-1.5 480p, 4 scenes x 8 latent frames, frame memory 4, every layer and step
        dict(name='scene-480p', kind='scene', lengths='8,8,8,8', grid='30x53', counts='128,128,128,128', pad=0,
             reps='0,10,21,31', halo=0, sides='adj', position='adjacent', rotated=False, **hunyuan),
        # a short uneven story at a low resolution with odd token and text counts, through the reference's own entry
        # (q / k already rotated, shared keys moved), padding text rows behind the valid ones
        dict(name='scene-ragged', kind='scene', lengths='5,2,7', grid='17x23', counts='77,201,64', pad=11,
             reps='0,6,13', halo=1, sides='prev', position='adjacent', rotated=True, **hunyuan),
        # bounded memory in place of shared frames, 480p: every denoising step after the first (warm centroids)
        dict(name='memory-480p-warm', kind='memory', lengths='8,8,8,8', grid='30x53', counts='128,128,128,128',
             budget=128, warm=True, **hunyuan),
        # bounded memory, first step of a request: the representatives are clustered from scratch in every layer
        dict(name='memory-first-step', kind='memory', lengths='5,3,6', grid='15x26', counts='90,128,41',
             budget=128, warm=False, **hunyuan),
        # Wan cross-attention of 16 scenes x 15 frames, each to its own 128-token sentence (every block of the step)
        dict(name='wan-cross', kind='cross', lengths=','.join(['15'] * 16), tokens=880, text=128, heads=24, dim=128),
        # the RMSNorm + RoPE of q and k ahead of every Wan self-attention, 3 scenes x 11 frames at 704x1280
        dict(name='wan-qk', kind='qk', rows=29040, heads=24, dim=128),
        # attention split over key sets (a rank's half scene against its local and its received keys), then merged
        dict(name='split-keys', kind='split', rows=8480, local=8739, far=8879, **hunyuan),
        # frame memory of one denoising step: pool the observed layer's 480p hidden states, choose the representatives
        dict(name='frame-memory', kind='frames', lengths='8,8,8,8', tokens=1590, width=2048, budget=4, pool='all'),
        # the FlashAttention drop-in on a batch of short ragged sequences (text, image prompts, thumbnails)
        dict(name='packed-short', kind='packed', q='1,77,256,33,410,128,699,5,300,64,512,190',
             k='128,77,300,65,410,1,899,640,33,257,512,31', **hunyuan),
        # the dense drop-in at head_dim 64
        dict(name='dense-64', kind='dense', batch=2, q_rows=3001, k_rows=3001, heads=16, dim=64),
        # a whole transformer pass: two blocks of the Wan2.2-TI2V-5B shape on a thumbnail-sized 3-scene latent
        dict(name='dit-pass', kind='dit', lengths='4,5,4', grid='11x20', text=128, halo=2, sides='next', blocks=2),
    ]


# the largest listed case bounds every drawn one
_MAX_FLOPS, _MAX_BYTES = 7.4e12, 3.0e9


def draw(rng):
    while True:
        case = _draw(rng)
        w = work(case)
        if w['flops'] <= _MAX_FLOPS and w['bytes'] <= _MAX_BYTES:
            return case


def _span(rng, lo, hi):
    """an integer of [lo, hi], spread over its logarithm"""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _text(xs):
    return ','.join(str(x) for x in xs)


def _draw(rng):
    kind = rng.choice(['scene', 'scene', 'scene', 'memory', 'memory', 'cross', 'qk', 'split', 'frames', 'packed',
                       'dense', 'dit'])
    if kind in ('scene', 'memory'):
        n = rng.randint(2, 6)
        lengths = [rng.randint(2, 12) for _ in range(n)]
        grid = f'{rng.randint(6, 30)}x{rng.randint(6, 53)}'
        counts = [rng.randint(5, 256) for _ in range(n)]
        heads, dim = rng.choice([(16, 128), (16, 128), (24, 128), (12, 64), (3, 128)])
        if kind == 'memory':
            return dict(kind=kind, lengths=_text(lengths), grid=grid, counts=_text(counts),
                        budget=rng.choice([32, 128, 128, 200]), warm=rng.random() < 0.6, heads=heads, dim=dim)
        total = sum(lengths)
        reps = sorted(rng.sample(range(total), min(total, rng.randint(1, 4))))
        return dict(kind=kind, lengths=_text(lengths), grid=grid, counts=_text(counts), pad=rng.choice([0, 0, 9]),
                    reps=_text(reps), halo=rng.choice([0, 0, 1]), sides=rng.choice(['adj', 'prev', 'next']),
                    position=rng.choice(['adjacent', 'source']), rotated=rng.random() < 0.3, heads=heads, dim=dim)
    if kind == 'cross':
        n = rng.randint(1, 16)
        return dict(kind=kind, lengths=_text([rng.randint(3, 15) for _ in range(n)]), tokens=_span(rng, 60, 1590),
                    text=rng.choice([64, 128, 200, 256, 333, 512]), heads=24, dim=128)
    if kind == 'qk':
        return dict(kind=kind, rows=_span(rng, 500, 100000), heads=24, dim=128)
    if kind == 'split':
        return dict(kind=kind, rows=_span(rng, 200, 13000), local=_span(rng, 300, 13000), far=_span(rng, 300, 13000),
                    heads=rng.choice([16, 24, 8]), dim=128)
    if kind == 'frames':
        n = rng.randint(2, 16)
        return dict(kind=kind, lengths=_text([rng.randint(2, 15) for _ in range(n)]), tokens=_span(rng, 60, 1590),
                    width=rng.choice([2048, 2048, 3072]), budget=rng.randint(2, 6),
                    pool=rng.choice(['all', 'all', 'boundary']))
    if kind == 'packed':
        n = rng.randint(1, 24)
        return dict(kind=kind, q=_text([_span(rng, 1, 1500) for _ in range(n)]),
                    k=_text([_span(rng, 1, 1500) for _ in range(n)]), heads=rng.choice([16, 24, 8]),
                    dim=rng.choice([128, 128, 64]))
    if kind == 'dense':
        rows = _span(rng, 100, 8000)
        return dict(kind=kind, batch=rng.randint(1, 4), q_rows=rows,
                    k_rows=rows if rng.random() < 0.5 else _span(rng, 64, 8000), heads=rng.choice([12, 16]),
                    dim=rng.choice([64, 64, 128]))
    n = rng.randint(1, 4)
    return dict(kind='dit', lengths=_text([rng.randint(3, 6) for _ in range(n)]),
                grid=f'{rng.randint(6, 13)}x{rng.randint(8, 20)}', text=rng.choice([64, 128, 333]),
                halo=rng.choice([1, 2]), sides=rng.choice(['adj', 'prev', 'next']), blocks=rng.randint(1, 2))


# ---------------------------------------------------------------------------------------------------------------------
# sizes of a case

def _ints(text):
    return [int(x) for x in text.split(',')]


def _tokens(case):
    a, b = case['grid'].split('x')
    return int(a) * int(b)


def _ranges(lengths):
    out, at = [], 0
    for n in lengths:
        out.append((at, at + n))
        at += n
    return out


def _extra(case):
    """scene -> the representatives outside it"""
    reps = _ints(case['reps'])
    return {j: [f for f in reps if not a <= f < b] for j, (a, b) in enumerate(_ranges(_ints(case['lengths'])))}


def _halo(ranges, j, halo, sides):
    out = []
    if j > 0 and sides != 'next':
        a, b = ranges[j - 1]
        out += range(max(a, b - halo), b)
    if j + 1 < len(ranges) and sides != 'prev':
        a, b = ranges[j + 1]
        out += range(a, min(b, a + halo))
    return out


def _shared(case, j):
    """the frames scene j reads beyond its own, in order: halo, then the representatives"""
    ranges = _ranges(_ints(case['lengths']))
    halo = _halo(ranges, j, case['halo'], case['sides'])
    return halo + [f for f in _extra(case)[j] if f not in halo]


def _groups(case):
    """(boundary keys, groups of like keys) of a memory case"""
    B = sum(min(n, 2) for n in _ints(case['lengths'])) * _tokens(case)
    return B, max(2, min(3 * case['budget'], B // 6))


def work(case):
    kind = case['kind']
    if kind in ('scene', 'memory'):
        lengths, T, counts = _ints(case['lengths']), _tokens(case), _ints(case['counts'])
        H, D = case['heads'], case['dim']
        rows = sum(lengths) * T + sum(counts)
        flops = 0
        for j, n in enumerate(lengths):
            own = n * T + counts[j]
            flops += 4 * counts[j] * own * H * D
            if kind == 'scene':
                flops += 4 * n * T * (own + len(_shared(case, j)) * T) * H * D
            else:
                far = case['budget'] * (len(lengths) - 1) // len(lengths)
                flops += 4 * n * T * (own + far) * H * D
        nbytes = 4 * rows * H * D * 2
        if kind == 'scene' and not case['rotated']:
            nbytes += 2 * sum(lengths) * T * D * 4
        if kind == 'memory':
            flops += 2 * _groups(case)[0] * case['budget'] * H * D
            nbytes += 2 * case['budget'] * H * D * 4
        return dict(bytes=nbytes, flops=flops)
    if kind == 'cross':
        n, width = sum(_ints(case['lengths'])) * case['tokens'], case['heads'] * case['dim']
        text = len(_ints(case['lengths'])) * case['text']
        return dict(bytes=2 * (n + text) * width * 2, flops=4 * n * case['text'] * width)
    if kind == 'qk':
        n, width = case['rows'], case['heads'] * case['dim']
        return dict(bytes=4 * n * width * 2 + 2 * n * case['dim'] * 4, flops=2 * n * width * 7)
    if kind == 'split':
        n, width, keys = case['rows'], case['heads'] * case['dim'], case['local'] + case['far']
        return dict(bytes=n * width * 2 + 2 * keys * width * 2 + n * width * 4 + n * case['heads'] * 4,
                    flops=4 * n * keys * width)
    if kind == 'frames':
        frames, width = sum(_ints(case['lengths'])), case['width']
        return dict(bytes=frames * case['tokens'] * width * 2 + frames * width * 4,
                    flops=frames * case['tokens'] * width)
    if kind == 'packed':
        q, k, width = _ints(case['q']), _ints(case['k']), case['heads'] * case['dim']
        return dict(bytes=2 * (sum(q) + sum(k)) * width * 2, flops=4 * sum(a * b for a, b in zip(q, k)) * width)
    if kind == 'dense':
        width = case['heads'] * case['dim']
        return dict(bytes=2 * case['batch'] * (case['q_rows'] + case['k_rows']) * width * 2,
                    flops=4 * case['batch'] * case['q_rows'] * case['k_rows'] * width)
    lengths, T, d, ffn = _ints(case['lengths']), _tokens(case), 3072, 14336
    S, text, ranges = sum(lengths) * T, len(lengths) * case['text'], _ranges(lengths)
    block = 6 * 2 * S * d * d + 2 * 2 * text * d * d + 2 * 2 * S * d * ffn
    for j, n in enumerate(lengths):
        keys = (n + len(_halo(ranges, j, case['halo'], case['sides']))) * T
        block += 4 * n * T * (keys + case['text']) * d
    ends = 2 * 2 * S * d * 192 + 2 * text * d * (4096 + d)
    weights = case['blocks'] * (8 * d * d + 2 * d * ffn) + 2 * d * 192 + d * (4096 + d) + d * (256 + d + 6 * d)
    return dict(bytes=2 * weights + 2 * 2 * S * 192 + 2 * text * 4096, flops=case['blocks'] * block + ends)


def tolerance(case):
    kind = case['kind']
    if kind == 'qk':
        return dict(rel=4e-3)                    # bf16 results: a few elements fall on the other side of a rounding
    if kind == 'frames':
        return dict(rel=1e-5)                    # fp32 sums; the chosen frames are the same
    if kind == 'dit':
        return dict(rel=2e-2)                    # bf16 through two blocks
    return dict(rel=1e-2)                        # bf16 probabilities and outputs


# ---------------------------------------------------------------------------------------------------------------------
# inputs

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV).to(torch.bfloat16)


def _rope_table(frames, grid, D, theta=1e4):
    """the 3D rotary table of a video latent: temporal, height and width angles on separate pair groups of a head"""
    a, b = (int(x) for x in grid.split('x'))
    f, y, x = torch.meshgrid(torch.arange(frames), torch.arange(a), torch.arange(b), indexing='ij')
    nt, ny = D // 8, 3 * D // 16
    groups = [(f, nt), (y, ny), (x, D // 2 - nt - ny)]
    ang = torch.cat([p.reshape(-1, 1).float() * (theta ** (-torch.arange(n).float() / n)) for p, n in groups], 1)
    return tuple(t.repeat_interleave(2, 1).contiguous().to(DEV) for t in (ang.cos(), ang.sin()))


def _scene_positions(case):
    """temporal position of every frame under scene RoPE: its place in its scene, one up after the first scene"""
    out = []
    for j, n in enumerate(_ints(case['lengths'])):
        out += [i + (j > 0) for i in range(n)]
    return out


def _table_frames(case):
    lengths = _ints(case['lengths'])
    return max(sum(lengths), max(n + 1 + len(_shared(case, j)) for j, n in enumerate(lengths)))


def _rotate(x, cos, sin, rows):
    """rows of x [n, H, D] rotated at the given rows of the table, in float64"""
    x, c, s = x.double(), cos[rows].double()[:, None], sin[rows].double()[:, None]
    even, odd = x[..., 0::2], x[..., 1::2]
    turned = torch.stack([-odd, even], -1).flatten(-2)
    return x * c + turned * s


def _token_rows(positions, T):
    return (torch.as_tensor(positions, device=DEV)[:, None] * T + torch.arange(T, device=DEV)).flatten()


def _scene_inputs(case, seed):
    g = _gen(seed)
    S, Le = sum(_ints(case['lengths'])) * _tokens(case), sum(_ints(case['counts'])) + case['pad']
    H, D = case['heads'], case['dim']
    q, k, v = (_randn(g, S, H, D) for _ in range(3))
    eq, ek, ev = (_randn(g, Le, H, D) for _ in range(3))
    cos, sin = _rope_table(_table_frames(case), case['grid'], D)
    if case['rotated']:
        rows = _token_rows(_scene_positions(case), _tokens(case))
        q, k = (_rotate(x, cos, sin, rows).to(torch.bfloat16) for x in (q, k))
    return q, k, v, eq, ek, ev, cos, sin


def _memory_inputs(case, seed):
    """q, k, v, eq, ek, ev, and for a warm call the previous step's centroids. The boundary frames' keys come in groups
    of like neighbours, as patches of a frame do; the previous step's groups lay elsewhere."""
    g = _gen(seed)
    lengths, T, H, D = _ints(case['lengths']), _tokens(case), case['heads'], case['dim']
    S, Le = sum(lengths) * T, sum(_ints(case['counts']))
    q, k, v = (_randn(g, S, H, D) for _ in range(3))
    eq, ek, ev = (_randn(g, Le, H, D) for _ in range(3))
    B, n = _groups(case)
    centre = torch.randn(n, H, D, generator=g, device=DEV)
    group = torch.arange(B, device=DEV) * n // B
    rows = _boundary_rows(case)[0]
    k[rows] = (0.8 * centre[group] + 0.6 * torch.randn(B, H, D, generator=g, device=DEV)).to(torch.bfloat16)
    c0 = None
    if case['warm']:
        M = min(case['budget'], B)
        before = 0.8 * centre + 0.6 * torch.randn(n, H, D, generator=g, device=DEV)
        before = F.normalize(before, dim=-1)
        own = torch.arange(n, device=DEV) * M // n
        c0 = torch.zeros(M, H, D, device=DEV).index_add_(0, own, before)
        c0 = (c0 / torch.bincount(own, minlength=M).clamp_min(1)[:, None, None]).transpose(0, 1).contiguous()
    return q, k, v, eq, ek, ev, c0


def _boundary_rows(case):
    """(token rows of every scene's first and last frame, the scene of each row)"""
    T, rows, scene = _tokens(case), [], []
    for j, (a, b) in enumerate(_ranges(_ints(case['lengths']))):
        for f in dict.fromkeys((a, b - 1)):
            rows.append(torch.arange(f * T, (f + 1) * T))
            scene += [j] * T
    return torch.cat(rows).to(DEV), torch.tensor(scene, device=DEV)


def _qk_inputs(case, seed):
    g = _gen(seed)
    n, C, D = case['rows'], case['heads'] * case['dim'], case['dim']
    q, k = _randn(g, 1, n, C), _randn(g, 1, n, C)
    wq, wk = (1 + 0.1 * torch.randn(C, generator=g, device=DEV) for _ in range(2))
    ang = torch.rand(n, D // 2, generator=g, device=DEV) * 2 * math.pi
    cos, sin = (t.repeat_interleave(2, 1)[None, :, None].contiguous() for t in (ang.cos(), ang.sin()))
    return q, k, wq.to(torch.bfloat16), wk.to(torch.bfloat16), cos, sin


def _split_inputs(case, seed):
    g = _gen(seed)
    H, D = case['heads'], case['dim']
    return [_randn(g, n, H, D) for n in (case['rows'], case['local'], case['local'], case['far'], case['far'])]


def _frames_inputs(case, seed):
    """hidden states of frames that look alike within a scene"""
    g = _gen(seed)
    lengths, T, C = _ints(case['lengths']), case['tokens'], case['width']
    scene = torch.repeat_interleave(torch.arange(len(lengths)), torch.tensor(lengths)).to(DEV)
    look = torch.randn(len(lengths), C, generator=g, device=DEV)[scene]
    look = look + 0.4 * torch.randn(sum(lengths), C, generator=g, device=DEV)
    hs = torch.empty(sum(lengths) * T, C, dtype=torch.bfloat16, device=DEV)
    for f in range(sum(lengths)):
        hs[f * T:(f + 1) * T] = (look[f] + torch.randn(T, C, generator=g, device=DEV)).to(torch.bfloat16)
    return hs


def _dit_parts(case, seed):
    from onereel_amd import wan_dit as WD
    from onereel_amd.layout import SceneLayout
    g = _gen(seed)
    lengths, T = _ints(case['lengths']), _tokens(case)
    a, b = (int(x) for x in case['grid'].split('x'))
    cfg = WD.DiTConfig(blocks=case['blocks'])
    lay = SceneLayout(lengths, halo=case['halo'], sides=case['sides'])
    model = WD.WanDiT(cfg, lay, T, case['text'], torch.device(DEV), seed=seed)
    latent = _randn(g, sum(lengths) * T, cfg.in_channels * cfg.patch)
    text = _randn(g, len(lengths) * case['text'], cfg.text_dim)
    rotary = tuple(x.to(DEV) for x in WD.wan_rope_table(sum(lengths), a, b, cfg.dim // cfg.heads))
    return model, latent, text, rotary


def prepare(case, seed):
    kind = case['kind']
    state = dict(case=case)
    if kind in ('scene', 'memory'):
        from onereel_amd import hunyuan15 as HY
        from onereel_amd.layout import SceneLayout
        lengths, counts = _ints(case['lengths']), _ints(case['counts'])
        if kind == 'scene':
            *x, cos, sin = _scene_inputs(case, seed)
            lay = SceneLayout(lengths, halo=case['halo'], sides=case['sides'], extra=_extra(case))
            ctx = HY.Context(lay, cfg=False, shared_pos=case['position'], scene_rope=True, T=_tokens(case))
            state.update(cos=cos, sin=sin)
            ctx._rot_full = (cos, sin)           # what Processor.__call__ leaves for Processor.scene
        else:
            *x, c0 = _memory_inputs(case, seed)
            ctx = HY.Context(SceneLayout(lengths, halo=0), cfg=False, scene_rope=True, memory=case['budget'],
                             T=_tokens(case))
            state.update(c0=c0, memory=HY.memory_attention(ctx).memory)
        ctx.counts, ctx.fwd = {True: counts}, 1
        state.update(x=x, proc=HY.Processor(ctx, 0))
    elif kind == 'cross':
        from onereel_amd import wan as W
        from onereel_amd.layout import SceneLayout
        g = _gen(seed)
        lengths, H, D = _ints(case['lengths']), case['heads'], case['dim']
        ctx = W.Context(SceneLayout(lengths, halo=0), T=case['tokens'], text_len=case['text'])
        n, m = sum(lengths) * case['tokens'], len(lengths) * case['text']
        state.update(ctx=ctx, x=[_randn(g, r, H, D) for r in (n, m, m)])
    elif kind == 'qk':
        state.update(x=_qk_inputs(case, seed))
    elif kind == 'split':
        from onereel_amd import attention as A
        n = case['rows']
        state.update(x=_split_inputs(case, seed), cu_q=A.cu_seqlens([n], DEV),
                     cu_k=[A.cu_seqlens([case[w]], DEV) for w in ('local', 'far')])
    elif kind == 'frames':
        from onereel_amd.frame_memory import FrameMemory
        from onereel_amd.layout import SceneLayout
        lay = SceneLayout(_ints(case['lengths']), halo=0)
        fm = FrameMemory(budget=case['budget'], candidates=case['pool'])
        fm.reset(lay, 30)
        frame = torch.arange(lay.n_frames * case['tokens'], device=DEV) // case['tokens']
        state.update(fm=fm, frame=frame, hs=_frames_inputs(case, seed))
    elif kind == 'packed':
        state.update(x=_packed_inputs(case, seed))
    elif kind == 'dense':
        state.update(x=_dense_inputs(case, seed))
    else:
        model, latent, text, rotary = _dit_parts(case, seed)
        state.update(model=model, latent=latent, text=text, rotary=rotary)
    return state


def _packed_inputs(case, seed):
    g = _gen(seed)
    H, D = case['heads'], case['dim']
    return [tuple(_randn(g, n, H, D) for n in (a, b, b)) for a, b in zip(_ints(case['q']), _ints(case['k']))]


def _dense_inputs(case, seed):
    g = _gen(seed)
    return [_randn(g, case['batch'], n, case['heads'], case['dim'])
            for n in (case['q_rows'], case['k_rows'], case['k_rows'])]


# ---------------------------------------------------------------------------------------------------------------------
# one pass

def run(state):
    case = state['case']
    kind = case['kind']
    if kind == 'scene':
        if case['rotated']:
            return state['proc'].scene(*state['x'])
        return state['proc'].scene_raw(*state['x'], state['cos'], state['sin'])
    if kind == 'memory':
        # a first step starts from no centroids, a later one from the previous step's
        memory = state['memory']
        memory.centroids = {(0, True): state['c0'].clone()} if case['warm'] else {}
        out, text = state['proc'].memory(*state['x'])
        return out, text, memory.centroids[(0, True)]
    if kind == 'cross':
        from onereel_amd import wan as W
        return W.cross_ranges(state['ctx'], *state['x'])
    if kind == 'qk':
        from onereel_amd import wan as W
        q, k, wq, wk, cos, sin = state['x']
        return W._qk(q, k, wq, wk, 1e-6, cos, sin, case['heads'])
    if kind == 'split':
        from onereel_amd import attention as A
        q, k, v, fk, fv = state['x']
        n = q.shape[0]
        o, lse = A.varlen_lse(q, k, v, state['cu_q'], state['cu_k'][0], n, k.shape[0], check=False)
        far, far_lse = A.varlen_lse(q, fk, fv, state['cu_q'], state['cu_k'][1], n, fk.shape[0], check=False)
        return A.merge_lse(o.float(), lse, far, far_lse)
    if kind == 'frames':
        fm = state['fm']
        fm.collect(state['frame'], state['hs'])
        sums, counts = fm.sums[fm.layer], fm.counts[fm.layer]
        fm.finish()
        return sums, counts, fm.pending
    if kind == 'packed':
        from onereel_amd import attention as A
        return A.packed(state['x'])
    if kind == 'dense':
        from onereel_amd import attention as A
        return A.dense(*state['x'])
    return state['model'].forward(state['latent'], 500.0, state['text'], state['rotary'])


# ---------------------------------------------------------------------------------------------------------------------
# the same pass in float64 torch

def _attend(q, k, v, lse=False):
    """softmax(q k^T / sqrt(D)) v of q [n, H, D] over k / v [m, H, D], one head and a bounded score block at a time"""
    n, H, D = q.shape
    out = torch.empty(n, H, D, dtype=torch.float64, device=q.device)
    top = torch.empty(H, n, dtype=torch.float64, device=q.device)
    step = max(1, (1 << 26) // max(1, k.shape[0]))
    for h in range(H):
        kh, vh = k[:, h].double().contiguous(), v[:, h].double().contiguous()
        for a in range(0, n, step):
            s = q[a:a + step, h].double().contiguous() @ kh.T.contiguous() * D ** -0.5
            if lse:
                top[h, a:a + step] = torch.logsumexp(s, 1)
            out[a:a + step, h] = torch.softmax(s, 1) @ vh
    return (out, top) if lse else out


def _exact_scene(case, seed):
    q, k, v, eq, ek, ev, cos, sin = _scene_inputs(case, seed)
    T, place = _tokens(case), _scene_positions(case)
    own_rows = _token_rows(place, T)
    if not case['rotated']:
        q, plain = _rotate(q, cos, sin, own_rows), _rotate(k, cos, sin, own_rows)
    else:
        plain = k.double()
    ov = torch.empty(q.shape, dtype=torch.float64, device=DEV)
    ot = torch.zeros(eq.shape, dtype=torch.float64, device=DEV)
    at = 0
    for j, ((a, b), c) in enumerate(zip(_ranges(_ints(case['lengths'])), _ints(case['counts']))):
        own, sent = slice(a * T, b * T), slice(at, at + c)
        at += c
        shared = _shared(case, j)
        ks, vs = [plain[own], ek[sent].double()], [v[own], ev[sent]]
        last = place[b - 1]
        for f in shared:
            sl = slice(f * T, (f + 1) * T)
            moved = plain[sl]
            if case['position'] == 'adjacent':
                to = last + sum(x <= f for x in shared)
                if case['rotated']:
                    d = to - place[f]
                    base = max(0, -d)
                    moved = _rotate(_rotate(k[sl], cos, -sin, _token_rows([base], T)), cos, sin,
                                    _token_rows([base + d], T))
                else:
                    moved = _rotate(k[sl], cos, sin, _token_rows([to], T))
            ks.append(moved)
            vs.append(v[sl])
        n_own = (b - a) * T + c
        keys, values = torch.cat(ks), torch.cat(vs)
        ov[own] = _attend(q[own], keys, values)
        ot[sent] = _attend(eq[sent], keys[:n_own], values[:n_own])
    return ov, ot


def _exact_memory(case, seed):
    q, k, v, eq, ek, ev, c0 = _memory_inputs(case, seed)
    T, H, D = _tokens(case), case['heads'], case['dim']
    rows, scene = _boundary_rows(case)
    B = rows.numel()
    M = min(case['budget'], B)
    x = F.normalize(k[rows].double(), dim=-1).transpose(0, 1).contiguous()
    if c0 is None:
        start = torch.linspace(0, B - 1, M).round().long().to(DEV)
        c = x[:, start].clone()
    else:
        c = c0.double()
    reps = []
    for h in range(H):
        for it in range((50 if c0 is None else 2) + 1):
            d = (x[h] ** 2).sum(1)[:, None] - 2 * x[h] @ c[h].T.contiguous() + (c[h] ** 2).sum(1)[None]
            z = d.argmin(1)
            if it == (50 if c0 is None else 2):
                break
            count = torch.bincount(z, minlength=M)
            mean = torch.zeros(M, D, dtype=torch.float64, device=DEV).index_add_(0, z, x[h])
            new = torch.where((count > 0)[:, None], mean / count.clamp_min(1)[:, None], c[h])
            if torch.allclose(new, c[h], rtol=0, atol=1e-12):
                break
            c[h] = new
        near = d.gather(1, z[:, None])[:, 0]
        order = torch.argsort(near, stable=True)
        first = torch.full((M,), B, device=DEV).scatter_reduce_(0, z[order], torch.arange(B, device=DEV), 'amin')
        reps.append(order[first[first < B]])
    ov = torch.empty(q.shape, dtype=torch.float64, device=DEV)
    ot = torch.zeros(eq.shape, dtype=torch.float64, device=DEV)
    at = 0
    for j, ((a, b), n) in enumerate(zip(_ranges(_ints(case['lengths'])), _ints(case['counts']))):
        own, sent = slice(a * T, b * T), slice(at, at + n)
        at += n
        keys, values = torch.cat([k[own], ek[sent]]), torch.cat([v[own], ev[sent]])
        ot[sent] = _attend(eq[sent], keys, values)
        for h in range(H):
            far = rows[reps[h][scene[reps[h]] != j]]
            ov[own, h:h + 1] = _attend(q[own, h:h + 1], torch.cat([keys[:, h:h + 1], k[far, h:h + 1]]),
                                       torch.cat([values[:, h:h + 1], v[far, h:h + 1]]))
    return ov, ot, c


def _exact_frames(case, seed):
    hs = _frames_inputs(case, seed)
    lengths, T, C = _ints(case['lengths']), case['tokens'], case['width']
    n = sum(lengths)
    sums = torch.stack([hs[f * T:(f + 1) * T].double().sum(0) for f in range(n)])
    feats = F.normalize(sums / T, dim=-1)
    cand = list(range(n))
    if case['pool'] == 'boundary':
        cand = sorted({f for a, b in _ranges(lengths) for f in (a, b - 1)})
    x, k = feats[torch.tensor(cand, device=DEV)], min(case['budget'], len(cand))
    centre = [0]
    for _ in range(k - 1):
        centre.append(int((1 - x @ x[centre].T.contiguous()).min(1).values.argmax()))
    c = x[centre].clone()
    for _ in range(20):
        z = (x @ c.T.contiguous()).argmax(1)
        new = torch.stack([F.normalize(x[z == i].mean(0), dim=0) if bool((z == i).any()) else c[i] for i in range(k)])
        if torch.allclose(new, c, rtol=0, atol=1e-13):
            break
        c = new
    sim = x @ c.T.contiguous()
    z = sim.argmax(1)
    reps = []
    for i in range(k):
        mine = (z == i).nonzero().flatten()
        if mine.numel():
            reps.append(cand[int(mine[sim[mine, i].argmax()])])
    return sums, torch.full((n,), float(T), dtype=torch.float64, device=DEV), sorted(reps)


def _norm_rope(x, w, eps, heads, cos=None, sin=None):
    y = x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps) * w.double()
    y = y.unflatten(-1, (heads, -1))
    if cos is None:
        return y
    c, s = cos.reshape(-1, 1, y.shape[-1]).double()[..., 0::2], sin.reshape(-1, 1, y.shape[-1]).double()[..., 1::2]
    a, b = y[..., 0::2], y[..., 1::2]
    return torch.stack([a * c - b * s, a * s + b * c], -1).flatten(-2)


def _exact_dit(case, seed):
    model, latent, text, (cos, sin) = _dit_parts(case, seed)
    cfg, lengths, T = model.cfg, _ints(case['lengths']), _tokens(case)
    ranges, H, eps = _ranges(lengths), cfg.heads, cfg.eps

    def lin(layer, x):
        return x @ layer.weight.double().T.contiguous() + layer.bias.double()

    def norm(x):
        return F.layer_norm(x, (cfg.dim,), eps=eps)

    half = cfg.freq_dim // 2
    freq = torch.exp(-math.log(10000.0) * torch.arange(half, device=DEV, dtype=torch.float64) / half)
    temb = lin(model.time_out, F.silu(lin(model.time_in, torch.cat([torch.cos(500.0 * freq), torch.sin(500.0 * freq)]))))
    temb6 = lin(model.time_proj, F.silu(temb)).view(6, cfg.dim)
    ctx = lin(model.text_out, F.gelu(lin(model.text_in, text.double()), approximate='tanh'))
    x = lin(model.patch_embed, latent.double())
    for blk in model.blocks:
        shift, scale, gate, c_shift, c_scale, c_gate = (blk.scale_shift_table.double() + temb6).chunk(6, 0)
        n = norm(x) * (1 + scale) + shift
        at = blk.attn1
        q = _norm_rope(lin(at.to_q, n), at.norm_q.weight, at.norm_q.eps, H, cos, sin)
        k = _norm_rope(lin(at.to_k, n), at.norm_k.weight, at.norm_k.eps, H, cos, sin)
        v = lin(at.to_v, n).unflatten(-1, (H, -1))
        o = []
        for j, (a, b) in enumerate(ranges):
            frames = list(range(a, b)) + _halo(ranges, j, case['halo'], case['sides'])
            keys = _token_rows(frames, T)
            o.append(_attend(q[a * T:b * T], k[keys], v[keys]))
        x = x + lin(at.to_out[0], torch.cat(o).flatten(1)) * gate
        n = norm(x) * blk.norm2_w.double() + blk.norm2_b.double()
        at = blk.attn2
        q = _norm_rope(lin(at.to_q, n), at.norm_q.weight, at.norm_q.eps, H)
        k = _norm_rope(lin(at.to_k, ctx), at.norm_k.weight, at.norm_k.eps, H)
        v = lin(at.to_v, ctx).unflatten(-1, (H, -1))
        L = case['text']
        o = [_attend(q[a * T:b * T], k[j * L:(j + 1) * L], v[j * L:(j + 1) * L]) for j, (a, b) in enumerate(ranges)]
        x = x + lin(at.to_out[0], torch.cat(o).flatten(1))
        n = norm(x) * (1 + c_scale) + c_shift
        x = x + lin(blk.ffn_out, F.gelu(lin(blk.ffn_in, n), approximate='tanh')) * c_gate
    shift, scale = (model.scale_shift_table.double() + temb[None]).chunk(2, 0)
    return lin(model.proj_out, norm(x) * (1 + scale) + shift)


@torch.no_grad()
def exact(case, seed):
    kind = case['kind']
    if kind == 'scene':
        return _exact_scene(case, seed)
    if kind == 'memory':
        return _exact_memory(case, seed)
    if kind == 'cross':
        g = _gen(seed)
        lengths, H, D, L, T = _ints(case['lengths']), case['heads'], case['dim'], case['text'], case['tokens']
        q, k, v = (_randn(g, r, H, D) for r in (sum(lengths) * T, len(lengths) * L, len(lengths) * L))
        return torch.cat([_attend(q[a * T:b * T], k[j * L:(j + 1) * L], v[j * L:(j + 1) * L])
                          for j, (a, b) in enumerate(_ranges(lengths))])
    if kind == 'qk':
        q, k, wq, wk, cos, sin = _qk_inputs(case, seed)
        return tuple(_norm_rope(x[0].double(), w, 1e-6, case['heads'], cos, sin)[None] for x, w in ((q, wq), (k, wk)))
    if kind == 'split':
        q, k, v, fk, fv = _split_inputs(case, seed)
        return _attend(q, torch.cat([k, fk]), torch.cat([v, fv]), lse=True)
    if kind == 'frames':
        return _exact_frames(case, seed)
    if kind == 'packed':
        return tuple(_attend(q, k, v) for q, k, v in _packed_inputs(case, seed))
    if kind == 'dense':
        q, k, v = _dense_inputs(case, seed)
        return torch.stack([_attend(q[b], k[b], v[b]) for b in range(case['batch'])])
    return _exact_dit(case, seed)
