"""The work that users of vnlbhip have it do, as cases that can be timed and
compared: whole clips through vnlbhip.Basic / vnlbhip.Final in both forms,
output frames one at a time, host clips, motion-guided search, replayed
stages of small clips, and one training batch of the candidate proposer.

A case names a profile (the vnlb arguments), a form and a path (the entry
points it goes through) and the clip's size.  exact() restates the VNLB
stages and the proposer network in float64 with torch alone.
"""
import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "vapoursynth-vnlb_amd"))

import vnlbhip  # noqa: E402
from vnlbhip import proposer as learned  # noqa: E402
from vnlbhip.flow import MVToolsAnalysis, VectorClip  # noqa: E402
from vnlbhip.params import BASIC, FINAL, parse_stage_parameters  # noqa: E402

DEV = "cuda:0"

# vnlb arguments of both stages; "final" holds what Final takes instead.
PROFILES = {
    # The plugin's own defaults: 8x8x1 patches, 8 neighbours, step 8, 19x19 windows over 3 frames.
    "defaults": dict(sigma=10),
    # The denoising configuration for grey clips: 8x8x2 patches, 16 neighbours, step 4, 5 frames.
    "temporal": dict(sigma=20, block_size=8, block_step=4, group_size=16, bm_range=9, patch_time=2, radius=2, rank=16,
                     tau=0),
    # The benchmark configuration: coupled YUV, groups that widen up to four times.
    "chroma": dict(sigma=15, block_size=8, block_step=4, group_size=16, bm_range=9, patch_time=2, radius=2, rank=16,
                   tau=200, cap_factor=4.0, model_cap_factor=1.0, chroma=1),
    # The same with a truncated model, which denoises more.
    "chroma_rank4": dict(sigma=15, block_size=8, block_step=4, group_size=16, bm_range=9, patch_time=2, radius=2,
                         rank=4, tau=200, cap_factor=4.0, model_cap_factor=1.0, chroma=1),
    # 25x25 windows on grey clips.
    "wide": dict(sigma=20, block_size=8, block_step=4, group_size=16, bm_range=12, patch_time=2, radius=2, rank=16,
                 tau=0),
    # The 4K configuration: 25x25 windows over 7 frames.
    "full": dict(sigma=25, block_size=8, block_step=4, group_size=16, bm_range=12, patch_time=2, radius=3, rank=16,
                 tau=200, cap_factor=4.0, model_cap_factor=1.0, chroma=1),
    # One model per channel.
    "uncoupled": dict(sigma=15, block_size=8, block_step=6, group_size=12, bm_range=5, patch_time=1, radius=1, rank=8,
                      chroma=0),
    # The tuned profile of the reference's tests: large groups, rank 39.
    "tuned": dict(sigma=20, block_size=8, block_step=4, bm_range=9, patch_time=2, radius=1, rank=39, tau=0,
                  group_size=100, final=dict(group_size=60)),
}

# Share of the anchors whose group is filtered (the others are skipped
# because their patch was already denoised), at least.
ACTIVE = 0.25


def listed():
    def clip(name, profile, form, width, height, frames, channels, path="clip"):
        return dict(name=name, path=path, profile=profile, form=form, width=width, height=height, frames=frames,
                    channels=channels)

    return [
        # Trying the filter on a small grey clip with every argument at its default: latency and launches.
        clip("grays_256_defaults", "defaults", "plain", 256, 256, 5, 1),
        # An interactive preview: a small clip denoised again and again in the same buffers, stages replayed.
        clip("yuv_preview_replayed", "chroma", "fast", 320, 180, 5, 3, path="replay"),
        # One batch of the candidate proposer's training: features, forward, loss and backward.
        dict(name="proposer_batch_64", path="train", width=480, height=270, frames=6, anchors=64, group=128),
        # A numpy clip through host memory, ragged size, truncated model.
        clip("yuv_host_rank4", "chroma_rank4", "fast", 501, 283, 6, 3, path="host"),
        # Odd-sized YUV with one model per channel, the default form.
        clip("yuv_odd_uncoupled", "uncoupled", "plain", 717, 403, 7, 3),
        # The tuned profile's large groups and models.
        clip("gray_tuned_rank39", "tuned", "plain", 160, 120, 5, 1),
        # A standard-definition grey clip whose search follows motion vectors.
        clip("gray_sd_guided", "temporal", "plain", 720, 480, 6, 1, path="guided"),
        # A standard-definition grey clip with wide windows.
        clip("gray_sd_wide", "wide", "fast", 720, 576, 10, 1),
        # Frames asked for one after the other, as a player or an encoder pulls them.
        clip("yuv_720p_frames", "chroma", "fast", 1280, 720, 8, 3, path="frames"),
        # An ordinary clip in the default form.
        clip("yuv_720p_plain", "chroma", "plain", 1280, 720, 8, 3),
        # The benchmark clip.
        clip("yuv_1080p_fast", "chroma", "fast", 1920, 1080, 16, 3),
        # The largest frames.
        clip("yuv_2160p_fast", "full", "fast", 3840, 2160, 5, 3),
    ]


# (path, profiles, forms, channels, width range, frame range) of drawn cases.
KINDS = [
    ("clip", ("defaults",), ("plain", "fast"), (1, 3), (96, 1920), (3, 12)),
    ("clip", ("temporal", "wide"), ("plain", "fast"), (1,), (96, 1280), (4, 10)),
    ("clip", ("chroma", "chroma_rank4"), ("fast",), (3,), (160, 1920), (4, 16)),
    ("clip", ("chroma", "chroma_rank4"), ("plain",), (3,), (160, 1280), (4, 8)),
    ("clip", ("full",), ("fast",), (3,), (320, 2560), (4, 7)),
    ("clip", ("uncoupled",), ("plain", "fast"), (3,), (96, 1280), (3, 8)),
    ("clip", ("tuned",), ("plain", "fast"), (1,), (96, 200), (4, 6)),
    ("replay", ("chroma", "temporal"), ("fast",), (1, 3), (96, 480), (4, 6)),
    ("host", ("chroma_rank4", "temporal"), ("plain", "fast"), (1, 3), (160, 720), (4, 8)),
    ("guided", ("temporal",), ("plain", "fast"), (1,), (160, 960), (4, 8)),
    ("frames", ("chroma", "temporal"), ("fast", "plain"), (1, 3), (160, 1280), (4, 8)),
    ("train", (), (), (), (160, 960), (4, 8)),
]


def draw(rng):
    path, profiles, forms, channels, width, frames = rng.choice(KINDS)
    w = int(round(math.exp(rng.uniform(math.log(width[0]), math.log(width[1])))))
    h = max(72, int(round(w * rng.uniform(0.5, 0.8))))
    f = rng.randint(*frames)
    if path == "train":
        return dict(path=path, width=w, height=h, frames=f, anchors=rng.choice((16, 32, 64, 96, 128)), group=128)
    return dict(path=path, profile=rng.choice(profiles), form=rng.choice(forms), width=w, height=h, frames=f,
                channels=rng.choice(channels))


# --- inputs ---------------------------------------------------------------

def _generator(seed):
    gen = torch.Generator(device="cpu")
    gen.manual_seed(int(seed))
    return gen


def _clip(case, seed):
    """A noisy clip [frames, channels, height, width] on the GPU: luma of
    three gratings and six rectangles under a random sub-pixel translation
    per frame, smooth chroma, Gaussian noise of the profile's sigma.  Returns
    (clip, translations)."""
    gen = _generator(seed)

    def uniform(low, high, n=1):
        return (torch.rand(n, generator=gen, dtype=torch.float64) * (high - low) + low).tolist()

    width, height, frames = case["width"], case["height"], case["frames"]
    channels = case.get("channels", 1)
    cw, ch = width + 8, height + 8
    yy = torch.arange(ch, device=DEV, dtype=torch.float64)[:, None]
    xx = torch.arange(cw, device=DEV, dtype=torch.float64)[None, :]

    def grating(theta, period, phase):
        return torch.sin(2.0 * math.pi * (xx * math.cos(theta) + yy * math.sin(theta)) / period + phase)

    planes = []
    luma = sum(grating(*uniform(0, math.pi), *uniform(4, 32), *uniform(0, 2 * math.pi)) for _ in range(3))
    luma = (luma / 3.0 + 1.0) * 0.5
    for _ in range(6):
        rw, rh = int(uniform(cw / 16, cw / 3)[0]), int(uniform(ch / 16, ch / 3)[0])
        x0, y0 = int(uniform(0, cw - rw)[0]), int(uniform(0, ch - rh)[0])
        luma[y0:y0 + rh, x0:x0 + rw] = uniform(0, 1)[0]
    planes.append(luma)
    for _ in range(channels - 1):
        planes.append(0.5 + 0.1 * grating(*uniform(0, math.pi), *uniform(64, 256), *uniform(0, 2 * math.pi)))
    moves = [tuple(uniform(-2.0, 2.0, 2)) for _ in range(frames)]
    out = torch.empty((frames, channels, height, width), device=DEV)
    for t, (ox, oy) in enumerate(moves):
        x0, y0 = math.floor(ox) + 3, math.floor(oy) + 3
        ax, ay = ox - math.floor(ox), oy - math.floor(oy)
        for c, p in enumerate(planes):
            a = p[y0:y0 + height + 1, x0:x0 + width + 1]
            rows = a[:, :-1] * (1 - ax) + a[:, 1:] * ax
            out[t, c] = (rows[:-1] * (1 - ay) + rows[1:] * ay).float()
    noise = torch.Generator(device=DEV)
    noise.manual_seed(int(seed))
    sigma = PROFILES[case["profile"]]["sigma"] if "profile" in case else 20
    out += torch.randn(out.shape, generator=noise, device=DEV) * (sigma / 255.0)
    return out, moves


def _vectors(case, seed, moves, backwards):
    """An MVTools vector clip (8x8 blocks overlapping by 4, half pixels) of
    the clip's translations, one block in eight off by a few pixels."""
    gen = torch.Generator(device="cpu")
    gen.manual_seed(int(seed) * 2 + int(backwards))
    width, height, frames = case["width"], case["height"], case["frames"]
    nx, ny = (width - 4) // 4, (height - 4) // 4
    vectors = np.zeros((frames, ny, nx, 2), np.int32)
    valid = np.ones(frames, np.uint8)
    for f in range(frames):
        g = f + 1 if backwards else f - 1
        if not 0 <= g < frames:
            valid[f] = 0
            continue
        for axis in (0, 1):
            vectors[f, :, :, axis] = round(2.0 * (moves[f][axis] - moves[g][axis]))
        off = torch.randint(-8, 9, (ny, nx, 2), generator=gen).numpy()
        stray = torch.rand((ny, nx, 1), generator=gen).numpy() < 0.125
        vectors[f] += np.where(stray, off, 0).astype(np.int32)
    analysis = MVToolsAnalysis(block_size_x=8, block_size_y=8, pel=2, level_count=1, delta_frame=1,
                               backwards=backwards, width=width, height=height, overlap_x=4, overlap_y=4,
                               block_count_x=nx, block_count_y=ny, bits_per_sample=8, chroma_ratio_x=1,
                               chroma_ratio_y=1, padding_x=8, padding_y=8)
    return VectorClip(analysis, vectors, valid)


def _arguments(case):
    basic = {k: v for k, v in PROFILES[case["profile"]].items() if k != "final"}
    return basic, {**basic, **PROFILES[case["profile"]].get("final", {})}


def _training_rows(case, seed):
    """Packed anchors and candidates of a training batch and its targets:
    per anchor 16 near positives, then candidates all over a 25x25 window."""
    gen = _generator(seed + 7)
    anchors, group = case["anchors"], case["group"]
    width, height, frames = case["width"], case["height"], case["frames"]

    def integers(low, high, shape):
        return torch.randint(low, high, shape, generator=gen)

    ax, ay = integers(12, width - 20, (anchors, 1)), integers(12, height - 20, (anchors, 1))
    af = integers(0, frames - 1, (anchors, 1))
    dx, dy = integers(-12, 13, (anchors, group)), integers(-12, 13, (anchors, group))
    dx[:, :16] = dx[:, :16] // 4
    dy[:, :16] = dy[:, :16] // 4
    cf = torch.clamp(af + integers(-2, 3, (anchors, group)), 0, frames - 2)
    a = (ax | (ay << 12) | (af << 24)).expand(anchors, group)
    c = (ax + dx) | ((ay + dy) << 12) | (cf << 24)
    targets = torch.zeros((anchors, group))
    targets[:, :16] = 1.0 / 16.0
    return (a.reshape(-1).to(torch.int32).to(DEV), c.reshape(-1).to(torch.int32).to(DEV),
            targets.reshape(-1).to(DEV))


def _weights(seed):
    """Proposer weights after some training: He-uniform layers, small biases."""
    rng = np.random.default_rng(seed)

    def uniform(limit, n):
        return rng.uniform(-limit, limit, n)

    return np.concatenate([uniform(math.sqrt(6 / 128), 256 * 128), uniform(0.05, 256),
                           uniform(math.sqrt(6 / 256), 256 * 256), uniform(0.05, 256),
                           uniform(math.sqrt(6 / 256), 256), uniform(0.05, 1)]).astype(np.float32)


def prepare(case, seed):
    clip, moves = _clip(case, seed)
    if case["path"] == "train":
        net = learned.Proposer(0, seed=seed)
        net.set_params(_weights(seed))
        anchors, candidates, targets = _training_rows(case, seed)
        return dict(case=case, clip=clip, net=net, anchors=anchors, candidates=candidates, targets=targets)
    basic, final = _arguments(case)
    state = dict(case=case, clip=clip, basic_args=basic, final_args=final)
    if case["path"] in ("replay", "frames"):
        context = vnlbhip.Context(0)
        context.set_form(case["form"])
        bp, fp = parse_stage_parameters(BASIC, basic), parse_stage_parameters(FINAL, final)
        state.update(context=context, bp=bp, fp=fp, basic=torch.empty_like(clip), final=torch.empty_like(clip))
        if case["path"] == "replay":
            context.set_graph(True)
        else:
            shape = tuple(clip.shape)
            state["caches"] = (context.frame_cache(BASIC, bp, *shape), context.frame_cache(FINAL, fp, *shape))
    elif case["path"] == "host":
        state["clip"] = clip.cpu().numpy()
    elif case["path"] == "guided":
        state["mvfw"] = _vectors(case, seed, moves, False)
        state["mvbw"] = _vectors(case, seed, moves, True)
    return state


def run(state):
    case, clip = state["case"], state["clip"]
    path = case["path"]
    if path == "train":
        net = state["net"]
        x = net.features(clip, 2, state["anchors"], state["candidates"])
        grads, losses = net.gradients(x, state["targets"], case["group"])
        return {"scores": net.scores(x), "grads": grads, "losses": losses}
    if path == "replay":
        context = state["context"]
        basic = context.stage(BASIC, state["bp"], clip, out=state["basic"])
        final = context.stage(FINAL, state["fp"], clip, basic, out=state["final"])
    elif path == "frames":
        basic, final = state["basic"], state["final"]
        for cache in state["caches"]:  # the clip is new to them
            cache.invalidate()
        for t in range(case["frames"]):
            state["caches"][0].render(t, clip, out=basic[t])
        for t in range(case["frames"]):
            state["caches"][1].render(t, clip, basic, out=final[t])
    else:
        extra = {k: state[k] for k in ("mvfw", "mvbw") if k in state}
        basic = vnlbhip.Basic(clip, **state["basic_args"], **extra, form=case["form"])
        final = vnlbhip.Final(clip, basic, **state["final_args"], **extra, form=case["form"])
    return {"basic": basic, "final": final}


# --- what a pass cannot do without ----------------------------------------

def work(case):
    """The clip (and, for Final, the Basic estimate) read once, the outputs
    written once; two operations per sample of every candidate distance, and
    the group models and estimates of the anchors that are filtered."""
    if case["path"] == "train":
        rows = case["anchors"] * case["group"]
        forward = 2.0 * rows * (128 * 256 + 256 * 256 + 256)
        return {"bytes": case["frames"] * case["width"] * case["height"] * 4.0 + rows * 16.0, "flops": 4.0 * forward}
    width, height, frames, channels = case["width"], case["height"], case["frames"], case["channels"]
    flops = 0.0
    for stage, args in zip((BASIC, FINAL), _arguments(case)):
        p = parse_stage_parameters(stage, args)
        anchors = (width / p.proc_step) * (height / p.proc_step) * (frames - p.patch_time + 1)
        candidates = p.search_window ** 2 * min(p.search_bwd + p.search_fwd + 1, frames - p.patch_time + 1)
        patch = p.patch_size ** 2 * p.patch_time
        matched = patch * (channels if stage == FINAL else 1)
        dim = patch * channels
        model = dim * p.similar * (p.similar + 1) + 4.0 * p.similar * p.rank * dim
        flops += anchors * (2.0 * candidates * matched + ACTIVE * model)
    return {"bytes": 5.0 * frames * channels * width * height * 4.0, "flops": flops}


# Largest relative errors of whole stages: four times what the stages were
# measured to be off from exact(), which takes every sum and every decision in
# float64.  Neighbours at nearly equal distances change places when sums are
# taken in another order, and with them the groups that are filtered at all;
# where the model is truncated (rank below its rows, or eigenvalues beside the
# variance threshold) components near the cut change sides too.
STAGE_ERROR = {
    "plain": {"defaults": 1e-4, "temporal": 5e-5, "chroma": 2e-5, "chroma_rank4": 4e-3, "wide": 5e-5, "full": 2e-5,
              "uncoupled": 1.2e-3, "tuned": 2e-4},
    "fast": {"defaults": 2.5e-4, "temporal": 2e-4, "chroma": 1e-4, "chroma_rank4": 4e-3, "wide": 2e-4, "full": 2e-4,
             "uncoupled": 1.2e-3, "tuned": 4e-4},
}


def tolerance(case):
    if case["path"] == "train":
        return {"rel": 1e-2, "max": 0.5}  # bf16 operands and hidden activations
    rel = STAGE_ERROR[case["form"]][case["profile"]]
    return {"rel": rel, "max": 0.3 if rel > 1e-3 else 0.05}


# --- the same in float64 ---------------------------------------------------

def _span(center, axis, patch, window):
    """The search range around center, shifted into the frame."""
    half, top = (window - 1) // 2, axis - patch
    start, end = center - half, center + half
    shift = start.clamp(max=0) + (end - top).clamp(min=0)
    return (start - shift).clamp(min=0), (end - shift).clamp(max=top)


def _schedule(p, anchor, frames):
    top = frames - p.patch_time
    start, end = anchor - p.search_bwd, anchor + p.search_fwd
    shift = min(0, start) + max(0, end - top)
    low, high = max(0, start - shift), min(top, end - shift)
    return [anchor, *range(anchor + 1, high + 1), *range(anchor - 1, low - 1, -1)]


def _grid(p, width, height, frames, anchor):
    top_x, top_y, step = width - p.patch_size, height - p.patch_size, p.proc_step
    phase_y = 0 if anchor == frames - p.patch_time else anchor
    y = torch.arange(top_y + 1, device=DEV)[:, None]
    x = torch.arange(top_x + 1, device=DEV)[None, :]
    phase_x = torch.where(y == top_y, 0, phase_y + y // step)
    on = (y == 0) | (y == top_y) | (y % step == phase_y % step)
    on = on & ((x == 0) | (x == top_x) | (x % step == phase_x % step))
    y, x = torch.nonzero(on, as_tuple=True)
    return x, y


def _follow(clip, frame, middle, x, y):
    """One step along a vector clip: the vector of the block nearest to the
    patch's middle, rounded to whole pixels, halves away from zero."""
    a = clip.analysis
    if not clip.valid[frame]:
        return x, y

    def nearest(at, block, overlap, count):
        shifted = at - block // 2
        step = block - overlap
        index = torch.sign(shifted) * ((shifted.abs() + step // 2) // step)
        return index.clamp(0, count - 1)

    bx = nearest(x + middle, a.block_size_x, a.overlap_x, a.block_count_x)
    by = nearest(y + middle, a.block_size_y, a.overlap_y, a.block_count_y)
    v = torch.from_numpy(clip.vectors[frame]).to(DEV).long()[by, bx]
    v = torch.sign(v) * ((v.abs() + a.pel // 2) // a.pel)
    return (x + v[:, 0]).clamp(0, a.width - 1), (y + v[:, 1]).clamp(0, a.height - 1)


def _centers(p, x, y, anchor, frame, mvfw, mvbw):
    if mvfw is None:
        return x, y
    walk = [(mvbw, f) for f in range(anchor, frame)] or [(mvfw, f) for f in range(anchor, frame, -1)]
    for clip, f in walk:
        x, y = _follow(clip, f, p.patch_size // 2, x, y)
    return x, y


def _patches(clip, size):
    """A view [frames, y, x, channels, size, size] of every patch."""
    return clip.unfold(2, size, 1).unfold(3, size, 1).permute(0, 2, 3, 1, 4, 5)


def _rows(view, pt, f, y, x):
    """Patches [..., channels, time, size, size] at origins f, y, x."""
    return torch.stack([view[f + t, y, x] for t in range(pt)], dim=-3)


def _matches(p, view, anchor, x, y, spans, cap):
    """Neighbours of the anchors: frame, y, x [A, limit] and counts [A]."""
    found = []
    per_anchor = sum(int((s[2][0] - s[1][0] + 1) * (s[4][0] - s[3][0] + 1)) for s in spans)
    dim = view.shape[3] * p.patch_size ** 2
    chunk = max(1, int(6e7 // (per_anchor * dim)))
    for at in range(0, x.numel(), chunk):
        ax, ay = x[at:at + chunk], y[at:at + chunk]
        cf, cy, cx = [], [], []
        for frame, x0, x1, y0, y1 in spans:
            nx, ny = int(x1[0] - x0[0]) + 1, int(y1[0] - y0[0]) + 1
            grid_y = (y0[at:at + chunk, None] + torch.arange(ny, device=DEV))[:, :, None]
            grid_x = (x0[at:at + chunk, None] + torch.arange(nx, device=DEV))[:, None, :]
            cy.append(grid_y.expand(-1, ny, nx).reshape(ax.numel(), -1))
            cx.append(grid_x.expand(-1, ny, nx).reshape(ax.numel(), -1))
            cf.append(torch.full_like(cy[-1], frame))
        cf, cy, cx = torch.cat(cf, 1), torch.cat(cy, 1), torch.cat(cx, 1)
        distance = 0
        for t in range(p.patch_time):
            diff = view[cf + t, cy, cx] - view[anchor + t, ay, ax][:, None]
            distance = distance + diff.square_().sum(dim=(2, 3, 4))
        distance, order = torch.sort(distance, dim=1, stable=True)
        limit = min(cap, distance.shape[1])
        k = min(p.similar, limit)
        reach = distance[:, k - 1:k].clamp(min=p.tau)
        counts = (distance[:, :limit] <= reach).sum(dim=1)
        order = order[:, :limit]
        found.append((cf.gather(1, order), cy.gather(1, order), cx.gather(1, order), counts))
    return [torch.cat(v) for v in zip(*found)]


def _active(p, anchor, x, y, mf, my, mx, counts, width, height):
    """Anchors that are filtered: each filtered one clears its neighbours in
    its own frame, and the pixels beside them, from those that follow."""
    none = width * height
    here = (mf == anchor) & (torch.arange(mf.shape[1], device=DEV) < counts[:, None])
    at, far = my * width + mx, 2 * p.patch_size
    beside = [(here, at), (here & (my > far), at - width), (here & (my < height - far), at + width),
              (here & (mx > far), at - 1), (here & (mx < width - far), at + 1)]
    cleared = torch.cat([torch.where(m, q, none) for m, q in beside], dim=1).cpu().numpy()
    own = (y * width + x).tolist()
    mask = np.ones(none + 1, bool)
    kept = []
    for a, q in enumerate(own):
        if mask[q]:
            kept.append(a)
            mask[cleared[a]] = False
    return torch.tensor(kept, device=DEV, dtype=torch.long)


def _eigen(matrices):
    """Eigenvalues in descending order and eigenvectors (columns) of symmetric
    matrices [..., n, n]: Jacobi sweeps of n - 1 rounds of disjoint pairs, all
    matrices at once."""
    n = matrices.shape[-1]
    even = n + n % 2
    flat = matrices.reshape(-1, n, n)
    a = torch.zeros((even, even, flat.shape[0]), dtype=flat.dtype, device=DEV)  # problems innermost
    a[:n, :n] = flat.permute(1, 2, 0)
    v = torch.eye(even, dtype=a.dtype, device=DEV)[:, :, None].expand_as(a).clone()
    off = ~torch.eye(even, dtype=torch.bool, device=DEV)[:, :, None]
    limit = 1e-13 * a.abs().amax(dim=(0, 1))
    ring = torch.arange(1, even)
    rounds = torch.stack([torch.cat([torch.zeros(1, dtype=torch.long), ring.roll(k)]) for k in range(even - 1)]).to(DEV)
    for _ in range(12):
        if not bool(((a.abs() > limit) & off).any()):
            break
        for order in rounds:
            p, q = order[:even // 2], order[even // 2:].flip(0)
            pivot = a[p, q]
            tau = (a[q, q] - a[p, p]) / (2 * torch.where(pivot == 0, 1.0, pivot))
            t = torch.where(tau < 0, -1.0, 1.0) / (tau.abs() + torch.sqrt(1 + tau * tau))
            t = torch.where(pivot == 0, 0.0, t)
            c = 1 / torch.sqrt(1 + t * t)
            s = t * c
            for m in (a, v):  # rows: A <- J' A, V' <- J' V'
                left, right = m[p], m[q]
                m[p] = c[:, None] * left - s[:, None] * right
                m[q] = s[:, None] * left + c[:, None] * right
            left, right = a[:, p], a[:, q]
            a[:, p] = c * left - s * right
            a[:, q] = s * left + c * right
    values, order = torch.sort(a.diagonal(dim1=0, dim2=1)[:, :n], dim=1, descending=True)
    vectors = v[:n, :n].permute(2, 1, 0).gather(2, order[:, None, :].expand_as(flat))
    return values.reshape(matrices.shape[:-1]), vectors.reshape(matrices.shape)


def _wiener(p, final, noisy, basic, counts, coupled):
    """Filtered rows and weights of groups [G, cap, C, D] (float64)."""
    groups, cap, channels, each = noisy.shape
    held = torch.arange(cap, device=DEV) < counts[:, None]
    models, d = (1, channels * each) if coupled else (channels, each)

    def by_model(v):
        return v.reshape(groups, cap, models, d).transpose(1, 2)

    size = counts.clamp(max=max(p.similar, math.ceil(p.similar * p.model_cap_factor)) if p.model_cap_factor else cap)
    model = (torch.arange(cap, device=DEV) < size[:, None])[:, None, :, None]
    share = size[:, None, None, None].double()
    same = ((noisy == noisy[:, :1]) | ~held[:, :, None, None]).all(dim=3).all(dim=2).all(dim=1) & (counts > 1)
    flat = torch.zeros(groups, dtype=torch.bool, device=DEV)
    if final and p.flat_areas:
        values = held[:, :, None, None].double()
        n = counts.double()[:, None] * each
        first = (noisy * values).sum(dim=(1, 3))
        second = (noisy.square() * values).sum(dim=(1, 3))
        flat = ((second - first * first / n) / (n - 1)).mean(dim=1) < p.sigma * p.sigma * p.gamma
    rows = by_model(noisy)
    center = (rows * model).sum(dim=2, keepdim=True) / share
    members = rows - center
    if final:
        guide = by_model(basic)
        guide_center = (guide * model).sum(dim=2, keepdim=True) / share
        center = torch.where(flat[:, None, None, None], guide_center, center)
        members = guide - guide_center
    # The dual problem.
    x = (members * model)[:, :, :int(size.max())]
    values, vectors = _eigen(x @ x.transpose(2, 3) / share)
    values, vectors = values[..., :p.rank], vectors[..., :p.rank]
    floor = 128 * float(np.finfo(np.float32).eps)
    basis = vectors.transpose(2, 3) @ x
    basis = basis / basis.norm(dim=3, keepdim=True).clamp(min=1e-300) * (values > floor)[..., None]
    sigma2 = p.beta * p.sigma * p.sigma
    noise2 = p.beta * p.sigma_basic ** 2 if final else sigma2
    variance = values - values.clamp(max=noise2) if noise2 > 0 else values
    gain = torch.where(variance > p.variance_threshold * sigma2, 1 / (1 + sigma2 / variance), 0.0)
    output = (((rows - center) @ basis.transpose(2, 3)) * gain[:, :, None]) @ basis + center
    # Group precision, membership and volume.
    signal = (values - noise2).clamp(min=0)
    trace = (signal / (signal + sigma2)).sum(dim=2, keepdim=True)
    log_weight = -p.weight_alpha * torch.log(p.weight_epsilon + d / share[..., 0] + trace)
    match2 = p.sigma_basic ** 2 if final else p.sigma ** 2
    member2 = max(match2, p.membership_noise_floor * p.sigma * p.sigma)
    volume = torch.log1p(signal / member2).sum(dim=2, keepdim=True) / d
    shadow = (members @ basis.transpose(2, 3)).square()
    left = (members.square().sum(dim=3) - shadow.sum(dim=3)).clamp(min=0)
    score = ((shadow / (signal + member2)[:, :, None]).sum(dim=3) + left / member2 - d) / math.sqrt(2 * d)
    nearest = score.masked_fill(~held[:, None], math.inf).min(dim=2, keepdim=True).values
    log_weight = log_weight - p.weight_beta * ((score - nearest).clamp(min=0) + volume)
    log_weight = log_weight.mean(dim=1)
    bypass = -p.weight_alpha * torch.log(p.weight_epsilon + d / share[:, 0, :, 0])
    log_weight = torch.where(same[:, None], bypass, log_weight)
    weight = torch.exp(log_weight.clamp(-80, 80)) * held
    output = output.transpose(1, 2).reshape(noisy.shape)
    return torch.where(same[:, None, None, None], noisy, output), weight


def _window(p):
    center = 0.5 * (p.patch_size - 1)
    r = (torch.arange(p.patch_size, device=DEV, dtype=torch.float64) - center) / max(center, 0.5)
    raw = torch.exp(-0.5 * (r[:, None] ** 2 + r[None, :] ** 2))
    return (raw / raw.max()) ** p.weight_gamma


def _exact_stage(p, final, clip, guide, mvfw, mvbw):
    frames, channels, height, width = clip.shape
    coupled = p.couple_channels and channels > 1
    cap = p.search_window ** 2 * (p.search_bwd + p.search_fwd + 1)
    if p.similar_cap_factor:
        cap = min(cap, max(p.similar, math.ceil(p.similar * p.similar_cap_factor)))
    if p.tau == 0:
        cap = min(cap, p.similar)  # only the nearest are kept, ties aside
    size, pt = p.patch_size, p.patch_time
    matched = _patches(guide if final else clip[:, :1], size)
    noisy_view = _patches(clip, size)
    basic_view = _patches(guide, size) if final else None
    window = _window(p)
    total = torch.zeros((channels + 1) * frames * height * width, dtype=torch.float64, device=DEV)
    plane = height * width
    place = (torch.arange(size, device=DEV)[:, None] * width + torch.arange(size, device=DEV)[None, :])
    times = torch.arange(pt, device=DEV)
    place = place + (times * (channels + 1) * plane)[:, None, None]
    place = place + (torch.arange(channels + 1, device=DEV) * plane)[:, None, None, None]
    for anchor in range(frames - pt + 1):
        x, y = _grid(p, width, height, frames, anchor)
        spans = []
        for frame in _schedule(p, anchor, frames):
            cx, cy = _centers(p, x, y, anchor, frame, mvfw, mvbw)
            spans.append((frame, *_span(cx, width, size, p.search_window), *_span(cy, height, size, p.search_window)))
        mf, my, mx, counts = _matches(p, matched, anchor, x, y, spans, cap)
        keep = _active(p, anchor, x, y, mf, my, mx, counts, width, height)
        chunk = max(1, int(2e8 // (mf.shape[1] * channels * pt * size * size)))
        for at in range(0, keep.numel(), chunk):
            pick = keep[at:at + chunk]
            f, gy, gx, n = mf[pick], my[pick], mx[pick], counts[pick]
            noisy = _rows(noisy_view, pt, f, gy, gx)
            shape = noisy.shape
            flat_shape = (shape[0], shape[1], channels, pt * size * size)
            basic = _rows(basic_view, pt, f, gy, gx).reshape(flat_shape) if final else None
            output, weight = _wiener(p, final, noisy.reshape(flat_shape), basic, n, coupled)
            # An anchor frame's stack has slots for search_bwd frames before it and search_fwd + Pt - 1 after it.
            slot = f[:, :, None] + times - anchor + p.search_bwd
            held = (slot >= 0) & (slot < p.search_bwd + p.search_fwd + pt)
            weight = weight[:, :, None, None, None, None] * held[:, :, None, :, None, None] * window
            values = torch.cat([output.reshape(shape) * weight, weight.expand(*shape[:2], 1, *shape[3:])], dim=2)
            index = ((f * (channels + 1)) * plane + gy * width + gx)[:, :, None, None, None, None] + place
            total.index_add_(0, index.reshape(-1), values.reshape(-1))
    total = total.reshape(frames, channels + 1, height, width)
    weight = total[:, channels:]
    return torch.where(weight > 0, total[:, :channels] / weight.clamp(min=1e-300), clip)


def _exact_batch(case, seed):
    clip, _ = _clip(case, seed)
    anchors, candidates, targets = _training_rows(case, seed)
    clip = clip.double()
    boxes = _patches(clip, 8)[:, :, :, 0]

    def means(packed):
        p = packed.long() & 0xFFFFFFFF
        at = [boxes[(p >> 24) + t, (p >> 12) & 0xFFF, p & 0xFFF] for t in range(2)]
        return torch.stack([v.reshape(-1, 4, 2, 4, 2).mean(dim=(2, 4)) for v in at], dim=1).reshape(-1, 32), p

    (a, pa), (c, pc) = means(anchors), means(candidates)
    x = torch.zeros((a.shape[0], 128), dtype=torch.float64, device=DEV)
    x[:, :32], x[:, 32:64], x[:, 64:96] = a - 0.5, c - 0.5, (a - c).abs() * 4
    for k, (shift, mask, scale) in enumerate(((0, 0xFFF, 16.0), (12, 0xFFF, 16.0), (24, 0xFF, 4.0))):
        x[:, 96 + k] = (((pc >> shift) & mask) - ((pa >> shift) & mask)).double() / scale
    x[:, 99] = (a - c).square().sum(dim=1) * 4
    flat = torch.from_numpy(_weights(seed).astype(np.float64)).to(DEV).requires_grad_()
    w1, b1, w2, b2, w3, b3 = flat.split([256 * 128, 256, 256 * 256, 256, 256, 1])
    h = torch.relu(x @ w1.reshape(256, 128).T + b1)
    h = torch.relu(h @ w2.reshape(256, 256).T + b2)
    scores = h @ w3 + b3
    logs = torch.log_softmax(scores.reshape(-1, case["group"]), dim=1)
    losses = -(targets.double().reshape(-1, case["group"]) * logs).sum(dim=1)
    losses.mean().backward()
    return {"scores": scores.detach(), "grads": flat.grad, "losses": losses.detach()}


# Terms of distances and group models that take about 15 seconds in float64.
EXACT_TERMS = 8e11


def exact(case, seed):
    if case["path"] == "train":
        return _exact_batch(case, seed)
    terms = 0.0
    for stage, args in zip((BASIC, FINAL), _arguments(case)):
        p = parse_stage_parameters(stage, args)
        anchors = case["width"] * case["height"] / p.proc_step ** 2 * case["frames"]
        candidates = p.search_window ** 2 * (p.search_bwd + p.search_fwd + 1)
        matched = p.patch_size ** 2 * p.patch_time * (case["channels"] if stage == FINAL else 1)
        terms += anchors * (candidates * matched + 1.5e4 * p.similar)
    if terms > EXACT_TERMS:
        return None
    clip, moves = _clip(case, seed)
    mvfw = mvbw = None
    if case["path"] == "guided":
        mvfw, mvbw = _vectors(case, seed, moves, False), _vectors(case, seed, moves, True)
    basic_args, final_args = _arguments(case)
    clip = clip.double()
    basic = _exact_stage(parse_stage_parameters(BASIC, basic_args), False, clip, None, mvfw, mvbw)
    final = _exact_stage(parse_stage_parameters(FINAL, final_args), True, clip, basic, mvfw, mvbw)
    return {"basic": basic, "final": final}
