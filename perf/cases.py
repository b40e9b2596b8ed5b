"""Performance cases of the KV transfer path, through its public entry points.

Kinds of work (`"kind"` of a case):

``cycle``   one save, prefix query and load through ``PegaEngine``: what the
            server does when a prompt is offloaded and comes back later.  The
            pinned pool is small enough that saves evict older blocks, the
            state a server is in after its first minutes.
``load``    prefix query and load of blocks that ``turns`` earlier saves have
            stored (a conversation is saved turn by turn and comes back whole).
``blocks``  the block-ID transfer handle (``BlockTransfer``) that an embedder
            drives itself, with a dense or padded host image.
``descs``   a descriptor batch through one of the two transfer backends.

Blocks are paged KV cache blocks: ``layers`` layers of ``segments`` (2 = K and V
in separate regions, 1 = one latent tensor) fragments of ``frag`` bytes.
"""

from __future__ import annotations

import math

import numpy as np
import torch

from pegaflow_amd.engine import LayerSave, PegaEngine
from pegaflow_amd.layout import KVCacheLayout
from pegaflow_amd.runtime import Event, PinnedMemory, Stream
from pegaflow_amd.transfer import BlockTransfer, LayerBlocks, build_backend, desc_array, TransferMode

KIB, MIB = 1 << 10, 1 << 20


def listed():
    return [
        # Layer-by-layer save of 256 tokens from a model's forward hooks: one
        # layer per call, the smallest call a worker makes.
        {"name": "layer_save_1mib", "kind": "blocks", "way": "save", "layers": 1, "segments": 2,
         "frag": 32 * KIB, "blocks": 16, "ids": "random", "pad": 0, "events": False, "window": 0},
        # One more cached block found at decode time: 32 layers x 1 block.
        {"name": "decode_load_2mib", "kind": "load", "layers": 32, "segments": 2,
         "frag": 32 * KIB, "blocks": 1, "turns": 1, "ids": "random", "page_first": False},
        # A short chat turn (256 tokens) offloaded and brought back.
        {"name": "chat_turn_cycle", "kind": "cycle", "layers": 32, "segments": 2,
         "frag": 32 * KIB, "blocks": 16, "ids": "random", "page_first": False},
        # A conversation of eight saved turns comes back in one load.
        {"name": "multiturn_load", "kind": "load", "layers": 32, "segments": 2,
         "frag": 32 * KIB, "blocks": 192, "turns": 8, "ids": "random", "page_first": False},
        # Two 10K-token prompts (2 x 625 blocks), Llama-3.1-8B shape.
        {"name": "prompt_cycle", "kind": "cycle", "layers": 32, "segments": 2,
         "frag": 32 * KIB, "blocks": 1250, "ids": "random", "page_first": False},
        # One 4K-token prompt in fp8, Llama-3-70B shape, half its ids in runs.
        {"name": "fp8_prompt_cycle", "kind": "cycle", "layers": 80, "segments": 2,
         "frag": 16 * KIB, "blocks": 256, "ids": "runs", "page_first": False},
        # One 10K-token prompt, DeepSeek-V3 latent cache, pages of all layers.
        {"name": "mla_page_first_cycle", "kind": "cycle", "layers": 61, "segments": 1,
         "frag": 72 * KIB, "blocks": 157, "ids": "random", "page_first": True},
        # A 5K-token prefix loaded layer by layer under the forward pass, with a
        # completion event for every layer.
        {"name": "layerwise_load", "kind": "blocks", "way": "load", "layers": 32, "segments": 2,
         "frag": 32 * KIB, "blocks": 313, "ids": "random", "pad": 0, "events": True, "window": 0},
        # Cache groups of unlike size: every sixth layer keeps the whole prompt,
        # the sliding-window layers keep their last eight blocks.
        {"name": "hybrid_roundtrip", "kind": "blocks", "way": "both", "layers": 48, "segments": 2,
         "frag": 32 * KIB, "blocks": 625, "ids": "random", "pad": 0, "events": False, "window": 8},
        # Long lists of 1 KiB blocks over 61 layers: the per-block cost of the
        # engine's bookkeeping.
        {"name": "small_blocks_cycle", "kind": "cycle", "layers": 61, "segments": 1,
         "frag": KIB, "blocks": 1024, "ids": "random", "page_first": False},
        # Shuffled 4 KiB fragments through the default backend, both ways.
        {"name": "descs_direct_4k", "kind": "descs", "mode": "direct", "frag": 4 * KIB,
         "blocks": 16384, "ids": "random"},
        # Fragments that are no multiple of 16 bytes, so that most of them
        # start off a 16-byte boundary.
        {"name": "ragged_roundtrip", "kind": "blocks", "way": "both", "layers": 16, "segments": 2,
         "frag": 1000, "blocks": 777, "ids": "random", "pad": 0, "events": False, "window": 0},
    ]


# Payload of the largest listed case, one way.
LARGEST = 32 * 1250 * 64 * KIB


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["cycle", "cycle", "load", "load", "blocks", "blocks", "descs"])
    payload = _log_uniform(rng, MIB, LARGEST // 4)
    if kind == "descs":
        frag = rng.choice([4 * KIB, 4 * KIB, 4112, 1000, _log_uniform(rng, 512, 128 * KIB)])
        return {"kind": kind, "mode": rng.choice(["direct", "kernel"]), "frag": frag,
                "blocks": max(1, min(65536, payload // frag)), "ids": rng.choice(["random", "runs"])}
    frag = rng.choice([16 * KIB, 32 * KIB, 72 * KIB, 16 * _log_uniform(rng, 64, 8192),
                       16 * _log_uniform(rng, 64, 8192), 4 * _log_uniform(rng, 128, 4096)])
    segments = rng.choice([1, 2])
    layers = _log_uniform(rng, 1, 80)
    # No more list entries than the longest listed lists hold.
    blocks = payload // (layers * segments * frag)
    blocks = max(1, min(blocks, 65536 // layers, 16384))
    case = {"kind": kind, "layers": layers, "segments": segments, "frag": frag, "blocks": blocks,
            "ids": rng.choice(["random", "runs"])}
    if kind == "blocks":
        case["way"] = rng.choice(["save", "load", "both"])
        case["pad"] = rng.choice([0, 0, 512])
        case["events"] = rng.random() < 0.25
        case["window"] = rng.choice([0, 0, 0, max(1, blocks // 50)])
    else:
        case["page_first"] = segments == 1 and rng.random() < 0.4
        if kind == "load":
            case["turns"] = min(blocks, _log_uniform(rng, 1, 16))
    return case


def _values(shape_bytes, frag, generator):
    """Cache contents: bf16 N(0, 1), or fp8 e4m3 bytes without its NaN
    encodings for the 16 KiB fragments of the fp8 shape and for odd sizes."""
    if frag == 16 * KIB or frag % 2:
        data = torch.randint(0, 254, shape_bytes, dtype=torch.uint8, device="cuda", generator=generator)
        return torch.where(data >= 127, data + 1, data)
    shape = (*shape_bytes[:-1], shape_bytes[-1] // 2)
    return torch.randn(shape, dtype=torch.bfloat16, device="cuda", generator=generator)


def _ids(rng, pool, n, how):
    """`n` distinct slots of a pool: a random choice, or half of them in runs of
    8 to 64 as they come from a pool that is not yet fragmented."""
    if how == "random":
        return rng.permutation(pool)[:n].astype(np.int64)
    taken, out, left = np.zeros(pool, dtype=bool), [], n // 2
    for start in rng.permutation(pool // 64):
        if left <= 0:
            break
        length = min(left, int(rng.integers(8, 65)))
        run = np.arange(start * 64, start * 64 + length)
        taken[run] = True
        out.append(run)
        left -= length
    free = rng.permutation(np.flatnonzero(~taken))
    have = sum(len(r) for r in out)
    out += [free[i:i + 1] for i in range(n - have)]
    order = rng.permutation(len(out))
    return np.concatenate([out[i] for i in order]).astype(np.int64)


class _Worker:
    """What a worker thread of an embedding program keeps for its lifetime: a
    stream, a block transfer handle and the two descriptor backends."""

    def __init__(self):
        self.stream = Stream()
        self.transfer = BlockTransfer()
        self.backends = {name: build_backend(TransferMode.from_name(name))
                         for name in ("direct", "kernel")}


_worker = None


def worker():
    global _worker
    if _worker is None:
        torch.cuda.current_stream()  # torch opens the device before the library does
        _worker = _Worker()
    return _worker


def _new_cache(case, pool, generator):
    shape = (case["layers"], case["segments"], pool, case["frag"])
    return _values(shape, case["frag"], generator)


def prepare(case, seed):
    generator = torch.Generator(device="cuda").manual_seed(seed)
    rng = np.random.default_rng(seed)
    if case["kind"] == "descs":
        state = _prepare_descs(case, rng, generator)
    elif case["kind"] == "blocks":
        state = _prepare_blocks(case, rng, generator)
    else:
        state = _prepare_engine(case, rng, generator)
    torch.cuda.synchronize()
    return state


def run(state):
    return state["run"](state)


# -- through the engine -----------------------------------------------------------


def _prepare_engine(case, rng, generator):
    n, layers, segments, frag = (case[k] for k in ("blocks", "layers", "segments", "frag"))
    # Blocks are saved from the lower half of the cache and come back into the
    # upper half.
    half = n + n // 4 + 64
    cache = _new_cache(case, 2 * half, generator)
    per_layer = segments * 2 * half * frag
    payload = n * layers * segments * frag
    # Room for two or three saves: later ones evict the oldest blocks.
    engine = PegaEngine(pool_size=int(payload * (2.5 if case["kind"] == "cycle" else 2)) + 32 * MIB)
    names = [f"model.layers.{i}.attn" for i in range(layers)]
    base = cache.data_ptr()
    engine.register_context_layer_batch(
        "model", "shared", torch.cuda.current_device(), 0, 0, 1, 1, names,
        [base + i * per_layer for i in range(layers)], [per_layer] * layers, [2 * half] * layers,
        [frag] * layers, [2 * half * frag if segments == 2 else 0] * layers, [segments] * layers,
        page_first=case["page_first"])
    state = {"engine": engine, "names": names, "cache": cache, "passes": 0,
             "save_ids": _ids(rng, half, n, case["ids"]).tolist(),
             "load_ids": (_ids(rng, half, n, case["ids"]) + half).tolist(),
             "digests": [rng.bytes(24) for _ in range(n)]}
    if case["kind"] == "cycle":
        state["run"] = _run_cycle
    else:
        state["hashes"] = [bytes(8) + d for d in state["digests"]]
        state["run"] = _run_load
        torch.cuda.synchronize()
        turns = case["turns"]
        for t in range(turns):
            part = slice(t * n // turns, (t + 1) * n // turns)
            _save(state, state["save_ids"][part], state["hashes"][part])
    return state


def _save(state, ids, hashes):
    state["engine"].batch_save_kv_blocks(
        "model", 0, 0, torch.cuda.current_device(),
        [LayerSave(name, ids, hashes) for name in state["names"]])


def _run_load(state):
    engine = state["engine"]
    hits, lease = engine.query_prefix("model", state["hashes"])
    task = engine.batch_load_kv_blocks_multi_layer(
        "model", 0, torch.cuda.current_device(), [state["names"]], lease, [state["load_ids"]])
    task.wait()
    task.close()
    return [hits, state["cache"]]


def _run_cycle(state):
    # Another request's tokens: other hashes each time.
    state["passes"] += 1
    salt = state["passes"].to_bytes(8, "little")
    state["hashes"] = [salt + d for d in state["digests"]]
    _save(state, state["save_ids"], state["hashes"])
    return _run_load(state)


# -- through the block transfer handle ----------------------------------------------


def _prepare_blocks(case, rng, generator):
    n, n_layers, segments, frag = (case[k] for k in ("blocks", "layers", "segments", "frag"))
    w = worker()
    pool = n + n // 2 + 64
    source = _new_cache(case, pool, generator)
    target = torch.zeros_like(source) if case["way"] != "save" else None
    counts = [n if case["window"] == 0 or i % 6 == 0 else min(n, case["window"]) for i in range(n_layers)]
    stride = -(-frag // case["pad"]) * case["pad"] if case["pad"] else frag
    host = PinnedMemory(sum(counts) * segments * stride)
    if case["way"] == "save":
        host.as_numpy()[:] = 0  # the image is the output, its padding with it
    region = pool * frag
    save_ids, load_ids = (_ids(rng, pool, n, case["ids"]).astype(np.uint32) for _ in range(2))

    def layers(cache, ids):
        out, at = [], 0
        for i, count in enumerate(counts):
            layout = KVCacheLayout(cache.data_ptr() + i * segments * region, segments * region, pool,
                                   frag, region if segments == 2 else 0, segments)
            offsets = [at + s * count * stride for s in range(segments)]
            out.append(LayerBlocks(layout, ids[:count],
                                   tuple(host.host_ptr + o for o in offsets),
                                   tuple(host.device_ptr + o for o in offsets),
                                   (count * stride,) * segments, stride))
            at += segments * count * stride
        return out

    image = torch.from_numpy(host.as_numpy())
    image.owner = host  # the view keeps the pinned memory
    state = {"host": host, "image": image, "source": source, "target": target, "way": case["way"],
             "save": layers(source, save_ids), "run": _run_blocks,
             "load": layers(target, load_ids) if target is not None else None,
             "events": [Event() for _ in counts] if case["events"] else None}
    if case["way"] == "load":
        torch.cuda.synchronize()
        w.transfer.save(state["save"], w.stream)
    return state


def _run_blocks(state):
    w = worker()
    if state["events"]:
        w.transfer.set_layer_events(state["events"])
    out = None
    if state["way"] != "load":
        w.transfer.save(state["save"], w.stream)
        out = state["image"]
    if state["way"] != "save":
        w.transfer.load(state["load"], w.stream)
        out = state["target"]
    if state["events"]:
        w.transfer.set_layer_events(None)
    return out


# -- through the descriptor backends --------------------------------------------------


def _prepare_descs(case, rng, generator):
    worker()
    n, frag = case["blocks"], case["frag"]
    pool = n + n // 2 + 64
    source = _values((pool, frag), frag, generator)
    target = torch.zeros_like(source)
    host = PinnedMemory(n * frag)

    def descs(cache):
        at = np.arange(n, dtype=np.uint64) * np.uint64(frag)
        ids = _ids(rng, pool, n, case["ids"]).astype(np.uint64)
        return desc_array(np.uint64(cache.data_ptr()) + ids * np.uint64(frag),
                          np.uint64(host.host_ptr) + at, np.uint64(host.device_ptr) + at, frag)

    return {"host": host, "source": source, "target": target, "mode": case["mode"],
            "save": descs(source), "load": descs(target), "run": _run_descs}


def _run_descs(state):
    w = worker()
    backend = w.backends[state["mode"]]
    backend.d2h(state["save"], w.stream)
    backend.h2d(state["load"], w.stream)
    return state["target"]


# -- what a pass cannot do without ------------------------------------------------------


def work(case):
    blocks = case["blocks"] * case.get("layers", 1)
    if case.get("window"):
        full = (case["layers"] + 5) // 6
        blocks = full * case["blocks"] + (case["layers"] - full) * min(case["blocks"], case["window"])
    payload = blocks * case.get("segments", 1) * case["frag"]
    # Each direction reads the payload on one side and writes it on the other.
    directions = 2 if case["kind"] in ("cycle", "descs") or case.get("way") == "both" else 1
    return {"bytes": 2 * directions * payload, "flops": 0}


def tolerance(case):
    # Bytes are moved, not computed.
    return "exact"
