"""Timed cases of the framework's main paths, through the Python package's
public entry points.

A program that uses the package keeps worlds on the GPU, ticks them and draws
them into texture layers; it loads and saves chunks, stamps rigid bodies,
moves particles and asks for outlines.  Each case is one such call sequence:

  frame      one frame of a running game: tick, (island check,) texture pass
  run        a new world simulated for a while, then drawn or saved
  batch      many worlds of uneven sizes advanced together, each drawn
  bodies     a frame with rigid bodies: stamp, tick, unstamp
  mesh       solid outlines of every chunk, for the host's physics engine
  particles  a frame of free-fall particles with a new burst, then drawn
  pack       chunk images of a region encoded and copied out, for a save file
  unpack     chunk images of a region decoded into the grid, then drawn

Sizes follow the benchmark and the tests: 512^2, 4096^2 and 16384^2 worlds,
batches of worlds with sides from 256 to 2048, up to 200 bodies, tens of
thousands of particles, 128x128 chunks.
"""
import ctypes
import math

import numpy as np
import torch

import falling_sand_engine_amd as fsg

CHUNK = 128
MOST_UPDATES = 16384 * 16384 * 16  # cell-updates of the largest run

_context = None


def context():
    """The program's one context (one stream, one block cache)."""
    global _context
    if _context is None:
        _context = fsg.Context(0)
    return _context


class Owner:
    """Keeps a world open for as long as the state or one of its textures is
    in use."""

    world = None

    def __init__(self, width, height, seed, **config):
        self.world = fsg.World(context(), width, height, seed, fsg.default_config(**config))

    def __del__(self):
        if self.world is not None:
            self.world.close()


class Texels:
    """A world's texture layer in device memory, for torch.as_tensor."""

    def __init__(self, owner, layer):
        w = owner.world
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (w.height, w.width), "typestr": "<i4", "version": 2,
                                         "data": (w.layer_ptr(layer), False), "strides": None}


def texture(owner, layer):
    """The layer as an int32 tensor over the world's own memory."""
    return torch.as_tensor(Texels(owner, layer), device="cuda")


def world_state(case, seed, layers=fsg.LAYER_CELLS, **config):
    """A generated world with its layers allocated, as a program has it after
    its first frame."""
    config.setdefault("reactions", 0 if case["kind"] == 3 else 1)
    config.setdefault("temp_every", case.get("temp_every", 1))
    if case.get("temp_every", 1) > 2:
        config.setdefault("temp_phase", 2)
    config.setdefault("chunk_skip", case.get("skip", 0))
    owner = Owner(case["width"], case["height"], seed, **config)
    owner.world.generate(case["kind"], seed)
    owner.world.render(layers)
    one = (fsg.LAYER_CELLS, fsg.LAYER_EMISSION, fsg.LAYER_FIRE)
    return {"case": case, "seed": seed, "owner": owner, "world": owner.world,
            "textures": [texture(owner, v) for v in one if layers & v]}


# --- frame ------------------------------------------------------------------
def prepare_frame(case, seed):
    layers = fsg.LAYER_CELLS
    if case["layers"] == 3:
        layers |= fsg.LAYER_EMISSION | fsg.LAYER_FIRE
    s = world_state(case, seed, layers)
    w, h = case["width"], case["height"]
    if case["zone"]:  # the game ticks the world less a one-chunk frame
        s["world"].tickZone = (CHUNK, CHUNK, w - 2 * CHUNK, h - 2 * CHUNK)
    s["world"].tick(64)
    rng = np.random.default_rng(seed)
    s["seeds"] = [(int(x), int(y)) for x, y in zip(rng.integers(0, w, 256), rng.integers(0, h, 256))]
    vw, vh = min(case["view_w"], w), min(case["view_h"], h)
    s["view"] = ((w - vw) // 2, (h - vh) // 2, vw, vh)
    s["layers"], s["frame"] = layers, 0
    return s


def run_frame(s):
    case, w = s["case"], s["world"]
    w.tick(1)
    out = {}
    if case["check"]:  # the reference checks one random cell a tick for a loose island
        r = w.physicsCheck([s["seeds"][s["frame"] % 256]])[0]
        out["island"] = [r["status"], r["count"], r["box"]]
    s["frame"] += 1
    moved = w.render(s["layers"], rect=s["view"], fire_mat=fsg.MAT_LAVA, stats=bool(case["census"]))
    if moved:
        out["moved"] = np.array(moved["moved"] + [moved["fire_cells"]], np.int64)
    out["textures"] = s["textures"]
    return out


# --- run --------------------------------------------------------------------
def prepare_run(case, seed):
    return world_state(case, seed, fsg.LAYER_CELLS | fsg.LAYER_EMISSION)


def run_run(s):
    case, w = s["case"], s["world"]
    w.generate(case["kind"], s["seed"])
    w.tick(case["ticks"])
    if case["save"]:
        return w.download()
    w.render(fsg.LAYER_CELLS | fsg.LAYER_EMISSION)
    return s["textures"]


# --- batch ------------------------------------------------------------------
def batch_sizes(case, rng):
    """Sides log-uniform between the case's, aspect ratio in [0.5, 2]."""
    sizes = []
    for _ in range(case["worlds"]):
        side = math.exp(rng.uniform(math.log(case["side_lo"]), math.log(case["side_hi"])))
        a = math.sqrt(rng.uniform(0.5, 2.0))
        sizes.append((max(64, round(side * a / case["step"]) * case["step"]),
                      max(64, round(side / a / case["step"]) * case["step"])))
    return sizes


def prepare_batch(case, seed):
    sizes = batch_sizes(case, np.random.default_rng(case["worlds"]))
    worlds = [world_state({"kind": 4, "width": w, "height": h, "skip": case["skip"]}, seed + i)
              for i, (w, h) in enumerate(sizes)]
    return {"case": case, "worlds": worlds}


def run_batch(s):
    case = s["case"]
    worlds = [m["world"] for m in s["worlds"]]
    for m in s["worlds"]:
        m["world"].generate(4, m["seed"])
    fsg.batch_step(context(), worlds, case["ticks"])
    for w in worlds:
        w.render(fsg.LAYER_CELLS)
    return [m["textures"][0] for m in s["worlds"]]


# --- bodies -----------------------------------------------------------------
def prepare_bodies(case, seed):
    """Stone and wood bodies with holes, rocking about their places."""
    s = world_state(case, seed)
    s["world"].tick(64)
    rng = np.random.default_rng(seed)
    n, lo, hi = case["bodies"], case["body_lo"], case["body_hi"]
    shape = np.random.default_rng(n).integers(lo, hi + 1, (n, 2))
    offset = np.concatenate([[0], np.cumsum(shape[:, 0] * shape[:, 1])])
    total = int(offset[-1])
    mats = rng.choice([fsg.MAT_STONE, fsg.MAT_WOOD], total)
    mats[rng.random(total) < 0.1] = fsg.MAT_AIR
    px = mats.astype(np.uint64) | (np.uint64(320) << np.uint64(16))
    px |= rng.integers(0, 2**32, total, dtype=np.uint64) << np.uint64(32)
    px[mats == fsg.MAT_AIR] = 0
    at = rng.uniform(0, 1, (n, 2)) * [case["width"], case["height"]]
    turn = rng.uniform(0, 2 * math.pi, n)
    s["poses"] = []
    for k in range(32):
        d = math.sin(2 * math.pi * k / 32)
        s["poses"].append([fsg.body_from_pose(at[b, 0] + 8 * d, at[b, 1] + 4 * d, turn[b] + 0.2 * d, int(shape[b, 1]),
                                              int(shape[b, 0]), int(offset[b])) for b in range(n)])
    s["pixels"], s["frame"] = px, 0
    s["displaced"] = np.zeros((512, 3), np.uint64)  # the frame's displaced cells, for new particles
    return s


def run_bodies(s):
    w = s["world"]
    r = w.stamp_bodies(s["poses"][s["frame"] % 32], s["pixels"], displaced_cap=512)
    s["frame"] += 1
    w.tick(1)
    w.render(fsg.LAYER_CELLS)  # the frame is drawn while the bodies are in the grid
    s["pixels"] = w.unstamp_bodies(s["pixels"].size)
    if r["displaced_cells"]:
        s["displaced"][:len(r["displaced_cells"])] = r["displaced_cells"]
    return {"counts": [r["placed"], r["unplaced"], r["displaced"]], "displaced": s["displaced"].view(np.int64),
            "hits": [np.array(r["hits_sand"], np.int64), np.array(r["hits_soup"], np.int64)],
            "pixels": s["pixels"].view(np.int64), "texture": s["textures"][0]}


# --- mesh -------------------------------------------------------------------
def prepare_mesh(case, seed):
    """Basin terrain with loose stone scattered over it, and every chunk of
    the world as a region."""
    s = world_state(case, seed)
    w = s["world"]
    cells = w.download()
    rng = np.random.default_rng(seed)
    loose = rng.random(cells.shape, dtype=np.float32) < case["loose"]
    cells[loose] = np.uint64(fsg.make_cell(fsg.MAT_STONE, 320, 0xFF808080))
    w.upload(cells)
    at = [(x, y, min(CHUNK, case["width"] - x), min(CHUNK, case["height"] - y))
          for y in range(0, case["height"], CHUNK) for x in range(0, case["width"], CHUNK)]
    s["regions"] = (fsg._abi.MeshRegion * len(at))(*[fsg._abi.MeshRegion(*r) for r in at])
    # the program's own arrays for the outlines of a frame
    s["loops"] = np.zeros((cells.size // 8, ctypes.sizeof(fsg._abi.MeshLoop) // 4), np.int32)
    s["vertices"] = np.zeros((cells.size, 2), np.float32)
    return s


def run_mesh(s):
    loops, vertices = ctypes.c_uint32(), ctypes.c_uint32()
    L, w = fsg.lib(), s["world"]
    fsg.check(L.fsg_world_mesh(w.handle, s["regions"], len(s["regions"]), ctypes.byref(loops),
                               ctypes.byref(vertices)), "fsg_world_mesh")
    fsg.check(L.fsg_world_mesh_download(w.handle, s["loops"].ctypes.data, len(s["loops"]), s["vertices"].ctypes.data,
                                        len(s["vertices"])), "fsg_world_mesh_download")
    return [loops.value, vertices.value, np.frombuffer(s["regions"], np.int32), s["loops"], s["vertices"]]


# --- particles --------------------------------------------------------------
PARTICLE = np.dtype([("f", np.float32, 9), ("lifetime", np.int32), ("flags", np.uint32), ("state", np.uint32),
                     ("cell", np.uint64)], align=False)


def burst(rng, n, width, height):
    """n sand, water and oil cells thrown about in the upper half."""
    a = np.zeros(n, PARTICLE)
    a["f"][:, 0] = rng.uniform(1, width - 1, n)
    a["f"][:, 1] = rng.uniform(1, height * 0.5, n)
    a["f"][:, 2:4] = rng.uniform(-1, 1, (n, 2))
    a["f"][:, 5] = 0.1
    a["cell"] = rng.choice([fsg.MAT_SAND, fsg.MAT_WATER, fsg.MAT_OIL], n).astype(np.uint64) | np.uint64(320 << 16)
    a["cell"] |= np.uint64(0xFF808080 << 32)
    return list((fsg._abi.Particle * n).from_buffer_copy(a.tobytes()))


def prepare_particles(case, seed):
    s = world_state(case, seed)
    rng = np.random.default_rng(seed)
    s["world"].particles_add(burst(rng, case["particles"], case["width"], case["height"]))
    for _ in range(20):  # under way
        s["world"].particles_tick()
    s["bursts"] = [burst(rng, case["burst"], case["width"], case["height"]) for _ in range(16)]
    s["frame"] = 0
    return s


def run_particles(s):
    w = s["world"]
    w.particles_add(s["bursts"][s["frame"] % 16])
    s["frame"] += 1
    alive, landed = w.particles_tick()
    w.render(fsg.LAYER_CELLS)
    return [alive, landed, s["textures"][0]]


# --- pack, unpack -----------------------------------------------------------
def prepare_pack(case, seed):
    case = dict(case, width=case["chunks_x"] * CHUNK, height=case["chunks_y"] * CHUNK)
    s = world_state(case, seed)
    s["world"].tick(16)
    # a save buffer of the cells' own size
    s["buffer"] = np.zeros(case["chunks_x"] * case["chunks_y"] * 8 * CHUNK * CHUNK, np.uint8)
    return s


def run_pack(s):
    case, w = s["case"], s["world"]
    sizes = w.pack(0, 0, case["chunks_x"], case["chunks_y"], download=False)
    fsg.check(fsg.lib().fsg_world_pack_download(w.handle, s["buffer"].ctypes.data, s["buffer"].size),
              "fsg_world_pack_download")
    return [np.array(sizes, np.int64), s["buffer"]]


def prepare_unpack(case, seed):
    s = prepare_pack(case, seed)
    c, w = s["case"], s["world"]
    s["images"] = w.pack(0, 0, c["chunks_x"], c["chunks_y"])
    w.generate(1, seed)
    return s


def run_unpack(s):
    c, w = s["case"], s["world"]
    status, phase, _, _ = w.unpack(0, 0, c["chunks_x"], c["chunks_y"], s["images"])
    w.render(fsg.LAYER_CELLS)
    return [status, phase, s["textures"][0]]


# ----------------------------------------------------------------------------
def listed():
    return [
        # a small game: one tick and its texture, the smallest call, all latency
        {"name": "frame 512", "op": "frame", "kind": 1, "width": 512, "height": 512, "skip": 0, "zone": False,
         "check": False, "census": False, "layers": 1, "view_w": 512, "view_h": 512},
        # the reference's frame on a large world: zone, island check, the three layers of the screen, census
        {"name": "frame 4096", "op": "frame", "kind": 2, "width": 4096, "height": 4096, "skip": 1, "zone": True,
         "check": True, "census": True, "layers": 3, "view_w": 1920, "view_h": 1080},
        # the small benchmark world, simulated and saved
        {"name": "run 512", "op": "run", "kind": 1, "width": 512, "height": 512, "ticks": 1000, "skip": 0,
         "temp_every": 1, "save": True},
        # a world between the sizes, of odd sides, at the reference's temperature cadence
        {"name": "run 1000x611", "op": "run", "kind": 2, "width": 1000, "height": 611, "ticks": 300, "skip": 0,
         "temp_every": 4, "save": True},
        # the reacting benchmark world, with dirty-chunk skipping
        {"name": "run 4096 skip", "op": "run", "kind": 2, "width": 4096, "height": 4096, "ticks": 200, "skip": 1,
         "temp_every": 1, "save": False},
        # the all-active benchmark world, the largest
        {"name": "run 16384", "op": "run", "kind": 3, "width": 16384, "height": 16384, "ticks": 16, "skip": 0,
         "temp_every": 1, "save": False},
        # environments of uneven sizes advanced together
        {"name": "batch 32", "op": "batch", "worlds": 32, "side_lo": 256, "side_hi": 2048, "step": 64, "ticks": 64,
         "skip": 1},
        # a frame with rigid bodies
        {"name": "bodies 100", "op": "bodies", "kind": 2, "width": 2048, "height": 1536, "bodies": 100, "body_lo": 16,
         "body_hi": 48, "skip": 1},
        # the physics engine's outlines of broken terrain
        {"name": "mesh 2048", "op": "mesh", "kind": 2, "width": 2048, "height": 2048, "loose": 0.2},
        # debris in the air
        {"name": "particles 40k", "op": "particles", "kind": 2, "width": 4096, "height": 4096, "particles": 40000,
         "burst": 256},
        # a region saved, and a region loaded
        {"name": "pack 16x16", "op": "pack", "kind": 4, "chunks_x": 16, "chunks_y": 16},
        {"name": "unpack 16x16", "op": "unpack", "kind": 4, "chunks_x": 16, "chunks_y": 16},
    ]


def draw(rng):
    def spread(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def sides(lo, hi):
        side, a = spread(lo, hi), math.sqrt(rng.uniform(0.5, 2.0))
        w, h = max(lo // 2, int(side * a)), max(lo // 2, int(side / a))
        return (w, h) if rng.random() < 0.5 else (max(64, w // 64 * 64), max(64, h // 64 * 64))

    op = rng.choice(["frame"] * 2 + ["run"] * 5 + ["batch"] * 2 + ["bodies", "mesh", "particles", "pack", "unpack"])
    if op == "frame":
        w, h = sides(384, 4096)
        w, h = max(w, 384), max(h, 384)
        return {"op": op, "kind": rng.choice([1, 2, 4]), "width": w, "height": h, "skip": rng.randrange(2),
                "zone": rng.random() < 0.5, "check": rng.random() < 0.5, "census": rng.random() < 0.5,
                "layers": rng.choice([1, 3]), "view_w": rng.choice([640, 1280, 1920]),
                "view_h": rng.choice([360, 720, 1080])}
    if op == "run":
        w, h = sides(128, 8192)
        ticks = max(4, min(spread(16, 1000), MOST_UPDATES // (w * h)))
        return {"op": op, "kind": rng.choice([1, 2, 3, 4]), "width": w, "height": h, "ticks": ticks,
                "skip": rng.randrange(2), "temp_every": rng.choice([1, 1, 4]), "save": w * h <= 1 << 20}
    if op == "batch":
        return {"op": op, "worlds": rng.randint(2, 48), "side_lo": rng.choice([64, 128, 256]),
                "side_hi": rng.choice([512, 1024, 2048]), "step": rng.choice([1, 64]), "ticks": spread(8, 128),
                "skip": rng.randrange(2)}
    if op == "bodies":
        w, h = sides(512, 3072)
        lo = rng.randint(4, 32)
        return {"op": op, "kind": rng.choice([1, 2, 4]), "width": w, "height": h, "bodies": spread(1, 200),
                "body_lo": lo, "body_hi": lo + rng.randint(0, 32), "skip": rng.randrange(2)}
    if op == "mesh":
        w, h = sides(384, 3072)
        return {"op": op, "kind": rng.choice([1, 2, 4]), "width": w, "height": h,
                "loose": round(rng.choice([0.0, rng.uniform(0.01, 0.5)]), 3)}
    if op == "particles":
        w, h = sides(1024, 4096)
        return {"op": op, "kind": rng.choice([1, 2, 4]), "width": w, "height": h, "particles": spread(500, 60000),
                "burst": spread(16, 256)}
    return {"op": op, "kind": rng.choice([1, 2, 4]), "chunks_x": spread(1, 24), "chunks_y": spread(1, 24)}


PREPARE = {"frame": prepare_frame, "run": prepare_run, "batch": prepare_batch, "bodies": prepare_bodies,
           "mesh": prepare_mesh, "particles": prepare_particles, "pack": prepare_pack, "unpack": prepare_unpack}
RUN = {"frame": run_frame, "run": run_run, "batch": run_batch, "bodies": run_bodies, "mesh": run_mesh,
       "particles": run_particles, "pack": run_pack, "unpack": run_unpack}


def prepare(case, seed):
    s = PREPARE[case["op"]](case, seed)
    s["op"] = case["op"]
    return s


def run(state):
    return RUN[state["op"]](state)


def exact(case, seed):
    """Cells, texels, counts and images are whole numbers; the outlines'
    vertices are corners of cells, chosen and not computed."""
    return None


def work(case):
    """Bytes: a tick reads and writes each cell (8 bytes); drawing reads a cell
    and writes a 4-byte texel per layer.  No floating-point work."""
    op = case["op"]
    if op == "batch":
        n = sum(w * h for w, h in batch_sizes(case, np.random.default_rng(case["worlds"])))
        return {"bytes": n * (16 * case["ticks"] + 12), "flops": 0}
    if op in ("pack", "unpack"):  # the cells, and images of about a ninth of the 28-byte records
        n = case["chunks_x"] * case["chunks_y"] * CHUNK * CHUNK
        return {"bytes": n * (8 + 3) + (12 * n if op == "unpack" else 0), "flops": 0}
    n = case["width"] * case["height"]
    if op == "frame":
        view = min(case["view_w"], case["width"]) * min(case["view_h"], case["height"])
        return {"bytes": 16 * n + view * (8 + 4 * case["layers"] + (8 if case["census"] else 0)), "flops": 0}
    if op == "run":
        return {"bytes": 16 * n * case["ticks"] + (8 if case["save"] else 16) * n, "flops": 0}
    if op == "bodies":  # each pixel in and out, the grid cell under it read and written each way
        side = (case["body_lo"] + case["body_hi"]) / 2
        return {"bytes": 28 * n + int(case["bodies"] * side * side) * 48, "flops": 0}
    if op == "mesh":
        return {"bytes": 8 * n, "flops": 0}
    return {"bytes": 12 * n + 112 * (case["particles"] + case["burst"]), "flops": 0}
