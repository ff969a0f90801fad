"""Performance cases of the neural ray query and its companions, through the Python interface.

listed() names the cases, draw() gives more of the same ranges; prepare() makes a case's inputs and
what a program keeps between calls (scene, weights, trainer, workspace), run() is one call as a
program makes it, work() the bytes and operations it cannot do without, exact() the result in 64
bits where it is a computed number (it needs no part of the package).

Device buffers are torch tensors: torch is imported first, so the library binds torch's HIP
runtime and both share the device and its default stream.
"""
import ctypes
import math
import weakref
from collections import namedtuple

import numpy as np
import torch

import nbvh_amd as nb
from nbvh_amd import _ffi

# MLP 96 -> 64 x 4 -> 8 of both network shapes in use, per segment.
FLOP_PER_SEGMENT = 2 * (96 * 64 + 3 * 64 * 64 + 64 * 8)
PRECISIONS = {"fp32": nb.PREC_FP32, "fp16": nb.PREC_FP16, "bf16": nb.PREC_BF16, "fp8": nb.PREC_FP8}
# The two network shapes that the MFMA and training kernels serve: the benchmark's grid and that
# of the reference's shipped chess model.
NETWORKS = {"16x2": dict(n_levels=16, n_features_per_level=2, log2_hashmap_size=19, base_resolution=16,
                         per_level_scale=1.5),
            "8x4": dict(n_levels=8, n_features_per_level=4, log2_hashmap_size=18, base_resolution=8,
                        per_level_scale=2.0)}
FLT_MAX = float(np.finfo(np.float32).max)


def listed():
    return [
        # The smallest request a server gets: 4,096 camera rays of one tile. Launch latency, weight
        # staging and a nearly empty chip.
        dict(name="request_4k", kind="frame", width=64, height=64, network="16x2", precision="fp16", tables=1e-4),
        # An ordinary frame of the benchmark: 1024 x 1024 camera rays, FP16 matrix cores.
        dict(name="frame_1m", kind="frame", width=1024, height=1024, network="16x2", precision="fp16", tables=1e-4),
        # The same frame through the FP32 query, the path that is bit-exact with the oracle.
        dict(name="frame_1m_fp32", kind="frame", width=1024, height=1024, network="16x2", precision="fp32",
             tables=1e-4),
        # The other network shape on a frame whose sides are no multiples of 8 (no tiled claim
        # order, a last wave that is not full), BF16.
        dict(name="frame_odd_8x4_bf16", kind="frame", width=1013, height=691, network="8x4", precision="bf16",
             tables=1e-4),
        # The largest query: a wavefront of incoherent closest-hit and shadow rays over 64 objects
        # in one two-part launch, traced in the coherence order.
        dict(name="wavefront_4m", kind="wavefront", closest=1 << 21, shadow=1 << 21, network="16x2",
             precision="fp16", sort=True, tables=1e-4),
        # The triangle query beside it: incoherent rays over a triangle BVH that no cache holds.
        dict(name="triangles_1m", kind="triangles", closest=1 << 20, shadow=0),
        # A whole path-traced frame of the object alone, 1 sample per pixel, 5 vertices.
        dict(name="path_1080p", kind="path", width=1920, height=1080, network="16x2", precision="fp16", hybrid=False,
             tables=1e-4),
        # A whole frame of the object inside a triangle environment, sides no multiples of 8, FP32.
        dict(name="path_odd_hybrid_fp32", kind="path", width=957, height=541, network="16x2", precision="fp32",
             hybrid=True, tables=1e-4),
        # The network alone on encoded segments (the replacement of the reference's inference call).
        dict(name="network_1m", kind="network", n=1 << 20, network="16x2", precision="fp16", tables=0.1),
        # Four training steps of the ordinary batch: forward, backward and Adam; the loss is read
        # after the last.
        dict(name="train_64k", kind="train", n=1 << 16, steps=4, network="16x2", tables=1e-4),
        # Four steps of a small odd batch on the other network shape.
        dict(name="train_odd_8x4", kind="train", n=10007, steps=4, network="8x4", tables=1e-4),
        # The image error of a validation run, at its usual frame size.
        dict(name="flip_1080p", kind="flip", width=1920, height=1080),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frame", "frame", "frame", "wavefront", "triangles", "path", "network", "train", "flip"])
    net = rng.choice(["16x2", "16x2", "8x4"])
    prec = rng.choice(["fp16", "fp16", "bf16", "fp32", "fp8"])
    if kind in ("frame", "path", "flip"):
        pixels = _log(rng, 4096, 1 << 20 if kind == "frame" else 1 << 19)
        width = max(16, int(math.sqrt(pixels * rng.uniform(0.5, 2.0))))
        if rng.random() < 0.4:
            width, height = -(-width // 8) * 8, -(-max(16, pixels // width) // 8) * 8
        else:
            height = max(16, pixels // width) | 1
        if kind == "flip":
            return dict(kind=kind, width=width, height=height)
        case = dict(kind=kind, width=width, height=height, network=net, precision=prec, tables=1e-4)
        if kind == "path":
            case["precision"], case["hybrid"] = rng.choice(["fp16", "fp32"]), rng.random() < 0.5
        return case
    if kind == "wavefront":
        return dict(kind=kind, closest=_log(rng, 1 << 12, 1 << 20), shadow=_log(rng, 1 << 12, 1 << 20), network=net,
                    precision=prec, sort=rng.random() < 0.6, tables=1e-4)
    if kind == "triangles":
        return dict(kind=kind, closest=_log(rng, 1 << 12, 1 << 20), shadow=rng.choice([0, _log(rng, 1 << 12, 1 << 19)]))
    if kind == "network":
        return dict(kind=kind, n=_log(rng, 1 << 10, 1 << 20), network=net, precision=prec, tables=0.1)
    return dict(kind=kind, n=_log(rng, 1 << 11, 1 << 16), steps=4, network=net, tables=1e-4)


# ---------------------------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------------------------
Buffer = namedtuple("Buffer", "ptr nbytes")  # what path_params takes as a workspace


class State:
    """What a program keeps: the library's objects, closed with the state, and the call's tensors."""

    def __init__(self, case):
        self.case = case
        self.ctx = nb.Context()
        self._owned = [self.ctx]
        weakref.finalize(self, State._close, self._owned)

    @staticmethod
    def _close(owned):
        while owned:
            owned.pop().close()

    def own(self, obj):
        self._owned.append(obj)
        return obj


def _config(case):
    return nb.network_config(**NETWORKS[case["network"]])


def _weights(case, seed):
    """Tables U(+-case["tables"]) and Kaiming-uniform matrices, as numpy float32. The visibility
    row is centred on the mean activation it meets: without that an untrained network sees nothing
    at all or everything, depending on the seed, while a trained one decides about half of the
    segments either way."""
    n_table, _ = nb.network_param_counts(_config(case))
    g = torch.Generator(device="cuda").manual_seed(seed)
    tables = (torch.rand(n_table, generator=g, device="cuda") * 2 - 1) * case["tables"]
    r = np.random.default_rng(seed)
    mlp = [r.uniform(-1, 1, (o, i)) * math.sqrt(6.0 / i) for o, i in ((64, 96), (64, 64), (64, 64), (64, 64), (8, 64))]
    h = r.normal(size=(1024, 96))
    for w in mlp[:-1]:
        h = np.maximum((h[:, None, :] * w).sum(-1), 0.0)  # no BLAS: the same bits everywhere
    h = h.mean(0)
    mlp[-1][0] -= (mlp[-1][0] * h).sum() / (h * h).sum() * h
    return tables.cpu().numpy(), np.concatenate([w.ravel() for w in mlp]).astype(np.float32)


def _rays(o, d, tmax):
    r = torch.empty(len(o), 8, device="cuda")
    r[:, 0:3], r[:, 3], r[:, 4:7], r[:, 7] = o, 1e-4, d, tmax
    return r


def _directions(n, g):
    d = torch.randn(n, 3, generator=g, device="cuda")
    return d / d.norm(dim=1, keepdim=True)


def _object(st, case, seed):
    """The benchmark's object: a displaced icosphere of 81,920 triangles, N-BVH of 256 leaves."""
    sc = st.own(nb.Scene(st.ctx, *nb.icosphere(6, seed=7 + seed, amplitude=0.1)))
    sc.build_nbvh(256)
    sc.load_network_model(_config(case), *_weights(case, seed))
    return sc


def _camera(seed, width, height):
    r = np.random.default_rng(seed)
    eye = r.normal(size=3)
    eye *= 3.0 / np.linalg.norm(eye)
    return nb.camera_look_at(eye, (0, 0, 0), (0, 1, 0) if abs(eye[1]) < 2.5 else (1, 0, 0), 45.0, width, height)


def _field(seed):
    """64 displaced spheres in the unit cube, about a million triangles."""
    return nb.sphere_field(64, seed=5 + seed, freq_range=(20, 34))


def _field_rays(verts, tris, n_closest, n_shadow, seed):
    """Incoherent rays from uniform origins, and shadow rays from the surfaces to 8 lights."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    closest = _rays(torch.rand(n_closest, 3, generator=g, device="cuda"), _directions(n_closest, g), FLT_MAX)
    v, t = torch.from_numpy(verts).cuda().double(), torch.from_numpy(tris.astype(np.int64)).cuda()
    lights = torch.rand(8, 3, generator=g, device="cuda").double() * 1.5 - 0.25
    tri = t[torch.randint(0, len(t), (n_shadow,), generator=g, device="cuda")]
    a, b, c = v[tri[:, 0]], v[tri[:, 1]], v[tri[:, 2]]
    w = torch.rand(n_shadow, 2, generator=g, device="cuda").double()
    w = torch.where(w.sum(1, keepdim=True) > 1, 1 - w, w)
    p = a + (b - a) * w[:, :1] + (c - a) * w[:, 1:]
    nrm = torch.linalg.cross(b - a, c - a)
    nrm = nrm / nrm.norm(dim=1, keepdim=True).clamp_min(1e-30)
    to = lights[torch.randint(0, 8, (n_shadow,), generator=g, device="cuda")] - p
    o = p + 1e-4 * torch.sign((to * nrm).sum(1, keepdim=True)) * nrm
    dist = to.norm(dim=1, keepdim=True)
    return closest, _rays(o.float(), (to / dist).float(), dist[:, 0].float())


def _encode(rays, mint, maxt, lo, hi):
    """The three points (entry, middle, exit) of segments, in the encoding box, float32 [n, 9]."""
    lo, hi = (torch.from_numpy(np.asarray(x, np.float32)).cuda() for x in (lo, hi))
    center, extent = (hi + lo) * 0.5, (hi - lo) * float(np.float32(1.0 + 1e-4) + np.float32(1e-5))
    po = rays[:, 0:3] + mint[:, None] * rays[:, 4:7]
    pi = rays[:, 0:3] + maxt[:, None] * rays[:, 4:7]
    eo, ei = (po - center) / extent + 0.5, (pi - center) / extent + 0.5
    return torch.cat([eo, 0.5 * eo + 0.5 * ei, ei], dim=1).contiguous()


def _segments(sc, n, seed):
    """n segments through the leaves of the scene's N-BVH: device rays, entries and exits."""
    rays, mint, maxt = nb.leaf_segments(sc.nbvh(), n, seed=seed)
    return (torch.from_numpy(rays.view(np.float32).reshape(n, 8)).cuda(), torch.from_numpy(mint).cuda(),
            torch.from_numpy(maxt).cuda())


def _environment():
    """A floor and four spheres around the object, as triangles."""
    vs = [np.array([[-3, -1.3, -3], [3, -1.3, -3], [3, -1.3, 3], [-3, -1.3, 3]], np.float32)]
    ts, off = [np.array([[0, 2, 1], [0, 3, 2]], np.uint32)], 4
    for i, c in enumerate([(1.6, -0.8, 0.2), (-1.5, -0.7, -0.4), (0.3, 1.5, -0.9), (-0.2, -0.9, 1.6)]):
        v, t = nb.geosphere(12, seed=40 + i, amplitude=0.05, center=c, radius=0.45)
        vs.append(v)
        ts.append(t + np.uint32(off))
        off += len(v)
    return np.concatenate(vs), np.concatenate(ts)


def _flip_images(case, seed):
    """Two noisy accumulation images of a smooth scene, 4 samples a pixel."""
    w, h = case["width"], case["height"]
    g = torch.Generator(device="cuda").manual_seed(seed)
    y, x = torch.meshgrid(torch.linspace(0, 1, h, device="cuda"), torch.linspace(0, 1, w, device="cuda"),
                          indexing="ij")
    k = torch.rand(3, 2, generator=g, device="cuda") * 24 + 2
    base = torch.stack([0.5 + 0.4 * torch.sin(k[c, 0] * x + k[c, 1] * y) for c in range(3)], dim=-1)
    images = []
    for noise in (0.01, 0.08):
        rgb = (base + noise * torch.randn(h, w, 3, generator=g, device="cuda")).clamp_min(0.0) * 4.0
        images.append(torch.cat([rgb, torch.full((h, w, 1), 4.0, device="cuda")], dim=-1).contiguous())
    return images


def prepare(case, seed):
    st = State(case)
    kind = case["kind"]
    if kind == "flip":
        st.images = _flip_images(case, seed)
        st.map = torch.empty(case["height"], case["width"], device="cuda")
    elif kind == "frame":
        w, h = case["width"], case["height"]
        st.module = nb.NeuralBVHModule(st.ctx, _object(st, case, seed))
        st.rays = torch.empty(w * h, 8, device="cuda")
        st.ctx.raygen(_camera(seed, w, h), w, h, st.rays.data_ptr())
        st.hits = torch.empty(w * h, 12, device="cuda")
        st.params = st.module.params(precision=PRECISIONS[case["precision"]], image_width=w)
    elif kind in ("wavefront", "triangles"):
        verts, tris = _field(seed)
        sc = st.own(nb.Scene(st.ctx, verts, tris))
        st.module = nb.NeuralBVHModule(st.ctx, sc)
        if kind == "wavefront":
            sc.build_nbvh(4096)
            sc.load_network_model(_config(case), *_weights(case, seed))
            st.params = st.module.params(precision=PRECISIONS[case["precision"]], sort_rays=case["sort"])
        else:
            st.params = st.module.params(kind=nb.QUERY_TRIANGLE_CLOSEST)
        n = (case["closest"], case["shadow"])
        st.rays = [r for r in _field_rays(verts, tris, max(n[0], 1), max(n[1], 1), seed)]
        st.hits = [torch.empty(m, 12, device="cuda") for m in n]
        st.parts = [(st.rays[k].data_ptr(), n[k], st.hits[k].data_ptr(), k == 1) for k in (0, 1) if n[k]]
    elif kind == "path":
        w, h = case["width"], case["height"]
        st.module = nb.NeuralBVHModule(st.ctx, _object(st, case, seed))
        st.environment = st.own(nb.Scene(st.ctx, *_environment())) if case["hybrid"] else None
        st.camera = _camera(seed, w, h)
        st.image = torch.empty(h, w, 4, device="cuda")
        opts = dict(precision=PRECISIONS[case["precision"]], max_depth=5, rr_start_depth=3)
        size = st.module.path_trace_workspace_size(st.module.path_params(w, h, **opts), w, h, st.environment)
        st.workspace = torch.empty(size, dtype=torch.uint8, device="cuda")
        st.params = st.module.path_params(w, h, workspace=Buffer(st.workspace.data_ptr(), size), **opts)
    else:
        sc = _object(st, case, seed)
        st.module = nb.NeuralBVHModule(st.ctx, sc)
        n = case["n"] * (case["steps"] if kind == "train" else 1)
        rays, mint, maxt = _segments(sc, n, seed)
        st.inputs = _encode(rays, mint, maxt, *sc.bbox())
        if kind == "train":
            st.targets = torch.empty(n, 8, device="cuda")
            st.ctx.check(_ffi.lib().nbvh_segment_labels(
                st.ctx.handle, sc.handle, ctypes.c_void_p(rays.data_ptr()), ctypes.c_void_p(mint.data_ptr()),
                ctypes.c_void_p(maxt.data_ptr()), n, ctypes.c_void_p(st.targets.data_ptr()), None))
            st.trainer = st.own(nb.Trainer(st.ctx, sc, max_batch=case["n"]))
        else:
            st.outputs, st.logits = torch.empty(n, 8, device="cuda"), torch.empty(n, 8, device="cuda")
    torch.cuda.synchronize()
    return st


# ---------------------------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------------------------
def _records(hits):
    """A hit buffer's fields: distances, ids (triangle, node, info word), and the rest."""
    return {"t": hits[:, 0], "ids": hits.view(torch.int32)[:, 1:4], "normal": hits[:, 4:7], "logit": hits[:, 7],
            "albedo": hits[:, 8:11]}


def run(st):
    case, kind = st.case, st.case["kind"]
    if kind == "frame":
        st.module.query_device(st.params, st.rays.data_ptr(), len(st.rays), st.hits.data_ptr())
        return _records(st.hits)
    if kind in ("wavefront", "triangles"):
        st.module.query_parts_device(st.params, st.parts)
        return [_records(h) for h in st.hits if len(h)]
    if kind == "path":
        st.module.path_trace_params_device(st.params, st.camera, case["width"], case["height"], st.image.data_ptr(),
                                           st.environment, stats=False)
        return st.image
    if kind == "network":
        st.module.network_inference_device(PRECISIONS[case["precision"]], st.inputs.data_ptr(), case["n"],
                                           st.outputs.data_ptr(), st.logits.data_ptr())
        return {"outputs": st.outputs, "logits": st.logits}
    if kind == "train":
        n, loss = case["n"], None
        for k in range(case["steps"]):
            loss = st.trainer.step_device(st.inputs[k * n].data_ptr(), st.targets[k * n].data_ptr(), n,
                                          want_loss=k + 1 == case["steps"])
        return {"loss": torch.tensor(loss), "mlp": st.trainer.get(nb.TRAIN_MLP)}
    mean = ctypes.c_float()
    st.ctx.check(_ffi.lib().nbvh_flip(
        st.ctx.handle, ctypes.c_void_p(st.images[0].data_ptr()), ctypes.c_void_p(st.images[1].data_ptr()),
        case["width"], case["height"], 0.0, ctypes.c_void_p(st.map.data_ptr()), ctypes.byref(mean), None))
    return {"mean": torch.tensor(mean.value), "map": st.map}


# ---------------------------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    if kind == "flip":
        # Two images in, the map out; the filters as separable passes (21 + 21 taps of 4 Gaussians,
        # 19 + 19 of the 4 feature responses, two images).
        n = case["width"] * case["height"]
        return {"bytes": n * 36, "flops": n * 2 * 2 * (4 * 42 + 4 * 38)}
    if kind == "triangles":
        # Rays in, records out, the triangles and their tree once; two box tests (24) on about 20
        # levels of nodes and two triangle tests (45) a ray.
        n, tris = case["closest"] + case["shadow"], 64 * 20 * 27 * 27
        return {"bytes": n * 80 + tris * (12 + 6 + 2 * 32), "flops": n * (20 * 48 + 2 * 45)}
    entries, features = {"16x2": (6513496, 2), "8x4": (1348096, 4)}[case["network"]]
    half = case.get("precision", "fp32") != "fp32"
    weights = entries * features * (2 if half else 4) + 18944 * (2 if half else 4)
    # One network evaluation: the MLP and the interpolation of 8 corners by 96 features.
    segment = FLOP_PER_SEGMENT + 2 * 8 * 96
    if kind == "network":
        return {"bytes": case["n"] * (36 + 64) + weights, "flops": case["n"] * segment}
    if kind == "train":
        # Forward, two products backward; inputs and targets once, the tables' weights, moments and
        # counts read and written once a step.
        n = case["n"]
        return {"bytes": case["steps"] * (n * 68 + entries * features * 32), "flops": case["steps"] * n * 3 * segment}
    if kind == "wavefront":
        n = case["closest"] + case["shadow"]
        return {"bytes": n * 80 + weights + 8191 * 32, "flops": n * 2 * segment}
    n = case["width"] * case["height"]
    if kind == "path":  # the object fills about a third of the frame; paths go on from its hits
        return {"bytes": n * 16 + weights + 511 * 32, "flops": n * 1.6 * segment}
    return {"bytes": n * 80 + weights + 511 * 32, "flops": n * segment}


# ---------------------------------------------------------------------------------------------
# Results in 64 bits
# ---------------------------------------------------------------------------------------------
def exact(case, seed):
    """The network, the training steps and the image error in float64. Hit records and frames have
    no such value: which segment a ray accepts is decided in the query's own precision (nearest
    accepted depth, visibility sign), and a decision that falls the other way is another hit."""
    kind = case["kind"]
    if kind == "flip":
        return _exact_flip(*_flip_images(case, seed))
    if kind not in ("network", "train"):
        return None
    st = prepare(case, seed)  # the inputs alone
    tables, mlp = (torch.from_numpy(w).cuda().double() for w in _weights(case, seed))
    grid, n = NETWORKS[case["network"]], case["n"]
    if kind == "network":
        z = torch.cat([_forward(grid, tables, _matrices(mlp), x)[0] for x in st.inputs.split(1 << 17)])
        return {"outputs": torch.sigmoid(z), "logits": z}
    return _exact_train(grid, tables, mlp, st.inputs.view(-1, n, 9), st.targets.view(-1, n, 8).double())


def _matrices(mlp):
    sizes = [(64, 96), (64, 64), (64, 64), (64, 64), (8, 64)]
    return [m.view(s) for m, s in zip(mlp.split([a * b for a, b in sizes]), sizes)]


def _levels(grid):
    """(scale, resolution, size, first entry, dense) of each level, formed in float32."""
    out, first, top = [], 0, 1 << grid["log2_hashmap_size"]
    log2s = np.log2(np.float32(grid["per_level_scale"]))
    for level in range(grid["n_levels"]):
        scale = np.exp2(np.float32(level) * log2s) * np.float32(grid["base_resolution"]) - np.float32(1)
        res = int(math.ceil(float(scale))) + 1
        size = min(-(-res ** 3 // 8) * 8, top)
        out.append((float(np.float32(scale)), res, size, first, res ** 3 <= size))
        first += size
    return out


def _corners_of(grid, x):
    """Per point and level: the corners' entries [n, 8] and weights [n, 8]. Positions are rounded
    to float32 as the grid defines them (one rounding of scale * x + 0.5), the rest is float64."""
    for p in range(3):
        for scale, res, size, first, dense in _levels(grid):
            pos = (x[:, 3 * p:3 * p + 3].double() * scale + 0.5).float()
            cell = torch.floor(pos)
            frac, cell = (pos - cell).double(), cell.long()
            idx, wgt = [], []
            for c in range(8):
                bit = [(c >> d) & 1 for d in range(3)]
                q = [cell[:, d] + bit[d] for d in range(3)]
                if dense:
                    i = (q[0] + q[1] * res + q[2] * res * res) % size
                else:
                    i = (q[0] ^ (q[1] * 2654435761 & 0xFFFFFFFF) ^ (q[2] * 805459861 & 0xFFFFFFFF)) & (size - 1)
                w = [frac[:, d] if bit[d] else 1 - frac[:, d] for d in range(3)]
                idx.append(i + first)
                wgt.append(w[0] * w[1] * w[2])
            yield torch.stack(idx, 1), torch.stack(wgt, 1)


def _forward(grid, tables, mats, x):
    """Logits, the layers' activations, the corners of a batch."""
    t = tables.view(-1, grid["n_features_per_level"])
    corners = list(_corners_of(grid, x))
    act = [torch.cat([(t[i] * w[:, :, None]).sum(1) for i, w in corners], dim=1)]
    for m in mats[:-1]:
        act.append(torch.relu(act[-1] @ m.T))
    return act[-1] @ mats[-1].T, act, corners


def _exact_train(grid, tables, mlp, inputs, targets):
    """The steps' Adam updates on the composite loss (cross entropy of the visibility; L1 depth, L1
    linearised normal and relative L2 albedo where the target is visible), in float64."""
    lr, b1, b2, eps, l2 = (float(np.float32(v)) for v in (1e-2, 0.9, 0.999, 1e-8, 1e-8))
    moments = {k: [torch.zeros_like(w), torch.zeros_like(w), torch.zeros_like(w)]
               for k, w in (("tables", tables), ("mlp", mlp))}
    loss = 0.0

    def adam(w, g, state, live):
        m, v, count = state
        m[live] = b1 * m[live] + (1 - b1) * g[live]
        v[live] = b2 * v[live] + (1 - b2) * g[live] ** 2
        count[live] += 1
        rate = lr * torch.sqrt(1 - b2 ** count[live]) / (1 - b1 ** count[live])
        w[live] -= rate * m[live] / (torch.sqrt(v[live]) + eps)

    for x, t in zip(inputs, targets):
        mats = _matrices(mlp)
        z, act, corners = _forward(grid, tables, mats, x)
        y, n = torch.sigmoid(z), len(x)
        p = y[:, :1].clamp(1e-5, 1 - 1e-5)
        values = [-(t[:, :1] * torch.log(p) + (1 - t[:, :1]) * torch.log(1 - p))]
        dy = [-(t[:, :1] - p) / (p - p * p)]
        keep = (t[:, :1] >= 0.5).double()
        d = y[:, 1:2] - t[:, 1:2]
        values.append(keep * d.abs())
        dy.append(keep * torch.copysign(torch.ones_like(d), d))
        d = ((y[:, 2:5] * 2 - 1) / 0.1) * 0.5 + 0.5 - t[:, 2:5]
        values.append(keep * d.abs())
        dy.append(keep * torch.copysign(torch.ones_like(d), d) / 0.1)
        d, den = y[:, 5:8] - t[:, 5:8], y[:, 5:8] ** 2 + 1e-2
        values.append(keep * d * d / den)
        dy.append(keep * 2 * d / den)
        loss = torch.cat(values, 1).sum() / (n * 8)
        delta = torch.cat(dy, 1) / (n * 8) * y * (1 - y)
        grads = []
        for layer in range(4, -1, -1):
            grads.append((delta.T @ act[layer]).reshape(-1))
            back = delta @ mats[layer]
            delta = back * (act[layer] > 0) if layer else back
        f = grid["n_features_per_level"]
        g_tables = torch.zeros_like(tables).view(-1, f)
        for k, (idx, wgt) in enumerate(corners):
            g_tables.index_add_(0, idx.reshape(-1), (wgt[:, :, None] * delta[:, None, k * f:k * f + f]).reshape(-1, f))
        g_tables, g_mlp = g_tables.view(-1), torch.cat(grads[::-1]) + l2 * mlp
        adam(tables, g_tables, moments["tables"], g_tables != 0)
        adam(mlp, g_mlp, moments["mlp"], torch.ones_like(mlp, dtype=torch.bool))
    return {"loss": loss, "mlp": mlp}


def _filter(img, k):
    """Correlation of an image [h, w] with a small kernel, edge pixels replicated."""
    r = len(k) // 2
    h, w = img.shape
    pad = torch.nn.functional.pad(img[None, None], (r, r, r, r), mode="replicate")[0, 0]
    out = torch.zeros_like(img)
    for dy in range(2 * r + 1):
        for dx in range(2 * r + 1):
            out += float(k[dy, dx]) * pad[dy:dy + h, dx:dx + w]
    return out


def _exact_flip(ref, test):
    """LDR-FLIP (Andersson et al., HPG 2020) at 0.7 m from a 0.7 m wide monitor of 3840 pixels."""
    ppd = 3840.0 * math.pi / 180.0
    to_xyz = torch.tensor([[10135552 / 24577794, 8788810 / 24577794, 4435075 / 24577794],
                           [2613072 / 12288897, 8788810 / 12288897, 887015 / 12288897],
                           [1425312 / 73733382, 8788810 / 73733382, 70074185 / 73733382]], dtype=torch.float64)
    to_rgb = torch.tensor([[3.241003275, -1.537398934, -0.498615861], [-0.969224334, 1.875930071, 0.041554224],
                           [0.055639423, -0.204011202, 1.057148933]], dtype=torch.float64)
    white = torch.tensor([0.950428545, 1.0, 1.088900371], dtype=torch.float64)
    inv_white = torch.tensor([1.052156925, 1.0, 0.918357670], dtype=torch.float64)
    to_xyz, to_rgb, white, inv_white = (m.to(ref.device) for m in (to_xyz, to_rgb, white, inv_white))

    def hunt_lab(rgb):
        f = rgb @ to_xyz.T * inv_white
        d = 6.0 / 29.0
        f = torch.where(f > d ** 3, f.clamp_min(1e-30) ** (1.0 / 3.0), f / (3 * d * d) + 4.0 / 29.0)
        light = 116 * f[..., 1] - 16
        return light, 0.01 * light * 500 * (f[..., 0] - f[..., 1]), 0.01 * light * 200 * (f[..., 1] - f[..., 2])

    def difference(a, b):
        return ((a[0] - b[0]).abs() + torch.sqrt((a[1] - b[1]) ** 2 + (a[2] - b[2]) ** 2)) ** 0.7

    def squares(r):
        y, x = np.mgrid[-r:r + 1, -r:r + 1].astype(np.float64)
        return x, x * x + y * y

    sensitivity, radius = [], math.ceil(3 * math.sqrt(0.04 / (2 * math.pi ** 2)) * ppd)
    for a1, b1, a2, b2 in ((1.0, 0.0047, 0.0, 1e-5), (1.0, 0.0053, 0.0, 1e-5), (34.1, 0.04, 13.5, 0.025)):
        d2 = squares(radius)[1] / ppd ** 2
        k = sum(a * math.sqrt(math.pi / b) * np.exp(-math.pi ** 2 * d2 / b) for a, b in ((a1, b1), (a2, b2)))
        sensitivity.append(k / k.sum())
    sd = 0.5 * 0.082 * ppd
    x, d2 = squares(math.ceil(3 * sd))
    gauss, detectors = np.exp(-d2 / (2 * sd * sd)), []
    for k in (-x * gauss, (x * x / (sd * sd) - 1) * gauss):
        k = np.where(k > 0, k / k[k > 0].sum(), np.where(k < 0, k / -k[k < 0].sum(), 0.0))
        detectors.append(k)
    labs, edges, points = [], [], []
    for img in (ref, test):
        c = img.double()
        c = torch.where(c[..., 3:] > 0, c[..., :3] / c[..., 3:].clamp_min(1e-30), torch.zeros_like(c[..., :3]))
        c = torch.where(c <= 0.0031308, 12.92 * c, 1.055 * c.clamp_min(0.0031308) ** (1 / 2.4) - 0.055).clamp(0, 1)
        c = torch.where(c <= 0.04045, c / 12.92, ((c + 0.055) / 1.055) ** 2.4)
        xyz = c @ to_xyz.T * inv_white
        lum = xyz[..., 1]
        ycc = [116 * lum - 16, 500 * (xyz[..., 0] - lum), 200 * (lum - xyz[..., 2])]
        y, cx, cz = (_filter(ch, k) for ch, k in zip(ycc, sensitivity))
        y = (y + 16) / 116
        rgb = torch.stack([cx / 500 + y, y, y - cz / 200], dim=-1) * white @ to_rgb.T
        labs.append(hunt_lab(rgb.clamp(0, 1)))
        edges.append(torch.hypot(_filter(lum, detectors[0]), _filter(lum, detectors[0].T)))
        points.append(torch.hypot(_filter(lum, detectors[1]), _filter(lum, detectors[1].T)))
    pure = torch.eye(3, dtype=torch.float64, device=ref.device)
    cmax = float(difference(hunt_lab(pure[1]), hunt_lab(pure[2])))
    dec = difference(*labs)
    dec = torch.where(dec < 0.4 * cmax, 0.95 / (0.4 * cmax) * dec, 0.95 + (dec - 0.4 * cmax) / (0.6 * cmax) * 0.05)
    feature = torch.maximum((edges[0] - edges[1]).abs(), (points[0] - points[1]).abs()) / math.sqrt(2)
    error = dec ** (1 - torch.sqrt(feature))
    return {"mean": error.mean(), "map": error}
