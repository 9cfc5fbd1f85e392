"""The workloads this library's speed is measured on, each through its public
entry points (slam-hands_amd/slk.py over the C ABI of include/slk.h) on device
memory held by torch.

A DROID-SLAM host calls the library in four places: for every video frame
(decode, encode, motion filter), for every frontend update pass (correlation
of the window's edges, update operator, GraphAgg, bundle adjustment), for
every graph update (proximity factors), and in the backend (bundle adjustment
over all keyframes). The listed cases take one or more calls from each, from a
3-edge correlation on a small odd map to the 200-keyframe adjustment; sizes
and distributions are those of slam-hands_amd/workloads.py and the tests.

  listed()             the cases
  draw(rng)            another case of the same ranges
  prepare(case, seed)  inputs, weights and handles on the GPU
  run(state)           one pass, as a host program calls it
  work(case)           bytes and operations of a pass
  tolerance(case)      distance another correct implementation may have
  exact(case, seed)    the outputs in 64-bit arithmetic
"""
from __future__ import annotations

import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "slam-hands_amd"))

import slk  # noqa: E402

C = 128                # feature channels
ALPHA = 1.0 / 16.0     # correlation scale of the reference
MIN_DEPTH = 0.25
DEV = "cuda"
F64 = torch.float64


# ------------------------------------------------------------------- cases --
def listed():
    return [
        # one video frame: 1080p NV12 from the decoder to the 384x512 network
        # input, then both encoders (every frame of a video takes this)
        dict(name="frame_1080p", kind="frame", src_h=1080, src_w=1920, H=384, W=512),
        # the motion filter of every video frame: single-edge correlation
        # against the last keyframe and one update step at batch 1
        dict(name="motion_filter", kind="motion_filter", h=48, w=64, half=True),
        # the smallest correlation call: the first edges of a new window on a
        # small odd-sized map, fp32 features
        dict(name="corr_small", kind="corr", h=29, w=43, frames=3, edges=3, half=False, flow=8.0),
        # the frontend window: 12 keyframes, 48 edges, fp16 features as a
        # DROID-SLAM host stores them
        dict(name="corr_window", kind="corr", h=48, w=64, frames=12, edges=48, half=True, flow=8.0),
        # the high-resolution window: 16 keyframes of 54x96, 64 edges, fp32
        dict(name="corr_highres", kind="corr", h=54, w=96, frames=16, edges=64, half=False,
             flow=8.0),
        # update operator on the few edges of a new keyframe, odd-sized map
        dict(name="update_few", kind="update", h=37, w=51, edges=5),
        # update operator of the frontend window
        dict(name="update_window", kind="update", h=48, w=64, edges=48),
        # GraphAgg of the window: keyframe means of the edges' features, the
        # damping network, its rows written back
        dict(name="graph_agg", kind="graph_agg", h=48, w=64, frames=12, edges=48),
        # bundle adjustment of the frontend window, three iterations
        dict(name="ba_window", kind="ba", h=48, w=64, frames=12, edges=48, iters=3, lm=1e-4,
             ep=0.1, motion_only=False),
        # the pose-only adjustment of the pipeline host, two iterations
        dict(name="ba_motion", kind="ba", h=48, w=64, frames=12, edges=48, iters=2, lm=1e-4,
             ep=0.1, motion_only=True),
        # the backend: 200 keyframes, 2000 edges, five iterations
        dict(name="ba_backend", kind="ba", h=48, w=64, frames=200, edges=2000, iters=5, lm=1e-5,
             ep=1e-2, motion_only=False),
        # proximity factors over the backend's graph
        dict(name="proximity", kind="proximity", h=48, w=64, frames=200, edges=2000),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frame", "motion_filter", "corr", "corr", "update", "update", "graph_agg",
                       "ba", "ba", "proximity"])
    h, w = rng.randint(20, 54), rng.randint(24, 96)
    if kind == "frame":
        src_h = 2 * rng.randint(180, 540)
        return dict(kind=kind, src_h=src_h, src_w=2 * rng.randint(240, 960),
                    H=8 * rng.randint(24, 54), W=8 * rng.randint(30, 96))
    if kind == "motion_filter":
        return dict(kind=kind, h=h, w=w, half=rng.random() < 0.7)
    if kind == "corr":
        frames = rng.randint(3, 16)
        return dict(kind=kind, h=h, w=w, frames=frames,
                    edges=min(_log_int(rng, 2, 64), frames * (frames - 1)),
                    half=rng.random() < 0.5, flow=rng.uniform(1.0, 8.0))
    if kind == "update":
        return dict(kind=kind, h=min(h, 48), w=min(w, 64), edges=_log_int(rng, 1, 48))
    if kind == "graph_agg":
        frames = rng.randint(2, 24)
        return dict(kind=kind, h=min(h, 48), w=min(w, 64), frames=frames,
                    edges=frames * min(rng.randint(1, 5), frames - 1))
    if kind == "ba":
        frames = _log_int(rng, 5, 180)
        return dict(kind=kind, h=min(h, 48), w=min(w, 64), frames=frames,
                    edges=frames * min(rng.randint(4, 9), frames - 1),
                    iters=rng.randint(2, 5), lm=1e-4, ep=0.1, motion_only=rng.random() < 0.25)
    frames = _log_int(rng, 12, 200)
    return dict(kind=kind, h=min(h, 48), w=min(w, 64), frames=frames,
                edges=frames * rng.randint(4, 10))


# ------------------------------------------------------------------ inputs --
def _gen(seed, salt):
    g = torch.Generator(device=DEV)
    g.manual_seed(1000003 * int(seed) + salt)
    return g


def _normal(g, *shape):
    return torch.randn(*shape, device=DEV, generator=g)


def _uniform(g, lo, hi, *shape):
    return torch.rand(*shape, device=DEV, generator=g) * (hi - lo) + lo


def _grid(h, w, dtype=torch.float32):
    y, x = torch.meshgrid(torch.arange(h, device=DEV, dtype=dtype),
                          torch.arange(w, device=DEV, dtype=dtype), indexing="ij")
    return torch.stack([x.reshape(-1), y.reshape(-1)])


def _edges(frames, edges, seed):
    """Directed edges of a keyframe window or graph: each keyframe with its
    nearest neighbours in time (cyclically, as the window's workload has it),
    and, for graphs of 64 keyframes and more, neighbours up to 2 apart and
    random long-range pairs up to the count."""
    ii, jj = [], []
    if frames < 64:
        for d in range(1, frames // 2 + 1):
            for i in range(frames):
                for j in sorted({(i + d) % frames, (i - d) % frames}):
                    ii.append(i)
                    jj.append(j)
        return np.asarray(ii[:edges], np.int32), np.asarray(jj[:edges], np.int32)
    for d in (1, 2):
        for i in range(frames - d):
            ii += [i, i + d]
            jj += [i + d, i]
    rng = np.random.default_rng(seed + 5)
    have = set(zip(ii, jj))
    while len(ii) < edges:
        i, j = (int(v) for v in rng.integers(0, frames, size=2))
        if abs(i - j) > 2 and (i, j) not in have:
            have.add((i, j))
            ii.append(i)
            jj.append(j)
    return np.asarray(ii, np.int32), np.asarray(jj, np.int32)


def _conv_weights(layers, seed):
    """{name: (w, b)} float32 on the host, w ~ N(0, 1/fan_in), b ~ N(0, 0.1)."""
    rng = np.random.default_rng(seed)
    out = {}
    for name, co, ci, k in layers:
        w = rng.standard_normal((co, ci, k, k), dtype=np.float32) / np.float32(math.sqrt(ci * k * k))
        out[name] = (w, 0.1 * rng.standard_normal(co, dtype=np.float32))
    return out


ENC_LAYERS = [("conv1", 32, 3, 7, 2)]
for _s, _ci, _co, _st in (("layer1", 32, 32, 1), ("layer2", 32, 64, 2), ("layer3", 64, 128, 2)):
    ENC_LAYERS += [(_s + "_0_conv1", _co, _ci, 3, _st), (_s + "_0_conv2", _co, _co, 3, 1)]
    if _st == 2:
        ENC_LAYERS += [(_s + "_0_downsample_0", _co, _ci, 1, 2)]
    ENC_LAYERS += [(_s + "_1_conv1", _co, _co, 3, 1), (_s + "_1_conv2", _co, _co, 3, 1)]
ENC_LAYERS += [("conv2", None, 128, 1, 1)]


def _enc_weights(prefix, out_dim, seed):
    return _conv_weights([(f"{prefix}_{n}", co or out_dim, ci, k)
                          for n, co, ci, k, _ in ENC_LAYERS], seed)


def _poses(g, n, rot=0.05, trans=0.1, fixed=2):
    """n world->camera poses [t, q(xyzw)] near identity, the first `fixed` ones at it."""
    v = _normal(g, n, 3).double() * rot
    th = v.norm(dim=1, keepdim=True).clamp_min(1e-12)
    q = torch.cat([v / th * torch.sin(th / 2), torch.cos(th / 2)], 1)
    p = torch.cat([_normal(g, n, 3).double() * trans, q], 1)
    if fixed:
        p[:fixed] = torch.tensor([0, 0, 0, 0, 0, 0, 1.0], device=DEV, dtype=F64)
    return p.float()


def _intrinsics(h, w):
    return torch.tensor([60.0 * w / 64, 60.0 * h / 48, w / 2.0, h / 2.0], device=DEV)


def _ba_inputs(case, seed):
    h, w, n = case["h"], case["w"], case["frames"]
    g = _gen(seed, 3)
    ii, jj = _edges(n, case["edges"], seed)
    poses = _poses(g, n)
    disps = _uniform(g, 0.2, 2.0, n, h * w)
    intr = _intrinsics(h, w)
    di, dj = (torch.from_numpy(v.astype(np.int64)).to(DEV) for v in (ii, jj))
    # targets: the exact reprojection, off by half a pixel of noise
    R, t = _relative(poses.double(), di, dj)
    X = _transform(R, t, disps.double()[di], intr.double(), h, w)
    fx, fy, cx, cy = intr.double().unbind()
    proj = torch.stack([fx * X[0] / X[2] + cx, fy * X[1] / X[2] + cy], 1).clamp(-1e6, 1e6)
    target = (proj + 0.5 * _normal(g, *proj.shape)).float().contiguous()
    weight = _uniform(g, 0.0, 1.0, *proj.shape).square().contiguous()
    eta = torch.full((n, h * w), 1e-6, device=DEV)
    return dict(poses=poses, disps=disps, intr=intr, target=target, weight=weight, eta=eta, ii=ii,
                jj=jj, ii_dev=di.int(), jj_dev=dj.int(), t0=2, t1=n)


def _update_inputs(case, seed):
    g = _gen(seed, 4)
    h, w, B = case["h"], case["w"], case["edges"]
    return dict(corr=_normal(g, B, 196, h, w), motion=_uniform(g, -8.0, 8.0, B, 4, h, w),
                net=_uniform(g, -1.0, 1.0, B, 128, h, w), inp=_normal(g, B, 128, h, w))


def _image(g, H, W):
    """An 8-bit luma or chroma plane with smooth structure and noise."""
    y = torch.arange(H, device=DEV, dtype=torch.float32)[:, None]
    x = torch.arange(W, device=DEV, dtype=torch.float32)[None, :]
    ph = _uniform(g, 0.0, 6.28, 2)
    v = 127 + 90 * torch.sin(x / 37.0 + ph[0]) * torch.cos(y / 51.0 + ph[1]) + 8 * _normal(g, H, W)
    return v.clamp(16, 240).to(torch.uint8).contiguous()


def _frame_inputs(case, seed):
    g = _gen(seed, 6)
    sh, sw = case["src_h"], case["src_w"]
    return dict(y=_image(g, sh, sw), uv=_image(g, sh // 2, sw))


def _corr_inputs(case, seed):
    g = _gen(seed, 1)
    h, w, n, B = case["h"], case["w"], case["frames"], case["edges"]
    fmaps = _normal(g, n, C, h, w)
    if case["half"]:
        fmaps = fmaps.half()
    ii, jj = _edges(n, B, seed)
    a = case["flow"]
    coords = (_grid(h, w)[None] + _uniform(g, -a, a, B, 2, h * w)).contiguous()
    return dict(fmaps=fmaps, ii=ii, jj=jj, coords=coords)


def _motion_inputs(case, seed):
    g = _gen(seed, 2)
    h, w = case["h"], case["w"]
    f = _normal(g, 2, C, h, w)
    return dict(f=f.half() if case["half"] else f, net=_uniform(g, -1.0, 1.0, 128, h, w),
                inp=_normal(g, 128, h, w).relu())


def _graph_agg_inputs(case, seed):
    g = _gen(seed, 7)
    ii, _ = _edges(case["frames"], case["edges"], seed)
    agg = _normal(g, case["edges"], 128, case["h"], case["w"]).relu().half().float()
    return dict(agg=agg, ii=ii)


def _proximity_inputs(case, seed):
    g = _gen(seed, 8)
    n, h, w = case["frames"], case["h"], case["w"]
    poses = _poses(g, n, rot=0.02, trans=0.01, fixed=0)
    poses[:, 0] += 0.02 * torch.arange(n, device=DEV)
    ii, jj = _edges(n, case["edges"], seed)
    return dict(poses=poses, disps=_uniform(g, 0.2, 2.0, n, h * w), intr=_intrinsics(h, w), ii=ii,
                jj=jj)


_UPDATE_LAYERS = [("update_corr_encoder_0", 128, 196, 1), ("update_corr_encoder_2", 128, 128, 3),
                  ("update_flow_encoder_0", 128, 4, 7), ("update_flow_encoder_2", 64, 128, 3),
                  ("update_gru_convz", 128, 448, 3), ("update_gru_convr", 128, 448, 3),
                  ("update_gru_convq", 128, 448, 3), ("update_gru_convz_glo", 128, 128, 1),
                  ("update_gru_convr_glo", 128, 128, 1), ("update_gru_convq_glo", 128, 128, 1),
                  ("update_gru_w", 128, 128, 1), ("update_weight_0", 128, 128, 3),
                  ("update_weight_2", 3, 128, 3), ("update_delta_0", 128, 128, 3),
                  ("update_delta_2", 3, 128, 3), ("update_agg_conv1", 128, 128, 3),
                  ("update_agg_conv2", 128, 128, 3), ("update_agg_eta_0", 1, 128, 3)]
_ETA_LAYERS = ("update_agg_conv2", "update_agg_eta_0")


def _update_weights(seed):
    return _conv_weights(_UPDATE_LAYERS, 17 + seed)


# ----------------------------------------------------------------- prepare --
def prepare(case, seed):
    kind = case["kind"]
    s = dict(case=case)
    if kind == "frame":
        s.update(_frame_inputs(case, seed))
        H, W = case["H"], case["W"]
        s["fnet"] = slk.Encoder(H, W, 128, True)
        s["fnet"].set_weights(_enc_weights("fnet", 128, seed), "fnet")
        s["cnet"] = slk.Encoder(H, W, 256, False)
        s["cnet"].set_weights(_enc_weights("cnet", 256, seed + 1), "cnet")
        s["bgr"] = torch.empty(H, W, 3, device=DEV)
        s["fmap"] = torch.empty(128, H // 8, W // 8, device=DEV, dtype=torch.float16)
        s["net"] = torch.empty(128, H // 8, W // 8, device=DEV)
        s["inp"] = torch.empty(128, H // 8, W // 8, device=DEV)
        return s
    h, w = case["h"], case["w"]
    if kind == "motion_filter":
        s.update(_motion_inputs(case, seed))
        s["ctx"] = slk.Context(h, w, C=C, max_batch=1, corr_scale=ALPHA)
        s["um"] = slk.UpdateModule(1, h, w)
        s["um"].set_weights(_update_weights(seed))
    elif kind == "corr":
        s.update(_corr_inputs(case, seed))
        s["ctx"] = slk.Context(h, w, C=C, max_batch=case["edges"], corr_scale=ALPHA)
        s["out"] = torch.empty(case["edges"], 196, h, w, device=DEV)
    elif kind == "update":
        s.update(_update_inputs(case, seed))
        B = case["edges"]
        s["um"] = slk.UpdateModule(B, h, w)
        s["um"].set_weights(_update_weights(seed))
        s["delta"] = torch.empty(B, 3, h, w, device=DEV)
        s["weight"] = torch.empty(B, 3, h, w, device=DEV)
        s["agg"] = torch.empty(B, 128, h, w, device=DEV)
    elif kind == "graph_agg":
        s.update(_graph_agg_inputs(case, seed))
        n = case["frames"]
        s["ctx"] = slk.Context(h, w, C=C, max_batch=1, corr_scale=ALPHA)
        s["um"] = slk.UpdateModule(max(n, 1), h, w)
        s["um"].set_weights(_update_weights(seed))
        s["kf_agg"] = torch.empty(n, 128, h, w, device=DEV)
        s["active"] = torch.empty(n, dtype=torch.int32, device=DEV)
        s["eta"] = torch.empty(n, h * w, device=DEV)
        s["damping"] = torch.full((n, h * w), 1e-6, device=DEV)
    elif kind == "ba":
        s.update(_ba_inputs(case, seed))
        s["ctx"] = slk.Context(h, w, C=C, max_batch=1, corr_scale=ALPHA)
    elif kind == "proximity":
        s.update(_proximity_inputs(case, seed))
        n = case["frames"]
        s["ctx"] = slk.Context(h, w, C=C, max_batch=1, corr_scale=ALPHA)
        s["cap"] = 2 * n * (n + 3)
        s["new_ii"] = np.zeros(s["cap"], np.int32)
        s["new_jj"] = np.zeros(s["cap"], np.int32)
        s["dists"] = np.zeros((n, n), np.float32)
    else:
        raise ValueError(kind)
    return s


# --------------------------------------------------------------------- run --
def _run_frame(s):
    c = s["case"]
    slk.nv12_to_bgr(s["y"].data_ptr(), s["uv"].data_ptr(), s["bgr"].data_ptr(), c["src_w"],
                    c["src_h"], c["src_w"], c["src_w"], c["W"], c["H"])
    slk.encode_frame(s["fnet"], s["cnet"], s["bgr"].data_ptr(), s["fmap"].data_ptr(),
                     s["net"].data_ptr(), s["inp"].data_ptr())
    return {"bgr": s["bgr"], "fmap": s["fmap"], "net": s["net"], "inp": s["inp"]}


def _run_motion_filter(s):
    f = s["f"]
    return s["um"].motion_filter(s["ctx"], f[0].data_ptr(), f[1].data_ptr(), s["net"].data_ptr(),
                                 s["inp"].data_ptr(),
                                 dtype=slk.SLK_F16 if s["case"]["half"] else slk.SLK_F32)


def _run_corr(s):
    s["ctx"].batch_build_and_sample_correlation(
        s["fmaps"].data_ptr(), s["ii"], s["jj"], s["coords"].data_ptr(), s["out"].data_ptr(),
        dtype=slk.SLK_F16 if s["case"]["half"] else slk.SLK_F32)
    return s["out"]


def _run_update(s):
    # the GRU state is updated in place: a pass starts from the edges' stored states
    net = s["net"].clone()
    s["um"].forward(s["corr"].data_ptr(), s["motion"].data_ptr(), net.data_ptr(),
                    s["inp"].data_ptr(), s["delta"].data_ptr(), s["weight"].data_ptr(),
                    s["agg"].data_ptr(), s["case"]["edges"])
    return {"net": net, "delta": s["delta"], "weight": s["weight"], "agg": s["agg"]}


def _run_graph_agg(s):
    c = s["case"]
    HW = c["h"] * c["w"]
    L = slk.lib()
    num = ctypes.c_int(0)
    slk.check(L.slk_scatter_mean(s["ctx"].ptr, s["kf_agg"].data_ptr(), s["agg"].data_ptr(),
                                 s["ii"].ctypes.data, c["edges"], 128 * HW,
                                 s["active"].data_ptr(), None, ctypes.byref(num), None))
    s["um"].compute_eta(s["kf_agg"].data_ptr(), s["eta"].data_ptr(), num.value)
    slk.check(L.slk_scatter_rows(s["damping"].data_ptr(), s["eta"].data_ptr(),
                                 s["active"].data_ptr(), num.value, HW, None))
    return {"mean": s["kf_agg"][:num.value], "eta": s["eta"][:num.value], "damping": s["damping"]}


def _run_ba(s):
    c = s["case"]
    # the adjustment works in place: a pass refines a copy of the estimate
    poses, disps = s["poses"].clone(), s["disps"].clone()
    s["ctx"].ba_iterate_n(poses.data_ptr(), disps.data_ptr(), s["intr"].data_ptr(),
                          s["target"].data_ptr(), s["weight"].data_ptr(), s["eta"].data_ptr(),
                          s["ii_dev"].data_ptr(), s["jj_dev"].data_ptr(), s["ii"], s["jj"],
                          s["t0"], s["t1"], c["lm"], c["ep"], c["iters"],
                          motion_only=c["motion_only"])
    return {"poses": poses, "disps": disps}


def _run_proximity(s):
    n = s["case"]["frames"]
    n_new, n_es = ctypes.c_int(0), ctypes.c_int(0)
    slk.check(slk.lib().slk_proximity_factors(
        s["ctx"].ptr, s["poses"].data_ptr(), s["disps"].data_ptr(), s["intr"].data_ptr(), n, 0, 0,
        2, 3, 20.0, 0.3, s["ii"].ctypes.data, s["jj"].ctypes.data, len(s["ii"]), None, None, 0, 0,
        s["new_ii"].ctypes.data, s["new_jj"].ctypes.data, s["cap"], ctypes.byref(n_new),
        ctypes.byref(n_es), s["dists"].ctypes.data, None))
    # the covisibility matrix a host keeps, with the new edges entered
    covis = np.zeros((n, n), np.uint8)
    m = n_new.value
    covis[s["new_ii"][:m], s["new_jj"][:m]] = 1
    return {"dists": s["dists"], "covis": covis}


_RUN = dict(frame=_run_frame, motion_filter=_run_motion_filter, corr=_run_corr, update=_run_update,
            graph_agg=_run_graph_agg, ba=_run_ba, proximity=_run_proximity)


def run(state):
    return _RUN[state["case"]["kind"]](state)


# -------------------------------------------------------------------- work --
def _conv_flops(layers, skip=()):
    """Operations per output pixel of a list of (name, co, ci, k)."""
    return sum(2.0 * co * ci * k * k for name, co, ci, k in layers if name not in skip)


def _corr_flops(px, edges, feat):
    """8x8 cells of 4 levels, 49 bilinear samples of each, per source pixel."""
    return edges * px * (4 * 64 * 2.0 * C + 4 * 49 * 7) + feat


def work(case):
    kind = case["kind"]
    if kind == "frame":
        H, W = case["H"], case["W"]
        flops, px = 0.0, {}
        res = {"conv1": 4, "layer1": 4, "layer2": 16, "layer3": 64, "conv2": 64}
        for name, co, ci, k, _ in ENC_LAYERS:
            per = H * W / res[name.split("_")[0]]
            for out_dim in (128, 256):
                flops += 2.0 * (co or out_dim) * ci * k * k * per
        weights = sum(2.0 * ((co or 192) * ci * k * k) for _, co, ci, k, _ in ENC_LAYERS) * 2
        hw = H * W / 64
        return {"bytes": case["src_h"] * case["src_w"] * 1.5 + 12.0 * H * W + weights
                + hw * (128 * 2 + 256 * 4), "flops": flops}
    px = case["h"] * case["w"]
    if kind == "motion_filter":
        e = 2 if case["half"] else 4
        skip = _ETA_LAYERS + ("update_agg_conv1", "update_weight_0", "update_weight_2")
        glo = [n for n, *_ in _UPDATE_LAYERS if n.endswith("_glo")]
        weights = 2.0 * _conv_flops(_UPDATE_LAYERS, skip) / 2
        return {"bytes": 2.0 * C * px * e + 2.0 * 128 * px * 4 + weights,
                "flops": px * _conv_flops(_UPDATE_LAYERS, skip + tuple(glo))
                + _corr_flops(px, 1, 0.0)}
    if kind == "corr":
        e = 2 if case["half"] else 4
        B = case["edges"]
        frames = min(case["frames"], 2 * B)
        return {"bytes": float(frames * C * px * e + B * px * (8 + 196 * 4)),
                "flops": _corr_flops(px, B, 0.0)}
    if kind == "update":
        B = case["edges"]
        glo = tuple(n for n, *_ in _UPDATE_LAYERS if n.endswith("_glo"))
        weights = _conv_flops(_UPDATE_LAYERS, _ETA_LAYERS)
        return {"bytes": 4.0 * B * px * (196 + 4 + 128 + 128 + 128 + 3 + 3 + 128) + weights,
                "flops": B * px * _conv_flops(_UPDATE_LAYERS, _ETA_LAYERS + glo)}
    if kind == "graph_agg":
        n, B = case["frames"], case["edges"]
        return {"bytes": 4.0 * px * (128 * B + 128 * n + 2 * n),
                "flops": 128.0 * px * B
                + n * px * 2.0 * 9 * (128 * 128 + 128)}
    if kind == "ba":
        n, M, P = case["frames"], case["edges"], case["frames"] - 2
        # a pixel of an edge: projection, Jacobians and its share of the 12x12
        # Hessian (symmetric), E rows and, with depths, the Schur products of
        # its keyframe's rows
        per = 100.0 + 2 * 2 * 27 + 2 * 2 * 12
        rows = 1 + M / n
        schur = 0.0 if case["motion_only"] else n * px * (6 * rows) * (6 * rows + 1)
        return {"bytes": 4.0 * (M * px * 4 + n * px * 3 + 14 * n),
                "flops": case["iters"] * (M * px * per + schur + (6.0 * P) ** 3 / 3)}
    n = case["frames"]
    return {"bytes": 4.0 * (n * px + 7 * n + n * n) + n * n, "flops": 50.0 * n * n * px}


# --------------------------------------------------------------- tolerance --
def tolerance(case):
    """About four times the distance measured between the library and the
    64-bit result (2-norm, relative), with the largest difference that the
    data types give."""
    kind = case["kind"]
    if kind == "frame":          # 3.4e-3 on fmap: 16 layers of fp16 activations, normalised
        return {"rel": 1.2e-2, "max": 0.3}
    if kind == "motion_filter":  # 6e-5: the mean of one update step's flow
        return {"rel": 3e-4, "max": 3e-4}
    if kind == "corr":           # 1.5e-7: fp32 sums of exact or 22-bit products
        return {"rel": 1e-6, "max": 2e-5}
    if kind == "update":         # 6e-4: fp16 activations through eight layers
        return {"rel": 2.5e-3, "max": 0.03}
    if kind == "graph_agg":      # 2.1e-4: fp16 activations through two layers
        return {"rel": 8e-4, "max": 8e-3}
    if kind == "ba":             # 3e-8: 64 bits inside, fp32 poses and depths
        return {"rel": 1e-6, "max": 2e-5}
    # 7e-8: fp32 sums; the selection may differ at near ties of the distances
    return {"rel": 1e-6, "max": 1e-5, "differ": 0.005}


# ------------------------------------------------------------------- exact --
def _conv64(x, w, b, stride=1):
    """2-D cross-correlation in float64, zero padding k//2; x [B, ci, H, W]."""
    w, b = torch.from_numpy(w).to(DEV, F64), torch.from_numpy(b).to(DEV, F64)
    B, ci, H, W = x.shape
    k = w.shape[-1]
    p = k // 2
    Ho, Wo = (H + 2 * p - k) // stride + 1, (W + 2 * p - k) // stride + 1
    xp = torch.nn.functional.pad(x, (p, p, p, p))
    out = b[None, :, None].expand(B, -1, Ho * Wo).clone()
    for ky in range(k):
        for kx in range(k):
            v = xp[:, :, ky:ky + stride * (Ho - 1) + 1:stride, kx:kx + stride * (Wo - 1) + 1:stride]
            v = v.reshape(B, ci, Ho * Wo).contiguous()
            wt = w[:, :, ky, kx].contiguous()
            for e in range(B):
                out[e] += wt @ v[e]
    return out.reshape(B, -1, Ho, Wo)


def _inorm64(x):
    m = x.mean(dim=(2, 3), keepdim=True)
    v = ((x - m) ** 2).mean(dim=(2, 3), keepdim=True)
    return (x - m) / torch.sqrt(v + 1e-5)


def _encoder64(img, P, norm):
    n = _inorm64 if norm else (lambda v: v)
    x = n(_conv64(img, *P["conv1"], stride=2)).relu()
    for st, stride in (("layer1", 1), ("layer2", 2), ("layer3", 2)):
        for blk in (0, 1):
            s, name = (stride if blk == 0 else 1), f"{st}_{blk}_"
            y = n(_conv64(x, *P[name + "conv1"], stride=s)).relu()
            y = n(_conv64(y, *P[name + "conv2"])).relu()
            if name + "downsample_0" in P:
                x = n(_conv64(x, *P[name + "downsample_0"], stride=s))
            x = (x + y).relu()
    return _conv64(x, *P["conv2"])


def _nv12_64(y, uv, sw, sh, W, H):
    """Bilinear luma, nearest chroma, BT.709, clamped to 0..255. The sample
    positions are the float32 ones: they select pixels."""
    f = torch.float32

    def axis(n_src, n_dst):
        s = (torch.arange(n_dst, device=DEV, dtype=f) + 0.5) * n_src / n_dst - 0.5
        lo = torch.floor(s)
        i0 = lo.long()
        return s, i0.clamp_min(0), (i0 + 1).clamp_max(n_src - 1), (s - lo).double()

    sx, x0, x1, wx = axis(sw, W)
    sy, y0, y1, wy = axis(sh, H)
    Y = y.double()

    def at(r, c):
        return Y[r[:, None], c[None, :]]

    wx, wy = wx[None, :], wy[:, None]
    Yv = (1 - wy) * ((1 - wx) * at(y0, x0) + wx * at(y0, x1)) \
        + wy * ((1 - wx) * at(y1, x0) + wx * at(y1, x1))
    ux = (((sx + 0.5).long() // 2) * 2).clamp(0, sw - 2)
    uy = ((sy + 0.5).long() // 2).clamp(0, sh // 2 - 1)
    U = uv.double()[uy[:, None], ux[None, :]] - 128
    V = uv.double()[uy[:, None], ux[None, :] + 1] - 128
    out = torch.stack([Yv + 1.8556 * U, Yv - 0.1873 * U - 0.4681 * V, Yv + 1.5748 * V], -1)
    return out.clamp(0, 255)


def _exact_frame(case, seed):
    s = _frame_inputs(case, seed)
    bgr = _nv12_64(s["y"], s["uv"], case["src_w"], case["src_h"], case["W"], case["H"])
    mean = torch.tensor([0.406, 0.456, 0.485], device=DEV, dtype=F64)
    std = torch.tensor([0.225, 0.224, 0.229], device=DEV, dtype=F64)
    img = ((bgr / 255 - mean) / std).flip(-1).permute(2, 0, 1)[None].contiguous()
    Pf = {k[5:]: v for k, v in _enc_weights("fnet", 128, seed).items()}
    Pc = {k[5:]: v for k, v in _enc_weights("cnet", 256, seed + 1).items()}
    fmap, cmap = _encoder64(img, Pf, True)[0], _encoder64(img, Pc, False)[0]
    return {"bgr": bgr, "fmap": fmap, "net": torch.tanh(cmap[:128]), "inp": cmap[128:].relu()}


def _lookup64(fi, fj, coords, h, w):
    """[196, h*w] lookup of one edge; fi, fj [C, h*w] and coords [2, h*w] float64."""
    HW = h * w
    lev = (ALPHA * (fi.t().contiguous() @ fj)).reshape(HW, 1, h, w)
    out = torch.zeros(196, HW, device=DEV, dtype=F64)
    ar = torch.arange(8, device=DEV)
    for l in range(4):
        if l:
            lev = torch.nn.functional.avg_pool2d(lev, 2, 2)
        H2, W2 = lev.shape[-2:]
        x, y = coords[0] / (1 << l), coords[1] / (1 << l)
        dx, dy = (x - x.floor())[:, None, None], (y - y.floor())[:, None, None]
        xs, ys = x.floor().long()[:, None] - 3 + ar, y.floor().long()[:, None] - 3 + ar
        ok = ((xs >= 0) & (xs < W2))[:, :, None] & ((ys >= 0) & (ys < H2))[:, None, :]
        at = (ys[:, None, :] * W2 + xs[:, :, None]).clamp(0, H2 * W2 - 1)
        v = torch.gather(lev.reshape(HW, -1), 1, at.reshape(HW, 64)).reshape(HW, 8, 8) * ok
        o = (1 - dx) * (1 - dy) * v[:, :7, :7] + dx * (1 - dy) * v[:, 1:, :7] \
            + (1 - dx) * dy * v[:, :7, 1:] + dx * dy * v[:, 1:, 1:]
        out[l * 49:(l + 1) * 49] = o.reshape(HW, 49).t()
    return out


def _exact_corr(case, seed):
    s = _corr_inputs(case, seed)
    h, w = case["h"], case["w"]
    f = s["fmaps"].double().reshape(case["frames"], C, h * w)
    out = torch.empty(case["edges"], 196, h * w, device=DEV, dtype=F64)
    for e in range(case["edges"]):
        out[e] = _lookup64(f[int(s["ii"][e])], f[int(s["jj"][e])], s["coords"][e].double(), h, w)
    return out.reshape(-1, 196, h, w)


def _update64(P, corr, motion, net, inp):
    """The update operator without its 16-bit roundings; tensors [B, c, h, w]."""
    def cv(name, x):
        return _conv64(x, *P["update_" + name])

    c = cv("corr_encoder_2", cv("corr_encoder_0", corr).relu()).relu()
    f = cv("flow_encoder_2", cv("flow_encoder_0", motion).relu()).relu()
    rest = torch.cat([inp, c, f], 1)
    glo = (torch.sigmoid(cv("gru_w", net)) * net).mean(dim=(2, 3), keepdim=True)
    x = torch.cat([net, rest], 1)
    z = torch.sigmoid(cv("gru_convz", x) + cv("gru_convz_glo", glo))
    r = torch.sigmoid(cv("gru_convr", x) + cv("gru_convr_glo", glo))
    q = torch.tanh(cv("gru_convq", torch.cat([r * net, rest], 1)) + cv("gru_convq_glo", glo))
    net = (1 - z) * net + z * q
    delta = cv("delta_2", cv("delta_0", net).relu())
    weight = torch.sigmoid(cv("weight_2", cv("weight_0", net).relu()))
    return net, delta, weight, cv("agg_conv1", net).relu()


def _exact_update(case, seed):
    s, P = _update_inputs(case, seed), _update_weights(seed)
    outs = []
    for e in range(case["edges"]):
        outs.append(_update64(P, *(s[k][e:e + 1].double() for k in ("corr", "motion", "net",
                                                                    "inp"))))
    net, delta, weight, agg = (torch.cat(v) for v in zip(*outs))
    return {"net": net, "delta": delta, "weight": weight, "agg": agg}


def _exact_motion_filter(case, seed):
    s, P = _motion_inputs(case, seed), _update_weights(seed)
    h, w = case["h"], case["w"]
    f = s["f"].double().reshape(2, C, h * w)
    corr = _lookup64(f[0], f[1], _grid(h, w, F64), h, w).reshape(1, 196, h, w)
    motion = torch.zeros(1, 4, h, w, device=DEV, dtype=F64)
    _, delta, _, _ = _update64(P, corr, motion, s["net"][None].double(), s["inp"][None].double())
    return float(torch.sqrt(delta[0, 0] ** 2 + delta[0, 1] ** 2).mean())


def _exact_graph_agg(case, seed):
    s, P = _graph_agg_inputs(case, seed), _update_weights(seed)
    ii = torch.from_numpy(s["ii"].astype(np.int64)).to(DEV)
    act = torch.unique(ii)
    mean = torch.stack([s["agg"][ii == a].double().mean(0) for a in act])
    e = _conv64(_conv64(mean, *P["update_agg_conv2"]).relu(), *P["update_agg_eta_0"])
    eta = 0.01 * torch.log1p(torch.exp(e)).reshape(len(act), -1)
    damping = torch.full((case["frames"], case["h"] * case["w"]), 1e-6, device=DEV, dtype=F64)
    damping[act] = eta
    return {"mean": mean, "eta": eta, "damping": damping}


def _skew(v):
    z = torch.zeros_like(v[..., 0])
    return torch.stack([torch.stack([z, -v[..., 2], v[..., 1]], -1),
                        torch.stack([v[..., 2], z, -v[..., 0]], -1),
                        torch.stack([-v[..., 1], v[..., 0], z], -1)], -2)


def _rot(q):
    """Rotation matrices of quaternions [.., (x, y, z, w)]."""
    K = _skew(q[..., :3])
    return torch.eye(3, device=DEV, dtype=q.dtype) + 2 * q[..., 3:, None] * K + 2 * (K @ K)


def _qmul(a, b):
    av, aw, bv, bw = a[..., :3], a[..., 3:], b[..., :3], b[..., 3:]
    return torch.cat([aw * bv + bw * av + torch.linalg.cross(av, bv),
                      aw * bw - (av * bv).sum(-1, keepdim=True)], -1)


def _relative(poses, i, j):
    """R, t of pose[j] * pose[i]^-1."""
    conj = torch.tensor([-1.0, -1, -1, 1], device=DEV, dtype=poses.dtype)
    R = _rot(_qmul(poses[j, 3:], poses[i, 3:] * conj))
    return R, poses[j, :3] - (R @ poses[i, :3, None])[..., 0]


def _transform(R, t, disp, intr, h, w):
    """(X, Y, Z) [M, h*w] of the unit-depth rays moved by (R, t * disp)."""
    g = _grid(h, w, disp.dtype)
    rx, ry = (g[0] - intr[2]) / intr[0], (g[1] - intr[3]) / intr[1]
    return [R[:, k, 0, None] * rx + R[:, k, 1, None] * ry + R[:, k, 2, None] + t[:, k, None] * disp
            for k in range(3)]


def _ba_step64(poses, disps, s, case):
    """One damped Gauss-Newton step on poses t0..t1-1 and the inverse depths
    of the keyframes with edges (Schur complement over the depths)."""
    h, w, HW = case["h"], case["w"], case["h"] * case["w"]
    ii, jj = s["ii_dev"].long(), s["jj_dev"].long()
    t0, P = s["t0"], s["t1"] - s["t0"]
    fx, fy = s["intr"].double()[:2]
    cx, cy = s["intr"].double()[2:]
    S = torch.zeros(P, P, 6, 6, device=DEV, dtype=F64)
    b = torch.zeros(P, 6, device=DEV, dtype=F64)
    depth = []  # per keyframe: its pose rows, E, Q, w
    for k in torch.unique(ii).tolist():
        e = torch.nonzero(ii == k)[:, 0]
        m = len(e)
        R, t = _relative(poses, ii[e], jj[e])
        d = disps[k][None].expand(m, HW)
        X, Y, Z = _transform(R, t, d, s["intr"].double(), h, w)
        ok = (Z >= MIN_DEPTH).double()
        iz = torch.where(Z >= MIN_DEPTH, 1 / Z, torch.zeros_like(Z))
        u, v = X * iz, Y * iz
        res = torch.stack([s["target"][e, 0].double() - (fx * u + cx),
                           s["target"][e, 1].double() - (fy * v + cy)], -1)
        wt = 1e-3 * s["weight"][e].double().permute(0, 2, 1) * ok[..., None]
        zero = torch.zeros_like(Z)
        Jj = torch.stack([
            torch.stack([fx * d * iz, zero, -fx * u * d * iz, -fx * u * v, fx * (1 + u * u),
                         -fx * v], -1),
            torch.stack([zero, fy * d * iz, -fy * v * d * iz, -fy * (1 + v * v), fy * u * v,
                         fy * u], -1)], -2)                                  # [m, HW, 2, 6]
        Jz = torch.stack([fx * (t[:, 0, None] - t[:, 2, None] * u) * iz,
                          fy * (t[:, 1, None] - t[:, 2, None] * v) * iz], -1)  # [m, HW, 2]
        Ad = torch.zeros(m, 6, 6, device=DEV, dtype=F64)
        Ad[:, :3, :3] = Ad[:, 3:, 3:] = R
        Ad[:, :3, 3:] = _skew(t) @ R
        Ji = -(Jj.reshape(m, HW * 2, 6) @ Ad).reshape(m, HW, 2, 6)
        JJ = torch.cat([Ji, Jj], -1).reshape(m, HW * 2, 12)
        WJ = JJ * wt.reshape(m, HW * 2, 1)
        Hs = WJ.transpose(1, 2).contiguous() @ JJ
        vs = (WJ * res.reshape(m, HW * 2, 1)).sum(1)
        Es = (WJ.reshape(m, HW, 2, 12) * Jz[..., None]).sum(2)               # [m, HW, 12]
        own = k - t0
        rows, E = [], []
        if 0 <= own < P:
            rows.append(own)
            E.append(Es[:, :, :6].sum(0))
            S[own, own] += Hs[:, :6, :6].sum(0)
            b[own] += vs[:, :6].sum(0)
        for q, p in enumerate((jj[e] - t0).tolist()):
            if not 0 <= p < P:
                continue
            S[p, p] += Hs[q, 6:, 6:]
            b[p] += vs[q, 6:]
            if 0 <= own < P:
                S[own, p] += Hs[q, :6, 6:]
                S[p, own] += Hs[q, 6:, :6]
            if p in rows:
                E[rows.index(p)] = E[rows.index(p)] + Es[q, :, 6:]
            else:
                rows.append(p)
                E.append(Es[q, :, 6:])
        if case["motion_only"]:
            continue
        Cq = (wt * Jz * Jz).sum((0, 2))
        wq = (wt * res * Jz).sum((0, 2))
        Q = 1 / (Cq + 0.2 * s["eta"][k].double() + 1e-7)
        if rows:
            En = torch.cat(E, 1)                                            # [HW, 6 rows]
            blk = En.t().contiguous() @ (Q[:, None] * En)
            at = torch.tensor(rows, device=DEV)
            n = len(rows)
            S[at[:, None], at[None, :]] -= blk.reshape(n, 6, n, 6).permute(0, 2, 1, 3)
            b[at] -= (En.t().contiguous() @ (Q * wq)).reshape(n, 6)
            depth.append((k, at, En, Q, wq))
        else:
            depth.append((k, None, None, Q, wq))
    A = S.permute(0, 2, 1, 3).reshape(6 * P, 6 * P).clone()
    A.diagonal().add_(case["ep"] + case["lm"] * A.diagonal())
    dx = torch.linalg.solve(A, b.reshape(-1)).reshape(P, 6)
    disps = disps.clone()
    for k, at, En, Q, wq in depth:
        dw = 0 if at is None else En @ dx[at].reshape(-1)
        disps[k] = disps[k] + Q * (wq - dw)
    tau, phi = dx[:, :3], dx[:, 3:]
    th = phi.norm(dim=1, keepdim=True).clamp_min(1e-30)
    K = _skew(phi)
    a, c = ((1 - torch.cos(th)) / th ** 2)[..., None], ((th - torch.sin(th)) / th ** 3)[..., None]
    a = torch.where(th[..., None] > 1e-4, a, torch.full_like(a, 0.5))
    c = torch.where(th[..., None] > 1e-4, c, torch.full_like(c, 1 / 6))
    V = torch.eye(3, device=DEV, dtype=F64) + a * K + c * (K @ K)
    dq = torch.cat([torch.sin(th / 2) / th * phi, torch.cos(th / 2)], 1)
    free = poses[t0:t0 + P]
    poses = poses.clone()
    poses[t0:t0 + P] = torch.cat([(_rot(dq) @ free[:, :3, None])[..., 0]
                                  + (V @ tau[..., None])[..., 0], _qmul(dq, free[:, 3:])], 1)
    return poses, disps


def _exact_ba(case, seed):
    s = _ba_inputs(case, seed)
    poses, disps = s["poses"].double(), s["disps"].double()
    for _ in range(case["iters"]):
        poses, disps = _ba_step64(poses, disps, s, case)
    return {"poses": poses, "disps": disps}


def _exact_proximity(case, seed):
    """The distances; the selection is of whole values and follows from them."""
    s = _proximity_inputs(case, seed)
    n, h, w, beta = case["frames"], case["h"], case["w"], 0.3
    poses, intr = s["poses"].double(), s["intr"].double()
    fx, fy, cx, cy = intr.unbind()
    g = _grid(h, w, F64)
    out = torch.empty(n, n, device=DEV, dtype=F64)
    jj = torch.arange(n, device=DEV)
    eye = torch.eye(3, device=DEV, dtype=F64).expand(n, 3, 3)
    for i in range(n):
        R, t = _relative(poses, torch.full_like(jj, i), jj)
        num = den = 0.0
        for wgt, rot in ((beta, R), (1 - beta, eye)):
            X, Y, Z = _transform(rot, t, s["disps"][i].double()[None], intr, h, w)
            d = torch.sqrt((fx * X / Z + cx - g[0]) ** 2 + (fy * Y / Z + cy - g[1]) ** 2)
            ok = Z > MIN_DEPTH
            num = num + wgt * torch.where(ok, d, torch.zeros_like(d)).sum(1)
            den = den + wgt * ok.double().sum(1)
        out[i] = torch.where(den / (h * w) < 0.75, torch.full_like(num, 1000.0), num / den)
    return {"dists": out, "covis": None}


_EXACT = dict(frame=_exact_frame, motion_filter=_exact_motion_filter, corr=_exact_corr,
              update=_exact_update, graph_agg=_exact_graph_agg, ba=_exact_ba,
              proximity=_exact_proximity)


def exact(case, seed):
    return _EXACT[case["kind"]](case, seed)
