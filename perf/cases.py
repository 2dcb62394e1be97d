"""The work that a user of the library has it do, as cases that can be timed.

A frame is primary paths, colours and one shadow ray per pixel of a camera over a seeded
coloured terrain. An edit pass applies sphere / box / paint editors (or copies) one by one or
fused, is followed by the frame that shows its result and taken back by undo, so that a pass can
be run again. A collection drops the nodes an undone batch left behind. Terrains and loaded DAGs
are kept per process, as a program keeps the scene it shows; cameras and editors come from the
seed.
"""
from __future__ import annotations

import math
from collections import OrderedDict

import numpy as np
import torch

from hashdag_amd import CameraView, DAGInfo, DAGTracer, Geometry, HashDAG, TerrainParams, generate_terrain
from hashdag_amd.graph import FrameGraph
from hashdag_amd.workload import cameras, copy_edits, mixed_edits, sphere_edits

# A case: what = frame | edit | copy | graph | gc; the terrain (levels, footprint, colors); the
# frame (width, height, fog, schedule: 0 = the default launch, else the step count of the
# hand-over launch that the autotuner settles on); the editors (edits, rmin, rmax, fused).


def _case(what, levels, footprint, width, height, *, colors=True, fog=0.0, schedule=0, edits=0, rmin=2.0, rmax=64.0,
          fused=True, **more):
    return {"what": what, "levels": levels, "footprint": footprint, "colors": colors, "width": width, "height": height,
            "fog": fog, "schedule": schedule, "edits": edits, "rmin": rmin, "rmax": rmax, "fused": fused, **more}


def listed():
    return [
        # a thumbnail of a small scene: launches and latency
        _case("frame", 13, 256, 128, 72, name="frame_thumb"),
        # an odd window over a shallow scene, seen through fog
        _case("frame", 13, 1024, 1283, 717, fog=40.0, name="frame_fog_odd"),
        # a preview window over a deep scene with the default launch
        _case("frame", 16, 4096, 640, 360, name="frame_preview"),
        # one brush stroke of an interactive session: one small editor, its frame, undo
        _case("edit", 16, 4096, 640, 360, edits=1, rmin=4.0, rmax=16.0, fused=False, name="edit_brush"),
        # an edit request of the serving loop: a few dozen editors fused into one pass
        _case("edit", 16, 4096, 1280, 720, edits=48, rmin=2.0, rmax=128.0, name="edit_request"),
        # copy tool: regions copied elsewhere, one pass each
        _case("copy", 16, 4096, 640, 360, edits=2, rmin=48.0, rmax=48.0, name="edit_copy"),
        # a frame of a game loop: editors and the frame after them replayed as one captured graph
        _case("graph", 16, 4096, 1280, 720, edits=8, rmin=4.0, rmax=48.0, schedule=128, name="graph_frame"),
        # a script of spheres on a binary scene, one pass per editor
        _case("edit", 12, 4096, 320, 180, colors=False, edits=24, rmin=8.0, rmax=64.0, fused=False,
              name="edit_script_binary"),
        # the frame the benchmark times, with the launch it settles on, over a large scene
        _case("frame", 15, 16384, 1920, 1080, schedule=128, name="frame_1080p"),
        # thousands of mixed editors fused into one pass over a large scene
        _case("edit", 15, 16384, 1280, 720, edits=4096, rmin=2.0, rmax=256.0, schedule=128, name="edit_batch"),
        # collecting the nodes that an undone batch left in the table
        _case("gc", 17, 8192, 640, 360, edits=32, rmin=2.0, rmax=64.0, name="collect"),
        # a 4K frame of the deepest scene
        _case("frame", 17, 8192, 3840, 2160, schedule=128, name="frame_4k"),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    what = rng.choice(["frame", "frame", "frame", "edit", "edit", "edit", "copy", "graph", "gc"])
    footprint = 1 << rng.randint(8, 13)  # terrains are a power of two wide
    levels = rng.randint(13, 17)
    schedule = rng.choice([0, 128])
    if what == "frame":
        return _case("frame", levels, footprint, _log_uniform(rng, 64, 3840), _log_uniform(rng, 64, 2160),
                     fog=rng.choice([0.0, 0.0, 20.0]), schedule=schedule)
    width, height = _log_uniform(rng, 64, 1280), _log_uniform(rng, 64, 720)
    if what == "copy":
        r = float(_log_uniform(rng, 8, 64))
        return _case("copy", levels, footprint, width, height, edits=rng.randint(1, 3), rmin=r, rmax=r,
                     schedule=schedule)
    rmax = float(_log_uniform(rng, 8, 128))
    if what == "graph":
        return _case("graph", levels, footprint, width, height, edits=rng.randint(1, 16), rmax=rmax / 2,
                     schedule=schedule)
    if what == "gc":
        return _case("gc", levels, footprint, width, height, edits=_log_uniform(rng, 1, 64), rmax=rmax,
                     schedule=schedule)
    if rng.random() < 0.4:  # one pass per editor
        return _case("edit", levels, footprint, width, height, edits=_log_uniform(rng, 1, 24), rmax=rmax / 2,
                     fused=False, schedule=schedule)
    return _case("edit", levels, footprint, width, height, edits=_log_uniform(rng, 2, 1024), rmax=rmax,
                 schedule=schedule)


_scenes: OrderedDict = OrderedDict()
_KEPT = 2  # terrains and DAGs kept loaded


def _terrain(case):
    return TerrainParams(levels=case["levels"], footprint=case["footprint"], colors=case["colors"])


def _dag(case):
    """The loaded DAG of the case's terrain. Collections get one of their own: they move every node."""
    key = (case["levels"], case["footprint"], case["colors"], case["what"] == "gc")
    dag = _scenes.pop(key, None)
    if dag is None:
        while len(_scenes) >= _KEPT:
            _scenes.popitem(last=False)
        scene = generate_terrain(_terrain(case))
        dag = HashDAG(Geometry.fit(case["levels"], scene.level_words, headroom=2.0))  # room for edits
        dag.load_scene(scene)
    _scenes[key] = dag
    return dag


def _edits(case, params, seed):
    n, lo, hi = case["edits"], case["rmin"], case["rmax"]
    if case["what"] == "copy":
        return copy_edits(params, n, seed=seed, radius=hi)
    if not case["fused"]:
        return sphere_edits(params, n, seed=seed, rmin=lo, rmax=hi)
    return mixed_edits(params, n, seed=seed, rmin=lo, rmax=hi)


def _camera_at(edit, footprint, seed):
    """A camera that looks down at an editor's centre."""
    where = edit[4] if len(edit) > 4 else edit[1]
    away = max(4.0 * edit[2], footprint / 16)
    yaw = float(np.random.default_rng(seed).uniform(0.0, 2.0 * math.pi))
    x, y, z = where
    pos = (x - away * math.sin(yaw) * 0.7, y + away * 0.7, z - away * math.cos(yaw) * 0.7)
    return CameraView.look(pos, yaw, -math.pi / 4)


def prepare(case, seed):
    params, dag = _terrain(case), _dag(case)
    s = {"what": case["what"], "dag": dag, "info": DAGInfo.unit(case["levels"]), "fog": case["fog"],
         "colors": case["colors"], "fused": case["fused"], "schedule": case["schedule"],
         "tracer": DAGTracer(case["width"], case["height"])}
    s["tracer"].set_schedule(dag, 2 if case["schedule"] else 0, case["schedule"])
    if case["what"] == "frame":
        s["camera"] = cameras(params, 1, seed=seed)[0]
        return s
    dag.remove_stale_nodes()  # a session starts from a collected table
    s["edits"] = _edits(case, params, seed)
    s["camera"] = _camera_at(s["edits"][0], case["footprint"], seed)
    if case["what"] == "graph":
        s["graph"] = FrameGraph(dag, s["tracer"], case["edits"])
    return s


def _frame(s):
    tracer, dag = s["tracer"], s["dag"]
    p = tracer.resolve_paths(s["camera"], s["info"], dag)
    if s["colors"]:
        tracer.resolve_colors(dag)
        tracer.resolve_shadows(s["camera"], s["info"], dag, 1.0, s["fog"], params=p)
        return {"paths": tracer.paths, "colors": tracer.colors}
    return {"paths": tracer.paths}


def run(s):
    dag = s["dag"]
    if s["what"] == "frame":
        return _frame(s)
    if s["what"] == "graph":
        from hashdag_amd import ray_params

        tracer = s["tracer"]
        p = ray_params(s["camera"], s["info"], dag.geometry.levels, tracer.width, tracer.height)
        st, _ = s["graph"].launch(s["edits"], p)
        out = {"paths": tracer.paths, "colors": tracer.colors}
        dag.undo()
    else:
        st = dag.edit_batch(s["edits"], fused=s["fused"])
        if s["what"] == "gc":
            dag.undo()
            out = {"live": dag.remove_stale_nodes()["live_nodes"], **_frame(s)}
        else:
            out = _frame(s)
            for _ in range(st.passes):
                dag.undo()
    return {**out, "voxels": int(st.num_voxels), "leaves": int(st.leaves_rebuilt), "encoded": int(st.colors_encoded)}


def work(case):
    """A frame writes a path and a colour per pixel, from a leaf and a colour block at least. An
    edit rewrites the shells of its editors: per voxel of a shell a colour read and written, and
    per 16 of them a leaf and its share of the nodes above it. A collection reads and writes the
    words of every live node (about 0.3 per column of the terrain)."""
    n = case["width"] * case["height"]
    nbytes = n * ((16 + 4 + 8 + 8) if case["colors"] else (16 + 8))
    lo, hi = case["rmin"], case["rmax"]
    if case["edits"]:
        if case["fused"] and hi > lo:  # radius log-uniform
            r2 = (hi * hi - lo * lo) / (2.0 * math.log(hi / lo))
        else:  # uniform
            r2 = (hi * hi + hi * lo + lo * lo) / 3.0
        shell = 4.0 * math.pi * r2 * case["edits"]
        nbytes += shell * ((16 if case["colors"] else 0) + 1.5)
    if case["what"] == "gc":
        nbytes += 2 * 4 * 0.3 * case["footprint"] ** 2
    return {"bytes": float(nbytes), "flops": 0.0}


def exact(case, seed):
    return None  # every output is a whole number
