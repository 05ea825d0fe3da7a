"""The measured cases: what a user of the framework has it do, through its public entry points.

A case is a dict of plain values with a "kind":

  top2        rs.bf_match_top2 on one or a few image pairs; a single pair is filtered as well (ratio test, cross-check)
  top1        rs.bf_match, both directions, 8-bit or 4-bit descriptors
  two_view    the batched hot path over the C ABI with task tables kept: top-2 match, filter and keypoint gather, seeded
              samples, 8-point F RANSAC, finish
  verify      the verification of pairs whose correspondences are in hand: 8-point F, 4-point H, or the default pair
              solver (7-point F, DEGENSAC, relative pose from F and H)
  batch       one launch of the captured pipeline over a batch of uneven pairs, either solver, with the affine match
              filter, lens undistortion and pose stages when asked
  cashash     cascade hashing: the registration of new images and the search against one train image, exact over the
              bucket union or re-ranked from the 128-bit remap
  guided      guided sampling and scoring with a proposal's weights
  train       one optimiser step of the proposal network
  forward     the proposal network's probabilities

Descriptors are the package's synthetic SIFT-like recipe (noisy true matches among fresh descriptors), keypoints one
two-view geometry per pair with outliers, focal 2000 px, images of 4000 x 3000.
"""
import ctypes
import math
import random

import numpy as np
import torch

import rapidsfm_amd as rs
from rapidsfm_amd import cashash, learned, ops, proposal, synth
from rapidsfm_amd._abi import BfTask, BfTop2Task, Camera, FilterTask, FinishTask, RansacTask, SampleTask, check, lib
from rapidsfm_amd.pipeline import SOLVERS, PipelineConfig, PipelinePair

DEV = "cuda"
VP = ctypes.c_void_p
CAM = (synth.FOCAL, synth.FOCAL, synth.WIDTH / 2, synth.HEIGHT / 2)
LENS = (-0.08, 0.02, 0.0005, -0.0003, 0.0)
# the reference's thresholds for images of this size: two-sided line test and homography test
T_LINE, T_PLANE = 0.008 * synth.HEIGHT, 0.005 * synth.HEIGHT


def listed():
    return [
        # two thumbnails or low-texture images: the smallest call, launches and latency
        {"name": "match_1k", "kind": "top2", "pairs": 1, "nA": 1000, "nB": 1187, "even": 1.0},
        # one ordinary pair matched both ways, as the reference's matcher is called
        {"name": "match_top1_8k", "kind": "top1", "bits": 8, "pairs": 1, "nA": 8192, "nB": 8192},
        # one pair of large images with the 4-bit descriptors that save memory there
        {"name": "match_u4_16k", "kind": "top1", "bits": 4, "pairs": 1, "nA": 16384, "nB": 15411},
        # the benchmark's step: matched and verified pairs per second at 8K keypoints
        {"name": "two_view_8k", "kind": "two_view", "pairs": 32, "nA": 8192, "nB": 8192, "hyp": 4096},
        # one small pair verified as soon as it was matched
        {"name": "verify_f8_one", "kind": "verify", "model": "f8", "pairs": 1, "n": 600, "hyp": 4096, "inliers": 0.5},
        # a project's candidate pairs of mixed sizes, affine filter before the 8-point solver
        {"name": "batch_f8", "kind": "batch", "solver": "f8", "pairs": 64, "lo": 1024, "hi": 16384, "hyp": 4096,
         "affine": True, "lens": False},
        # the same through the default pair solver, with lens distortion and poses
        {"name": "batch_degensac", "kind": "batch", "solver": "degensac", "pairs": 32, "lo": 1024, "hi": 8192,
         "hyp": 4096, "affine": False, "lens": True},
        # cascade hashing of new images against one train image, exact over the bucket union
        {"name": "cashash_union", "kind": "cashash", "mode": "union", "queries": 2, "nQ": 8192, "nT": 8192, "tables": 8},
        # the cascade-hashing paper's form: six tables, the eight Hamming-nearest re-ranked
        {"name": "cashash_rerank", "kind": "cashash", "mode": "rerank", "queries": 1, "nQ": 8192, "nT": 8192, "tables": 6},
        # guided verification of a group of pairs with 70% outliers
        {"name": "guided", "kind": "guided", "pairs": 12, "n": 2400, "hyp": 4096},
        # one step of the proposal network's training
        {"name": "train_8k", "kind": "train", "n": 8192},
        # the network over the matches of a whole project's batch
        {"name": "forward_1m", "kind": "forward", "n": 1 << 20},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["top2", "top2", "top1", "top1", "two_view", "verify", "verify", "batch", "batch", "cashash",
                       "cashash", "guided", "train", "forward"])
    if kind == "top2":
        n = _log(rng, 100, 16384)
        return {"kind": kind, "pairs": rng.randint(1, max(1, min(8, (8192 // n) ** 2))), "nA": n,
                "nB": _log(rng, max(100, n // 4), min(16384, 4 * n)), "even": round(rng.uniform(0.3, 1.0), 3)}
    if kind == "top1":
        n = _log(rng, 100, 16384)
        return {"kind": kind, "bits": rng.choice([8, 4]), "pairs": rng.randint(1, max(1, min(16, (12000 // n) ** 2))),
                "nA": n, "nB": _log(rng, max(100, n // 4), min(16384, 4 * n))}
    if kind == "two_view":
        n = _log(rng, 512, 8192)
        return {"kind": kind, "pairs": rng.randint(2, 32), "nA": n, "nB": rng.randint(max(256, n // 2), n),
                "hyp": rng.choice([1000, 2048, 4096])}
    if kind == "verify":
        return {"kind": kind, "model": rng.choice(["f8", "f8", "h4", "degensac"]), "pairs": rng.randint(1, 4),
                "n": _log(rng, 100, 8000), "hyp": _log(rng, 256, 8192), "inliers": round(rng.uniform(0.25, 0.8), 3)}
    if kind == "batch":
        hi = _log(rng, 2048, 16384)
        return {"kind": kind, "solver": rng.choice(["f8", "degensac"]), "pairs": rng.randint(4, 32),
                "lo": rng.randint(256, hi // 2), "hi": hi, "hyp": rng.choice([1024, 2048, 4096]),
                "affine": rng.random() < 0.5, "lens": rng.random() < 0.5}
    if kind == "cashash":
        n = _log(rng, 1000, 16384)
        return {"kind": kind, "mode": rng.choice(["union", "rerank"]), "queries": rng.randint(1, 2), "nQ": n,
                "nT": _log(rng, max(500, n // 3), min(16384, 3 * n)), "tables": rng.choice([6, 8])}
    if kind == "guided":
        return {"kind": kind, "pairs": rng.randint(1, 12), "n": _log(rng, 200, 4000), "hyp": rng.choice([1024, 2048, 4096])}
    if kind == "train":
        return {"kind": kind, "n": _log(rng, 1000, 65536)}
    return {"kind": kind, "n": _log(rng, 1000, 1 << 20)}


# ---- sizes of a case (fixed by the case: another seed gives other values, not other shapes)


def _pair_sizes(case):
    """(nA, nB) of every pair."""
    r = random.Random(repr(sorted((k, v) for k, v in case.items() if k != "name")))
    if case["kind"] == "batch":
        return [(r.randint(case["lo"], case["hi"]), r.randint(case["lo"], case["hi"])) for _ in range(case["pairs"])]
    e = case.get("even", 1.0)
    f = lambda n: n if e == 1.0 else max(1, int(n * r.uniform(e, 1.0)))  # noqa: E731
    return [(f(case["nA"]), f(case["nB"])) for _ in range(case["pairs"])]


def _verify_sizes(case):
    r = random.Random(case["n"] * 31 + case["pairs"])
    return [case["n"] if p == 0 else max(60, int(case["n"] * r.uniform(0.4, 1.0))) for p in range(case["pairs"])]


# ---- inputs


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) & 0x7FFFFFFFFFFFFFFF)
    return g


def _descriptors(seed, nA, nB, copy_frac):
    """Query and train descriptors: copy_frac of the queries are noisy copies of distinct train rows."""
    g = _gen(seed)
    b, vb = synth.sift_like(g, nB, DEV)
    a, _ = synth.sift_like(g, nA, DEV)
    m = min(int(round(copy_frac * nA)), nB)
    at = torch.randperm(nA, generator=g, device=DEV)[:m]
    src = torch.randperm(nB, generator=g, device=DEV)[:m]
    a[at] = synth.sift_like(g, m, DEV, base=vb[src])[0]
    return a, b


def _correspondences(seed, n, inliers, plane=0.0):
    """float32 (n, 4): inliers of one two-view geometry (a share of them on one plane), the rest uniform, shuffled; and which
    rows are inliers."""
    rng = np.random.default_rng(seed)
    view = synth.TwoView(rng)
    k = max(8, int(round(n * inliers)))
    p = view.points(rng, k)
    if plane:
        on = int(k * plane)
        K = np.array([[synth.FOCAL, 0, synth.WIDTH / 2], [0, synth.FOCAL, synth.HEIGHT / 2], [0, 0, 1]])
        H = K @ (view.R + np.outer(view.t, [0.1, -0.05, 1.0]) / 20.0) @ np.linalg.inv(K)
        q = np.column_stack([p[:on, :2], np.ones(on)]) @ H.T
        p[:on, 2:] = q[:, :2] / q[:, 2:]
    p = p + synth.NOISE_PX * rng.normal(size=p.shape)
    o = rng.uniform((0, 0) * 2, (synth.WIDTH, synth.HEIGHT) * 2, (max(0, n - k), 4))
    at = rng.permutation(n)
    good = np.arange(n) < k
    return torch.from_numpy(np.concatenate([p, o])[:n][at].astype(np.float32)).to(DEV), torch.from_numpy(good[at]).to(DEV)


def _matched_pair(seed, nA, nB):
    p = synth.make_pair(seed, nA, nB, copy_frac=0.3, geo_frac=0.7, device=DEV)
    kp = lambda k: torch.from_numpy(np.ascontiguousarray(p[k][:, :2])).to(DEV)  # noqa: E731
    return p["descA"], p["descB"], kp("kpA"), kp("kpB")


class _Rows:
    """Rows of several pairs in one buffer, each pair's part 256-byte aligned."""

    def __init__(self, sizes, cols, dtype):
        per = cols * torch.empty(0, dtype=dtype).element_size()
        unit = 256 // math.gcd(256, per)
        self.at, n = [], 0
        for s in sizes:
            self.at.append(n * per)
            n += (s + unit - 1) // unit * unit
        self.buf = torch.zeros((max(1, n), cols), dtype=dtype, device=DEV)

    def ptr(self, i):
        return self.buf.data_ptr() + self.at[i]


def _stream():
    return VP(torch.cuda.current_stream().cuda_stream)


def _vp(arr):
    return ctypes.cast(arr, VP)


class _TwoView:
    """The task tables of the batched hot path, made once over fixed buffers, and its calls."""

    def __init__(self, pairs, hyp):
        P = self.P = len(pairs)
        self.pairs, self.H = pairs, hyp
        nA, nB = [p[0].shape[0] for p in pairs], [p[1].shape[0] for p in pairs]
        i32, f32, u8 = torch.int32, torch.float32, torch.uint8
        self.o = o = {"bestA": _Rows(nA, 2, i32), "secA": _Rows(nA, 2, i32), "bestB": _Rows(nB, 2, i32),
                      "pts": _Rows(nA, 4, f32), "count": _Rows([1] * P, 1, i32), "idx": _Rows([hyp] * P, 8, i32),
                      "counts": _Rows([hyp] * P, 1, i32), "models": _Rows([hyp] * P, 9, f32), "F": _Rows([1] * P, 9, f32),
                      "result": _Rows([1] * P, 4, i32), "mask": _Rows(nA, 1, u8)}
        self.top2, self.filt, self.samp = (BfTop2Task * P)(), (FilterTask * P)(), (SampleTask * P)()
        self.ran, self.fin = (RansacTask * P)(), (FinishTask * P)()
        for i, (a, b, ka, kb) in enumerate(pairs):
            q = {k: v.ptr(i) for k, v in o.items()}
            d = [t.data_ptr() for t in (a, b, ka, kb)]
            self.top2[i] = BfTop2Task(BfTask(nA[i], nB[i], d[0], d[1], q["bestA"], q["bestB"], None, None), q["secA"])
            self.filt[i] = FilterTask(q["bestA"], q["secA"], nA[i], q["bestB"], nB[i], None, q["count"], d[2], d[3], q["pts"])
            self.samp[i] = SampleTask(q["idx"], hyp, nA[i], q["count"], 77 + i)
            self.ran[i] = RansacTask(q["pts"], nA[i], q["count"], q["idx"], hyp, q["counts"], q["models"], None, None)
            self.fin[i] = FinishTask(q["pts"], nA[i], q["count"], q["idx"], q["counts"], q["models"], hyp, q["F"],
                                     q["result"], q["mask"])
        need = ctypes.c_size_t(0)
        check(lib.rsfm_bf_match_top2_workspace_size(_vp(self.top2), P, ctypes.byref(need)), "workspace")
        self.need = need.value
        self.ws = torch.empty(self.need + 256, dtype=torch.uint8, device=DEV)
        self.wsp = (self.ws.data_ptr() + 255) // 256 * 256

    def run(self):
        s, P = _stream(), self.P
        check(lib.rsfm_bf_match_top2(_vp(self.top2), P, VP(self.wsp), self.need, s), "match")
        check(lib.rsfm_filter_matches_batch(_vp(self.filt), P, 4, 5, s), "filter")
        check(lib.rsfm_ransac_sample_indices_batch(_vp(self.samp), P, s), "sample")
        check(lib.rsfm_ransac_f8(_vp(self.ran), P, 1.0, 1, 0.0, 0.0, s), "ransac")
        check(lib.rsfm_ransac_f8_finish(_vp(self.fin), P, 1.0, 1, 0.0, 5000, 1, s), "finish")
        return {k: v.buf for k, v in self.o.items()}


class _Batch:
    """A pipeline handle over fixed buffers: one graph launch a pass."""

    def __init__(self, pairs, case):
        P, hyp = len(pairs), case["hyp"]
        self.pairs = pairs
        nA, nB = [p[0].shape[0] for p in pairs], [p[1].shape[0] for p in pairs]
        i32, f32, u8 = torch.int32, torch.float32, torch.uint8
        dg = case["solver"] == "degensac"
        one = [1] * P
        self.o = o = {"bestA": _Rows(nA, 2, i32), "secA": _Rows(nA, 2, i32), "bestB": _Rows(nB, 2, i32),
                      "matches": _Rows(nA, 3, i32), "count": _Rows(one, 1, i32), "pts": _Rows(nA, 4, f32),
                      "idx": _Rows([hyp] * P, 7 if dg else 8, i32), "counts": _Rows([hyp] * P, 1, i32),
                      "best": _Rows(one, 2, i32), "mask": _Rows(nA, 1, u8), "F": _Rows(one, 9, f32),
                      "result": _Rows(one, 4, i32)}
        if dg:
            o.update(H=_Rows(one, 9, f32), maskH=_Rows(nA, 1, u8), posesF=_Rows(one, 48, f32), poseF=_Rows(one, 10, i32),
                     posesH=_Rows(one, 96, f32), normalsH=_Rows(one, 24, f32), poseH=_Rows(one, 19, i32))
        arr = (PipelinePair * P)()
        lens = (ctypes.c_float * 10)(*(LENS + LENS))
        for i, (a, b, ka, kb) in enumerate(pairs):
            q = lambda k: o[k].ptr(i) if k in o else None  # noqa: E731
            arr[i] = PipelinePair(nA[i], nB[i], a.data_ptr(), b.data_ptr(), ka.data_ptr(), kb.data_ptr(), q("bestA"),
                                  q("secA"), q("bestB"), q("matches"), q("count"), q("pts"), q("idx"), q("counts"),
                                  q("best"), q("mask"), q("F"), q("H"), q("result"), q("maskH"), Camera(*CAM), Camera(*CAM),
                                  q("posesF"), q("poseF"), q("posesH"), q("normalsH"), q("poseH"),
                                  ctypes.cast(lens, VP) if case["lens"] else None, int(synth.WIDTH), int(synth.HEIGHT))
        cfg = PipelineConfig(hyp, T_LINE if dg else 1.0, 0 if dg else 1, 4, 5, 77, 0.0, 0.0, 0, 0, SOLVERS[case["solver"]],
                             T_PLANE, 8, 256, 0.95, 0.0, 5000, 0 if dg else 1, int(case["affine"]), 16, 256, 0.15, 2, 1)
        torch.cuda.synchronize()  # creation times the matcher's tilings on the inputs
        self.h = VP()
        check(lib.rsfm_pipeline_create(_vp(arr), P, ctypes.byref(cfg), ctypes.byref(self.h)), "create")

    def run(self):
        check(lib.rsfm_pipeline_run(self.h, _stream()), "run")
        return {k: v.buf for k, v in self.o.items()}

    def __del__(self):
        if getattr(self, "h", None):
            lib.rsfm_pipeline_destroy(self.h)


class _Verify:
    """Correspondences in hand: samples, hypotheses, the solver's end."""

    def __init__(self, case, seed):
        self.model, self.hyp = case["model"], case["hyp"]
        self.pts = [_correspondences(seed * 1009 + i, n, case["inliers"], 0.0 if self.model == "f8" else 0.6)[0]
                    for i, n in enumerate(_verify_sizes(case))]
        self.k = {"f8": 8, "h4": 4, "degensac": 7}[self.model]

    def run(self):
        idx = [torch.empty((self.hyp, self.k), dtype=torch.int32, device=DEV) for _ in self.pts]
        tasks = (SampleTask * len(self.pts))()
        for i, (p, x) in enumerate(zip(self.pts, idx)):
            tasks[i] = SampleTask(x.data_ptr(), self.hyp, p.shape[0], None, 77 + i)
        check(lib.rsfm_ransac_sample_indices_batch_k(_vp(tasks), len(self.pts), self.k, _stream()), "sample")
        prob = list(zip(self.pts, idx))
        if self.model == "h4":
            return [{k: v for k, v in o.items() if v is not None} for o in ops.ransac_h4(prob, 3.0)]
        if self.model == "f8":
            sc = ops.ransac_f8(prob, 1.0, want_models=True)
            fin = ops.ransac_f8_finish([(p, i, s["counts"], s["models"]) for (p, i), s in zip(prob, sc)], 1.0)
            return [dict(s, **{"final_" + k: v for k, v in f.items()}, idx=i) for s, f, i in zip(sc, fin, idx)]
        sc = ops.ransac_f7(prob, T_LINE, mode=0)
        dg = ops.degensac_refine([(p, i, s["counts"]) for (p, i), s in zip(prob, sc)], T_LINE, T_PLANE, mode=0)
        pf = ops.pose_from_f([(d["F"], CAM, CAM, p, d["mask_f"]) for p, d in zip(self.pts, dg)])
        ph = ops.pose_from_h([(d["H"], CAM, CAM, p, d["mask_h"]) for p, d in zip(self.pts, dg)])
        return [dict(d, counts=s["counts"], poses=f["poses"], pose=f["result"], pose_h=h["result"])
                for d, s, f, h in zip(dg, sc, pf, ph)]


class _CasHash:
    """New images hashed with the projections and biases in hand, then searched against the train image."""

    def __init__(self, case, seed):
        self.case = case
        self.w, base = synth.cashash_weights(3, 192, DEV)
        nQ, nT = case["nQ"], case["nT"]
        self.train, self.q = None, []
        for i in range(case["queries"]):
            a, b = _descriptors(seed * 1013 + i, nQ, nT, 0.3)
            if self.train is None:
                self.train = b
            else:  # the later queries copy rows of the same train image
                at = torch.arange(0, nQ, 4, device=DEV)
                noise = torch.randint(-3, 4, (at.numel(), 128), generator=_gen(seed + i), device=DEV)
                a[at] = (self.train[at % nT].int() + noise).clamp(0, 127).to(torch.uint8)
            self.q.append(a)
        self.bias = cashash.compute_bias(self.w, base, cashash.accumulate(self.train), nT)

    def run(self):
        c = self.case
        t = cashash.register_image(self.train, self.w, self.bias)
        qs = [cashash.register_image(q, self.w, self.bias) for q in self.q]
        if c["mode"] == "union":
            best = cashash.find_best_match(qs, t, c["tables"])
        else:
            best = cashash.find_best_match_rerank(qs, t, c["tables"], 8)
        return {"best": best, "codes": [i["codes"] for i in [t] + qs], "remap": [i["remap"] for i in [t] + qs],
                "ends": [i["ends"] for i in [t] + qs]}


def _features(seed, good):
    """Proposal features of matches: inliers have the lower ratio, and agree in scale and orientation."""
    g, n = _gen(seed), good.numel()
    x = torch.rand((n, 8), generator=g, device=DEV)
    x[:, 0] = torch.where(good, 0.55 + 0.2 * x[:, 0], 0.7 + 0.1 * x[:, 0])
    x[:, 1] = 0.2 + 0.4 * x[:, 1]
    x[:, 2:6] = x[:, 2:6] * 2 - 1
    e = torch.randn((n, 2), generator=g, device=DEV)
    x[:, 6:] = torch.where(good[:, None], 0.15 * e + 0.1, e * torch.tensor([1.2, 0.5], device=DEV))
    x[:, 7].clamp_(-1, 1)
    return x.contiguous()


class _Guided:
    def __init__(self, case, seed):
        self.hyp = case["hyp"]
        made = [_correspondences(seed * 1019 + i, n, 0.3) for i, n in enumerate(_verify_sizes(case))]
        self.pts = [p for p, _ in made]
        g = _gen(seed)  # what a trained proposal says: high for most inliers, plus the floor every match keeps
        self.w = [(torch.where(good, 0.75, 0.08) + 0.2 * torch.rand(good.numel(), generator=g, device=DEV) + 0.02)
                  .contiguous() for _, good in made]

    def run(self):
        idx = learned.sample_weighted([(w, self.hyp, 9 + i) for i, w in enumerate(self.w)])
        return [dict(o, idx=i) for o, i in zip(proposal.score(list(zip(self.pts, idx))), idx)]


class _Net:
    def __init__(self, case, seed):
        n = case["n"]
        good = torch.rand(n, generator=_gen(seed), device=DEV) < 0.4
        self.x, self.y = _features(seed + 1, good), good.float()
        self.params = learned.init_params(seed)
        self.train = case["kind"] == "train"
        self.opt = learned.Adam(self.params, lr=3e-3) if self.train else None

    def run(self):
        if not self.train:
            return learned.forward(self.params, self.x)
        g, loss = learned.grad(self.params, self.x, self.y)
        self.opt.step(g)
        return {"grad": g, "loss": loss, "params": self.params}


class _Top2:
    def __init__(self, pairs):
        self.pairs = pairs
        self.kept = torch.zeros((pairs[0][0].shape[0], 3), dtype=torch.int32, device=DEV)
        self.count = torch.zeros(1, dtype=torch.int32, device=DEV)

    def run(self):
        out = rs.bf_match_top2(self.pairs)
        if len(self.pairs) > 1:
            return out
        (a, s, b), (qa, qb) = out[0], self.pairs[0]
        check(lib.rsfm_filter_matches(a.data_ptr(), s.data_ptr(), qa.shape[0], b.data_ptr(), qb.shape[0], 4, 5,
                                      self.kept.data_ptr(), self.count.data_ptr(), None, 0, _stream()), "filter")
        return [a, s, b, self.kept, self.count]


class _Top1:
    def __init__(self, pairs, impl):
        self.pairs, self.impl = pairs, impl

    def run(self):
        return rs.bf_match(self.pairs, impl=self.impl)


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("top2", "top1"):
        pairs = [_descriptors(seed * 1021 + i, a, b, 0.3) for i, (a, b) in enumerate(_pair_sizes(case))]
        if kind == "top2":
            return _Top2(pairs)
        if case["bits"] == 4:
            pairs = [(rs.desc8b_to_4b(a), rs.desc8b_to_4b(b)) for a, b in pairs]
        return _Top1(pairs, "u4" if case["bits"] == 4 else "mfma")
    if kind in ("two_view", "batch"):
        pairs = [_matched_pair(seed * 1031 + i, a, b) for i, (a, b) in enumerate(_pair_sizes(case))]
        return _TwoView(pairs, case["hyp"]) if kind == "two_view" else _Batch(pairs, case)
    return {"verify": _Verify, "cashash": _CasHash, "guided": _Guided, "train": _Net, "forward": _Net}[kind](case, seed)


def run(state):
    return state.run()


# ---- what a pass cannot do without

# arithmetic of one hypothesis' fit and of one test of a correspondence, in operations
FIT = {"f8": 2000, "f7": 2500, "h4": 1500}
TEST = {"f8": 34, "f7": 3 * 60, "h4": 30}


def _match_work(sizes, per_row, row_bytes=128):
    flops = sum(2 * 128 * a * b for a, b in sizes)
    return flops, sum(row_bytes * (a + b) + 8 * (per_row * a + b) for a, b in sizes)


def _net_flops(n):
    return 2 * n * (8 * 64 + 2 * 64 * 64 + 64)


def work(case):
    kind = case["kind"]
    if kind in ("top2", "top1"):
        flops, by = _match_work(_pair_sizes(case), 2 if kind == "top2" else 1, 16 * case.get("bits", 8))
        return {"flops": flops, "bytes": by}
    if kind in ("two_view", "batch"):
        sizes, H = _pair_sizes(case), case["hyp"]
        flops, by = _match_work(sizes, 2)
        model = "f7" if case.get("solver") == "degensac" else "f8"
        kept = sum(0.25 * min(a, b) for a, b in sizes)  # matches that survive the filter, about
        flops += H * (kept * TEST[model] + len(sizes) * FIT[model])
        by += sum(8 * (a + b) for a, b in sizes) + len(sizes) * H * 36 + 33 * kept
        return {"flops": flops, "bytes": by}
    if kind == "verify":
        m, H = {"f8": "f8", "h4": "h4", "degensac": "f7"}[case["model"]], case["hyp"]
        n = sum(_verify_sizes(case))
        return {"flops": H * (n * TEST[m] + case["pairs"] * FIT[m]), "bytes": 17 * n + case["pairs"] * H * 36}
    if kind == "cashash":
        q, t, Q = case["nQ"], case["nT"], case["queries"]
        # the projections, and the exact distances of a bucket union of a few percent of the other image
        flops = 2 * 128 * 192 * (q * Q + t) + 2 * 128 * Q * q * t * (0.02 * case["tables"] if case["mode"] == "union" else 0)
        flops += 2 * 128 * 8 * Q * (q + t) if case["mode"] == "rerank" else 0
        return {"flops": flops, "bytes": (128 + 8 + 16 + 4 * 8) * (q * Q + t) + 8 * Q * (q + t) + 192 * 132}
    if kind == "guided":
        n, P, H = sum(_verify_sizes(case)), case["pairs"], case["hyp"]
        return {"flops": H * (n * TEST["f8"] + P * FIT["f8"]), "bytes": (16 + 4 + 1) * n + P * H * 36}
    n = case["n"]
    if kind == "train":
        return {"flops": 3 * _net_flops(n), "bytes": 36 * n + 28 * learned.N_PARAM}
    return {"flops": _net_flops(n), "bytes": 36 * n + 4 * learned.N_PARAM}


def tolerance(case):
    # everything but the network is whole numbers, or FP32/FP64 sums whose order the framework fixes: the same on every
    # run and equal to its CPU restatement bit for bit
    # bf16 weights, inputs and activations with FP32 sums: the probabilities are 1.2e-3 off their 64-bit values, the
    # gradient 4.9e-3
    if case["kind"] == "forward":
        return {"rel": 5e-3, "max": 0.1}
    if case["kind"] == "train":
        return {"rel": 2e-2, "max": 0.4}
    return "exact"


def _net64(p, x):
    o = learned
    W = lambda a, b, r: p[a:b].view(r, -1)  # noqa: E731
    h1 = torch.relu(x @ W(o.OFF_W1, o.OFF_B1, 64).T + p[o.OFF_B1:o.OFF_W2])
    h2 = torch.relu(h1 @ W(o.OFF_W2, o.OFF_B2, 64).T + p[o.OFF_B2:o.OFF_W3])
    h3 = torch.relu(h2 @ W(o.OFF_W3, o.OFF_B3, 64).T + p[o.OFF_B3:o.OFF_W4])
    return h3 @ p[o.OFF_W4:o.OFF_B4] + p[o.OFF_B4]


def exact(case, seed):
    """The network in 64 bits. The other kinds' floating results hang on whole-number decisions (which hypothesis wins, who
    its inliers are) that the framework takes in FP32 by contract, and have no value in 64 bits."""
    if case["kind"] not in ("train", "forward"):
        return None
    s = prepare(case, seed)
    p, x, y = s.params.double(), s.x.double(), s.y.double()
    if case["kind"] == "forward":
        return torch.sigmoid(_net64(p, x))
    p.requires_grad_(True)
    loss = torch.nn.functional.binary_cross_entropy_with_logits(_net64(p, x), y)
    g, = torch.autograd.grad(loss, p)
    # Adam's first step from zero moments
    return {"grad": g, "loss": loss.detach().reshape(1), "params": (p - 3e-3 * g / (g.abs() + 1e-8)).detach()}
