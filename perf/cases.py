"""Workloads of this framework for timing: what a data-parallel rank (or an offline replay) has it
do, through the public entry points, from buckets where launches count to the largest sets.

Five kinds of work, one ``prepare`` / ``run`` pair each:

``step``    one fused sparse step of one flat bucket (score -> exact top-k -> pack -> residual ->
            AdamW), any step variant, score, gradient dtype and state layout
``multi``   the same for several buckets in one call, each with its own top-k (per-bucket online path)
``plugin``  the optimizer / selection / backend plugins as an engine calls them: a full step with
            re-selection, or a sparse step on the index or the mask layout
``select``  exact top-k mask of one flat score array
``replay``  recorded steps of the offline replay: a group of configurations, optionally with the dense
            reference pass before it

A bucket is laid out as a transformer's parameter list (``_layers``) or as one of the two sets of
``sga_amd.shapes``; gradients are Student-t(3), Gaussian with a scale per tensor, or with repeated
magnitudes, as in the benchmark configurations.
"""
import math
from types import SimpleNamespace

import torch

from sga_amd.adamw import OptContext, ParamRecord, SgaAdamW, build_dir_table
from sga_amd.backends import (index_layout_pack, mask_layout_pack, mask_layout_unpack)
from sga_amd.clip import masked_clip_grad_norm
from sga_amd.config import set_args
from sga_amd.fused_step import FusedSparseStep, PackedState, fused_step_multi, k_for
from sga_amd.kernels import scatter_selected
from sga_amd.replay import select_topk_flat
from sga_amd.replay_dense import DenseReplay
from sga_amd.replay_group import Config, ReplayGroup
from sga_amd.selection import TopkSelection
from sga_amd.shapes import llama32_1b, qwen3_06b, segments_for
from sga_amd.support import compact_mask_u8

LLAMA_N, QWEN_N = 1_235_814_400, 596_049_920
# score x ratio x cycle length arms of the replay, in the order a group takes them
REPLAY_ARMS = "abs_g_blind:10:4 abs_g:1:1 update:1:4 abs_g:10:16 abs_g:0.1:4 update:0.1:16 " \
              "abs_g_blind:1:1 abs_g_blind:1:16"
REPLAY_STEPS = 16            # recorded steps of one pass: a whole number of every cycle length


def _step(name, n, **kw):
    case = {"name": name, "kind": "step", "n": n, "set": "layers", "grad": "bf16", "data": "student",
            "score": "abs_g", "ratio": 1.0, "variant": "two_sweep", "packed": False, "mask": False,
            "values": "bf16", "optimizer": "adamw"}
    case.update(kw)
    return case


def listed():
    return [
        # the smallest bucket: one small model's parameters, latency and launches count
        _step("step_small", 261_024),
        # 2^22 fp32 gradients, |g + r| at 1 %: the single-tensor configuration of the benchmark
        _step("step_4m_fp32", 1 << 22, grad="fp32", values="fp32", set="one"),
        # an ordinary DDP bucket of about 40 M coordinates with a ragged end; the buffer already
        # holds g + r (the reference's own contract), Adam-normalised score
        _step("step_40m_single_buffer", 40_013_477, grad="none", score="update"),
        # the Llama-3.2-1B set as one bucket, out of place on ping-pong state: the headline workload
        _step("step_llama1b_out", LLAMA_N, set="llama", score="update", variant="single_out"),
        # the Qwen3-0.6B set as eight buckets with a top 1 % each, mask layout, one call
        {"name": "multi_qwen06b", "kind": "multi", "n": QWEN_N, "set": "qwen", "buckets": 8,
         "grad": "bf16", "data": "scaled", "score": "abs_g", "ratio": 1.0, "mask": True,
         "values": "fp32"},
        # the cycle boundary of the plugin path: full step that emits the score, re-selection over the
        # per-parameter views, index compaction; four transformer layers
        {"name": "plugin_full_63m", "kind": "plugin", "n": 62_920_704, "phase": "full",
         "score": "update", "ratio": 1.0, "clip": 1.0},
        # the steps between boundaries: index pack, clip over the packed values, merge-join commit
        {"name": "plugin_sparse_index_63m", "kind": "plugin", "n": 62_920_704, "phase": "index",
         "score": "abs_g", "ratio": 1.0, "clip": 1.0},
        # the same on the mask layout and a small model, where host work and launches count
        {"name": "plugin_sparse_mask_1m", "kind": "plugin", "n": 1_150_187, "phase": "mask",
         "score": "abs_g", "ratio": 2.0, "clip": 1.0},
        # exact top-k of a billion scores, 5 % of the magnitudes repeated
        {"name": "select_1e9_ties", "kind": "select", "n": 1_000_000_000, "data": "ties", "ratio": 1.0},
        # top-k of one shard's branch scores, odd length
        {"name": "select_3m", "kind": "select", "n": 3_000_017, "data": "student", "ratio": 1.0},
        # offline replay of one of eight shards of the Qwen3-0.6B set, eight configurations
        {"name": "replay_g8_shard", "kind": "replay", "n": 74_506_240, "grad": "bf16", "configs": 8,
         "optimizer": "adamw", "dense": False},
        # a small recorded model: dense reference pass, then two configurations
        {"name": "replay_dense_small", "kind": "replay", "n": 1_500_003, "grad": "fp32", "configs": 2,
         "optimizer": "adamw", "dense": True},
    ]


def _log(rng, lo, hi):
    """Log-uniform, odd more often than not."""
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return min(hi, n | 1 if rng.random() < 0.6 else n)


def draw(rng):
    kind = rng.choice(["step", "step", "step", "multi", "plugin", "plugin", "plugin", "select", "select",
                       "replay"])
    ratio = round(math.exp(rng.uniform(math.log(0.1), math.log(10.0))), 3)
    if kind == "step":
        n = _log(rng, 150_000, LLAMA_N)
        packed = rng.random() < 0.25
        case = _step("", n, set=rng.choice(["layers", "layers", "one"]),
                     grad=rng.choice(["bf16", "bf16", "fp32"] if packed else ["bf16", "bf16", "fp32", "none"]),
                     data=rng.choice(["student", "scaled"]),
                     score=rng.choice(["abs_g", "abs_g", "update", "update", "coi", "abs_m"]),
                     ratio=ratio, variant=rng.choice(["two_sweep", "two_sweep", "single_out"]),
                     packed=packed, mask=rng.random() < 0.3, values=rng.choice(["bf16", "fp32"]),
                     optimizer=rng.choice(["adamw", "adamw", "adams"]))
    elif kind == "multi":
        case = {"kind": "multi", "n": _log(rng, 1_000_000, QWEN_N), "set": "layers",
                "buckets": rng.randint(2, 12), "grad": rng.choice(["bf16", "fp32"]),
                "data": rng.choice(["student", "scaled"]), "score": rng.choice(["abs_g", "update"]),
                "ratio": ratio, "mask": rng.random() < 0.5, "values": rng.choice(["bf16", "fp32"])}
    elif kind == "plugin":
        case = {"kind": "plugin", "n": _log(rng, 150_000, 400_000_000),
                "phase": rng.choice(["full", "index", "mask"]),
                "score": rng.choice(["abs_g", "update", "coi", "abs_m"]), "ratio": ratio,
                "clip": rng.choice([0.01, 1.0])}
    elif kind == "select":
        case = {"kind": "select", "n": _log(rng, 150_000, 1_000_000_000),
                "data": rng.choice(["student", "scaled", "ties"]), "ratio": ratio}
    else:
        case = {"kind": "replay", "n": _log(rng, 300_000, 70_000_000), "grad": rng.choice(["bf16", "fp32"]),
                "configs": rng.randint(1, 8), "optimizer": rng.choice(["adamw", "adams"]),
                "dense": rng.random() < 0.3}
    case.pop("name", None)
    return case


# ------------------------------------------------------------------- inputs
def _layers(n):
    """(name, numel) of a transformer of n parameters: whole layers of the widest hidden size that
    fits twice, the rest as the embedding in front."""
    h = 1024
    while h > 64 and 2 * (15 * h * h + 2 * h + 256) > n:
        h //= 2
    layer = [("in_norm", h), ("q", 2 * h * h), ("k", h * h), ("v", h * h), ("q_norm", 128),
             ("k_norm", 128), ("o", 2 * h * h), ("post_norm", h), ("gate", 3 * h * h),
             ("up", 3 * h * h), ("down", 3 * h * h)]
    per = sum(s for _, s in layer)
    count = min(28, (n - 1) // per)
    out = [("embed", n - count * per)]
    for i in range(count):
        out += [(f"l{i}.{name}", s) for name, s in layer]
    return out


def _shapes(case):
    which = case.get("set", "layers")
    if which == "llama":
        return llama32_1b()
    if which == "qwen":
        return qwen3_06b()
    return [("flat", case["n"])] if which == "one" else _layers(case["n"])


def _gen(seed, dev):
    return torch.Generator(device=dev).manual_seed(int(seed))


def _gradient(n, shapes, data, gen, dev, dtype=torch.float32, chunk=1 << 26):
    """Student-t(3) x 1e-3; Gaussian with a scale per tensor, log-uniform in [1e-5, 1e-2]; or
    Student-t with 5 % of the magnitudes repeated."""
    out = torch.empty(n, dtype=dtype, device=dev)
    if data == "scaled":
        scales = 10.0 ** (-5.0 + 3.0 * torch.rand(len(shapes), generator=gen, device=dev)).cpu()
        off = 0
        for (_name, s), std in zip(shapes, scales.tolist()):
            for a in range(off, off + s, chunk):
                b = min(off + s, a + chunk)
                out[a:b] = torch.randn(b - a, generator=gen, device=dev) * std
            off += s
        return out
    for a in range(0, n, chunk):
        b = min(n, a + chunk)
        z = torch.randn(b - a, generator=gen, device=dev)
        chi = torch.zeros(b - a, device=dev)
        for _ in range(3):
            chi += torch.randn(b - a, generator=gen, device=dev).square_()
        out[a:b] = z / torch.sqrt(chi / 3.0) * 1e-3
    if data == "ties":
        pairs = (n + 18) // 20
        out[0::20][:pairs] = out[1::20].clone()
    return out


def _moments(n, gen, dev, g_scale=1e-3):
    """p, m, v in the middle of a training run."""
    p = torch.randn(n, generator=gen, device=dev).mul_(0.02)
    m = torch.randn(n, generator=gen, device=dev).mul_(0.1 * g_scale)
    v = torch.rand(n, generator=gen, device=dev).add_(0.05).mul_(g_scale * g_scale)
    return p, m, v


# --------------------------------------------------------------------- step
_GRAD = {"bf16": torch.bfloat16, "fp32": torch.float32, "none": torch.float32}


def _prepare_step(case, seed, dev):
    n, gen = case["n"], _gen(seed, dev)
    shapes = _shapes(case)
    segs, total = segments_for(shapes)
    assert total == n
    k = k_for(n, case["ratio"])
    fs = FusedSparseStep(n, segs, dev, values_dtype=_GRAD[case["values"]], max_k=k,
                         want_mask=case["mask"])
    g = _gradient(n, shapes, case["data"], gen, dev, _GRAD[case["grad"]])
    p, m, v = _moments(n, gen, dev)
    if case["grad"] == "none":          # backward accumulated into the buffer that keeps the residual
        r, g = g, None
    else:
        r = torch.randn(n, generator=gen, device=dev).mul_(3e-4)
    cur = [r, p, m, v]
    single = case["variant"] == "single_out"
    if case["packed"]:
        cur = PackedState(n, dev).pack(*cur)
        nxt = PackedState(n, dev) if single else None
    else:
        nxt = [torch.empty_like(t) for t in cur] if single else None
    return {"case": case, "fs": fs, "g": g, "cur": cur, "nxt": nxt, "k": k, "t": 100,
            "packed_last": None}


def _run_step(s):
    case, fs = s["case"], s["fs"]
    s["t"] += 1
    if s["packed_last"] is not None:
        # single buffer (flat tensors only): the next backward lands where the last pack left zeros
        scatter_selected(s["cur"][0], s["packed_last"][0], s["packed_last"][1].float())
    kw = dict(k=s["k"], score=case["score"], optimizer=case["optimizer"])
    if s["nxt"] is not None:
        kw.update(single_sweep=True, out=s["nxt"], check=False)
    if case["packed"]:
        idx, values = fs.step_packed(s["g"], s["cur"], s["t"], **kw)
    else:
        idx, values = fs.step(s["g"], *s["cur"], s["t"], **kw)
    if s["nxt"] is not None:
        s["cur"], s["nxt"] = s["nxt"], s["cur"]
    if s["g"] is None:
        s["packed_last"] = (idx, values)
    state = s["cur"].data if case["packed"] else s["cur"]
    return {"idx": idx, "values": values, "mask": fs.mask, "state": state}


def _work_step(case):
    n, k = case["n"], k_for(case["n"], case["ratio"])
    g = {"bf16": 2, "fp32": 4, "none": 0}[case["grad"]]
    bytes_ = n * (g + 32 + (1 if case["mask"] else 0)) + k * (4 + (2 if case["values"] == "bf16" else 4))
    return {"bytes": bytes_, "flops": n * (30 if case["score"] in ("update", "coi") else 16)}


# -------------------------------------------------------------------- multi
def _bucket_cuts(case, segs, n):
    """Bucket boundaries at tensor boundaries, about n / buckets apart."""
    if case["set"] == "qwen":
        return [0, segs[1]["start"]] + [segs[1 + 11 * j]["start"] for j in range(4, 28, 4)] + [n]
    starts = [s["start"] for s in segs] + [n]
    cuts = [0]
    for b in range(1, case["buckets"]):
        at = min(starts, key=lambda s: abs(s - b * n // case["buckets"]))
        if at > cuts[-1] and at < n:
            cuts.append(at)
    return cuts + [n]


def _prepare_multi(case, seed, dev):
    n, gen = case["n"], _gen(seed, dev)
    shapes = _shapes(case)
    segs, _ = segments_for(shapes)
    cuts = _bucket_cuts(case, segs, n)
    g = _gradient(n, shapes, case["data"], gen, dev, _GRAD[case["grad"]])
    p, m, v = _moments(n, gen, dev)
    r = torch.randn(n, generator=gen, device=dev).mul_(3e-4)
    spans = list(zip(cuts[:-1], cuts[1:]))
    ks = [k_for(hi - lo, case["ratio"]) for lo, hi in spans]
    steppers = [FusedSparseStep(hi - lo, [dict(s, start=s["start"] - lo) for s in segs
                                          if lo <= s["start"] < hi], dev,
                                values_dtype=_GRAD[case["values"]], max_k=k, want_mask=case["mask"])
                for (lo, hi), k in zip(spans, ks)]
    views = [[t[lo:hi] for lo, hi in spans] for t in (g, r, p, m, v)]
    return {"case": case, "steppers": steppers, "views": views, "state": [r, p, m, v], "ks": ks, "t": 100}


def _run_multi(s):
    s["t"] += 1
    packs = fused_step_multi(s["steppers"], *s["views"], s["t"], ks=s["ks"], score=s["case"]["score"])
    return {"packs": packs, "masks": [fs.mask for fs in s["steppers"]], "state": s["state"]}


def _work_multi(case):
    return _work_step(dict(case, optimizer="adamw"))


# ------------------------------------------------------------------- plugin
def _prepare_plugin(case, seed, dev):
    n, gen = case["n"], _gen(seed, dev)
    shapes = _layers(n)
    segs, _ = segments_for(shapes)
    set_args(SimpleNamespace(sga_score=case["score"], sga_optimizer_residual_mean=False,
                             sga_optimizer_compact_search="table",
                             sga_optimizer_full_sync_inactive_lr_scale=1.0,
                             sga_selection_method="histogram",
                             sga_selection_ratio_percent=case["ratio"],
                             sga_selection_histogram_mode="exact"))
    g = _gradient(n, shapes, "student", gen, dev)
    p, m, v = _moments(n, gen, dev)
    bucket = SimpleNamespace(grad_data=g.clone(), active_mask_u8=None, extra_main_grads=[], support_index=0)
    records = []
    for s in segs:
        a, b = s["start"], s["start"] + s["n"]
        mp = SimpleNamespace(data=p[a:b], grad=bucket.grad_data[a:b])
        records.append(ParamRecord(None, mp, bucket, a, b, s["lr"], s["b1"], s["b2"], s["eps"], s["wd"], 100,
                                   _state={"exp_avg": m[a:b], "exp_avg_sq": v[a:b]}))
    st = {"case": case, "opt": SgaAdamW(), "sel": TopkSelection(), "bucket": bucket, "records": records,
          "g": g, "state": [p, m, v]}
    if case["phase"] != "full":
        k = k_for(n, case["ratio"])
        mask = select_topk_flat(g.abs() + torch.rand(n, generator=gen, device=dev).mul_(1e-3), k)[0]
        bucket.active_mask_u8 = mask.view(torch.uint8)
        idx = compact_mask_u8(bucket.active_mask_u8)
        st.update(idx=idx, fresh=g[idx.long()], values=torch.empty(k, device=dev),
                  support=SimpleNamespace(buckets=[SimpleNamespace(idx=idx, dir_table=build_dir_table(idx, n))]))
    return st


def _run_plugin(s):
    case, opt, bucket, records = s["case"], s["opt"], s["bucket"], s["records"]
    for r in records:
        r.step += 1
    if case["phase"] == "full":
        bucket.grad_data.copy_(s["g"])                                 # this step's backward
        norm, _ = masked_clip_grad_norm(records, case["clip"], was_full=True)
        opt.full_step(OptContext(records, "full", bucket_states=[bucket]))
        masks = s["sel"].select(SimpleNamespace(grad_views=[r.grad for r in records]))
        bucket.active_mask_u8 = torch.cat(masks)
        idx = compact_mask_u8(bucket.active_mask_u8)
        return {"norm": norm, "mask": bucket.active_mask_u8, "idx": idx, "dir": build_dir_table(idx, case["n"]),
                "score": bucket.grad_data, "state": s["state"]}
    # the backward of a step adds to the support's coordinates, which the last pack left at zero
    scatter_selected(bucket.grad_data, s["idx"], s["fresh"])
    if case["phase"] == "index":
        index_layout_pack(bucket.grad_data, s["idx"], s["values"], factor=0.5)
        values = {id(bucket): s["values"]}
        norm, coeff = masked_clip_grad_norm(records, case["clip"], was_full=False, compact_values=values)
        opt.sparse_step(OptContext(records, "sparse", support=s["support"], bucket_states=[bucket],
                                   apply_coeff=coeff, compact_values=values))
        return {"norm": norm, "coeff": coeff, "values": s["values"], "grad": bucket.grad_data,
                "state": s["state"]}
    payloads, idx = mask_layout_pack(bucket.grad_data, bucket.active_mask_u8, factor=0.5)
    mask_layout_unpack(bucket.grad_data, idx, payloads)
    norm, coeff = masked_clip_grad_norm(records, case["clip"], was_full=False)
    opt.sparse_step(OptContext(records, "sparse", bucket_states=[bucket], apply_coeff=coeff))
    return {"norm": norm, "coeff": coeff, "payload": torch.cat(payloads), "idx": idx, "grad": bucket.grad_data,
            "state": s["state"]}


def _work_plugin(case):
    n, k = case["n"], k_for(case["n"], case["ratio"])
    if case["phase"] == "full":      # g in; score, p, m, v out; p, m, v in; mask and index list out
        return {"bytes": n * (4 + 4 + 24 + 1) + k * 4, "flops": n * 30}
    # p, m, v in and out; per selected coordinate: its index, its gradient out and back in, its value
    per_k = 4 + 4 + 4 + 4
    extra = 9 if case["phase"] == "mask" else 0         # the mask, the gradient buffer read and cleared
    return {"bytes": n * (24 + extra) + k * per_k, "flops": n * 16}


# ------------------------------------------------------------------- select
def _prepare_select(case, seed, dev):
    n, gen = case["n"], _gen(seed, dev)
    score = _gradient(n, _layers(n), case["data"], gen, dev).abs_()
    return {"score": score, "k": k_for(n, case["ratio"])}


def _run_select(s):
    mask, thresh = select_topk_flat(s["score"], s["k"])
    return {"mask": mask, "thresh": thresh}


def _work_select(case):
    return {"bytes": case["n"] * 5, "flops": case["n"] * 2}


# ------------------------------------------------------------------- replay
def _arms(case):
    return [Config(s, float(r), int(t), optimizer=case["optimizer"])
            for s, r, t in (a.split(":") for a in REPLAY_ARMS.split()[:case["configs"]])]


def _prepare_replay(case, seed, dev):
    n, gen = case["n"], _gen(seed, dev)
    shapes = _layers(n)
    segs, _ = segments_for(shapes)
    entries = [{"a": s["start"], "n": s["n"], "b1": s["b1"], "b2": s["b2"], "eps": s["eps"], "wd": s["wd"],
                "group": 0} for s in segs]
    window = [_gradient(n, shapes, "student", gen, dev, _GRAD[case["grad"]]) for _ in range(REPLAY_STEPS)]
    w0, m0, v0 = _moments(n, gen, dev)
    base = window[0].float().abs_()
    arms = _arms(case)
    sel0 = [select_topk_flat(base, k_for(n, c.ratio))[0] for c in arms]
    group = ReplayGroup(entries, w0, m0, v0, sel0, arms, t0=100, window=1 << 20)
    dense = DenseReplay(entries, w0, m0, v0, 100, case["optimizer"]) if case["dense"] else None
    return {"case": case, "window": window, "group": group, "dense": dense}


def _run_replay(s):
    group, dense = s["group"], s["dense"]
    out = {}
    if dense is not None:
        meta = {"clip_grad": 1.0, "grad_norm": 1.5, "lr": [1e-4]}
        for t, g in enumerate(s["window"]):
            dense.step(t, g, meta)
        out["dense"] = [dense.w, dense.m, dense.v, dense.label,
                        [r["recon_grad_norm"] for r in dense.recon_steps[-REPLAY_STEPS:]]]
        del dense.recon_steps[:]
    for g in s["window"]:
        group.step(g, {"clip_grad": 1.0, "grad_norm": 1.5, "lr": 1e-4})
    out["state"] = [st.data for st in group.state]
    out["sel"] = [st.sel for st in group.state]
    out["coef"] = group.coef_d
    return out


def _work_replay(case):
    n, arms = case["n"], _arms(case)
    g = 2.0 if case["grad"] == "bf16" else 4.0
    per = 0.0                                           # bytes per coordinate of the whole pass
    for s in range(REPLAY_STEPS):
        per += g                                        # the recorded gradient, once for the group
        for c in arms:
            bnd, clean = s % c.T == 0, (s - 1) % c.T == 0       # clean: the residual is known to be zero
            per += 24.0 + (0.0 if clean else 4.0) + (0.0 if bnd and clean else 4.0) + 0.125
            if case["dense"] and c is arms[0]:
                per += g + 32.0                         # w, m, v and the label in and out
    return {"bytes": n * per, "flops": n * REPLAY_STEPS * len(arms) * 16}


# ----------------------------------------------------------------- interface
_PREPARE = {"step": _prepare_step, "multi": _prepare_multi, "plugin": _prepare_plugin,
            "select": _prepare_select, "replay": _prepare_replay}
_RUN = {"step": _run_step, "multi": _run_multi, "plugin": _run_plugin, "select": _run_select,
        "replay": _run_replay}
_WORK = {"step": _work_step, "multi": _work_multi, "plugin": _work_plugin, "select": _work_select,
         "replay": _work_replay}


def prepare(case, seed):
    return _RUN[case["kind"]], _PREPARE[case["kind"]](case, seed, torch.device("cuda:0"))


def run(state):
    fn, s = state
    return fn(s)


def work(case):
    return _WORK[case["kind"]](case)


def tolerance(case):
    # The fused steps and the select evaluate one chain of correctly rounded operations per
    # coordinate: any correct implementation gives the same bits.  The plugin steps and the replay
    # scale by a clip coefficient that comes from a 32- or 64-bit sum over the bucket, whose rounding
    # depends on the order of the sum (1e-6 relative in the coefficient, 1e-5 after a few steps); a
    # coordinate at a threshold may then fall on the other side.
    if case["kind"] in ("plugin", "replay"):
        return {"rel": 1e-5, "max": 1e-3, "differ": 1e-5}
    return "exact"
