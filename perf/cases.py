"""The workloads this library's speed is measured on: training steps and scoring calls of the extreme
classifier through the public entry points, from one small call to the largest benchmark shape.

A case is a dict of plain values; `kind` says which entry point a user's program calls:

  csr        XFCLayer.step_csr, the whole training step from a CSR label list
  coo        XFCLayer.xfc_backward, the same from the collator's row-sorted COO pair
  trainer    BCELossMultiNode as the reference's fit loop drives it (fp32 embeddings, `accum` micro-batches)
  master     XFCLayer(master_weights=True).xfc_backward, fp32 weights and momentum
  autograd   xfc_loss(...).backward() with the summed loss
  topk       XFCLayer.topk, the K best labels of every row
  gemm       the drop-in six-argument xfc_gemm: sigmoid(X.W^T), G^T.X and G.W
"""
from __future__ import annotations

import math

import torch

from renee_amd import BCELossMultiNode, XFCLayer, synth, xfc_gemm, xfc_loss

LR, MU = 0.05, 0.9
STEPS = ("csr", "coo", "trainer", "master", "autograd")


def listed():
    return [
        # a classifier of a few thousand labels (unit-test and smoke size): launches and host time count
        dict(name="coo_b64_4k", kind="coo", B=64, L=4097, d=768, kmax=8, kmean=2.3, zipf=1.1),
        # the small-batch configuration: 131,072 labels, 32 rows
        dict(name="csr_b32_131k", kind="csr", B=32, L=131072, d=768, kmax=8, kmean=2.3, zipf=1.1),
        # the usual training batch on a 131,073-label data set (an odd count), driven by the loss module
        dict(name="trainer_b512_131k", kind="trainer", B=512, L=131073, d=768, accum=1, kmax=8, kmean=2.3, zipf=1.1),
        # the headline configuration
        dict(name="csr_b512_1310k", kind="csr", B=512, L=1310720, d=768, kmax=20, kmean=5.0, zipf=1.0),
        # the largest data set that is trained as one step of 1024 rows, a ragged label count
        dict(name="coo_b1024_2812k", kind="coo", B=1024, L=2812281, d=768, kmax=30, kmean=8.0, zipf=0.9),
        # the reference's optimizer regime: fp32 weights and momentum beside the fp16 copy
        dict(name="master_b512_655k", kind="master", B=512, L=655363, d=768, kmax=20, kmean=5.0, zipf=1.0),
        # gradient accumulation over four micro-batches of 256 rows, with a 384-wide encoder
        dict(name="trainer_accum4_b1024_320k_d384", kind="trainer", B=1024, L=320001, d=384, accum=4, kmax=20, kmean=5.0,
             zipf=1.0),
        # the step as a differentiable scalar that also returns the loss; the last, partial batch of an epoch
        dict(name="autograd_b199_131k", kind="autograd", B=199, L=131072, d=768, kmax=8, kmean=2.3, zipf=1.1),
        # validation during training: the five best labels of 1024 rows over all labels
        dict(name="top5_b1024_2812k", kind="topk", B=1024, L=2812281, d=768, K=5),
        # final evaluation: the hundred best labels
        dict(name="top100_b512_1310k", kind="topk", B=512, L=1310720, d=768, K=100),
        # serving: a handful of queries at a time
        dict(name="top5_b16_131k", kind="topk", B=16, L=131072, d=768, K=5),
        # a program that keeps its own trainer and only calls the extension function
        dict(name="gemm_b512_131k", kind="gemm", B=512, L=131072, d=768),
    ]


LARGEST = 1024 * 2812281 * 768


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One case of the ranges above: 1 to 1024 rows (training from 8), 4,000 to 2.8 million labels, encoder
    widths from a 64-wide bottleneck to 1024."""
    while True:
        kind = rng.choice(["csr", "csr", "coo", "coo", "trainer", "master", "autograd", "topk", "topk", "topk", "gemm"])
        d = rng.choice([64, 128, 256, 384, 512, 768, 768, 768, 768, 1024])
        L = _log_int(rng, 4000, 2812281)
        B = _log_int(rng, 1 if kind == "topk" else 8, 1024)
        if rng.random() < 0.4:  # full batches are the common case
            B = rng.choice([32, 64, 128, 256, 512, 1024])
        case = dict(kind=kind, B=B, L=L, d=d)
        if kind == "topk":
            case["K"] = rng.choice([1, 3, 5, 5, 5, 10, 100, 100, 200])
        elif kind != "gemm":
            kmax = rng.choice([8, 20, 30])
            case.update(kmax=kmax, kmean=round(rng.uniform(2.0, kmax / 3), 2), zipf=rng.choice([0.9, 1.0, 1.1]))
        if kind == "trainer":
            case["accum"] = rng.choice([1, 1, 2, 4])
        if kind == "gemm":
            case["L"] = L = -(-L // 16) * 16  # the reference pads the label count for its extension
            if B % 8:
                case["B"] = B = -(-B // 8) * 8
        per_weight = 16 if kind == "gemm" else 18 if kind == "master" else 8
        if B * L * d <= LARGEST // 2 and per_weight * L * d <= 8 * 2812281 * 512:
            return case


def prepare(case, seed):
    dev = torch.device("cuda:0")
    kind, B, L, d = case["kind"], case["B"], case["L"], case["d"]
    X = synth.make_X(B, d, seed, dev, torch.float32)
    if kind == "gemm":
        W = synth.make_W(L, d, seed, dev, torch.float16)
        return dict(case=case, X=X.half(), W=W, out=torch.empty(B, L, device=dev, dtype=torch.float16),
                    grad=torch.empty(L, d, device=dev, dtype=torch.float32),
                    dX=torch.empty(B, d, device=dev, dtype=torch.float32))
    master = kind == "master"
    W = synth.make_W(L, d, seed, dev, torch.float32 if master else torch.float16)
    layer = XFCLayer(L, d, B, dev, lr=LR, momentum=MU, weight=W, master_weights=master)
    if kind == "topk":
        return dict(case=case, layer=layer, X=X.half())
    g = torch.Generator(device=dev)
    g.manual_seed(3000 + seed)
    step = 1 << 20
    for r0 in range(0, L, step):  # the momentum of a run under way
        layer.momentum_buffer[r0:r0 + step].normal_(0.0, 1e-3, generator=g)
    P = synth.make_positives(B, L, case["kmax"], case["kmean"], case["zipf"], seed)
    state = dict(case=case, layer=layer, X=X if kind in ("trainer", "autograd") else X.half())
    if kind == "csr":
        state.update(rowptr=torch.from_numpy(P.rowptr).to(dev), colidx=torch.from_numpy(P.colidx).to(dev))
        return state
    px, py = P.coo()
    if kind != "trainer":
        state.update(px=px.to(dev), py=py.to(dev))
    else:
        n = min(case["accum"], B)
        state["loss"] = BCELossMultiNode(layer, accum=n)
        state["micro"] = []
        for i in range(n):  # rows and their label pairs, micro-batch by micro-batch
            r0, r1 = B * i // n, B * (i + 1) // n
            p0, p1 = int(P.rowptr[r0]), int(P.rowptr[r1])
            state["micro"].append((r0, r1, (px[p0:p1] - r0).to(dev), py[p0:p1].to(dev)))
    if kind == "autograd":
        state["X"].requires_grad_(True)
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "gemm":
        X, W, out, grad, dX = (state[k] for k in ("X", "W", "out", "grad", "dX"))
        xfc_gemm(X, W.t(), out, 1.0, 0.0, True)
        xfc_gemm(out.t(), X, grad, 1.0, 0.0, False)
        xfc_gemm(out, W, dX, 1.0, 0.0, False)
        return dict(out=out, grad=grad, dX=dX)
    layer = state["layer"]
    if kind == "topk":
        values, labels = layer.topk(state["X"], case["K"])
        return dict(values=values, labels=labels)
    result = dict(weight=layer.xfc_weight, momentum=layer.momentum_buffer)
    if kind == "csr":
        result["grad_input"] = layer.step_csr(state["X"], state["rowptr"], state["colidx"])
    elif kind in ("coo", "master"):
        result["grad_input"] = layer.xfc_backward(state["X"], state["px"], state["py"])
        if kind == "master":
            result["master"] = layer.xfc_weight_master
    elif kind == "autograd":
        X = state["X"]
        X.grad = None
        loss = xfc_loss(X, layer, state["px"], state["py"], compute_loss=True)
        loss.backward()
        result.update(loss=loss, grad_input=X.grad)
    else:
        module = state["loss"]
        for r0, r1, px, py in state["micro"]:
            embed = module.gather_embed(state["X"][r0:r1])
            module.xfc_backward(embed, layer.outsoft[0:r1 - r0, :layer.numy], px, py, layer.grad_input[r0:r1])
        module.xfc_optimizer.step()
        result["grad_input"] = layer.grad_input[0:case["B"]]
    return result


def work(case):
    kind, B, L, d = case["kind"], case["B"], case["L"], case["d"]
    if kind == "topk":
        return dict(bytes=2 * L * d + 2 * B * d + 12 * B * case["K"], flops=2 * B * L * d)
    if kind == "gemm":  # X, W read; out, grad, dX written
        return dict(bytes=2 * L * d + 2 * B * d + 2 * B * L + 4 * L * d + 4 * B * d, flops=6 * B * L * d)
    per_weight = 18 if kind == "master" else 8  # weights and momentum read and written
    pairs = B * case["kmean"]
    embed = 4 if kind in ("trainer", "autograd") else 2
    return dict(bytes=per_weight * L * d + (embed + 4) * B * d + 16 * pairs, flops=6 * B * L * d)


def tolerance(case):
    """About four times the distance of each path from the same expressions in float64 (largest of the kinds below)."""
    if case["kind"] == "topk":
        if case["K"] <= 8:  # scores are fp32 sums; labels may change places where two scores differ by less than that
            return dict(rel=1e-5, max=1e-4, differ=1e-3)
        return dict(rel=1e-4, max=2e-3, differ=2e-3)  # scores are rounded to fp16: equal ones are ordered by label
    # G is rounded to fp16 once (2.2e-4 of its norm, 3e-4 in the momentum); so are the weights and the momentum unless they are kept in fp32
    return dict(rel=1.2e-3, max=6e-3)
