"""Calls of the two operators as programs make them: what is timed when this framework's speed is looked at.

A case is one call, or one training step, of `ttt_forward` / `ttt_backward` through `ttt_mlp_host`:

  call       "forward"   the forward scan alone: inference over a given sequence, or the forward of a step timed by itself
             "backward"  the remat backward alone, from the checkpoints that a forward left
             "train"     forward, zero-fill of the accumulating gradients where the caller has to do it, backward
             "autograd"  `ttt_mlp` and `torch.autograd.grad`: the differentiable call with everything it allocates
  B, NH, NC, cgs         batch, heads, mini-batches of 64 tokens, checkpoint group size
  eta_std    spread of the learning-rate logits (1 or 2, the benchmark's two values)
  wait       the operators block the host until the kernels are done (their default), or only enqueue
  overwrite  the backward overwrites the four accumulating gradients instead of adding to zeros
  workspace  the caller hands over the workspace of the multi-workgroup launches once instead of having it allocated per call
"""
import math
import os
import sys

import torch

_PKG = os.path.join(os.getcwd(), "ttt-tk_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import ttt_mlp_host as host  # noqa: E402

CS, F, HID = 64, 64, 256
STEP_FLOP = 2 * CS * F * HID            # one 64 x 64 x 256 contraction; 7 in the forward of a mini-batch, 21 in its remat backward
MOST_STEPS = 48 * 4096                  # (batch, head, mini-batch) steps of the largest calls

INPUTS = ("XQ", "XK", "XV", "last_eta", "ttt_norm_weight", "ttt_norm_bias", "W1", "b1", "W2", "b2")
CHECKPOINTS = ("W1_checkpoints", "b1_checkpoints", "W2_checkpoints", "b2_checkpoints")


def _case(name, call, B, NH, NC, cgs, eta_std=1.0, wait=True, overwrite=False, workspace=False):
    c = dict(call=call, B=B, NH=NH, NC=NC, cgs=cgs, eta_std=eta_std, wait=wait, overwrite=overwrite, workspace=workspace)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the smallest call: two heads, 256 tokens, a checkpoint before every mini-batch (the oracle's own configuration)
        _case("forward-256tok-2h", "forward", 1, 2, 4, 1),
        # a unit-test-sized differentiable call with a ragged last checkpoint group: allocation and launches are most of it
        _case("autograd-576tok-2x3h", "autograd", 2, 3, 9, 4),
        # inference over a prompt of 2,048 tokens with a dozen heads
        _case("forward-2k-12h", "forward", 1, 12, 32, 16),
        # a training step of a small model, 4,096 tokens, enqueued without waiting
        _case("train-4k-2x12h", "train", 2, 12, 64, 8, wait=False),
        # the benchmark's forward-only workload: 48 heads, 16,384 tokens
        _case("forward-16k-48h", "forward", 1, 48, 256, 16),
        # the backward of the same step
        _case("backward-16k-48h", "backward", 1, 48, 256, 16),
        # an odd number of heads in a batch of three, a sequence that no group size divides
        _case("backward-odd-3x17h", "backward", 3, 17, 77, 10, wait=False, overwrite=True),
        # 96 recurrences: a medium batch of 8,192-token sequences through autograd
        _case("autograd-8k-4x24h", "autograd", 4, 24, 128, 16),
        # 32 long recurrences with the caller's own workspace
        _case("backward-32k-2x16h", "backward", 2, 16, 512, 32, wait=False, workspace=True),
        # nearly a recurrence per compute unit, a ragged group, gradients overwritten
        _case("train-6k-5x40h", "train", 5, 40, 100, 16, wait=False, overwrite=True),
        # the benchmark's long sequence: 48 heads, 262,144 tokens
        _case("train-256k-48h", "train", 1, 48, 4096, 64, wait=False),
        # the benchmark's full chip: 384 recurrences of 32,768 tokens
        _case("train-32k-8x48h", "train", 8, 48, 512, 32, eta_std=2.0, wait=False),
    ]


def _log_uniform(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.5)))))))


def draw(rng):
    B = _log_uniform(rng, 1, 8)
    NH = _log_uniform(rng, 1, 64)
    NC = _log_uniform(rng, 4, min(4096, MOST_STEPS // (B * NH)))
    # group sizes around the square root of the sequence length, as the benchmark's: at most 64 checkpoints, groups of at most 64
    cgs = _log_uniform(rng, max(1, -(-NC // 64)), min(64, NC))
    return _case("", rng.choice(("forward", "backward", "train", "autograd")), B, NH, NC, cgs, eta_std=rng.choice((1.0, 2.0)),
                 wait=rng.random() < 0.5, overwrite=rng.random() < 0.3, workspace=rng.random() < 0.3)


def prepare(case, seed):
    B, NH, NC, cgs = (case[k] for k in ("B", "NH", "NC", "cgs"))
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(seed)

    def rn(*shape, std=1.0, dtype=torch.float32):
        return torch.empty(*shape, device=dev, dtype=dtype).normal_(0.0, std, generator=g)

    # activations ~N(0,1), weights ~N(0,0.02), step sizes sigmoid(N(0,eta_std)) / 64: the benchmark's distributions, with
    # biases and a norm affine as after some training
    t = {k: rn(B, NH, NC, CS, F, dtype=torch.bfloat16) for k in ("XQ", "XK", "XV")}
    t["last_eta"] = (torch.sigmoid(rn(B, NH, NC, CS, 1, std=case["eta_std"])) / CS).to(torch.bfloat16)
    t["ttt_norm_weight"] = 1.0 + rn(1, NH, 1, F, std=0.1)
    t["ttt_norm_bias"] = rn(1, NH, 1, F, std=0.1)
    t["W1"], t["b1"] = rn(B, NH, F, HID, std=0.02), rn(B, NH, 1, HID, std=0.02)
    t["W2"], t["b2"] = rn(B, NH, HID, F, std=0.02), rn(B, NH, 1, F, std=0.02)
    s = {"case": dict(case), "t": t, "workspace": None}
    if case["call"] != "forward":
        t["grad_L_XQW_mini_batch"] = rn(B, NH, NC, CS, F, dtype=torch.bfloat16)
    if case["call"] == "autograd":
        for k in INPUTS:
            t[k].requires_grad_(True)
    else:
        t.update(host.alloc_forward_buffers(B, NH, NC, cgs, dev))
    if case["call"] in ("backward", "train"):
        for k, shape in (("W1", (F, HID)), ("b1", (1, HID)), ("W2", (HID, F)), ("b2", (1, F))):
            t["grad_L_%s_last" % k] = rn(B, NH, *shape, std=1e-3)
        t.update(host.alloc_backward_buffers(B, NH, NC, cgs, dev, zero_fill=not case["overwrite"]))
    if case["workspace"]:
        need = host.workspace_bytes(B, NH, cgs)
        if need:
            s["workspace"] = torch.empty(need, dtype=torch.uint8, device=dev)
    if case["call"] == "backward":
        host.set_synchronize(True)
        host.forward(t, cgs)             # the checkpoints that the backward starts from
    return s


def run(s):
    case, t = s["case"], s["t"]
    host.set_synchronize(case["wait"])
    host.set_accumulate(not case["overwrite"])
    host.set_workspace(s["workspace"])
    cgs = case["cgs"]
    if case["call"] == "autograd":
        out = host.ttt_mlp(*[t[k] for k in INPUTS], cgs)
        grads = torch.autograd.grad(out, [t[k] for k in INPUTS], t["grad_L_XQW_mini_batch"])
        return {"Out": out.detach(), "grads": list(grads)}
    res = {}
    if case["call"] in ("forward", "train"):
        res["Out"] = host.forward(t, cgs)
        res.update({k: t[k] for k in CHECKPOINTS})
    if case["call"] in ("backward", "train"):
        if not case["overwrite"]:
            host.zero_accumulating_grads(t)
        host.backward(t, cgs)
        res.update({k: t[k] for k in host.GRAD_NAMES})
    return res


def work(case):
    pairs, NC, K = case["B"] * case["NH"], case["NC"], -(-case["NC"] // case["cgs"])
    tile, state = CS * F * 2, (2 * F * HID + HID + F) * 4
    step = pairs * NC
    nbytes = flops = 0
    if case["call"] != "backward":       # XQ, XK, XV, eta in; Out out; initial state in, checkpoints out
        nbytes += step * (4 * tile + 2 * CS) + pairs * state * (1 + K)
        flops += 7 * STEP_FLOP * step
    if case["call"] != "forward":        # XQ, XK, XV, dOut, eta in; dXQ, dXK, dXV, d eta out; checkpoints in, state gradients in and out
        nbytes += step * (7 * tile + 4 * CS) + pairs * state * (K + 2)
        flops += 21 * STEP_FLOP * step
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # operands of the matrix products, activations and most outputs are bf16; state and sums are fp32
    return {"rel": 1e-2}
