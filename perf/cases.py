"""Performance cases of the compile-once / invoke-many path.

A user builds or exports an ONNX graph, compiles it once with an ``Executor`` and then calls ``invoke`` with host
arrays for every request; outputs are written into the caller's arrays.  A pass here is one such ``invoke`` call,
copies to and from the device included, on an executor that stays alive from request to request.

Graphs are those of ``fluidml_amd.models`` with their seeded weights; requests (token ids, images) come from the seed.
"""
from __future__ import annotations

import functools
import math
import os
import tempfile

import numpy as np
import torch  # noqa: F401  (before fluidml_amd: the process then has one HIP runtime)

from fluidml_amd import fluidml, models

TEXT = ("small_encoder", "bert_base", "convbert_base", "gpt_neox")


def listed():
    return [
        # a two-layer encoder of the smoke test's size: nothing but launches, copies and the call itself
        {"name": "small_encoder_s32", "model": "small_encoder", "size": 32, "batch": 1, "bf16": False},
        # the headline configuration
        {"name": "bert_base_s128", "model": "bert_base", "size": 128, "batch": 1, "bf16": False},
        # a short query of odd length: embedding or classifying one sentence
        {"name": "bert_base_s37", "model": "bert_base", "size": 37, "batch": 1, "bf16": False},
        # the longest document the position table holds
        {"name": "bert_base_s512", "model": "bert_base", "size": 512, "batch": 1, "bf16": False},
        # mixed self-attention and dynamic convolution
        {"name": "convbert_base_s128", "model": "convbert_base", "size": 128, "batch": 1, "bf16": False},
        # decoder prefill at the configured context, logits of every position returned
        {"name": "gpt_neox_s256", "model": "gpt_neox", "size": 256, "batch": 1, "bf16": False},
        # prefill of a short prompt of odd length
        {"name": "gpt_neox_s77", "model": "gpt_neox", "size": 77, "batch": 1, "bf16": False},
        # the same prefill on the opt-in bf16 contractions
        {"name": "gpt_neox_s256_bf16", "model": "gpt_neox", "size": 256, "batch": 1, "bf16": True},
        # one image through a depthwise-separable network: many small layers
        {"name": "efficientnet_b0_224", "model": "efficientnet_b0", "size": 224, "batch": 1, "bf16": False},
        # one image through large convolutions and weight-bound fully connected layers
        {"name": "vgg16_224_b1", "model": "vgg16", "size": 224, "batch": 1, "bf16": False},
        # a batch of images: the most arithmetic
        {"name": "vgg16_224_b8", "model": "vgg16", "size": 224, "batch": 8, "bf16": False},
        # the same batch on the opt-in bf16 contractions
        {"name": "vgg16_224_b8_bf16", "model": "vgg16", "size": 224, "batch": 8, "bf16": True},
    ]


def draw(rng):
    def spread(low, high):
        return min(high, int(math.exp(rng.uniform(math.log(low), math.log(high + 1)))))

    model = rng.choice(["small_encoder", "bert_base", "bert_base", "convbert_base", "gpt_neox", "gpt_neox",
                        "efficientnet_b0", "vgg16", "vgg16"])
    case = {"model": model, "batch": 1, "bf16": model != "small_encoder" and rng.random() < 0.25}
    if model == "small_encoder":
        case["size"] = spread(4, 64)  # its position table
    elif model == "bert_base":
        case["size"] = spread(12, 512)
    elif model == "convbert_base":
        case["size"] = spread(12, 256)
    elif model == "gpt_neox":
        case["size"] = spread(12, 256)
    elif model == "efficientnet_b0":
        case["size"] = rng.randint(96, 224)  # sides that strides of two do not divide among them
    else:
        case["size"], case["batch"] = rng.randint(96, 224), rng.randint(1, 8)
    return case


def _net(case):
    model, size = case["model"], case["size"]
    if model == "small_encoder":
        return models.bert_base(seq=size, layers=2, hidden=128, heads=4, ffn=256, vocab=500, max_pos=64)
    if model == "efficientnet_b0":
        return models.efficientnet_b0(size)
    if model == "vgg16":
        return models.vgg16(case["batch"], size)
    return getattr(models, model)(seq=size)


def _request(case, seed):
    size = case["size"]
    if case["model"] == "gpt_neox":
        return models.gpt_neox_inputs(size, seed=seed)
    if case["model"] in TEXT:
        return models.bert_inputs(size, 500 if case["model"] == "small_encoder" else 30522, seed=seed)
    return models.image_input((case["batch"], 3, size, size), seed=seed)


@functools.lru_cache(maxsize=32)
def _compiled(key):
    """(executor, outputs' (name, shape, dtype)): what a serving process keeps for one model."""
    case = dict(key)
    net = _net(case)
    executor = fluidml.Executor.make_plain_greedy(case["model"])
    if case["bf16"]:
        executor.context().set_bf16(True)
    with tempfile.TemporaryDirectory() as folder:
        executor.compile(net.save(os.path.join(folder, "model.onnx")))
    return executor, [(v.name, v.shape, v.dtype) for v in net.outputs]


def prepare(case, seed):
    executor, outputs = _compiled(tuple(sorted((k, v) for k, v in case.items() if k != "name")))
    args = {k: np.ascontiguousarray(v) for k, v in _request(case, seed).items()}
    results = {name: np.zeros(shape, dtype) for name, shape, dtype in outputs}
    args.update(results)
    return {"executor": executor, "args": args, "results": results}


def run(state):
    state["executor"].invoke(state["args"])
    return state["results"]


@functools.lru_cache(maxsize=64)
def _work(key):
    net = _net(dict(key))
    tables, flops = set(), 0
    nbytes = sum(int(np.prod(v.shape)) * v.dtype.itemsize for v in net.inputs + net.outputs)
    for n in net.nodes:
        out = n.outputs[0]
        if n.op_type == "MatMul":
            flops += 2 * int(np.prod(out.shape)) * n.inputs[0].shape[-1]
        elif n.op_type == "Gemm":
            flops += 2 * int(np.prod(out.shape)) * n.inputs[0].shape[1]
        elif n.op_type == "Conv":
            flops += 2 * int(np.prod(out.shape)) * int(np.prod(n.inputs[1].shape[1:]))
        elif n.op_type == "Gather" and n.inputs[0].const is not None:  # the looked-up rows of an embedding table
            tables.add(n.inputs[0].name)
            nbytes += min(int(np.prod(out.shape)), int(np.prod(n.inputs[0].shape))) * out.dtype.itemsize
    nbytes += sum(v.const.nbytes for v in net.initializers if v.name not in tables)
    return nbytes, flops


def work(case):
    nbytes, flops = _work(tuple(sorted((k, v) for k, v in case.items() if k not in ("name", "bf16"))))
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # fp32: sums of up to 25088 terms in another order, through up to twelve layers; bf16: 8 bits of mantissa in the
    # operands of every contraction, where a sum in another order can round a value the other way
    return {"rel": 1e-2} if case["bf16"] else {"rel": 3e-5}
