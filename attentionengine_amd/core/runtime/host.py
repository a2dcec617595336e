"""Binding of ``csrc/_ae_host.so``: the native host path of repeated calls (csrc/ae_host.cpp says what it does).

An operator owns one ``Host``.  Its Python code runs the first call of a shape -- compiles, plans, tunes, checks --
and hands what it decided to ``add_forward`` / ``add_backward``; later calls of that shape go through ``Host.run``,
which returns None whenever they do not match a plan.  There is no fallback for a library that was not built:
``new_host`` raises, as ``hip_rt.lib()`` does.
"""
from __future__ import annotations

import importlib.util
import os
import os.path as osp
import threading

import torch

from . import hip_rt as rt

HOST_PATH = osp.join(rt.CSRC_DIR, "_ae_host.so")
# kinds of a plan (enum Kind of ae_host.cpp)
PREFILL, PREFILL_SPLIT, DECODE, MLA, MLA_PAGED = range(5)

_module = None
_lock = threading.Lock()


def _load():
    global _module
    if _module is None:
        with _lock:
            if _module is None:
                if not osp.exists(HOST_PATH):
                    raise rt.AEError(f"{HOST_PATH} is missing: build it with `python -c 'import __graft_entry__ as g; "
                                     "g.build()'` (or attentionengine_amd/csrc/build.py)")
                rt.lib()                                   # libae_hip.so, which it links against
                spec = importlib.util.spec_from_file_location("_ae_host", HOST_PATH)
                module = importlib.util.module_from_spec(spec)
                spec.loader.exec_module(module)
                if module.ABI_VERSION != rt.AE_ABI_VERSION:
                    raise rt.AEError(f"{HOST_PATH} was built for C ABI version {module.ABI_VERSION}, this binding is written "
                                     f"for {rt.AE_ABI_VERSION}: rebuild it")
                _module = module
    return _module


def new_host(d, dv, dtype, customs, n_rowscales):
    """A ``Host`` for an operator with these head dims, custom inputs (their descriptors) and row scales."""
    in_dtype = sum(1 << i for i, c in enumerate(customs) if c.torch_dtype != torch.float32)
    return _load().Host(d, dv, dtype == torch.bfloat16, len(customs), in_dtype, n_rowscales)


def _handle(kernel):
    return kernel.handle.value if kernel is not None else 0


def add_forward(host, kind, B, Sq, Hq, Hkv, Skv, device, modules, kernel, cfg, combine=None, ccfg=None, n_split=1,
                kv_per_split=0, page=0, table=None, mask_block=(0, 0), env=(), o_rows=None, counters=0,
                tail_slots=0):
    """Hands a forward launch that has just run to ``host``.  ``env``: switches read at every call; the plan holds
    while they keep their values.  ``modules``: what the kernels live in.  ``o_rows``: partial results a split launch writes (None: one per row and split);
    ``counters``: arrival counters of a launch whose last workgroup merges; ``tail_slots``: see ae_attn_params."""
    host.add({"kind": kind, "B": B, "Sq": Sq, "Hq": Hq, "Hkv": Hkv, "Skv": Skv, "page": page, "device": device.index,
              "k0": _handle(kernel), "k1": _handle(combine), "cfg": bytes(cfg), "ccfg": None if ccfg is None else bytes(ccfg),
              "n_split": n_split, "kv_per_split": kv_per_split, "o_rows": o_rows, "counters": counters, "tail_slots": tail_slots, "table": table, "mask_bm": mask_block[0],
              "mask_bn": mask_block[1], "env": {n: os.environ.get(n, "") for n in env}, "keep": tuple(modules)})


def add_backward(host, B, Sq, Hq, Hkv, Skv, device, modules, delta, dkv, dq, cfg, n_rs, planes, tables=None, dkv_parts=0,
                 work_more=0, again=None, retry=0, skip=0):
    """Hands the backward launches of the forward plan with these extents to ``host``.  ``work_more``: fp32 values of the
    work buffer behind its planes; ``again``: weak reference to the operator that is called instead where they cannot be had,
    then for the next ``retry`` calls too, and for the first ``skip``."""
    host.add_backward({"B": B, "Sq": Sq, "Hq": Hq, "Hkv": Hkv, "Skv": Skv, "device": device.index,
                       "delta": _handle(delta), "dkv": _handle(dkv), "dq": _handle(dq), "cfg": bytes(cfg), "n_rs": n_rs,
                       "planes": planes, "dkv_parts": dkv_parts, "work_more": work_more, "table_dq": tables[0] if tables else None,
                       "table_dkv": tables[1] if tables else None, "keep": tuple(modules), "again": again,
                       "retry": retry, "skip": skip})
