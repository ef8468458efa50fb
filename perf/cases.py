"""Performance cases: the calls a program that serves a quantized checkpoint makes, timed one pass at a time.

Two models are served with this library: the dense hybrid model (hidden 5120, FFN 17408, IQ3_XXS
tensors with Q6_K / Q5_K / Q4_K ones beside them) and the mixture of experts (hidden 2048, 256 routed
experts of FF 512 and one shared, top-8).  A case is one block of one of them, called through
``thunderllamax_amd.ops`` the way the integration notes show, with weights uploaded and repacked
beforehand (``prepare``) and caller-owned buffers.

Kinds, and the range that ``draw`` takes each over:

* ``route``        router of a MoE layer: logits, top-8, gates, shared gate; P = 1..2048 positions
* ``ffn``          decode / speculative-verify FFN block: residual add + RMSNorm, gate+up+SwiGLU,
                   down + residual; M = 1..16 rows; tiled records, packed rows or the packed7 plane
* ``qkv``          decode q/k/v (IQ3_XXS or Q6_K q, Q4_K v) or GDN projections; M = 1..16
* ``head``         lm_head: Q5_K, Q6_K (fp16 activations, M = 1..16) or Q6_K with fp32 activations
* ``prefill_ffn``  FFN block of a prompt chunk: gate+up+SwiGLU, down + residual; M = 256..2048
* ``prefill_qkv``  merged q/k/v or GDN qkv + gate GEMM of a prompt chunk; M = 256..2048
* ``moe``          MoE layer, IQ4_XS experts; P = 1..2048; tiled slabs or GGUF rows
* ``moe_ckpt``     MoE layer, IQ3_S gate/up, Q6_K down, Q8_0 shared expert; P = 1..2048
"""
import math

import numpy as np
import torch

from thunderllamax_amd import formats, ops
from thunderllamax_amd._lib import (LAYOUT_PACK7, LAYOUT_PACKED, LAYOUT_RAW, LAYOUT_TILED, TYPE_IQ3_XXS, TYPE_Q4_K,
                                    TYPE_Q5_K, TYPE_Q6_K, V_Q4K)

DEV = "cuda"
HID, FFN = 5120, 17408              # the dense model
MHID, MFF, EXPERTS, TOPK = 2048, 512, 256, 8   # the mixture of experts
LAYOUTS = {"tiled": LAYOUT_TILED, "packed": LAYOUT_PACKED, "packed7": LAYOUT_PACK7, "raw": LAYOUT_RAW}
# bytes of a block, weights in it, offset of its fp16 scales (and how many follow each other)
BLOCKS = {"iq3xxs": (98, 256, 0, 1), "q6k": (210, 256, 208, 1), "q4k": (144, 256, 0, 2), "q5k": (176, 256, 0, 2),
          "iq4xs": (136, 256, 0, 1), "iq3s": (110, 256, 0, 1), "q8_0": (34, 32, 0, 1)}
# the dense model's tensors that a qkv / prefill_qkv call reads: (rows, class)
QKV = {"q6": ((12288, "q6k"), (1024, "iq3xxs"), (1024, "q4k")),
       "iq3": ((12288, "iq3xxs"), (1024, "iq3xxs"), (1024, "q4k")),
       "gdn": ((10240, "iq3xxs"), (6144, "iq3xxs"), (48, "iq3xxs"), (48, "iq3xxs"))}
PREFILL_QKV = {"q6": QKV["q6"], "iq3": QKV["iq3"], "gdn": ((10240, "q5k"), (6144, "iq3xxs"))}
HEADS = {"q5k": (248320, HID), "q6k": (151936, HID), "q6k_f32": (HID, HID), "q6k_f32_moe": (248320, MHID)}


def listed():
    return [
        # the router of one MoE layer at a small verify width: one short launch, 40 times a token
        {"name": "route_p4", "kind": "route", "P": 4},
        # plain decoding of the dense model: 64 such blocks a token
        {"name": "ffn_m1", "kind": "ffn", "M": 1, "layout": "tiled"},
        # the same at the widest speculative-verify width that the model is run with
        {"name": "ffn_m11", "kind": "ffn", "M": 11, "layout": "tiled"},
        # attention projections with three weight classes in one call, a mid verify width
        {"name": "qkv_q6_m4", "kind": "qkv", "M": 4, "mix": "q6"},
        # the dense model's head over the full vocabulary, once a step
        {"name": "head_q5k_m11", "kind": "head", "M": 11, "head": "q5k"},
        # the FFN block of a short prompt chunk, and of the usual one
        {"name": "prefill_ffn_m256", "kind": "prefill_ffn", "M": 256},
        {"name": "prefill_ffn_m2048", "kind": "prefill_ffn", "M": 2048},
        # the projections of a prompt chunk whose q is Q6_K
        {"name": "prefill_qkv_q6_m1024", "kind": "prefill_qkv", "M": 1024, "mix": "q6"},
        # a MoE layer at the verify width and over a whole prompt chunk
        {"name": "moe_p11", "kind": "moe", "P": 11, "layout": "tiled"},
        {"name": "moe_p2048", "kind": "moe", "P": 2048, "layout": "tiled"},
        # the checkpoint's own classes: plain decoding of a few sequences, and its 256-token chunk
        {"name": "moe_ckpt_p3", "kind": "moe_ckpt", "P": 3, "layout": "tiled"},
        {"name": "moe_ckpt_p256", "kind": "moe_ckpt", "P": 256, "layout": "tiled"},
    ]


def draw(rng):
    known = [{k: v for k, v in c.items() if k != "name"} for c in listed()]
    while True:
        case = _draw(rng)
        if case not in known:
            return case


def _draw(rng):
    def spread(lo, hi):   # whole numbers, even over their logarithm
        return min(hi, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))

    kind = rng.choice(["route", "ffn", "ffn", "qkv", "head", "prefill_ffn", "prefill_qkv", "moe", "moe", "moe_ckpt",
                       "moe_ckpt"])
    if kind == "route":
        return {"kind": kind, "P": spread(1, 2048)}
    if kind == "ffn":
        return {"kind": kind, "M": rng.randint(1, 16), "layout": rng.choice(["tiled", "tiled", "packed", "packed7"])}
    if kind == "qkv":
        return {"kind": kind, "M": rng.randint(1, 16), "mix": rng.choice(sorted(QKV))}
    if kind == "head":
        head = rng.choice(sorted(HEADS))
        return {"kind": kind, "M": 1 if head.startswith("q6k_f32") else rng.randint(1, 16), "head": head}
    if kind == "prefill_ffn":
        return {"kind": kind, "M": 256 * rng.randint(1, 8)}
    if kind == "prefill_qkv":
        return {"kind": kind, "M": 256 * rng.randint(1, 8), "mix": rng.choice(sorted(PREFILL_QKV))}
    return {"kind": kind, "P": spread(1, 2048), "layout": rng.choice(["tiled", "tiled", "tiled", "raw"])}


# ------------------------------------------------------------------ inputs (from the seed alone)
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(0x7157 + int(seed))
    return g


def _rows(g, cls, rows, k):
    """GGUF rows of a weight class, u8[rows][k / block * bytes]: uniform bytes, the blocks' fp16 scales |N(0,1)| * 1e-3."""
    nbytes, per, off, n = BLOCKS[cls]
    nb = k // per
    w = torch.randint(0, 256, (rows, nb, nbytes), dtype=torch.uint8, device=DEV, generator=g)
    d = (torch.randn(rows, nb, n, device=DEV, generator=g).abs() * 1e-3).half()
    w[:, :, off:off + 2 * n] = d.view(torch.uint8).view(rows, nb, 2 * n)
    return w.view(rows, nb * nbytes)


def _act16(g, m, k):
    """bf16 N(0,1) activations as fp16."""
    return torch.randn(m, k, device=DEV, generator=g).bfloat16().half()


def _inputs(case, seed):
    """The seed's inputs: GGUF weights, activations, residuals."""
    g = _gen(seed)
    kind = case["kind"]
    if kind == "route":
        P = case["P"]
        return {"wrt": torch.randn(EXPERTS, MHID, device=DEV, generator=g) * MHID ** -0.5,
                "wsh": torch.randn(MHID, device=DEV, generator=g) * MHID ** -0.5,
                "h": torch.randn(P, MHID, device=DEV, generator=g).bfloat16().float()}
    if kind == "ffn":
        M = case["M"]
        return {"wg": _rows(g, "iq3xxs", FFN, HID), "wu": _rows(g, "iq3xxs", FFN, HID),
                "wd": _rows(g, "iq3xxs", HID, FFN), "x": torch.randn(M, HID, device=DEV, generator=g),
                "attn": _act16(g, M, HID), "nw": 1 + 0.1 * torch.randn(HID, device=DEV, generator=g)}
    if kind == "qkv":
        return {"w": [_rows(g, cls, n, HID) for n, cls in QKV[case["mix"]]], "x": _act16(g, case["M"], HID)}
    if kind == "head":
        n, k = HEADS[case["head"]]
        w = _rows(g, "q5k" if case["head"] == "q5k" else "q6k", n, k)
        x = _act16(g, case["M"], k)
        return {"w": w, "x": x.float().view(-1) if case["head"].startswith("q6k_f32") else x}
    if kind == "prefill_ffn":
        M = case["M"]
        return {"wg": _rows(g, "iq3xxs", FFN, HID), "wu": _rows(g, "iq3xxs", FFN, HID),
                "wd": _rows(g, "iq3xxs", HID, FFN), "x": _act16(g, M, HID),
                "res": torch.randn(M, HID, device=DEV, generator=g)}
    if kind == "prefill_qkv":
        return {"w": [_rows(g, cls, n, HID) for n, cls in PREFILL_QKV[case["mix"]]], "x": _act16(g, case["M"], HID)}
    # MoE layers: hidden states of 0.05 * N(0,1) keep the fp16 parts of these weights in range
    P = case["P"]
    s = {"logits": torch.randn(P, EXPERTS, device=DEV, generator=g), "sg": torch.rand(P, device=DEV, generator=g),
         "x": (0.05 * torch.randn(P, MHID, device=DEV, generator=g)).bfloat16().float(),
         "res": torch.randn(P, MHID, device=DEV, generator=g)}
    if kind == "moe":   # expert e's 1024 gate/up rows, then the next expert's; the shared expert is the last one
        s["gu"] = _rows(g, "iq4xs", (EXPERTS + 1) * 2 * MFF, MHID)
        s["dn"] = _rows(g, "iq4xs", (EXPERTS + 1) * MHID, MFF)
    else:
        s["gu"] = _rows(g, "iq3s", EXPERTS * 2 * MFF, MHID)
        s["dn"] = _rows(g, "q6k", EXPERTS * MHID, MFF)
        s["shared"] = [_rows(g, "q8_0", MFF, MHID), _rows(g, "q8_0", MFF, MHID), _rows(g, "q8_0", MHID, MFF)]
        # the grid is a run-time table: 512 entries of four odd levels
        s["grid"] = 1.0 + 2.0 * torch.randint(0, 8, (512, 4), device=DEV, generator=g).float()
    return s


# ------------------------------------------------------------------ what a program keeps
def _iq3(raw, n, k, layout):
    """An IQ3_XXS tensor in the layout that the program serves it in."""
    packed = torch.empty_like(raw)
    ops.pack_iq3_rows(raw, packed, n, k)
    if layout == "packed":
        return packed
    if layout == "packed7":
        out = torch.empty(n * k // 2, dtype=torch.uint8, device=DEV)
        return ops.pack_w7(packed, out, n, k)
    out = torch.empty((n + 15) // 16 * 16 * 102 * (k // 256), dtype=torch.uint8, device=DEV)
    return ops.pack_iq3_tiled(packed, out, n, k)


def _q6pad(raw, n, k):
    return ops.pack_q6_pad(raw, torch.empty(n * 212 * (k // 256), dtype=torch.uint8, device=DEV), n, k)


def _table(slabs, count):
    size = slabs.numel() // count
    return torch.tensor([slabs.data_ptr() + e * size for e in range(count)], dtype=torch.int64, device=DEV)


def prepare(case, seed):
    kind = case["kind"]
    s = _inputs(case, seed)
    f16 = dict(dtype=torch.float16, device=DEV)
    if kind == "route":
        P = case["P"]
        return dict(s, kind=kind, eids=torch.empty(P, TOPK, dtype=torch.int16, device=DEV),
                    gates=torch.empty(P, TOPK, device=DEV), sg=torch.empty(P, device=DEV))
    st = {"kind": kind, "gridf": formats.gridf_tensor(DEV), "x": s["x"]}
    if kind == "ffn":
        M, lay = case["M"], case["layout"]
        st.update(layout=LAYOUTS[lay], wg=_iq3(s["wg"], FFN, HID, lay), wu=_iq3(s["wu"], FFN, HID, lay),
                  wd=_iq3(s["wd"], HID, FFN, lay), attn=s["attn"], nw=s["nw"], hh=torch.empty(M, HID, device=DEV),
                  hhx=torch.empty(M, HID, **f16), y=torch.empty(M, HID, device=DEV),
                  act=ops.tileord_empty(FFN, DEV) if lay == "tiled" else torch.empty(M, FFN, **f16))
    elif kind == "qkv":
        mix = case["mix"]
        st.update(mix=mix, out=[torch.empty(case["M"], n, **f16) for n, _ in QKV[mix]])
        lay = "packed" if mix == "q6" else "tiled"
        st["w"] = [_iq3(w, n, HID, lay) if cls == "iq3xxs" else _q6pad(w, n, HID) if cls == "q6k" else w
                   for w, (n, cls) in zip(s["w"], QKV[mix])]
    elif kind == "head":
        n, _ = HEADS[case["head"]]
        fp32 = case["head"].startswith("q6k_f32")
        st.update(head=case["head"], w=s["w"], out=torch.empty(n, device=DEV) if fp32 else torch.empty(case["M"], n, **f16))
    elif kind == "prefill_ffn":
        M = case["M"]
        st.update(wg=_iq3(s["wg"], FFN, HID, "packed7"), wu=_iq3(s["wu"], FFN, HID, "packed7"),
                  wd=_iq3(s["wd"], HID, FFN, "packed7"), res=s["res"], act=torch.empty(M, FFN, **f16),
                  y=torch.empty(M, HID, device=DEV))
    elif kind == "prefill_qkv":
        form = {"iq3xxs": (TYPE_IQ3_XXS, LAYOUT_PACK7), "q4k": (TYPE_Q4_K, LAYOUT_RAW),
                "q5k": (TYPE_Q5_K, LAYOUT_RAW), "q6k": (TYPE_Q6_K, LAYOUT_PACKED)}
        segs = PREFILL_QKV[case["mix"]]
        st["w"] = [_iq3(w, n, HID, "packed7") if cls == "iq3xxs" else _q6pad(w, n, HID) if cls == "q6k" else w
                   for w, (n, cls) in zip(s["w"], segs)]
        st.update(types=[form[c][0] for _, c in segs], layouts=[form[c][1] for _, c in segs],
                  out=[torch.empty(case["M"], n, **f16) for n, _ in segs])
    else:
        P, tiled = case["P"], case["layout"] == "tiled"
        count = EXPERTS + 1 if kind == "moe" else EXPERTS
        gu, dn = s["gu"], s["dn"]
        if tiled:
            pack_gu, pack_dn = ((ops.pack_iq4_tiled, ops.pack_iq4_tiled) if kind == "moe" else
                                (ops.pack_iq3s_tiled, ops.pack_q6k_tiled))
            gu = pack_gu(gu, torch.empty_like(gu), count * 2 * MFF, MHID)
            dn = pack_dn(dn, torch.empty_like(dn), count * MHID, MFF)
        tg, td = _table(gu, count), _table(dn, count)
        st.update(layout=LAYOUTS[case["layout"]], keep=(gu, dn), ptbl=tg[:EXPERTS].contiguous(),
                  ptbl_dn=td[:EXPERTS].contiguous(), logits=s["logits"], sg=s["sg"], res=s["res"],
                  y=torch.empty(P, MHID, device=DEV), scratch=ops.MoeScratch(P, DEV))
        if kind == "moe":
            st.update(ptbl_sh=torch.stack([tg[EXPERTS], td[EXPERTS]]), iq4nl=formats.iq4nl_tensor(DEV))
        else:
            st.update(shared=s["shared"], grid=s["grid"].reshape(-1).contiguous())
    return st


def run(s):
    kind = s["kind"]
    if kind == "route":
        ops.moe_route(s["wrt"], s["wsh"], s["h"], s["eids"], s["gates"], s["sg"])
        return {"eids": s["eids"], "gates": s["gates"], "sg": s["sg"]}
    if kind == "ffn":
        if s["layout"] == LAYOUT_TILED:   # the hand-off form between the two GEMVs
            ops.add_rms_f16(s["x"], s["attn"], s["nw"], s["hh"], s["hhx"])
            ops.ffn8(s["wg"], s["wu"], s["gridf"], s["hhx"], s["act"], LAYOUT_TILED, out_tileord=True)
            ops.down8(s["wd"], s["gridf"], s["act"], s["hh"], s["y"], LAYOUT_TILED, in_tileord=True)
        else:
            ops.ffn8_hh(s["wg"], s["wu"], s["gridf"], s["x"], s["attn"], s["nw"], s["hh"], s["hhx"], s["act"], s["layout"])
            ops.down8(s["wd"], s["gridf"], s["act"], s["hh"], s["y"], s["layout"])
        return {"hh": s["hh"], "y": s["y"]}
    if kind == "qkv":
        if s["mix"] == "gdn":
            ops.iq3_gemv_multi(s["w"], s["gridf"], s["x"], s["out"], LAYOUT_TILED)
        elif s["mix"] == "iq3":
            ops.aq3k8(*s["w"], s["gridf"], s["x"], *s["out"], layout=LAYOUT_TILED | V_Q4K)
        else:
            ops.aq6k8(*s["w"], s["gridf"], s["x"], *s["out"], layout=LAYOUT_PACKED | V_Q4K)
        return s["out"]
    if kind == "head":
        if s["head"] == "q5k":
            ops.head8(s["w"], s["x"], s["out"])
        elif s["head"] == "q6k":
            ops.q6k_gemv16(s["w"], s["x"], s["out"], LAYOUT_RAW)
        else:
            ops.h6k_gemv(s["w"], s["x"], s["out"], LAYOUT_RAW)
        return s["out"]
    if kind == "prefill_ffn":
        ops.pfg3_ffn(s["wg"], s["wu"], s["gridf"], s["x"], s["act"])
        ops.pfg3_iq3d(s["wd"], s["gridf"], s["act"], s["res"], s["y"])
        return {"act": s["act"], "y": s["y"]}
    if kind == "prefill_qkv":
        return ops.pfg3m(s["w"], s["out"], s["types"], s["layouts"], s["gridf"], s["x"])
    if kind == "moe":
        return ops.moe_layer(s["logits"], s["sg"], s["x"], s["res"], s["y"], s["ptbl"], s["ptbl_dn"], s["ptbl_sh"],
                             s["iq4nl"], s["scratch"], layout=s["layout"])
    return ops.moe_layer_ckpt(s["logits"], s["sg"], s["x"], s["res"], s["y"], s["ptbl"], s["ptbl_dn"], s["shared"],
                              s["grid"], s["scratch"], layout=s["layout"])


# ------------------------------------------------------------------ what a pass cannot do without
def _bytes(cls, rows, k):
    return rows * k // BLOCKS[cls][1] * BLOCKS[cls][0]


def work(case):
    kind = case["kind"]
    if kind == "route":
        P = case["P"]
        return {"bytes": 4 * (EXPERTS + 1) * MHID + P * (4 * MHID + 6 * TOPK + 4), "flops": 2 * P * (EXPERTS + 1) * MHID}
    if kind in ("ffn", "prefill_ffn"):
        M = case["M"]
        w = 3 * _bytes("iq3xxs", FFN, HID)
        # x (fp32 and the fp16 attention output, or fp16 and the fp32 residual), the SwiGLU output written and read, y
        io = M * (HID * (4 + 2 + 4 + 4) if kind == "ffn" else HID * (2 + 4 + 4)) + 4 * M * FFN
        return {"bytes": w + io, "flops": 2 * M * 3 * FFN * HID}
    if kind in ("qkv", "prefill_qkv"):
        segs = (QKV if kind == "qkv" else PREFILL_QKV)[case["mix"]]
        M, n = case["M"], sum(n for n, _ in segs)
        return {"bytes": sum(_bytes(c, n_, HID) for n_, c in segs) + 2 * M * (HID + n), "flops": 2 * M * n * HID}
    if kind == "head":
        n, k = HEADS[case["head"]]
        fp32 = case["head"].startswith("q6k_f32")
        return {"bytes": _bytes("q5k" if case["head"] == "q5k" else "q6k", n, k) + (4 if fp32 else 2) * case["M"] * (n + k),
                "flops": 2 * case["M"] * n * k}
    P = case["P"]
    hit = EXPERTS * (1 - (1 - TOPK / EXPERTS) ** P)   # experts that P positions reach
    if kind == "moe":
        w = (hit + 1) * (_bytes("iq4xs", 2 * MFF, MHID) + _bytes("iq4xs", MHID, MFF))
    else:
        w = hit * (_bytes("iq3s", 2 * MFF, MHID) + _bytes("q6k", MHID, MFF)) + 3 * _bytes("q8_0", MFF, MHID)
    io = P * (4 * EXPERTS + 4 + 3 * 4 * MHID)   # logits, shared gate, x, residual, y
    return {"bytes": int(w) + io, "flops": 2 * 3 * MFF * MHID * (TOPK + 1) * P}


# ------------------------------------------------------------------ tolerances
# About four times the distance from the 64-bit result: fp16 operands and outputs with fp32 sums are
# 2.1e-4 .. 2.9e-4 away where one GEMM ends in fp16, 5e-4 where an fp16 SwiGLU chain or fp16 parts are
# between two; the sums of fp32 operands 1e-7 .. 3e-7.
TOLERANCE = {"route": {"rel": 1e-6, "differ": 1e-3}, "ffn": {"rel": 2e-3}, "qkv": {"rel": 1e-3}, "head": {"rel": 1e-3},
             "prefill_ffn": {"rel": 2e-3}, "prefill_qkv": {"rel": 1.2e-3}, "moe": {"rel": 2.2e-3},
             "moe_ckpt": {"rel": 1.3e-3}}


def tolerance(case):
    if case.get("head", "").startswith("q6k_f32"):
        return {"rel": 1e-6}
    return dict(TOLERANCE[case["kind"]])


# ------------------------------------------------------------------ the same in 64 bits
def _h(b):
    """fp16 bytes u8[..., 2n] -> float64 [..., n]."""
    return b.contiguous().view(torch.float16).double()


def _nib(b):
    return b & 15, b >> 4


def _k4_scales(q):
    """The 8 six-bit (scale, min) pairs of a k-quant block's 12 bytes, int [..., 12]."""
    sc = torch.cat([q[..., 0:4] & 63, (q[..., 8:12] & 15) | (q[..., 0:4] >> 6 << 4)], -1)
    mn = torch.cat([q[..., 4:8] & 63, (q[..., 8:12] >> 4) | (q[..., 4:8] >> 6 << 4)], -1)
    return sc, mn


def _dequant(cls, rows, grid=None):
    """GGUF rows u8[n][...] -> their weights in 64 bits [n][k]."""
    nbytes = BLOCKS[cls][0]
    b = rows.view(rows.shape[0], -1, nbytes)
    n, nb = b.shape[:2]
    if cls == "iq3xxs":
        g = formats.gridf_tensor(b.device).view(256, 4).double()
        v = g[b[..., 2:66].long()].view(n, nb, 8, 4, 8)
        sw = b[..., 66:98].contiguous().view(torch.int32).long() & 0xFFFFFFFF
        sh = torch.tensor([0, 7, 14, 21], device=b.device)
        s7 = (sw[..., None] >> sh) & 127
        bits = (s7[..., None] >> torch.arange(7, device=b.device)) & 1
        bits = torch.cat([bits, bits.sum(-1, keepdim=True) & 1], -1)   # an even number of signs
        db = _h(b[..., 0:2]) * ((sw >> 28).double() + 0.5) * 0.5
        return (db[..., None, None] * v * (1 - 2 * bits)).view(n, -1)
    if cls == "iq3s":
        q = b[..., 2:66].long()
        hi = (b[..., 66:74].long()[..., None] >> torch.arange(8, device=b.device)) & 1
        v = grid.double()[q + 256 * hi.view(n, nb, 64)].view(n, nb, 8, 32)
        sg = (b[..., 74:106].long()[..., None] >> torch.arange(8, device=b.device)) & 1
        ls = torch.stack(_nib(b[..., 106:110].long()), -1).view(n, nb, 8)
        db = _h(b[..., 0:2]) * (1 + 2 * ls).double()
        return (db[..., None] * v * (1 - 2 * sg.view(n, nb, 8, 32))).view(n, -1)
    if cls == "iq4xs":
        kv = formats.iq4nl_tensor(b.device).double()
        i = torch.arange(8, device=b.device)
        hi = b[..., 2:4].contiguous().view(torch.int16).long() & 0xFFFF
        ls = torch.stack(_nib(b[..., 4:8].long()), -1).view(n, nb, 8) | (((hi >> (2 * i)) & 3) << 4)
        lo, up = _nib(b[..., 8:136].long().view(n, nb, 8, 16))
        return ((_h(b[..., 0:2]) * (ls - 32).double())[..., None] * kv[torch.cat([lo, up], -1)]).view(n, -1)
    if cls == "q6k":
        lo, up = _nib(b[..., 0:128].long().view(n, nb, 2, 1, 64))
        low = torch.cat([lo, up], -1).view(n, nb, 2, 4, 32)
        hi = (b[..., 128:192].long().view(n, nb, 2, 1, 32) >> torch.tensor([0, 2, 4, 6], device=b.device)[:, None]) & 3
        sc = b[..., 192:208].contiguous().view(torch.int8).double().view(n, nb, 16, 1)
        q = (low + 16 * hi - 32).double().view(n, nb, 16, 16)
        return (_h(b[..., 208:210])[..., None] * sc * q).view(n, -1)
    if cls in ("q4k", "q5k"):
        sc, mn = _k4_scales(b[..., 4:16].long())
        lo, up = _nib(b[..., nbytes - 128:].long().view(n, nb, 4, 32))
        q = torch.stack([lo, up], -2).view(n, nb, 8, 32)
        if cls == "q5k":
            q = q + (((b[..., 16:48].long()[:, :, None] >> torch.arange(8, device=b.device)[:, None]) & 1) << 4)
        d = _h(b[..., 0:4])
        return ((d[..., 0:1] * sc)[..., None] * q - (d[..., 1:2] * mn)[..., None]).view(n, -1)
    return (_h(b[..., 0:2]) * b[..., 2:34].contiguous().view(torch.int8).double()).view(n, -1)   # q8_0


def _matmul(x, cls, rows, grid=None, step=8192):
    """x . W^T with W's rows decoded a part at a time."""
    return torch.cat([x @ _dequant(cls, rows[i:i + step], grid).T for i in range(0, rows.shape[0], step)], 1)


def _swiglu(g, u):
    return g / (1 + torch.exp(-g)) * u


def exact(case, seed):
    kind = case["kind"]
    s = _inputs(case, seed)
    if kind == "route":
        h = s["h"].double()
        top, ids = torch.sort(h @ s["wrt"].double().T, dim=1, descending=True, stable=True)
        return {"eids": ids[:, :TOPK].short(), "gates": torch.softmax(top[:, :TOPK], 1),
                "sg": torch.sigmoid(h @ s["wsh"].double())}
    x = s["x"].double()
    if kind in ("ffn", "prefill_ffn"):
        hh, inp = s.get("res"), x
        if kind == "ffn":
            hh = x + s["attn"].double()
            inp = hh * torch.rsqrt((hh * hh).mean(1, keepdim=True) + 1e-6) * s["nw"].double()
        act = _swiglu(_matmul(inp, "iq3xxs", s["wg"]), _matmul(inp, "iq3xxs", s["wu"]))
        y = hh.double() + _matmul(act, "iq3xxs", s["wd"], step=2048)
        return {"hh": hh, "y": y} if kind == "ffn" else {"act": act, "y": y}
    if kind in ("qkv", "prefill_qkv"):
        segs = (QKV if kind == "qkv" else PREFILL_QKV)[case["mix"]]
        return [_matmul(x, cls, w) for w, (_, cls) in zip(s["w"], segs)]
    if kind == "head":
        out = _matmul(x.view(case["M"], -1), "q5k" if case["head"] == "q5k" else "q6k", s["w"])
        return out.view(-1) if case["head"].startswith("q6k_f32") else out
    P = case["P"]
    top, ids = torch.sort(s["logits"].double(), dim=1, descending=True, stable=True)
    ids, gates = ids[:, :TOPK], torch.softmax(top[:, :TOPK], 1)
    up, down = ("iq4xs", "iq4xs") if kind == "moe" else ("iq3s", "q6k")
    y = s["res"].double().clone()

    def expert(e, t):
        w = _dequant(up, s["gu"][e * 2 * MFF:(e + 1) * 2 * MFF], s.get("grid"))
        act = _swiglu(t @ w[:MFF].T, t @ w[MFF:].T)
        return act @ _dequant(down, s["dn"][e * MHID:(e + 1) * MHID]).T

    flat = ids.reshape(-1)
    order = torch.sort(flat, stable=True)[1]
    counts = np.bincount(flat.cpu().numpy(), minlength=EXPERTS)
    first = 0
    for e in range(EXPERTS):
        pairs = order[first:first + int(counts[e])]
        first += int(counts[e])
        if len(pairs):
            pos = pairs // TOPK
            y.index_add_(0, pos, gates.reshape(-1)[pairs, None] * expert(e, x[pos]))
    if kind == "moe":
        sh = expert(EXPERTS, x)
    else:
        wg, wu, wd = (_dequant("q8_0", w) for w in s["shared"])
        sh = _swiglu(x @ wg.T, x @ wu.T) @ wd.T
    return y + s["sg"].double().view(P, 1) * sh
