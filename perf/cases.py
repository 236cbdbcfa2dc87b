"""What the engine's speed is measured on: the calls a program around it makes, through the
package's public entry points, from a batch of a few hundred cells to the million-cell matrix.

Nine kinds of call, and what each stands for:
  project     qcsr_spmm: a quantized CSR as it arrives (no prepared projection) against fp16
              weights: embedding new cells while serving, or a structure that is used once.
  csr_f32     qcsr_spmm on an unquantized fp32 CSR with fp32 weights.
  prepared    ExecProjection.spmm: the same matrix projected again and again, its
              execution-order form prepared once.
  train       the backward pass of that projection: the gradient of every stored value
              (qcsr_spmm_bwd_values) and of the weights (qcsr_spmm_bwd_rhs, the transpose
              built once per structure).
  codec       one matrix decoded to fp32 and new values encoded into its structure.
  bell_bf16   Blocked-ELL in bf16 with packed weights and planned row-block groups.
  bell_quant  Blocked-ELL with packed codes and fp32 weights, row blocks in planned order.
  bell_plain  Blocked-ELL with fp16 or fp32 values in 8, 16 or 32 wide blocks against fp32
              weights of any width: the reference-semantics entry on lowered matrices.
  cpbp        the CP-BP warp-tile feature-weighted row reduction.

Inputs come from the package's seeded generators (single-cell shaped: log-normal row sizes,
Zipf gene popularity, log1p counts) or, where those have no such form, from torch's; sizes are
those of the benchmark's configurations and of the tests.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from cellerator_amd import (BellMatrix, Epilogue, QcsrMatrix, bell_block_major, bell_pack_rhs,
                            bell_plan_groups, bell_spmm, bell_spmm_grouped, cpbp_entry_rows,
                            cpbp_reduce_rows, qcsr_check_columns, qcsr_pack_gene_affine, qcsr_spmm,
                            qcsr_spmm_bwd_rhs, qcsr_spmm_bwd_values, qcsr_transpose)
from cellerator_amd import _native as N
from cellerator_amd import codec
from cellerator_amd.cpbp import build_tiles_device, contiguous_plan
from cellerator_amd.exec_order import ExecProjection
from cellerator_amd.synth import (BellConfig, CpbpConfig, QcsrConfig, dense_normal, generate_bell,
                                  generate_cpbp_host, generate_qcsr)


def listed():
    return [
        # a serving batch: a few hundred new cells through a fused bias + ReLU layer
        {"name": "project_serve", "kind": "project", "rows": 250, "cols": 20_000, "bits": 8, "policy": "gene",
         "mean": 2_000.0, "sigma": 0.5, "n": 64, "epilogue": True},
        # one sample's cells, row-offset codes, a wider layer
        {"name": "project_sample", "kind": "project", "rows": 30_011, "cols": 33_538, "bits": 4, "policy": "row",
         "mean": 1_500.0, "sigma": 0.6, "n": 128, "epilogue": False},
        # an atlas shard projected once
        {"name": "project_shard", "kind": "project", "rows": 250_007, "cols": 33_538, "bits": 4, "policy": "gene",
         "mean": 1_500.0, "sigma": 0.6, "n": 64, "epilogue": False},
        # the benchmark's smallest configuration: fp32 CSR over 2,000 selected genes
        {"name": "csr_f32", "kind": "csr_f32", "rows": 10_000, "cols": 2_000, "mean": 200.0, "n": 64},
        # the benchmark's 100k-cell 8-bit configuration, prepared
        {"name": "prepared_100k", "kind": "prepared", "rows": 100_000, "cols": 20_000, "bits": 8, "mean": 2_000.0,
         "sigma": 0.5, "n": 64, "head": 3_072},
        # the benchmark's headline: one million cells, 4-bit codes, prepared
        {"name": "prepared_1m", "kind": "prepared", "rows": 1_000_000, "cols": 33_538, "bits": 4, "mean": 1_500.0,
         "sigma": 0.6, "n": 64, "head": 2_048},
        # one backward pass over the 100k-cell configuration
        {"name": "train_100k", "kind": "train", "rows": 100_000, "cols": 20_000, "bits": 8, "mean": 2_000.0,
         "sigma": 0.5, "n": 64},
        # re-encoding a sample: decode every stored value, encode new ones
        {"name": "codec_50k", "kind": "codec", "rows": 50_003, "cols": 20_000, "bits": 4, "mean": 1_500.0,
         "sigma": 0.6},
        # the benchmark's Blocked-ELL configuration
        {"name": "bell_bf16", "kind": "bell_bf16", "rows": 500_000, "cols": 20_000, "n": 256},
        # its quantized form on a fifth of the cells
        {"name": "bell_quant", "kind": "bell_quant", "rows": 100_000, "cols": 20_000, "bits": 8, "n": 256},
        # a lowered matrix with 16 x 16 blocks, a ragged last row block
        {"name": "bell_plain", "kind": "bell_plain", "rows": 40_005, "cols": 20_000, "block": 16, "dtype": "f16",
         "slots": 64, "n": 64},
        # a quarter of the benchmark's CP-BP configuration
        {"name": "cpbp_500k", "kind": "cpbp", "rows": 500_000, "dtype": "f32", "width": 64},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["project", "project", "project", "csr_f32", "prepared", "prepared", "train", "codec",
                       "bell_bf16", "bell_quant", "bell_plain", "cpbp"])
    if kind == "project":
        return {"kind": kind, "rows": _log_int(rng, 60, 250_000), "cols": _log_int(rng, 2_000, 33_538),
                "bits": rng.choice([2, 4, 8]), "policy": rng.choice(["gene", "row"]),
                "mean": float(_log_int(rng, 200, 1_500)), "sigma": rng.uniform(0.3, 0.6),
                "n": rng.choice([64, 64, 128]), "epilogue": rng.random() < 0.3}
    if kind == "csr_f32":
        return {"kind": kind, "rows": _log_int(rng, 1_000, 100_000), "cols": _log_int(rng, 2_000, 20_000),
                "mean": float(_log_int(rng, 100, 800)), "n": rng.choice([32, 64, 128])}
    if kind == "prepared":
        n = rng.choice([64, 64, 128])
        return {"kind": kind, "rows": _log_int(rng, 20_000, 400_000 * 64 // n), "cols": _log_int(rng, 8_000, 33_538),
                "bits": rng.choice([4, 8]), "mean": float(_log_int(rng, 500, 2_000)), "sigma": rng.uniform(0.3, 0.6),
                "n": n, "head": rng.choice([2_048, 3_072])}
    if kind == "train":
        n = rng.choice([64, 64, 128])
        return {"kind": kind, "rows": _log_int(rng, 5_000, 100_000 * 64 // n), "cols": _log_int(rng, 2_000, 33_538),
                "bits": rng.choice([4, 8]), "mean": float(_log_int(rng, 200, 1_500)), "sigma": rng.uniform(0.3, 0.6),
                "n": n}
    if kind == "codec":
        return {"kind": kind, "rows": _log_int(rng, 1_000, 100_000), "cols": _log_int(rng, 2_000, 33_538),
                "bits": rng.choice([1, 2, 4, 8]), "mean": float(_log_int(rng, 200, 1_500)),
                "sigma": rng.uniform(0.3, 0.6)}
    if kind == "bell_bf16":
        return {"kind": kind, "rows": 32 * _log_int(rng, 300, 12_000), "cols": rng.randint(4_000, 20_000),
                "n": rng.choice([64, 128, 256])}
    if kind == "bell_quant":
        return {"kind": kind, "rows": 32 * _log_int(rng, 100, 3_000), "cols": rng.randint(4_000, 20_000),
                "bits": rng.choice([4, 8]), "n": rng.choice([64, 128, 256])}
    if kind == "bell_plain":
        return {"kind": kind, "rows": _log_int(rng, 1_000, 40_000), "cols": rng.randint(4_000, 20_000),
                "block": rng.choice([8, 16, 32]), "dtype": rng.choice(["f16", "f32"]), "slots": rng.randint(16, 64),
                "n": rng.choice([50, 64, 100, 128])}
    return {"kind": kind, "rows": _log_int(rng, 20_000, 400_000), "dtype": rng.choice(["f16", "f32"]),
            "width": rng.choice([32, 64])}


# ---- inputs ------------------------------------------------------------------------------


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _matrix(case, seed):
    """The stored matrix as it arrives: separate per-gene (or per-row) metadata."""
    f32 = case["kind"] == "csr_f32"
    m = generate_qcsr(QcsrConfig(
        "case", case["rows"], case["cols"], 0 if f32 else case["bits"], min(case["mean"], case["cols"] / 4.0),
        case.get("sigma", 0.0), row_dist=1 if f32 else 0, nnz_min=1, zipf_s=0.0 if f32 else 1.1,
        nb_mean=2.0, nb_size=0.5, seed=0xCE11E7A700001000 + seed))
    if case.get("policy") == "row":
        rows = torch.rand(m.rows, device="cuda", generator=_generator(seed)) * 0.5 + 0.2
        m = QcsrMatrix(m.rows, m.cols, m.bits, m.row_ptr, m.col_idx, packed_row_ptr=m.packed_row_ptr,
                       packed_values=m.packed_values, column_scales=m.column_scales, row_offsets=rows,
                       decode_policy=N.DECODE_COLUMN_SCALE_ROW_OFFSET)
    return m


def _weights(case, seed):
    dtype = torch.float32 if case["kind"] == "csr_f32" else torch.float16
    return dense_normal((case["cols"], case["n"]), 0.02, dtype, seed=77_000 + seed)


def _bias(case, seed):
    return dense_normal((case["n"],), 0.5, torch.float32, seed=88_000 + seed)


def _grad_out(case, seed):
    return dense_normal((case["rows"], case["n"]), 1.0, torch.float32, seed=99_000 + seed)


def _capacity(case):
    """Entries a program reserves for the per-entry outputs of matrices of this size, whatever
    their realised count (what lies past it stays zero)."""
    return int(case["rows"] * min(case["mean"], case["cols"] / 4.0) * 1.3) + 1_000


def _entries(case, m):
    cap = _capacity(case)
    if m.nnz > cap:
        raise ValueError(f"{m.nnz} entries exceed the reserved {cap}")
    return torch.zeros(cap, device="cuda")


def _new_values(case, m, seed):
    """fp32 values to encode: near the stored range, some past its ends."""
    return torch.rand(m.nnz, device="cuda", generator=_generator(seed)) * 3.0 + 0.3


def _bell_bf16(case, seed):
    return generate_bell(BellConfig("case", case["rows"], case["cols"], max_blocks=min(64, case["cols"] // 32),
                                    seed=0xCE11E7A700002000 + seed))


def _bell_codes(case, seed):
    g = _bell_bf16(case, seed)
    gen = _generator(seed)
    bits = case["bits"]
    stride = g.ell_cols * bits // 8
    codes = torch.randint(0, 256, (g.rows * stride,), dtype=torch.uint8, device="cuda", generator=gen)
    return BellMatrix(g.rows, g.cols, 32, g.ell_cols, g.block_col_idx, bits=bits,
                      decode_policy=N.DECODE_PER_GENE_AFFINE, row_stride_bytes=stride, packed_values=codes,
                      column_scales=torch.rand(g.cols, device="cuda", generator=gen) * 0.02 + 0.001,
                      column_offsets=torch.rand(g.cols, device="cuda", generator=gen) * 0.5)


def _bell_plain(case, seed):
    """Rows of `slots` ELL slots, three quarters of them valid on average, values 35% dense."""
    gen = _generator(seed)
    bs, slots, rows, cols = case["block"], case["slots"], case["rows"], case["cols"]
    rb, bcs = -(-rows // bs), -(-cols // bs)
    pool = torch.rand((64, bcs), device="cuda", generator=gen).argsort(dim=1)[:, :slots]
    idx = pool[torch.randint(0, 64, (rb,), device="cuda", generator=gen)]
    used = torch.randint(slots // 2, slots + 1, (rb, 1), device="cuda", generator=gen)
    idx = torch.where(torch.arange(slots, device="cuda") < used, idx, torch.full_like(idx, bcs)).sort(dim=1).values
    valid = idx < bcs
    idx = torch.where(valid, idx, torch.full_like(idx, -1)).to(torch.int32)
    dtype = torch.float16 if case["dtype"] == "f16" else torch.float32
    mask = valid.repeat_interleave(bs, dim=0)[:rows].repeat_interleave(bs, dim=1)
    vals = torch.rand((rows, slots * bs), device="cuda", generator=gen)
    vals = torch.where(mask & (vals < 0.35), torch.log1p(vals * 20.0), torch.zeros_like(vals)).to(dtype)
    return BellMatrix(rows, cols, bs, slots * bs, idx.contiguous(), values=vals)


def _bell_weights(case, seed):
    dtype = torch.bfloat16 if case["kind"] == "bell_bf16" else torch.float32
    return dense_normal((case["cols"], case["n"]), 0.02, dtype, seed=55_000 + seed)


def _cpbp_csr(case, seed):
    offs, feats, vals = generate_cpbp_host(CpbpConfig("case", case["rows"], seed=0xCE11E7A700003000 + seed))
    return offs, feats, vals.astype(np.float16) if case["dtype"] == "f16" else vals


def _cpbp_weights(seed):
    return dense_normal((20_000,), 1.0, torch.float32, seed=66_000 + seed)


def prepare(case, seed):
    kind = case["kind"]
    state = {"kind": kind}
    if kind in ("project", "csr_f32", "prepared", "train", "codec"):
        m = _matrix(case, seed)
        if kind == "codec":
            state.update(m=m, values=_new_values(case, m, seed), decoded=_entries(case, m),
                         packed=torch.zeros(_capacity(case) + case["rows"], dtype=torch.uint8, device="cuda"))
            return state
        if m.bits and m.decode_policy == N.DECODE_PER_GENE_AFFINE:
            m = qcsr_pack_gene_affine(m)  # the interleaved metadata a program keeps per generation
        m = qcsr_check_columns(m)
        state.update(m=m, w=_weights(case, seed), out=torch.empty((m.rows, case["n"]), device="cuda"))
        if kind == "prepared":
            state.update(proj=ExecProjection(m, case["head"]), m=None)
        if kind == "train":
            state.update(t=qcsr_transpose(m), g=_grad_out(case, seed), out=None,
                         gv=_entries(case, m), gw=torch.empty((m.cols, case["n"]), device="cuda"))
        if case.get("epilogue"):
            state["epilogue"] = Epilogue(kind=N.EPILOGUE_BIAS_RELU, bias=_bias(case, seed))
    elif kind == "cpbp":
        offs, feats, vals = _cpbp_csr(case, seed)
        t, _ = build_tiles_device(contiguous_plan(20_000, 25), offs, feats, vals, group_width=case["width"])
        state.update(t=t, rows=cpbp_entry_rows(t), w=_cpbp_weights(seed),
                     out=torch.empty(t.row_count, device="cuda"))
    else:
        w = _bell_weights(case, seed)
        out = torch.empty((case["rows"], case["n"]), device="cuda")
        if kind == "bell_bf16":
            m = _bell_bf16(case, seed)
            state.update(groups=bell_plan_groups(m), m=bell_block_major(m), w=bell_pack_rhs(w), n=case["n"], out=out)
        elif kind == "bell_quant":
            m = _bell_codes(case, seed)
            state.update(m=m, order=bell_plan_groups(m).order, w=w, out=out)
        else:
            state.update(m=_bell_plain(case, seed), w=w, out=out)
    return state


def run(state):
    kind = state["kind"]
    if kind in ("project", "csr_f32"):
        return qcsr_spmm(state["m"], state["w"], out=state["out"], epilogue=state.get("epilogue"))
    if kind == "prepared":
        return state["proj"].spmm(state["w"], out=state["out"])
    if kind == "train":
        qcsr_spmm_bwd_values(state["m"], state["g"], state["w"], out=state["gv"])
        return {"grad_values": state["gv"], "grad_rhs": qcsr_spmm_bwd_rhs(state["t"], state["g"], out=state["gw"])}
    if kind == "codec":
        codec.dequantize(state["m"], state["decoded"])
        return {"decoded": state["decoded"], "packed": codec.quantize(state["m"], state["values"], packed_out=state["packed"])}
    if kind == "bell_bf16":
        return bell_spmm_grouped(state["m"], state["w"], state["groups"], state["n"], out=state["out"])
    if kind == "bell_quant":
        return bell_spmm(state["m"], state["w"], out=state["out"], row_block_order=state["order"])
    if kind == "bell_plain":
        return bell_spmm(state["m"], state["w"], out=state["out"])
    return cpbp_reduce_rows(state["t"], state["rows"], state["w"], out=state["out"])


# ---- what a pass cannot do without -------------------------------------------------------


def work(case):
    kind, rows, n = case["kind"], case["rows"], case.get("n", 0)
    if kind in ("project", "csr_f32", "prepared", "train", "codec"):
        nnz = rows * min(case["mean"], case["cols"] / 4.0)
        code = 4.0 if kind == "csr_f32" else case["bits"] / 8.0
        structure = nnz * (4.0 + code) + rows * 8.0 + case["cols"] * 8.0
        if kind == "codec":  # both directions read the structure; 4 bytes a value each
            return {"bytes": 2.0 * structure + nnz * 8.0, "flops": 4.0 * nnz}
        wbytes = case["cols"] * n * (4 if kind == "csr_f32" else 2)
        if kind == "train":  # structure and values once for each gradient, G twice
            return {"bytes": nnz * (4.0 + 4.0) + nnz * 8.0 + 2.0 * rows * n * 4 + wbytes + case["cols"] * n * 4.0,
                    "flops": 4.0 * nnz * n}
        return {"bytes": structure + wbytes + rows * n * 4.0, "flops": 2.0 * nnz * n}
    if kind == "cpbp":
        nnz = rows * 380.0
        entries = rows * 70.0
        vb = 2.0 if case["dtype"] == "f16" else 4.0
        return {"bytes": nnz * vb + entries * 12.0 + rows * 8.0, "flops": 2.0 * nnz}
    if kind == "bell_plain":
        bs = case["block"]
        stored = rows * case["slots"] * 0.75 * bs
        vb = 2.0 if case["dtype"] == "f16" else 4.0
    else:
        stored = rows * 44.0 * 32.0
        vb = 2.0 if kind == "bell_bf16" else case["bits"] / 8.0
    wb = 2.0 if kind == "bell_bf16" else 4.0
    return {"bytes": stored * vb + case["cols"] * n * wb + rows * n * 4.0, "flops": 2.0 * stored * n}


def tolerance(case):
    if case["kind"] == "codec":
        return "exact"  # both directions are pinned bit for bit
    # fp32 products and sums in any order (fp16, bf16 and code operands widen exactly): the worst
    # case is 8.5e-7 off the 64-bit result, so two orders differ by about 1.2e-6
    return {"rel": 5e-6, "max": 1e-4}


# ---- the same results in 64 bits ---------------------------------------------------------


def _codes(m, r0, r1):
    """(row within the chunk, column, decoded value in float64) of rows [r0, r1)."""
    b, e = int(m.row_ptr[r0]), int(m.row_ptr[r1])
    ptr = m.row_ptr[r0:r1 + 1].long()
    row = torch.repeat_interleave(torch.arange(r1 - r0, device="cuda"), ptr[1:] - ptr[:-1])
    col = m.col_idx[b:e].long()
    if m.bits == 0:
        return row, col, m.values[b:e].double()
    local = torch.arange(b, e, device="cuda") - ptr[row]
    cpb = 8 // m.bits
    byte = m.packed_values[m.packed_row_ptr[r0:r1].long()[row] + local // cpb].long()
    code = (byte >> ((local % cpb) * m.bits)) & ((1 << m.bits) - 1)
    off = m.row_offsets[r0:r1].double()[row] if m.row_offsets is not None else m.column_offsets.double()[col]
    return row, col, code.double() * m.column_scales.double()[col] + off


def _chunks(rows, cols):
    step = max(1, (1 << 29) // max(cols, 1))
    return [(r, min(rows, r + step)) for r in range(0, rows, step)]


def _dense(m, r0, r1):
    row, col, x = _codes(m, r0, r1)
    d = torch.zeros((r1 - r0) * m.cols, dtype=torch.float64, device="cuda")
    d[row * m.cols + col] = x
    return d.view(r1 - r0, m.cols), row, col


def _exact_csr(case, seed):
    m = _matrix(case, seed)
    if case["kind"] == "codec":
        out = torch.zeros(_capacity(case), dtype=torch.float64, device="cuda")
        for r0, r1 in _chunks(m.rows, m.cols):
            out[int(m.row_ptr[r0]):int(m.row_ptr[r1])] = _codes(m, r0, r1)[2]
        return {"decoded": out, "packed": None}
    w = _weights(case, seed).double()
    if case["kind"] != "train":
        y = torch.cat([_dense(m, r0, r1)[0] @ w for r0, r1 in _chunks(m.rows, m.cols)])
        return torch.relu(y + _bias(case, seed).double()) if case.get("epilogue") else y
    g = _grad_out(case, seed).double()
    gv = torch.zeros(_capacity(case), dtype=torch.float64, device="cuda")
    gw = torch.zeros((m.cols, case["n"]), dtype=torch.float64, device="cuda")
    wt = w.t().contiguous()
    for r0, r1 in _chunks(m.rows, m.cols):
        d, row, col = _dense(m, r0, r1)
        gw += d.t().contiguous() @ g[r0:r1]
        gv[int(m.row_ptr[r0]):int(m.row_ptr[r1])] = (g[r0:r1] @ wt)[row, col]
    return {"grad_values": gv, "grad_rhs": gw}


def _exact_bell(case, seed):
    kind, n = case["kind"], case["n"]
    m = {"bell_bf16": _bell_bf16, "bell_quant": _bell_codes, "bell_plain": _bell_plain}[kind](case, seed)
    w = _bell_weights(case, seed).double()
    bs, slots = m.block_size, m.ell_cols // m.block_size
    rb = -(-m.rows // bs)
    bcs = -(-m.cols // bs)
    wz = torch.zeros(((bcs + 1) * bs, n), dtype=torch.float64, device="cuda")  # the last block column is zero
    wz[: m.cols] = w
    idx = m.block_col_idx.view(rb, slots).long()
    idx = torch.where(idx < 0, torch.full_like(idx, bcs), idx)
    out = torch.empty((m.rows, n), dtype=torch.float64, device="cuda")
    step = max(1, (1 << 28) // (slots * bs * n))
    for b0 in range(0, rb, step):
        b1 = min(rb, b0 + step)
        r0, r1 = b0 * bs, min(m.rows, b1 * bs)
        gene = (idx[b0:b1, :, None] * bs + torch.arange(bs, device="cuda")).view(b1 - b0, slots * bs)
        if m.bits:
            byte = m.packed_values.view(m.rows, m.row_stride_bytes)[r0:r1].long()
            cpb = 8 // m.bits
            code = torch.stack([(byte >> (k * m.bits)) & ((1 << m.bits) - 1) for k in range(cpb)], dim=2)
            code = code.reshape(r1 - r0, m.ell_cols).double()
            g = torch.clamp(gene, max=m.cols - 1).repeat_interleave(bs, dim=0)[: r1 - r0]
            x = code * m.column_scales.double()[g] + m.column_offsets.double()[g]
        else:
            x = m.values[r0:r1].double()
        full = torch.zeros(((b1 - b0) * bs, slots * bs), dtype=torch.float64, device="cuda")
        full[: r1 - r0] = x
        y = torch.bmm(full.view(b1 - b0, bs, slots * bs), wz[gene])
        out[r0:r1] = y.reshape(-1, n)[: r1 - r0]
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind.startswith("bell"):
        return _exact_bell(case, seed)
    if kind == "cpbp":
        offs, feats, vals = _cpbp_csr(case, seed)
        w = _cpbp_weights(seed).cpu().numpy().astype(np.float64)
        prod = vals.astype(np.float64) * w[feats]
        return torch.from_numpy(np.add.reduceat(prod, offs[:-1].astype(np.int64)))
    return _exact_csr(case, seed)
