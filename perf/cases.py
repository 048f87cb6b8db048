"""Performance cases of the uplink LDPC decode path and of the DL encode path
beside it, each one pass through the public entry points of aerial_amd (the
Python layer over the C ABI of include/cuphy_hip.h).

A case is a dict of plain values; "kind" names the entry point:

  tb      LdpcDecoder.decode_tb      the drop-in: TBs of one configuration in one launch
  slot    BatchDecoder.replay        a slot of different UEs as one captured batch
  load    BatchDecoder.replay        a fully loaded slot of one configuration
  derate  DeRateMatch.run            de-rate-matching + HARQ combining
  crc     CrcDecode.run              CB and TB CRC, TB assembly
  encode  LdpcEncoder.encode_words   DL: bit-packed LDPC encoder
  dlrm    dl_rate_match              DL: rate matching and scrambling
  cells   SlotDecoder.replay         fused receive chain, many equal cells
  ues     SlotDecoder.launch         fused receive chain, different UEs, retransmission combined
  serve   HarqServer.serve_trace     HARQ engine: a burst of TBs served to the end

Shapes (which UEs a slot holds) come from the case, the data (payloads,
noise) from the seed.  Data is made as a transmitter and a channel make it:
random payloads with their CRCs, encoded, rate-matched, BPSK-AWGN LLRs.
"""
import os
import sys

import numpy as np
import torch

_PKG = os.path.abspath("aerial-cuda-accelerated-ran_amd")  # of the tree that is the working folder
if _PKG not in sys.path:
    sys.path.insert(1, _PKG)

from aerial_amd import _lib as L  # noqa: E402
from aerial_amd.batch import BatchDecoder  # noqa: E402
from aerial_amd.decoder import LdpcDecodeConfig, LdpcDecoder  # noqa: E402
from aerial_amd.encoder import LdpcEncoder, dl_rate_match  # noqa: E402
from aerial_amd.pusch import CrcDecode, DeRateMatch, make_tb_params  # noqa: E402
from aerial_amd.server import HarqServer, RV_SEQUENCE, serving_specs  # noqa: E402
from aerial_amd.slot import SLOT_CB_WORDS, SlotDecoder, SlotTb  # noqa: E402
from aerial_amd.workloads import (LIFTING_SIZES, TransportBlock, encode, fill_tb, mb_for_rate, nrows, nsys,  # noqa: E402
                                  num_edges)

QAM_STRIDE = 8
CRC24A, CRC24B, CRC16 = (0x864CFB, 24), (0x800063, 24), (0x1021, 16)
_FLOAT = {"fp16": torch.float16, "fp32": torch.float32, "int8": torch.int8}
_BYTES = {"fp16": 2, "fp32": 4, "int8": 1}


def listed():
    return [
        # the smallest call: one short code block (a VoIP or control-sized TB), where latency counts
        {"name": "tb_one_small_cb", "kind": "tb", "bg": 2, "Z": 64, "mb": 20, "tbs": 1, "ncb": 1, "dtype": "fp16",
         "iters": 10, "et": False, "soft": False, "esn0": 2.0},
        # one TB of 8 large low-rate code blocks in binary32, as the reference CPU path decodes it
        {"name": "tb_8cb_fp32", "kind": "tb", "bg": 1, "Z": 384, "mb": 46, "tbs": 1, "ncb": 8, "dtype": "fp32",
         "iters": 10, "et": False, "soft": False, "esn0": 1.0},
        # an ordinary mixed slot: 16 UEs of any base graph, lifting size and rate
        {"name": "slot_16_ues", "kind": "slot", "shape_seed": 2, "ues": 16, "z_min": 64, "max_cbs": 24,
         "dtype": "fp16", "iters": 10, "et": False},
        # a fully loaded slot: 20 cells of 100 MHz, 256QAM, R = 0.93
        {"name": "load_20_cells", "kind": "load", "bg": 1, "Z": 384, "R": 0.93, "tbs": 20, "ncb": 140,
         "dtype": "fp16", "iters": 10, "et": False, "esn0": 8.0},
        # the same slot's HARQ buffers: a first transmission and its retransmission combined
        {"name": "derate_20_cells", "kind": "derate", "bg": 1, "Z": 384, "tbs": 20, "ncb": 140, "Kp": 8448,
         "Qm": 8, "Nl": 4, "E": 9088, "fp": 3, "tx": 2, "descr": False},
        # filler bits, an odd size, repetition and descrambling, binary32 buffers
        {"name": "derate_descrambled", "kind": "derate", "bg": 2, "Z": 208, "tbs": 8, "ncb": 25, "Kp": 2056,
         "Qm": 4, "Nl": 2, "E": 10808, "fp": 0, "tx": 1, "descr": True},
        # CB and TB CRC of the full slot
        {"name": "crc_20_cells", "kind": "crc", "bg": 1, "Z": 384, "tbs": 20, "ncb": 140, "Kp": 8448},
        # DL: the full slot's code blocks encoded
        {"name": "encode_20_cells", "kind": "encode", "bg": 1, "Z": 384, "tbs": 20, "ncb": 140, "puncture": True},
        # DL: the full slot rate-matched and scrambled
        {"name": "dlrm_20_cells", "kind": "dlrm", "bg": 1, "Z": 384, "tbs": 20, "ncb": 140, "Kp": 8448, "Qm": 8,
         "Nl": 4, "E": 9088, "rv": 0, "scramble": True},
        # the largest: 64 cells' receive chain from int8 LLRs, large TBs and one-CB TBs beside them
        {"name": "cells_64_int8", "kind": "cells", "cells": 64, "ncb": 140, "small": 28, "dtype": "int8", "iters": 8,
         "et": True, "snr": 8.0},
        # receive chain of different UEs, descrambled, first transmission and retransmission
        {"name": "ues_64_harq", "kind": "ues", "shape_seed": 11, "ues": 64, "dtype": "fp16", "iters": 10, "et": True,
         "descr": True},
        # serving: a burst of TBs from 32 cells through the HARQ engine, retransmissions included
        {"name": "serve_burst", "kind": "serve", "shape_seed": 41, "tbs": 384, "cells": 32, "iters": 10},
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(lo * (hi / lo) ** rng.random()))

    kind = rng.choice(["tb", "slot", "load", "derate", "crc", "encode", "dlrm", "cells", "ues", "serve"])
    bg = rng.choice([1, 1, 2])
    Z = rng.choice([z for z in LIFTING_SIZES if z >= 24])
    K = nsys(bg) * Z
    if kind == "tb":
        return {"kind": kind, "bg": bg, "Z": Z, "mb": log_int(4, nrows(bg)), "tbs": rng.randint(1, 32),
                "ncb": rng.randint(1, 16), "dtype": rng.choice(["fp16", "fp16", "fp32"]), "iters": rng.randint(4, 12),
                "et": rng.random() < 0.3, "soft": rng.random() < 0.3, "esn0": round(rng.uniform(0.0, 6.0), 2)}
    if kind == "slot":
        return {"kind": kind, "shape_seed": rng.randrange(1 << 20), "ues": log_int(4, 128),
                "z_min": rng.choice([2, 24, 64]), "max_cbs": rng.choice([4, 24, 24]),
                "dtype": rng.choice(["fp16", "fp16", "fp32"]), "iters": rng.randint(6, 10), "et": rng.random() < 0.3}
    if kind == "load":
        return {"kind": kind, "bg": bg, "Z": Z, "R": round(rng.uniform(0.35, 0.93), 3), "tbs": rng.randint(2, 20),
                "ncb": rng.randint(16, 120), "dtype": rng.choice(["fp16", "fp16", "fp32"]),
                "iters": rng.randint(5, 10), "et": rng.random() < 0.3, "esn0": round(rng.uniform(2.0, 9.0), 2)}
    Qm, Nl = rng.choice([2, 4, 6, 8]), rng.choice([1, 2, 4])
    Kp = K - 8 * rng.randrange(0, max(1, Z // 8))
    Kp -= Kp % 8
    E = int(Kp / rng.uniform(0.3, 0.95))
    E -= E % (Qm * Nl)
    if kind == "derate":
        return {"kind": kind, "bg": bg, "Z": Z, "tbs": log_int(1, 32), "ncb": log_int(1, 100), "Kp": Kp, "Qm": Qm,
                "Nl": Nl, "E": E, "fp": rng.choice([0, 1, 2, 3, 3]), "tx": rng.choice([1, 2]),
                "descr": rng.random() < 0.5}
    if kind == "crc":
        return {"kind": kind, "bg": bg, "Z": Z, "tbs": log_int(1, 64), "ncb": log_int(1, 140), "Kp": Kp}
    if kind == "encode":
        return {"kind": kind, "bg": bg, "Z": Z, "tbs": log_int(1, 64), "ncb": log_int(1, 100),
                "puncture": rng.random() < 0.8}
    if kind == "dlrm":
        return {"kind": kind, "bg": bg, "Z": Z, "tbs": log_int(1, 32), "ncb": log_int(1, 100), "Kp": Kp, "Qm": Qm,
                "Nl": Nl, "E": E, "rv": rng.choice([0, 0, 1, 2, 3]), "scramble": rng.random() < 0.7}
    if kind == "cells":
        return {"kind": kind, "cells": log_int(1, 48), "ncb": rng.randint(20, 150), "small": rng.randint(0, 32),
                "dtype": rng.choice(["int8", "int8", "fp16", "fp32"]), "iters": rng.randint(6, 10),
                "et": rng.random() < 0.8, "snr": round(rng.uniform(5.0, 11.0), 2)}
    if kind == "ues":
        return {"kind": kind, "shape_seed": rng.randrange(1 << 20), "ues": log_int(4, 128),
                "dtype": rng.choice(["int8", "fp16"]), "iters": rng.randint(6, 10), "et": rng.random() < 0.8,
                "descr": rng.random() < 0.7}
    return {"kind": kind, "shape_seed": rng.randrange(1 << 20), "tbs": log_int(16, 384), "cells": 32,
            "iters": rng.randint(6, 10)}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _powers(n, poly):
    """x^j mod g for j < n, as n integers."""
    g, deg = poly
    top, mask = 1 << (deg - 1), (1 << deg) - 1
    out = np.zeros(n, np.int64)
    v = 1
    for j in range(n):
        out[j] = v
        v = ((v << 1) & mask) ^ (g if v & top else 0)
    return out


def _crc(bits, poly):
    """Remainders of the rows of a 0/1 device matrix, seen as polynomials
    (first column the highest power), as 0/1 float rows, MSB first."""
    n = bits.shape[1]
    p = _powers(n, poly)[::-1].copy()
    deg = poly[1]
    table = ((p[:, None] >> np.arange(deg - 1, -1, -1)) & 1).astype(np.float32)
    return torch.remainder(bits.float() @ torch.from_numpy(table).cuda(), 2.0)


def _mulmod(a, b, poly):
    g, deg = poly
    r = np.zeros_like(a)
    for i in range(deg - 1, -1, -1):
        r = np.where((r >> (deg - 1)) & 1, ((r << 1) & ((1 << deg) - 1)) ^ g, r << 1)
        r = r ^ (a if (b >> i) & 1 else 0)
    return r


def _bits_to_ints(bits):
    deg = bits.shape[1]
    w = torch.tensor([1 << (deg - 1 - i) for i in range(deg)], dtype=torch.float64, device=bits.device)
    return (bits.double() @ w).cpu().numpy().astype(np.int64)


def _code_blocks(n, bg, Z, C, Kp, gen):
    """n TBs of C code blocks of Kp bits each (payload, TB CRC, CB CRCs, then
    filler zeros): (n * C, nsys * Z) 0/1 bytes on the device."""
    K = nsys(bg) * Z
    info = torch.zeros((n * C, K), dtype=torch.uint8, device="cuda")
    if C == 1:
        poly = CRC16 if Kp - 16 <= 3824 else CRC24A
        info[:, :Kp - poly[1]] = torch.randint(0, 2, (n, Kp - poly[1]), generator=gen, device="cuda",
                                               dtype=torch.uint8)
        info[:, Kp - poly[1]:Kp] = _crc(info[:, :Kp], poly).to(torch.uint8)
        return info
    d = Kp - 24
    info[:, :d] = torch.randint(0, 2, (n * C, d), generator=gen, device="cuda", dtype=torch.uint8)
    last = torch.arange(C - 1, n * C, C, device="cuda")
    info[last, d - 24:d] = 0
    part = _bits_to_ints(_crc(info[:, :d], CRC24A)).reshape(n, C)
    step = int(_powers(d + 1, CRC24A)[d])
    r = np.zeros(n, np.int64)
    for c in range(C):
        r = _mulmod(r, step, CRC24A) ^ part[:, c]
    tb = ((r[:, None] >> np.arange(23, -1, -1)) & 1).astype(np.uint8)
    info[last, d - 24:d] = torch.from_numpy(tb).cuda()
    tail = torch.zeros((n * C, Kp), dtype=torch.uint8, device="cuda")
    tail[:, :d] = info[:, :d]
    info[:, d:Kp] = _crc(tail, CRC24B).to(torch.uint8)
    return info


def _selection(bg, Z, Kp, E, k0):
    """Circular-buffer positions of the E selected bits (filler skipped)."""
    N, K = (66 if bg == 1 else 50) * Z, nsys(bg) * Z
    lo, hi = Kp - 2 * Z, K - 2 * Z
    j = (k0 + np.arange((E // (N - (K - Kp)) + 2) * N)) % N
    return torch.from_numpy(j[(j < lo) | (j >= hi)][:E].astype(np.int64)).cuda()


def _gold(cinit, n):
    """The first n bits of the TS 38.211 5.2.1 sequence of cinit."""
    m = n + 1600
    x1, x2 = np.zeros(m + 62, np.uint8), np.zeros(m + 62, np.uint8)
    x1[0] = 1
    x2[:31] = (cinit >> np.arange(31)) & 1
    for i in range(0, m, 28):
        x1[i + 31:i + 59] = x1[i + 3:i + 31] ^ x1[i:i + 28]
        x2[i + 31:i + 59] = x2[i + 3:i + 31] ^ x2[i + 2:i + 30] ^ x2[i + 1:i + 29] ^ x2[i:i + 28]
    return x1[1600:m] ^ x2[1600:m]


def _channel(bits, Qm, snr_db, dtype, gen, sign=None):
    """(n, G) transmitted bits -> (n, G / Qm * 8) LLRs in the receiver's
    layout (8 slots per symbol), BPSK-AWGN; sign: the scrambling's +-1."""
    n, G = bits.shape
    sigma2 = 10.0 ** (-snr_db / 10.0) / 2.0
    x = 1.0 - 2.0 * bits.float()
    if sign is not None:
        x = x * sign
    y = x + torch.randn(x.shape, generator=gen, device="cuda") * float(np.sqrt(sigma2))
    buf = torch.zeros((n, G // Qm, QAM_STRIDE), device="cuda")
    buf[:, :, :Qm] = (y * (2.0 / sigma2)).view(n, G // Qm, Qm)
    buf = buf.view(n, -1)
    if dtype == torch.int8:
        return torch.clamp(torch.round(buf * 4.0), -127, 127).to(torch.int8)
    return buf.to(dtype).contiguous()


def _transmission(cw, n, C, bg, Z, Kp, Qm, E, k0):
    """Code words (n * C, all columns) -> (n, C * E) interleaved bits."""
    e = cw[:, 2 * Z:][:, _selection(bg, Z, Kp, E, k0)]
    return e.view(n * C, Qm, E // Qm).transpose(1, 2).reshape(n, C * E)


def _slot_shapes(case):
    rng = np.random.RandomState(case["shape_seed"])
    zs = [z for z in LIFTING_SIZES if z >= case["z_min"]]
    tbs = []
    for _ in range(case["ues"]):
        bg, Z = int(rng.randint(1, 3)), int(zs[rng.randint(len(zs))])
        R, ncb = float(rng.uniform(0.2, 0.93)), int(rng.randint(1, case["max_cbs"] + 1))
        esn0 = float(rng.uniform(-1.0, 8.0))
        mb, N = mb_for_rate(bg, Z, nsys(bg) * Z, R)
        tbs.append(TransportBlock(bg, Z, mb, ncb, min(N - 2 * Z, (nsys(bg) + mb - 2) * Z), esn0))
    return tbs


def _load_shapes(case):
    bg, Z = case["bg"], case["Z"]
    mb, N = mb_for_rate(bg, Z, nsys(bg) * Z, case["R"])
    return [TransportBlock(bg, Z, mb, case["ncb"], min(N - 2 * Z, (nsys(bg) + mb - 2) * Z), case["esn0"])
            for _ in range(case["tbs"])]


def _rm_params(case, rv, ndi):
    ps = []
    for u in range(case["tbs"]):
        p, _ = make_tb_params(case["bg"], case["Z"], case["ncb"], case["Kp"], case["Qm"], case["Nl"],
                              case["ncb"] * case["E"], rv, ndi=ndi, user_group=u)
        p.cinit = (0x1B5A3C7 * (u + 1)) & 0x7FFFFFFF
        ps.append(p)
    return ps


def _rm_inputs(case, seed):
    """This many transmissions' LLRs: the receiver's layout, one row per TB."""
    gen = _generator(seed)
    dtype = torch.float16 if case["fp"] in (1, 3) else torch.float32
    txs = []
    for _ in range(case["tx"]):
        bits = torch.randint(0, 2, (case["tbs"], case["ncb"] * case["E"]), generator=gen, device="cuda",
                             dtype=torch.uint8)
        txs.append(_channel(bits, case["Qm"], 2.0, dtype, gen))
    return txs


# groups of equal TBs of a fused slot: (how many, bg, Z, C, Kp, Qm, E, snr)
def _fused_groups(case):
    if case["kind"] == "cells":
        g = [(case["cells"], 1, 384, case["ncb"], 8448, 8, 9088, case["snr"])]
        if case["small"]:  # one-CB BG2 TBs at R = 0.5, the two sizes in turn
            half = case["cells"] * case["small"] // 2
            g += [(case["cells"] * case["small"] - half, 2, 104, 1, 1040, 8, 2080, case["snr"]),
                  (half, 2, 208, 1, 2080, 8, 4160, case["snr"])]
        return [x for x in g if x[0] > 0]
    out = []
    for bg, Z, C, Kp, Qm, _, E, snr in serving_specs(case.get("ues") or 64, case["shape_seed"]):
        Kp -= Kp % 8
        out.append((1, bg, Z, C, Kp, Qm, E, snr))
    return out


def _fused_rvs(case):
    return (0,) if case["kind"] == "cells" else (0, 2)


def _fused_data(case, seed, rvs):
    """Per group: LLRs of each transmission, one row per TB."""
    gen = _generator(seed)
    data = []
    t = 0
    for n, bg, Z, C, Kp, Qm, E, snr in _fused_groups(case):
        cw = encode(bg, Z, _code_blocks(n, bg, Z, C, Kp, gen))
        sign = None
        if case.get("descr"):
            sign = torch.from_numpy(np.stack([1.0 - 2.0 * _gold(_cinit(t + i), C * E) for i in range(n)])).float().cuda()
        txs = []
        for rv in rvs:
            p, _ = make_tb_params(bg, Z, C, Kp, Qm, 1, C * E, rv)
            bits = _transmission(cw, n, C, bg, Z, Kp, Qm, E, p.k0)
            txs.append(_channel(bits, Qm, snr, _FLOAT[case["dtype"]], gen, sign))
        data.append(txs)
        t += n
    return data


def _cinit(t):
    return (0x2A6F01 * (t + 1) + 77) & 0x7FFFFFFF


class _Outputs:
    """One slot's output buffers, a part of them for each TB."""

    def __init__(self, params):
        ncb = [int(p.num_CBs) for p in params]
        nby = [(p.num_CBs * SlotTb.data_bytes(p) + 15) // 16 * 16 for p in params]
        self.all = {"bits": torch.zeros((sum(ncb), SLOT_CB_WORDS), dtype=torch.int32, device="cuda"),
                    "cb_crc": torch.zeros(sum(ncb), dtype=torch.int32, device="cuda"),
                    "bytes": torch.zeros(sum(nby), dtype=torch.uint8, device="cuda"),
                    "tb_crc": torch.zeros(len(params), dtype=torch.int32, device="cuda"),
                    "iterations": torch.zeros(sum(ncb), dtype=torch.uint8, device="cuda")}
        self.tb = []
        c = b = 0
        for t in range(len(params)):
            a = self.all
            self.tb.append((a["bits"][c:c + ncb[t]], a["cb_crc"][c:c + ncb[t]], a["bytes"][b:b + nby[t]],
                            a["tb_crc"][t:t + 1], a["iterations"][c:c + ncb[t]]))
            c += ncb[t]
            b += nby[t]


def _prepare_fused(case, seed):
    groups, rvs = _fused_groups(case), _fused_rvs(case)
    data = _fused_data(case, seed, rvs)
    dec = LdpcDecoder()
    first = [make_tb_params(bg, Z, C, Kp, Qm, 1, C * E, 0)[0] for n, bg, Z, C, Kp, Qm, E, _ in groups for _ in range(n)]
    outs = _Outputs(first)
    harq = torch.zeros(sum(int(p.num_CBs * p.Ncb_padded) for p in first), dtype=torch.float16, device="cuda")
    plans = []
    for k, rv in enumerate(rvs):
        slot, t, at = [], 0, 0
        for (n, bg, Z, C, Kp, Qm, E, _), txs in zip(groups, data):
            mb = max(make_tb_params(bg, Z, C, Kp, Qm, 1, C * E, r)[1] for r in rvs[:k + 1])
            for i in range(n):
                p, _ = make_tb_params(bg, Z, C, Kp, Qm, 1, C * E, rv, ndi=1 if k == 0 else 0)
                p.cinit = _cinit(t)
                size = int(p.num_CBs * p.Ncb_padded)
                slot.append(SlotTb(p, txs[k][i], harq[at:at + size], mb, max_iterations=case["iters"],
                                   early_term=case["et"], llr_scale=0.25 if case["dtype"] == "int8" else 1.0,
                                   outputs=outs.tb[t], descramble=bool(case.get("descr"))))
                t += 1
                at += size
        plans.append(SlotDecoder(dec).build(slot))
    if case["kind"] == "cells":
        plans[0].launch()
        torch.cuda.synchronize()
        plans[0].capture()
    return {"kind": case["kind"], "dec": dec, "plans": plans, "keep": data, "out": dict(outs.all, harq=harq)}


def _prepare_serve(case, seed):
    groups = [g[1:] for g in _fused_groups(dict(case, ues=64))]
    data = _fused_data(dict(case, ues=64, dtype="fp16"), seed, RV_SEQUENCE)
    dec = LdpcDecoder()
    srv = HarqServer(dec, pool_bytes=1 << 30, max_inflight=3, max_tbs=2048, max_cbs=16384)
    n = case["tbs"]
    prm = [[make_tb_params(bg, Z, C, Kp, Qm, 1, C * E, rv, ndi=1 if k == 0 else 0)
            for k, rv in enumerate(RV_SEQUENCE)] for bg, Z, C, Kp, Qm, E, _ in groups]
    outs = _Outputs([prm[a % 64][0][0] for a in range(n)])
    entries = (L.HarqTraceEntry * (4 * n))()
    for a in range(n):
        mb = 4
        for k in range(4):
            p, m = prm[a % 64][k]
            mb = max(mb, m)
            e = entries[4 * a + k]
            e.req = srv.request((a % case["cells"], 1 + a // 16, a % 16), p, data[a % 64][k][0], outs.tb[a], mb,
                                max_iterations=case["iters"], early_term=True, last=k == 3, tag=4 * a + k)
            e.arrival_us = 0.0 if k == 0 else -1.0
            e.next = 4 * a + k + 1 if k < 3 else -1
    out = {k: v for k, v in outs.all.items() if k != "tb_crc"}  # the engine reports the TB CRCs itself
    return {"kind": "serve", "dec": dec, "srv": srv, "entries": entries, "keep": data, "out": out}


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("cells", "ues"):
        return _prepare_fused(case, seed)
    if kind == "serve":
        return _prepare_serve(case, seed)
    if kind == "derate":
        txs = _rm_inputs(case, seed)
        rm = DeRateMatch(fp_config=case["fp"], descrambling=case["descr"])
        prms = [_rm_params(case, (0, 2)[k], 1 if k == 0 else 0) for k in range(case["tx"])]
        size = case["ncb"] * int(prms[0][0].Ncb_padded)
        harq = torch.zeros((case["tbs"], size), dtype=torch.float16 if case["fp"] in (2, 3) else torch.float32,
                           device="cuda")
        return {"kind": kind, "rm": rm, "prms": prms, "llrs": [[x[u] for u in range(case["tbs"])] for x in txs],
                "harqs": [harq[u] for u in range(case["tbs"])], "out": harq}
    gen = _generator(seed)
    if kind == "tb":
        dec = LdpcDecoder()
        bg, Z, mb = case["bg"], case["Z"], case["mb"]
        tbs = [fill_tb(TransportBlock(bg, Z, mb, case["ncb"], (nsys(bg) + mb - 2) * Z, case["esn0"]), gen,
                       _FLOAT[case["dtype"]]) for _ in range(case["tbs"])]
        cfg = LdpcDecodeConfig(bg, Z, mb, llr_type=L.CUPHY_R_32F if case["dtype"] == "fp32" else L.CUPHY_R_16F,
                               max_iterations=case["iters"], flags=L.CUPHY_LDPC_DECODE_EARLY_TERM if case["et"] else 0)
        out = {"bits": torch.zeros((case["tbs"] * case["ncb"], tbs[0].out_words), dtype=torch.int32, device="cuda")}
        if case["soft"]:
            out["soft"] = torch.zeros((case["tbs"] * case["ncb"], nsys(bg) * Z), dtype=torch.float16, device="cuda")
        parts = {k: list(v.split(case["ncb"])) for k, v in out.items()}
        return {"kind": kind, "dec": dec, "cfg": cfg, "llrs": [tb.llr for tb in tbs], "parts": parts, "out": out}
    if kind in ("slot", "load"):
        dec = LdpcDecoder()
        tbs = _slot_shapes(case) if kind == "slot" else _load_shapes(case)
        for tb in tbs:
            fill_tb(tb, gen, _FLOAT[case["dtype"]])
            tb.info = None
        words = torch.zeros(sum(tb.ncb * tb.out_words for tb in tbs), dtype=torch.int32, device="cuda")
        at = 0
        for tb in tbs:
            tb.out = words[at:at + tb.ncb * tb.out_words].view(tb.ncb, tb.out_words)
            at += tb.ncb * tb.out_words
        bd = BatchDecoder(dec).build(tbs, llr_type=L.CUPHY_R_32F if case["dtype"] == "fp32" else L.CUPHY_R_16F,
                                     fp16_math=case["dtype"] == "fp16", max_iterations=case["iters"],
                                     flags=L.CUPHY_LDPC_DECODE_EARLY_TERM if case["et"] else 0)
        bd.capture()
        return {"kind": kind, "dec": dec, "bd": bd, "tbs": tbs, "out": words}
    if kind == "crc":
        bg, Z, C, Kp = case["bg"], case["Z"], case["ncb"], case["Kp"]
        prms = [make_tb_params(bg, Z, C, Kp, 2, 1, C * 2 * Kp, 0)[0] for _ in range(case["tbs"])]
        info = _code_blocks(case["tbs"], bg, Z, C, Kp, gen)
        bad = torch.rand(info.shape[0], generator=gen, device="cuda") < 0.05  # blocks the decoder got wrong
        info[bad, torch.randint(0, Kp, (int(bad.sum()),), generator=gen, device="cuda")] ^= 1
        padded = torch.zeros((info.shape[0], SLOT_CB_WORDS, 32), dtype=torch.int32, device="cuda")
        padded.view(info.shape[0], -1)[:, :info.shape[1]] = info
        words = torch.zeros((info.shape[0], SLOT_CB_WORDS), dtype=torch.int32, device="cuda")
        for b in range(32):
            words |= padded[:, :, b] << b
        nby = (C * SlotTb.data_bytes(prms[0]) + 3) // 4 * 4
        out = {"cb_crc": torch.zeros(info.shape[0], dtype=torch.int32, device="cuda"),
               "bytes": torch.zeros(case["tbs"] * nby, dtype=torch.uint8, device="cuda"),
               "tb_crc": torch.zeros(case["tbs"], dtype=torch.int32, device="cuda")}
        return {"kind": kind, "crc": CrcDecode(), "prms": prms, "words": words, "out": out}
    n_in = (nsys(case["bg"]) if kind == "encode" else (66 if case["bg"] == 1 else 50)) * case["Z"]
    words = torch.randint(-(1 << 31), 1 << 31, (case["tbs"], case["ncb"], (n_in + 31) // 32), generator=gen,
                          device="cuda", dtype=torch.int64).to(torch.int32)
    if n_in % 32:
        words[:, :, -1] &= (1 << (n_in % 32)) - 1
    rows = [words[t] for t in range(case["tbs"])]
    if kind == "encode":
        return {"kind": kind, "enc": LdpcEncoder(puncturing=case["puncture"]), "bg": case["bg"], "Z": case["Z"],
                "words": rows}
    return {"kind": kind, "prms": _rm_params(case, case["rv"], 1), "words": rows,
            "emax": (case["E"] + 31) // 32 * 32, "scramble": case["scramble"]}


def run(state):
    kind = state["kind"]
    if kind == "tb":
        state["dec"].decode_tb(state["cfg"], state["llrs"], state["parts"]["bits"], state["parts"].get("soft"))
    elif kind in ("slot", "load"):
        state["bd"].replay()
    elif kind == "derate":
        for prms, llrs in zip(state["prms"], state["llrs"]):
            state["rm"].run(prms, llrs, state["harqs"])
    elif kind == "crc":
        o = state["out"]
        state["crc"].run(state["prms"], state["words"], o["cb_crc"], o["bytes"], o["tb_crc"])
    elif kind == "encode":
        return state["enc"].encode_words(state["bg"], state["Z"], state["words"])
    elif kind == "dlrm":
        return dl_rate_match(state["prms"], state["words"], state["emax"], scrambling=state["scramble"])
    elif kind == "cells":
        state["plans"][0].replay()
    elif kind == "ues":
        for plan in state["plans"]:
            plan.launch()
    else:
        done = state["srv"].serve_trace(state["entries"], 0.0)
        got = np.frombuffer(done, dtype=np.dtype(L.HarqCompletion))
        return dict(state["out"], tb_crc=got["tb_crc"].copy(), status=got["status"].copy())
    return state["out"]


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _decode_work(bg, Z, mb, ncb, iters, et, in_bytes):
    """8 operations per edge and iteration (subtract, three for the minima,
    sign, two to select, add); with early termination at least one iteration."""
    return {"bytes": ncb * ((nsys(bg) + mb - 2) * Z * in_bytes + nsys(bg) * Z / 8),
            "flops": 8.0 * ncb * Z * num_edges(bg, mb) * (1 if et else iters)}


def _fused_work(groups, in_bytes, rvs):
    total = {"bytes": 0.0, "flops": 0.0}
    for n, bg, Z, C, Kp, Qm, E, _ in groups:
        harq = 2 * (nsys(bg) + nrows(bg)) * Z
        mb = max(make_tb_params(bg, Z, C, Kp, Qm, 1, C * E, rv)[1] for rv in rvs)
        total["bytes"] += n * C * (len(rvs) * E * in_bytes + harq + nsys(bg) * Z / 8 + Kp / 8)
        total["flops"] += n * C * 8.0 * Z * num_edges(bg, mb)
    return total


def work(case):
    kind = case["kind"]
    if kind in ("cells", "ues"):
        return _fused_work(_fused_groups(case), _BYTES[case["dtype"]], _fused_rvs(case))
    if kind == "serve":
        w = _fused_work([(1,) + g[1:] for g in _fused_groups(dict(case, ues=64))], 2, (0,))
        return {k: v * case["tbs"] / 64 for k, v in w.items()}
    if kind in ("slot", "load"):
        ws = [_decode_work(tb.bg, tb.Z, tb.mb, tb.ncb, case["iters"], case["et"], _BYTES[case["dtype"]])
              for tb in (_slot_shapes(case) if kind == "slot" else _load_shapes(case))]
        return {k: sum(w[k] for w in ws) for k in ("bytes", "flops")}
    bg, Z, ncb = case["bg"], case["Z"], case["tbs"] * case["ncb"]
    N = (66 if bg == 1 else 50) * Z
    if kind == "tb":
        w = _decode_work(bg, Z, case["mb"], ncb, case["iters"], case["et"], _BYTES[case["dtype"]])
        w["bytes"] += 2 * ncb * nsys(bg) * Z if case["soft"] else 0
        return w
    if kind == "derate":
        e_in, e_out = (2 if case["fp"] in (1, 3) else 4), (2 if case["fp"] in (2, 3) else 4)
        # the buffer written in full once, and what a retransmission adds to read and written again
        again = min(case["E"], N) * 2 * e_out if case["tx"] == 2 else 0
        return {"bytes": ncb * (case["tx"] * case["E"] * e_in + (N + 2 * Z) * e_out + again),
                "flops": float(ncb * case["tx"] * case["E"])}
    if kind == "crc":
        return {"bytes": ncb * (case["Kp"] / 8 * 2 + 4), "flops": 0.0}
    if kind == "encode":
        return {"bytes": ncb * (nsys(bg) * Z + N + (0 if case["puncture"] else 2 * Z)) / 8, "flops": 0.0}
    return {"bytes": ncb * 2 * case["E"] / 8, "flops": 0.0}


# ---------------------------------------------------------------------------
# 64-bit results: the HARQ buffers (everything else is bits and counts)
# ---------------------------------------------------------------------------
def _exact_combine(buf, llr, C, bg, Z, Kp, Qm, E, k0, scale, sign):
    """Add one transmission ((n, G / Qm * 8) LLRs) to (n, C, 2Z + Ncb) buffers."""
    n = llr.shape[0]
    x = llr.double().view(n, -1, QAM_STRIDE)[:, :, :Qm].reshape(n, -1) * scale
    if sign is not None:
        x = x * sign
    x = x.clamp(-10000.0, 10000.0).view(n, C, E // Qm, Qm).transpose(2, 3).reshape(n, C, E)
    pos = _selection(bg, Z, Kp, E, k0) + 2 * Z
    span = (66 if bg == 1 else 50) * Z - (nsys(bg) * Z - Kp)
    for i in range(0, E, span):
        at = pos[i:i + span]
        buf[:, :, at] = (buf[:, :, at] + x[:, :, i:i + span]).clamp(-10000.0, 10000.0)


def _exact_buffers(n, C, bg, Z, Kp):
    N, K = (66 if bg == 1 else 50) * Z, nsys(bg) * Z
    buf = torch.zeros((n, C, (N + 2 * Z + 7) // 8 * 8), dtype=torch.float64, device="cuda")
    buf[:, :, Kp:K] = 10000.0
    return buf


def exact(case, seed):
    kind = case["kind"]
    if kind == "derate":
        bg, Z, C, Kp, Qm, E = (case[k] for k in ("bg", "Z", "ncb", "Kp", "Qm", "E"))
        buf = _exact_buffers(case["tbs"], C, bg, Z, Kp)
        for k, llr in enumerate(_rm_inputs(case, seed)):
            prms = _rm_params(case, (0, 2)[k], 1)
            sign = None
            if case["descr"]:
                sign = torch.from_numpy(np.stack([1.0 - 2.0 * _gold(p.cinit, C * E) for p in prms])).cuda()
            _exact_combine(buf, llr, C, bg, Z, Kp, Qm, E, prms[0].k0, 1.0, sign)
        return buf.view(case["tbs"], -1)
    if kind in ("cells", "ues"):
        rvs = _fused_rvs(case)
        bufs, t = [], 0
        for (n, bg, Z, C, Kp, Qm, E, _), txs in zip(_fused_groups(case), _fused_data(case, seed, rvs)):
            buf = _exact_buffers(n, C, bg, Z, Kp)
            sign = None
            if case.get("descr"):
                sign = torch.from_numpy(np.stack([1.0 - 2.0 * _gold(_cinit(t + i), C * E) for i in range(n)])).cuda()
            for rv, llr in zip(rvs, txs):
                k0 = make_tb_params(bg, Z, C, Kp, Qm, 1, C * E, rv)[0].k0
                _exact_combine(buf, llr, C, bg, Z, Kp, Qm, E, k0, 0.25 if case["dtype"] == "int8" else 1.0, sign)
            bufs.append(buf.view(-1))
            t += n
        return {"harq": torch.cat(bufs), "bits": None, "cb_crc": None, "bytes": None, "tb_crc": None,
                "iterations": None}
    return None
