"""PUSCH back end around the decoder: de-rate-matching/HARQ combining and
CB/TB CRC checking through the C ABI (cuphySetupPuschRxRateMatch,
cuphySetupPuschRxCrcDecode), plus PerTbParams construction.

Mirrors pyAerial's LdpcDeRateMatch / CrcChecker (pyaerial/src/aerial/phy5g/
ldpc/derate_match.py, crc_check.py) and the parameter derivation of
pycuphy_ldpc_util.cpp:75-171; arrays are torch device tensors.
"""
import ctypes as C

import torch

from . import _hip
from . import _lib as L
from ._upload import UploadBlock, on_stream
from .decoder import _stream_handle

LLR_MAX_ABS = 10000.0


def k0_of(bg, rv, Ncb, Zc):
    """TS 38.212 Table 5.4.2.1-2 (pycuphy_ldpc_util.cpp:122-157)."""
    num = (0, 17, 33, 56) if bg == 1 else (0, 13, 25, 43)
    den = 66 if bg == 1 else 50
    return (num[rv] * Ncb // (den * Zc)) * Zc


def num_parity_nodes(bg, Zc, K, F, G, C, k0, Ncb):
    """mb covering the received parity (pycuphy_ldpc_util.cpp:117-157)."""
    Kd = K - F - 2 * Zc
    ncb_par = min(G // C + k0, Ncb)
    mb = (ncb_par - Kd + Zc - 1) // Zc
    return max(4, min(46 if bg == 1 else 42, mb))


def make_tb_params(bg, Zc, C, Kprime, Qm, Nl, G, rv, ndi=1, n_bbu_layers=None, layer_map=None, user_group=0,
                   first_cb=0, Nref=0):
    """PerTbParams of one TB (fields as setPerTbParams fills them)."""
    p = L.PerTbParams()
    p.ndi, p.rv, p.Qm, p.bg, p.Nl, p.num_CBs, p.Zc = ndi, rv, Qm, bg, Nl, C, Zc
    N = (66 if bg == 1 else 50) * Zc
    p.N = N
    p.Ncb = min(N, Nref) if Nref > 0 else N
    p.Ncb_padded = (N + 2 * Zc + 7) // 8 * 8
    p.G = G
    p.K = (22 if bg == 1 else 10) * Zc
    p.F = p.K - Kprime
    p.k0 = k0_of(bg, rv, p.Ncb, Zc)
    p.encodedSize = G
    p.firstCodeBlockIndex = first_cb
    p.nBBULayers = Nl if n_bbu_layers is None else n_bbu_layers
    lm = list(range(Nl)) if layer_map is None else layer_map
    for i in range(Nl):
        p.layer_map_array[i] = lm[i]
    p.userGroupIndex = user_group
    p.isDataPresent = 1
    mb = num_parity_nodes(bg, Zc, p.K, p.F, G, C, p.k0, p.Ncb)
    p.nZpBitsPerCb = mb * Zc + p.K
    return p, mb


def get_tb_size(num_symbols, num_prbs, num_layers, code_rate, mod_order, num_dmrs_cdm_grps_no_data1_symbols=0):
    """TS 38.214 5.1.3.2 transport block size and code-block count of an
    allocation (cuphyHipTransportBlockSize; pyAerial get_tb_size,
    util.py:171-333, with the code rate as a fraction)."""
    tbs, ncb = C.c_uint32(), C.c_uint32()
    L.check("cuphyHipTransportBlockSize",
            L.lib().cuphyHipTransportBlockSize(num_symbols, num_prbs, num_layers, code_rate, mod_order,
                                               num_dmrs_cdm_grps_no_data1_symbols, C.byref(tbs), C.byref(ncb)))
    return tbs.value, ncb.value


def set_per_tb_params(tb_size, code_rate, qam_mod, rate_match_len, rv, ndi=1, cinit=0, user_group=0, num_layers=1,
                      num_ue_grp_layers=None, layer_map=None, n_dmrs_cdm_grps_no_data=2, lbrm=None):
    """PerTbParams of a PUSCH TB from its size (bits, without CRC) and code
    rate, as pyAerial's setPerTbParams (pycuphy_ldpc_util.cpp:75-171) with
    the PUSCH pipeline's limited-buffer rate matching (lbrm = (n_PRB_LBRM,
    maxLayers, maxQm) or None).  Returns (params, parity nodes, info nodes Kb)."""
    p = L.PerTbParams()
    nl = num_layers
    ng = nl if num_ue_grp_layers is None else num_ue_grp_layers
    lm = (C.c_uint32 * L.MAX_N_LAYERS_PUSCH)(*(list(range(nl)) if layer_map is None else list(layer_map)))
    lb = None
    if lbrm is not None:
        lb = L.LbrmPrm(i_lbrm=1, maxLayers=lbrm[1], maxQm=lbrm[2], n_PRB_LBRM=lbrm[0])
    mb, kb = C.c_uint16(), C.c_uint16()
    L.check("cuphyHipSetPerTbParams",
            L.lib().cuphyHipSetPerTbParams(C.byref(p), tb_size, code_rate, qam_mod, ndi, rv, rate_match_len, cinit,
                                           user_group, nl, ng, lm, n_dmrs_cdm_grps_no_data,
                                           C.byref(lb) if lb is not None else None, C.byref(mb), C.byref(kb)))
    return p, mb.value, kb.value


def put_params(address, params):
    """PerTbParams array at a host address."""
    arr = (L.PerTbParams * len(params)).from_address(address)
    for i, p in enumerate(params):
        arr[i] = p
    return arr


class DeRateMatch:
    """cuphyCreate/Setup/DestroyPuschRxRateMatch + launch of its kernel nodes."""

    def __init__(self, fp_config=3, descrambling=False):
        """descrambling: negate LLR n of each TB where its Gold sequence
        (PerTbParams.cinit) has c(n) = 1, as cuphyCreatePuschRxRateMatch's
        descramblingOn."""
        self._lib = L.lib()
        self.h = C.c_void_p()
        L.check("cuphyCreatePuschRxRateMatch",
                self._lib.cuphyCreatePuschRxRateMatch(C.byref(self.h), fp_config, int(descrambling)))
        sz, al = C.c_size_t(), C.c_size_t()
        L.check("cuphyPuschRxRateMatchGetDescrInfo",
                self._lib.cuphyPuschRxRateMatchGetDescrInfo(C.byref(sz), C.byref(al)))
        self._desc_bytes = sz.value
        self.cfg = L.RateMatchLaunchCfg()

    def close(self):
        if self.h:
            self._lib.cuphyDestroyPuschRxRateMatch(self.h)
            self.h = C.c_void_p()

    def run(self, params, llr_in, harq_out, stream=None):
        """params: list of PerTbParams (UE index = list index); llr_in: one
        device tensor per user group; harq_out: one device tensor per UE."""
        n = len(params)
        idx = (C.c_uint16 * n)(*range(n))
        tin = (L.TensorPrm * len(llr_in))()
        for i, t in enumerate(llr_in):
            tin[i].pAddr = t.data_ptr()
        with on_stream(stream):
            blk = UploadBlock((self._desc_bytes, n * C.sizeof(L.PerTbParams), len(harq_out) * 8))
            prms = put_params(blk.host(1), params)
            ptrs = (C.c_uint64 * len(harq_out)).from_address(blk.host(2))
            for i, t in enumerate(harq_out):
                ptrs[i] = t.data_ptr()
            sh = _stream_handle(stream)
            st = self._lib.cuphySetupPuschRxRateMatch(
                self.h, n, idx, prms, blk.dev(1), tin, tin, C.cast(blk.dev(2), C.POINTER(C.c_void_p)),
                C.c_void_p(blk.host(0)), blk.dev(0), 0, C.c_void_p(C.addressof(self.cfg)), sh)
            L.check("cuphySetupPuschRxRateMatch", st)
            blk.send()
            # (the library's reset and clamp nodes are empty kernels: nothing to launch)
            _hip.launch_node(self.cfg.kernelNodeParamsDriver, sh)
        self._block = blk


class CrcDecode:
    """cuphyCreate/Setup/DestroyPuschRxCrcDecode + launch of CB and TB kernels."""

    def __init__(self, reverse_bytes=True):
        self._lib = L.lib()
        self.h = C.c_void_p()
        L.check("cuphyCreatePuschRxCrcDecode", self._lib.cuphyCreatePuschRxCrcDecode(C.byref(self.h), int(reverse_bytes)))
        sz, al = C.c_size_t(), C.c_size_t()
        L.check("cuphyPuschRxCrcDecodeGetDescrInfo", self._lib.cuphyPuschRxCrcDecodeGetDescrInfo(C.byref(sz), C.byref(al)))
        self._desc_bytes = sz.value
        self.cb_cfg = L.CrcDecodeLaunchCfg()
        self.tb_cfg = L.CrcDecodeLaunchCfg()

    def close(self):
        if self.h:
            self._lib.cuphyDestroyPuschRxCrcDecode(self.h)
            self.h = C.c_void_p()

    def run(self, params, cb_words, cb_crc, tb_bytes, tb_crc, stream=None):
        n = len(params)
        idx = (C.c_uint16 * n)(*range(n))
        with on_stream(stream):
            blk = UploadBlock((self._desc_bytes, n * C.sizeof(L.PerTbParams)))
            prms = put_params(blk.host(1), params)
            sh = _stream_handle(stream)
            st = self._lib.cuphySetupPuschRxCrcDecode(
                self.h, n, idx, C.c_void_p(cb_crc.data_ptr()), C.c_void_p(tb_bytes.data_ptr()),
                C.c_void_p(cb_words.data_ptr()), C.c_void_p(tb_crc.data_ptr()), prms, blk.dev(1),
                C.c_void_p(blk.host(0)), blk.dev(0), 0, C.c_void_p(C.addressof(self.cb_cfg)),
                C.c_void_p(C.addressof(self.tb_cfg)), sh)
            L.check("cuphySetupPuschRxCrcDecode", st)
            blk.send()
            _hip.launch_node(self.cb_cfg.kernelNodeParamsDriver, sh)
            _hip.launch_node(self.tb_cfg.kernelNodeParamsDriver, sh)
        self._block = blk
