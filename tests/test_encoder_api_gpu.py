"""LDPC encoder behind the reference's encoder API (cuphySetupLDPCEncode:
bit-packed tensors, puncturing, a subset of parity rows for rv 0, batched
TBs) and DL rate matching (cuphyHipDlRateMatch: bit selection, bit
interleaving, scrambling), bit-exact against the oracle's encoder (pinned
by the reference's MATLAB goldens and H c = 0) and the oracle's rate-matching
steps (TS 38.212 5.4.2.1 E split, k0, bit selection pinned by the
reference's textbook selection; TS 38.211 Gold sequence)."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def enc():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from aerial_amd.encoder import LdpcEncoder
    return LdpcEncoder(puncturing=True, max_tbs=8)


def nsys(bg):
    return 22 if bg == 1 else 10


def info_bits(bg, Z, ncw, seed, filler=0):
    rng = np.random.RandomState(seed)
    x = rng.randint(0, 2, (ncw, nsys(bg) * Z)).astype(np.uint8)
    if filler:
        x[:, nsys(bg) * Z - filler:] = 0
    return x


def words_to_bits(words, n):
    w = np.ascontiguousarray(words, dtype=np.int32).view(np.uint32)
    return np.unpackbits(w.view(np.uint8), axis=-1, bitorder="little")[..., :n]


# (bg, Z, puncture, num_rows (0: all), rv, TBs, code words, filler bits)
ENC_CASES = [(1, 384, 1, 0, 0, 1, 3, 0), (1, 384, 0, 0, 2, 2, 2, 224), (1, 2, 1, 0, 0, 1, 5, 0),
             (1, 15, 0, 0, 1, 1, 4, 0), (2, 384, 1, 0, 0, 3, 2, 96), (2, 7, 1, 0, 3, 1, 6, 0),
             (1, 208, 1, 8, 0, 2, 3, 0), (2, 104, 1, 6, 0, 1, 4, 40), (1, 64, 0, 20, 2, 1, 2, 0),
             (2, 36, 1, 2, 0, 1, 3, 0)]


@pytest.mark.parametrize("case", ENC_CASES)
def test_encoder_api_matches_oracle(enc, case):
    from aerial_amd.encoder import pack_bits
    bg, Z, punct, rows, rv, n_tbs, ncw, filler = case
    print("[case] encoder API BG%d Z=%d puncture=%d rows=%d rv=%d TBs=%d CWs=%d" % case[:7], flush=True)
    enc.puncturing = bool(punct)
    infos = [info_bits(bg, Z, ncw, 100 * sum(case) + t, filler) for t in range(n_tbs)]
    words = enc.encode_words(bg, Z, [pack_bits(torch.from_numpy(x.T.copy()).cuda()) for x in infos],
                             num_rows=rows, rv=rv)
    torch.cuda.synchronize()
    nrows = rows if (rv == 0 and 0 < rows < (46 if bg == 1 else 42)) else (46 if bg == 1 else 42)
    first = 2 * Z if punct else 0
    nbits = (nsys(bg) + nrows) * Z - first
    for t in range(n_tbs):
        got = words[t].cpu().numpy()
        bits = words_to_bits(got, got.shape[1] * 32)
        for c in range(ncw):
            cw = O.encode(bg, Z, infos[t][c])
            assert np.array_equal(bits[c, :nbits], cw[first:first + nbits]), (case, t, c)
            assert not bits[c, nbits:].any(), "bits after the code word are not zero"
    enc.puncturing = True


def dl_reference(params, cw_bits, cinit, scrambling):
    """Rate-matched bits of each CB from the oracle's steps: E_r, bit
    selection from k0 skipping the filler, interleaving f[j Qm + k] =
    e[k E/Qm + j], XOR with c(start_r + i)."""
    p = params
    cfg = O.rm_cfg(bg=p.bg, Zc=p.Zc, C=p.num_CBs, Qm=p.Qm, Nl=p.Nl, G=p.encodedSize, K=p.K, F=p.F, Ncb=p.Ncb,
                   Ncb_padded=0, k0=p.k0, ndi=1)
    Kd = p.K - p.F - 2 * p.Zc
    gold = O.gold(cinit, 0, p.encodedSize) if scrambling else None
    out, start = [], 0
    for r in range(p.num_CBs):
        E = O.rm_E(cfg, r)
        e = cw_bits[r][O.bit_select(E, Kd, p.F, p.k0, p.Ncb)]
        f = e.reshape(p.Qm, E // p.Qm).T.reshape(-1)
        if scrambling:
            f = f ^ gold[start:start + E]
        out.append(f)
        start += E
    return out


# (tbs, code rate, Qm, layers, rv, G, LBRM (n_PRB_LBRM, maxLayers, maxQm) or None, scrambling)
DL_CASES = [(8448 * 3 - 96, 0.9, 8, 2, 0, 3 * 9216, None, True),       # BG1 Zc=384, 3 CBs
            (7608, 0.3, 4, 1, 2, 2 * 9000, None, False),               # BG1 R < 0.67, one CB, k0 at rv 2
            (1200, 0.5, 2, 1, 3, 7000, None, True),                    # BG2, repetition (E > Ncb - F)
            (256, 0.2, 6, 1, 1, 1800, None, True),                     # BG2, small Zc, filler
            (120936, 0.66, 8, 4, 1, 184000, (51, 2, 6), True),         # limited buffer: Ncb < N, E > Ncb - F
            (40976, 0.8, 6, 3, 0, 3 * 17766, None, True)]              # uneven E split


@pytest.mark.parametrize("case", DL_CASES)
def test_dl_rate_match_matches_oracle(case):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from aerial_amd.encoder import dl_rate_match
    from aerial_amd.pusch import set_per_tb_params
    tbs, R, Qm, nl, rv, G, lbrm, scr = case
    print("[case] DL rate matching TBS=%d R=%.2f Qm=%d Nl=%d rv=%d G=%d lbrm=%s scr=%d" % case, flush=True)
    cinit = (0x51ED27 * (tbs % 977) + 3) & 0x7FFFFFFF
    p, _, _ = set_per_tb_params(tbs, R, Qm, G, rv, num_layers=nl, cinit=cinit, lbrm=lbrm)
    assert p.Ncb <= p.N and (lbrm is None) == (p.Ncb == p.N)
    rng = np.random.RandomState(tbs)
    cw = []
    for r in range(p.num_CBs):
        info = rng.randint(0, 2, p.K).astype(np.uint8)
        info[p.K - p.F:] = 0
        cw.append(O.encode(p.bg, p.Zc, info)[2 * p.Zc:2 * p.Zc + p.N])
    nw = (p.N + 31) // 32
    words = np.zeros((p.num_CBs, nw), np.uint32)
    for r in range(p.num_CBs):
        words[r] = O.pack_bits(cw[r])
    dev = torch.from_numpy(words.view(np.int32)).cuda()
    emax = ((max(O.rm_E(O.rm_cfg(bg=p.bg, Zc=p.Zc, C=p.num_CBs, Qm=Qm, Nl=nl, G=G, K=p.K, F=p.F, Ncb=p.Ncb,
                                         Ncb_padded=0, k0=0, ndi=1), r) for r in range(p.num_CBs)) + 31) // 32 + 1) * 32
    out = dl_rate_match([p], [dev], emax, scrambling=scr)
    torch.cuda.synchronize()
    ref = dl_reference(p, cw, cinit, scr)
    got = out.cpu().numpy()[0]
    for r in range(p.num_CBs):
        bits = words_to_bits(got[r], emax)
        E = ref[r].size
        assert np.array_equal(bits[:E], ref[r]), (case, r)
        assert not bits[E:].any(), (case, r)


def test_encode_then_rate_match_chain(enc):
    """Encoder API -> DL rate matching on the device equals the oracle's
    encoder -> rate-matching steps; the pyAerial-style encode() gives the
    same coded bits."""
    from aerial_amd.encoder import dl_rate_match, pack_bits
    from aerial_amd.pusch import set_per_tb_params
    print("[case] encoder API -> DL rate matching chain, TBS 60000", flush=True)
    tbs, R, Qm, G = 60000, 0.75, 6, 6 * 13500
    p, _, _ = set_per_tb_params(tbs, R, Qm, G, 2, cinit=12345)
    rng = np.random.RandomState(8)
    kp = p.K - p.F
    blocks = rng.randint(0, 2, (kp, p.num_CBs)).astype(np.uint8)
    cbs_dev = torch.from_numpy(blocks).cuda()
    coded = enc.encode([cbs_dev], [tbs], [R], [2])[0]                       # (N, C) bits
    info = torch.zeros((p.K, p.num_CBs), dtype=torch.uint8, device="cuda")
    info[:kp] = cbs_dev
    words = enc.encode_words(p.bg, p.Zc, [pack_bits(info)], rv=2)[0]
    out = dl_rate_match([p], [words], 32 * ((G // p.num_CBs + 40) // 32 + 1), scrambling=True)
    torch.cuda.synchronize()
    cw = []
    for r in range(p.num_CBs):
        full = np.zeros(p.K, np.uint8)
        full[:kp] = blocks[:, r]
        cw.append(O.encode(p.bg, p.Zc, full)[2 * p.Zc:2 * p.Zc + p.N])
    assert np.array_equal(coded.cpu().numpy().T, np.stack(cw))
    ref = dl_reference(p, cw, 12345, True)
    got = out.cpu().numpy()[0]
    for r in range(p.num_CBs):
        assert np.array_equal(words_to_bits(got[r], got.shape[1] * 32)[:ref[r].size], ref[r]), r


# (bg, Zc, CBs, K', Qm, layers, E per CB, rv, scrambling): fewer symbols than a
# word, remainders of 32 symbols, Qm = 1, runs that cross the filler hole and
# the wrap (short circles several times within a word), a sequence far from
# its start (2.5 M bits)
DL_EDGES = [(2, 2, 2, 16, 2, 1, 6, 0, True), (2, 2, 1, 16, 8, 1, 1000, 3, True), (1, 3, 2, 60, 1, 1, 31, 1, True),
            (1, 3, 1, 60, 6, 2, 504, 2, False), (2, 52, 3, 480, 1, 1, 2049, 0, True), (1, 384, 1, 8448, 8, 4, 9088, 0, True),
            (1, 208, 2, 4400, 4, 1, 4 * 33, 2, True), (1, 384, 100, 8424, 6, 1, 25344, 1, True)]


@pytest.mark.parametrize("case", DL_EDGES)
def test_dl_rate_match_edges(case):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from aerial_amd.encoder import dl_rate_match
    from aerial_amd.pusch import make_tb_params
    bg, Zc, C, Kp, Qm, Nl, E, rv, scr = case
    print("[case] DL rate matching BG%d Zc=%d CBs=%d K'=%d Qm=%d Nl=%d E=%d rv=%d scr=%d" % case, flush=True)
    p, _ = make_tb_params(bg, Zc, C, Kp, Qm, Nl, C * E, rv)
    p.cinit = (0x3C6EF35 * (E + 1)) & 0x7FFFFFFF
    cw = np.random.RandomState(E).randint(0, 2, (C, p.N)).astype(np.uint8)
    words = np.stack([O.pack_bits(x) for x in cw])
    emax = (E + 31) // 32 * 32 + 64
    out = dl_rate_match([p], [torch.from_numpy(words.view(np.int32)).cuda()], emax, scrambling=scr)
    torch.cuda.synchronize()
    got = out.cpu().numpy()[0]
    for r, ref in enumerate(dl_reference(p, cw, p.cinit, scr)):
        bits = words_to_bits(got[r], emax)
        assert np.array_equal(bits[:E], ref), (case, r)
        assert not bits[E:].any(), (case, r)


def _busy():
    """Keep the current stream busy for some milliseconds."""
    a = torch.full((4096, 4096), 1e-4, device="cuda")
    for _ in range(12):
        a = a @ a
    return a


def test_calls_on_another_stream(enc):
    """Inputs still being produced on the current stream, and outputs partly
    filled there (TBs of different numbers of code blocks), when the calls are
    launched on another stream."""
    from aerial_amd.encoder import dl_rate_match
    from aerial_amd.pusch import make_tb_params
    print("[case] encoder and DL rate matching launched on another stream", flush=True)
    rng = np.random.RandomState(3)
    enc.puncturing = True
    late, words, cws, params = [], [], [], []
    for t, C in enumerate((3, 1, 2)):
        p, _ = make_tb_params(2, 52, C, 480, 2, 1, C * 600, 0)
        p.cinit = 77 + t
        params.append(p)
        info = rng.randint(0, 2, (C, 520)).astype(np.uint8)
        info[:, 480:] = 0
        late.append(torch.from_numpy(np.stack([O.pack_bits(x) for x in info]).view(np.int32)).cuda())
        words.append(torch.zeros_like(late[-1]))
        cws.append([O.encode(2, 52, x)[104:104 + p.N] for x in info])
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    for _ in range(3):
        for w in words:
            w.zero_()
        keep = _busy()
        for w, x in zip(words, late):
            w.copy_(x)
        coded = [enc.encode_words(2, 52, [w], stream=s)[0] for w in words]
        s.synchronize()
        keep = _busy()
        coded = [c.clone() for c in coded]  # (on the current stream, after the work above)
        out = dl_rate_match(params, coded, 640, scrambling=True, stream=s)
        s.synchronize()
        got = out.cpu().numpy()
        for t, (p, cw) in enumerate(zip(params, cws)):
            for r, ref in enumerate(dl_reference(p, cw, p.cinit, True)):
                assert np.array_equal(words_to_bits(got[t, r], 640)[:ref.size], ref), (t, r)
            assert (got[t, len(cw):] == -1).all()
    del keep


def test_encode_words_captured():
    """A captured call replays with the addresses it was captured with, also
    after other calls of the same encoder."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from aerial_amd.encoder import LdpcEncoder
    print("[case] encode_words under capture", flush=True)
    enc = LdpcEncoder()
    rng = np.random.RandomState(4)
    x = [torch.from_numpy(rng.randint(0, 1 << 32, (3, 22 * 104 // 32 + 1), dtype=np.uint64).astype(np.uint32)
                          .view(np.int32)).cuda() for _ in range(4)]
    for t in x:
        t[:, -1] &= (1 << (22 * 104 % 32)) - 1
    want = [w.clone() for w in enc.encode_words(1, 104, x)]
    graphs, outs = [], []
    for k in (0, 2):
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            o = enc.encode_words(1, 104, x[k:k + 2])
        graphs.append(g)
        outs.append(o)
    for _ in range(3):
        for k, g in zip((0, 2), graphs):
            for o in outs[k // 2]:
                o.zero_()
            enc.encode_words(1, 104, x[3:])
            g.replay()
            torch.cuda.synchronize()
            assert all(torch.equal(o, w) for o, w in zip(outs[k // 2], want[k:k + 2]))


def test_encode_words_results_are_aligned(enc):
    """Each TB's words start on an address of their own, as separate tensors do
    (9 words per TB here: viewed as bytes of any width)."""
    print("[case] encode_words result alignment", flush=True)
    outs = enc.encode_words(2, 5, [torch.zeros((1, 2), dtype=torch.int32, device="cuda")] * 5)
    assert all(o.data_ptr() % 512 == 0 and o.is_contiguous() and o.storage_offset() % 4 == 0 for o in outs)


def test_calls_with_a_cuda_default_device(enc):
    """The uploads' host blocks are host memory whatever torch's default device."""
    from aerial_amd.encoder import dl_rate_match
    from aerial_amd.pusch import make_tb_params
    print("[case] encoder and DL rate matching, default device cuda", flush=True)
    p, _ = make_tb_params(2, 52, 2, 520, 2, 1, 2 * 600, 0)
    info = np.random.RandomState(6).randint(0, 2, (2, 520)).astype(np.uint8)
    words = torch.from_numpy(np.stack([O.pack_bits(x) for x in info]).view(np.int32)).cuda()
    enc.puncturing = True
    with torch.device("cuda"):
        out = dl_rate_match([p], enc.encode_words(2, 52, [words]), 640)
    torch.cuda.synchronize()
    cw = [O.encode(2, 52, x)[104:104 + p.N] for x in info]
    for r, ref in enumerate(dl_reference(p, cw, 0, False)):
        assert np.array_equal(words_to_bits(out.cpu().numpy()[0, r], 640)[:ref.size], ref), r
