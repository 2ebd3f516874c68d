"""Performance cases: what programs call this framework for, over the sizes they call it with.

Every case goes through the package's public entry points with device tensors, the outputs and
workspaces kept by the program where the entry point takes them. The shapes are those of the
benchmark and the tests (hidden 6144, dense inter 12288, expert inter 2048, 64 experts top-8, the
latent projections 576 and 1536 x 6144, 64 heads of 512 x 256); `draw` varies them.

Weights are random blocks whose scales give a weight rms of 1 / sqrt(in_dim) (log-normal over the
blocks), so that products, and the SwiGLU inputs made from them, are of order one as in a trained
model; activations are normal with one channel in 64 eight times larger.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import gpeed_amd as G

# ---- block formats --------------------------------------------------------------------------------

F32, F16, Q8_0, Q2_K, Q3_K, Q6_K, IQ3_XXS, IQ3_S, IQ2_S, IQ4_XS, BF16 = 0, 1, 8, 10, 11, 14, 18, 21, 22, 23, 30
NAMES = {F32: "f32", F16: "f16", Q8_0: "q8_0", Q2_K: "q2_k", Q3_K: "q3_k", Q6_K: "q6_k", IQ3_XXS: "iq3_xxs",
         IQ3_S: "iq3_s", IQ2_S: "iq2_s", IQ4_XS: "iq4_xs", BF16: "bf16"}
DTYPES = {v: k for k, v in NAMES.items()}
# weights per block, bytes per block, byte offset of d, rms of weight / d over uniform random codes
BLOCKS = {Q8_0: (32, 34, 0, 74.0), Q2_K: (256, 84, 80, 17.0), Q3_K: (256, 110, 108, 43.0),
          Q6_K: (256, 210, 208, 1370.0), IQ3_XXS: (256, 98, 0, 115.0), IQ3_S: (256, 110, 0, 166.0),
          IQ2_S: (256, 82, 0, 63.0), IQ4_XS: (256, 136, 0, 1290.0)}
SCALARS = {F32: torch.float32, F16: torch.float16, BF16: torch.bfloat16}

# The formats' codebooks, packed: 3 bits per value (IQ3_XXS levels below, IQ3_S 2v + 1), 2 bits (IQ2_S).
IQ3_LEVELS = (4, 12, 20, 28, 36, 44, 52, 62)
IQ2_LEVELS = (8, 25, 43, 0)
IQ4_LEVELS = (-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113)
IQ3_XXS_GRID = (
    "00000200400900b00f01001201902203b03d04104304804a05105505805a06106c07808008208408909009209909b09f0a90af0b"
    "d0c10c70c80ca0d50f810b11f12412f13b13d14114715a16a19d1b41c81cc1ce1e31f120120320820a21121321821a21c2272282"
    "4024224925025228128328828a2912982ba2c02c22d02d92e62f63013053283503543663793853d23e040040240940b410412416"
    "41942244144344544844a45145847347747848048248948f49049249f4a04ad4c14c84cc4f84fc51d52b54355756157c5c15c35c"
    "e5e560160860a61161362863563a6406426506596646666816836886956aa6ba6c96db71872773a74074675276d78c79e7b37db7"
    "f080480f81d81f82b82f87c89089f8a08b08b68c78e59049299349559639789c59c89ca9d8a0aa21a38a40a46a56a6da8ca9aaba"
    "ac2aebb08b13b17b3ab42b59ba8bd4be2c14c24c26c34c51c71c8fcb4cd8cded24d45d6ad9bdc3dd1e03e05e07e08e1ae2ae56e6"
    "0e8aea5eaaec0ecdedbef0f11f21f40f42f54f98")
IQ3_S_GRID = (
    "00000100200500700800900a00c00e01001101501b02002202502702902b03003203903c03f04004104204404804904d05005305"
    "705905d06407107507a08008108508708808b08e09109509809c0a20a50a70a90ab0b80bb0c30c90cd0d00d20d90db0de0e40e80"
    "ea0f70f90fd10010b10f11111411a12012312913814214415015215615b16116516717617b18618918b1991aa1b91c01c21c41d0"
    "1d21d61db1e81ec20020120220420820920b20d20f21021221921c21e22c22e23123a24024124324624824c25125825b26126826"
    "a27827e28028a28d28f29029429a2a02a32ad2b02ba2c12c42c72c82cb2d12d72d82dc2e12f22f830330530a30c31931b3223263"
    "2832c34134834b35135835a3693903943973a43a63c13c33c83ca3d13dd3e13f23f840040140340540740840a40c40e411413417"
    "41841a42142342542842a43743843b43d44044244844b44f45245545945c46246948148448749149349849f4a14ab4af4b94bc4c"
    "04c24c54c94d24d44d94db4e24e84f650150751051351a51d52153a53d54454955255f56056b5785805825875915ad5b15c55c95"
    "d65d85e35e860260960b60d60f61261961b61d62262462762963363964164364564c65165366067067a67e68068a69069a69c6a8"
    "6c16c86cc6d16d36d76d86e16e36e76ed6fb70370970e71271972a73073474174874a75575a76476e77b78e7a17c17c37d07d27d"
    "d80080480a81081481781a82182883884284784984b85285885d86386986d88188388888d89189b8a08af8b28b88c48c98cb8d08"
    "d28d98dd90090291491f92093994594795197298b99c9b09c89cd9d89e39e9a02a08a0ca12a20a24a27a2aa36a3ca41a43a45a4a"
    "a51a5aa7aa80a89a93a98a9eaabac2ac7ac8ad7ae4ae9af5afbb01b04b10b1ab26b4ab56b69b6bba2bc2bc4bd2c09c0bc0dc19c1"
    "bc30c40c50c57c74c8ac9cca2cadcb2cb8cc0ccccd1ce0d15d23d32d40d43d5cd70d85da0dc9dcbe00e04e07e10e12e1ee20e2ce"
    "32e42e49e54e63e65e81e84e88e8ee91e98ea9ec2edaeddeebf01f05f0bf10f28f52f62f82f99fc0")
IQ2_S_GRID = (
    "0000000200050008000a001100140016001900200022002500280041004400460049005000520055005800610064006600690080"
    "0082008500880091009400a000a500aa010101040106010901100112011501180121012401400142014501480151015401560159"
    "0160016501680181018401900192019501a101a40200020202050208021102140220022a02410244024602490250025502800285"
    "028a029402a20401040404060409041004120415041804210424042604290440044204450448044a045104540456045904600462"
    "0465048104840486048904900495049804a104a40500050205050508050a05110514051605190520052505280541054405460549"
    "05500552055505580561056405800582058505880591059405a00601060406060609061006150640064506480651065406600681"
    "068406900800080208050808081108140816081908200825082a0841084408460849085008520855085808610864088008850894"
    "08aa0901090409100912091509180921094009450948095109540960098109900a000a110a140a220a280a2a0a500a9910011004"
    "10061009101010121015101810211024102610401042104510481051105410561059106010621065106810811084108610901095"
    "109810a110a41100110211051108110a111111141116111911201122112511281141114411461149115011521155115811611164"
    "11801182118511881191119412011204120912101215122112241240124512511254128112841290140014021405140814111414"
    "14161419142014251428144114441446144914501452145514581461146414801482148514881491149414a01501150415061509"
    "15101512151515181521152415401542154515481551155415601581158415901600160516081611161416201641164416501680"
    "16aa1801180418061809181018151818182118401842184518481851185418601881188419001902190519081911191419201941"
    "19441950196919a21a041a101a401a562000200220052008201120142016201920202025202a2041204420502052205520642080"
    "208a209420aa2101210421102112211521212140214221452151215421602181218421902200220a22222228222a224422502288"
    "228a22a8240124042406240924102415241824212424244024422445244824512454246024812484249025002505250825112514"
    "252025412544255025662580260126042610264026592800280528112814284128442850288a28aa29012904291029952a0a2a22"
    "2a642a882a8a40014004400640094010401240154018401a4021402440264040404240454048404a405140544056405940604062"
    "40654081408440904095409840a140a4410041024105410841114114411641194120412241254141414441464149415041524155"
    "41584161416441804182418541884191419441a04201420442104212421542184224424042454248425142544260428142844400"
    "440244054408440a4411441444164419442044224425442844414444444644494450445244554458446144644480448244854488"
    "4491449444a045014504450645094510451245154518452145244540454245454548455145544560456a45814584459046004602"
    "46054608461146144620464146444650468046a54801480448094810481248154818482148244840484248454848485148544860"
    "488448904900490249054908491149144920494149444950498049964a014a044a104a4050005002500550085011501450165019"
    "50205022502550285041504450465049505050525055505850615064508050825085508850915094510151045106510951105112"
    "51155118512151245140514251455148515151545160518151845190520052055208521152145220524152445250526952805401"
    "54045406540954105412541554185421542454405442544554485451545454605481548454905500550255055508551155145520"
    "5541554455505580560156045610562656405800580258055808581158145820584158445850585a588059015904591059405a00"
    "5a195a855aa860016004600660106012601560186021602460406045604860516054606060846090610061026105610861116114"
    "612061416144615061806199620462106240625662a164006405640864116414642064416444645064806501650465106540654a"
    "6568659266006694680168046810686568986900692a6a426aa18000800280058008801180148019802080258041804480508052"
    "805580588061808080858091809481018104810981108112811581188121812481408142814581488151815481818184819081a9"
    "82008205820a82118214824182448250840184048406840984108412841584188421844084428445844884518454846084818484"
    "849085008502850585088511851485208541854485508580858a86018604861086298640880088058811881488418844885088a2"
    "89018904894089658a228a588a5a8a828aa290019004900990109012901590189024904090429045904890519054906090819084"
    "90909100910591119114914191449150915a920192049210924092a6940094029405940894119414942094419444945094809496"
    "9501950495109540959895a19600964696649801980498109826984098a99900994999529a90a000a005a00aa014a022a02aa041"
    "a044a050a0a2a0aaa140a165a202a20aa222a228a22aa282a288a28aa2a8a401a404a410a440a489a4a4a500a519a651a80aa828"
    "a8a2a954a986aa08aa0aaa20aa22aa28aa88aaaa")


def row_bytes(dtype: int, n: int) -> int:
    if dtype in SCALARS:
        return n * (4 if dtype == F32 else 2)
    return n // BLOCKS[dtype][0] * BLOCKS[dtype][1]


def random_rows(gen, dtype: int, n_rows: int, in_dim: int):
    """GGUF rows on the device: uint8 [n_rows, row_bytes]."""
    rms = 1.0 / math.sqrt(in_dim)
    if dtype in SCALARS:
        w = torch.randn(n_rows, in_dim, generator=gen, device="cuda") * rms
        return w.to(SCALARS[dtype]).view(torch.uint8).reshape(n_rows, -1)
    elems, nbytes, d_off, unit = BLOCKS[dtype]
    n = n_rows * in_dim // elems
    raw = torch.randint(0, 256, (n, nbytes), generator=gen, device="cuda", dtype=torch.uint8)
    offs = (d_off, d_off + 2) if dtype == Q2_K else (d_off,)
    for off in offs:
        d = torch.exp(0.3 * torch.randn(n, generator=gen, device="cuda")) * (rms / unit)
        raw[:, off:off + 2] = d.half().view(torch.uint8).reshape(n, 2)
    return raw.reshape(n_rows, -1)


def activations(gen, *shape):
    x = torch.randn(*shape, generator=gen, device="cuda")
    x[..., ::64] *= 8.0
    return x


def _grid(text: str, digits: int, values: int, bits: int, levels):
    """[entries, values] codebook from its packed text."""
    codes = np.array([int(text[i:i + digits], 16) for i in range(0, len(text), digits)], np.int64)
    lv = np.array(levels, np.int64)
    return np.stack([lv[(codes >> (bits * j)) & ((1 << bits) - 1)] for j in range(values)], 1)


_GRIDS: dict = {}


def grid(dtype: int):
    if dtype not in _GRIDS:
        g = {IQ3_XXS: lambda: _grid(IQ3_XXS_GRID, 3, 4, 3, IQ3_LEVELS),
             IQ3_S: lambda: _grid(IQ3_S_GRID, 3, 4, 3, range(1, 16, 2)),
             IQ2_S: lambda: _grid(IQ2_S_GRID, 4, 8, 2, IQ2_LEVELS),
             IQ4_XS: lambda: np.array(IQ4_LEVELS, np.int64)}[dtype]()
        _GRIDS[dtype] = torch.from_numpy(g).cuda()
    return _GRIDS[dtype]


def _d16(b, off: int):
    return b[:, off:off + 2].contiguous().view(torch.float16).double()


def _bits(v, n: int):
    """The low n bits of every value, as a last axis."""
    return (v.unsqueeze(-1) >> torch.arange(n, device=v.device)) & 1


def decode_blocks(dtype: int, raw):
    """float64 [blocks, weights] of uint8 [blocks, bytes]."""
    n = raw.shape[0]
    b = raw.long()
    if dtype == Q8_0:
        return _d16(raw, 0) * raw[:, 2:].contiguous().view(torch.int8).double()
    if dtype == Q6_K:
        ql, qh = b[:, :128].reshape(n, 2, 1, 2, 32), b[:, 128:192].reshape(n, 2, 1, 1, 32)
        hi2 = torch.arange(2, device=raw.device).reshape(1, 1, 2, 1, 1)  # quarters 2, 3: high nibbles
        lo2 = torch.arange(2, device=raw.device).reshape(1, 1, 1, 2, 1)
        v = ((ql >> (4 * hi2)) & 15) | (((qh >> (4 * hi2 + 2 * lo2)) & 3) << 4)
        sc = raw[:, 192:208].contiguous().view(torch.int8).double().reshape(n, 16, 1)
        return (_d16(raw, 208).reshape(n, 1, 1) * sc * (v - 32).double().reshape(n, 16, 16)).reshape(n, 256)
    if dtype in (Q2_K, Q3_K):
        j = torch.arange(4, device=raw.device).reshape(1, 1, 4, 1)
        qs = (b[:, 16:80] if dtype == Q2_K else b[:, 32:96]).reshape(n, 2, 1, 32)
        code = (qs >> (2 * j)) & 3
        if dtype == Q2_K:
            sc = b[:, :16].reshape(n, 16, 1)
            dl = _d16(raw, 80).reshape(n, 1, 1) * (sc & 15).double()
            ml = _d16(raw, 82).reshape(n, 1, 1) * (sc >> 4).double()
            # (the weight is rounded to float32 where the minimum is taken off)
            return (dl * code.double().reshape(n, 16, 16) - ml).float().double().reshape(n, 256)
        half = torch.arange(2, device=raw.device).reshape(1, 2, 1, 1)
        hbit = (b[:, :32].reshape(n, 1, 1, 32) >> (4 * half + j)) & 1
        v = code - 4 * (1 - hbit)
        low = torch.cat([b[:, 96:104] & 15, b[:, 96:104] >> 4], 1)
        top = torch.cat([(b[:, 104:108] >> s) & 3 for s in (0, 2, 4, 6)], 1)
        dl = _d16(raw, 108) * ((low | (top << 4)) - 32).double()
        return (dl.reshape(n, 16, 1) * v.double().reshape(n, 16, 16)).reshape(n, 256)
    if dtype == IQ4_XS:
        sh = (b[:, 2] | (b[:, 3] << 8)).unsqueeze(1)
        ib = torch.arange(8, device=raw.device)
        low = torch.stack([b[:, 4:8] & 15, b[:, 4:8] >> 4], 2).reshape(n, 8)
        ls = (low | (((sh >> (2 * ib)) & 3) << 4)) - 32
        q = b[:, 8:].reshape(n, 8, 16)
        v = grid(IQ4_XS)[torch.cat([q & 15, q >> 4], 2)]
        return ((_d16(raw, 0) * ls.double()).unsqueeze(2) * v.double()).reshape(n, 256)
    if dtype == IQ3_XXS:
        aux = b[:, 66:].reshape(n, 8, 4)
        aux = aux[..., 0] | (aux[..., 1] << 8) | (aux[..., 2] << 16) | (aux[..., 3] << 24)
        s7 = (aux.unsqueeze(2) >> (7 * torch.arange(4, device=raw.device))) & 127
        sg = _bits(s7, 7)
        sg = torch.cat([sg, sg.sum(-1, keepdim=True) & 1], -1).reshape(n, 8, 32)  # even parity
        v = grid(IQ3_XXS)[b[:, 2:66]].reshape(n, 8, 32)
        db = _d16(raw, 0) * (0.25 * (2 * (aux >> 28) + 1).double())
        return (db.unsqueeze(2) * (v * (1 - 2 * sg)).double()).reshape(n, 256)
    if dtype == IQ3_S:
        idx = b[:, 2:66] | (_bits(b[:, 66:74], 8).reshape(n, 64) << 8)
        sg = _bits(b[:, 74:106], 8).reshape(n, 8, 32)
        s = torch.stack([b[:, 106:] & 15, b[:, 106:] >> 4], 2).reshape(n, 8)
        v = grid(IQ3_S)[idx].reshape(n, 8, 32) * (1 - 2 * sg)
        return ((_d16(raw, 0) * (2 * s + 1).double()).unsqueeze(2) * v.double()).reshape(n, 256)
    if dtype == IQ2_S:
        qh = (b[:, 66:74].unsqueeze(2) >> (2 * torch.arange(4, device=raw.device))) & 3
        v = grid(IQ2_S)[b[:, 2:34] | (qh.reshape(n, 32) << 8)].reshape(n, 16, 16)
        sg = _bits(b[:, 34:66], 8).reshape(n, 16, 16)
        s = torch.stack([b[:, 74:] & 15, b[:, 74:] >> 4], 2).reshape(n, 16)
        dl = _d16(raw, 0) * (0.125 * (2 * s + 1).double())
        return (dl.unsqueeze(2) * (v * (1 - 2 * sg)).double()).reshape(n, 256)
    raise ValueError(dtype)


def decode_rows(dtype: int, rows, in_dim: int):
    """float64 [n_rows, in_dim] of GGUF rows."""
    if dtype in SCALARS:
        return rows.contiguous().view(SCALARS[dtype]).double().reshape(-1, in_dim)
    blocks = rows.reshape(-1, BLOCKS[dtype][1])
    step = 1 << 17
    return torch.cat([decode_blocks(dtype, blocks[i:i + step]) for i in range(0, blocks.shape[0], step)]).reshape(
        -1, in_dim)


# ---- the cases -------------------------------------------------------------------------------------

HIDDEN, INTER, EXPERT_INTER = 6144, 12288, 2048
LIMIT = 10.0


def listed():
    return [
        # One decode token through the absorbed per-head projections of attention: the smallest call of
        # a layer, a few microseconds of work.
        {"name": "heads_1tok", "kind": "heads", "heads": 64, "in": 256, "rows": 512},
        # One decode token through a latent projection, by name through the store.
        {"name": "q_a_1tok", "kind": "product", "dtype": "iq3_xxs", "tokens": 1, "in": HIDDEN, "rows": 1536, "row0": 0},
        # One decode token through a dense layer's MLP.
        {"name": "dense_mlp_1tok", "kind": "dense_mlp", "hidden": HIDDEN, "inter": INTER},
        # One decode token through an attention tensor the file keeps in six bits.
        {"name": "q6_k_1tok", "kind": "product", "dtype": "q6_k", "tokens": 1, "in": HIDDEN, "rows": HIDDEN, "row0": 0},
        # A decode batch of 20 sequences through an attention tensor kept in eight bits.
        {"name": "q8_0_20tok", "kind": "product", "dtype": "q8_0", "tokens": 20, "in": HIDDEN, "rows": HIDDEN,
         "row0": 0},
        # A ragged prefill chunk through a three-bit tensor that is not IQ3_XXS.
        {"name": "q3_k_509tok", "kind": "product", "dtype": "q3_k", "tokens": 509, "in": HIDDEN, "rows": HIDDEN,
         "row0": 0},
        # Continuous batching: 64 tokens through the batched MLP with the two latent projections of the
        # same activations.
        {"name": "mlp_64tok", "kind": "mlp", "hidden": HIDDEN, "inter": INTER, "tokens": 64, "x": "f32",
         "extra": "576,1536"},
        # A prefill chunk with bf16 activations through one dense projection.
        {"name": "gemm_bf16_512tok", "kind": "gemm", "tokens": 512, "in": HIDDEN, "rows": INTER},
        # A long ragged prompt with fp32 activations through one dense projection, by name.
        {"name": "up_1999tok", "kind": "product", "dtype": "iq3_xxs", "tokens": 1999, "in": HIDDEN, "rows": INTER,
         "row0": 0},
        # The routed step with its shared expert: one sequence, a decode batch, a prefill chunk.
        {"name": "moe_1tok", "kind": "moe", "tokens": 1, "experts": 64, "top_k": 8, "hidden": HIDDEN,
         "inter": EXPERT_INTER, "shared": True, "mode": 0},
        {"name": "moe_32tok", "kind": "moe", "tokens": 32, "experts": 64, "top_k": 8, "hidden": HIDDEN,
         "inter": EXPERT_INTER, "shared": True, "mode": 0},
        {"name": "moe_512tok", "kind": "moe", "tokens": 512, "experts": 64, "top_k": 8, "hidden": HIDDEN,
         "inter": EXPERT_INTER, "shared": True, "mode": 1},
    ]


def _log(rng, lo: int, hi: int) -> int:
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    kind = rng.choice(["product", "product", "product", "heads", "dense_mlp", "mlp", "gemm", "moe", "moe"])
    if kind == "product":
        dtype = rng.choice(["iq3_xxs", "iq3_xxs", "iq3_xxs"] + list(DTYPES))
        tokens = 1 if rng.random() < 0.25 else _log(rng, 1, 1024)
        small = dtype in ("q8_0", "f16", "bf16", "f32")  # formats with blocks of 32 or less: any multiple of 32
        in_dim = 32 * _log(rng, 16, 384) if small else 256 * _log(rng, 2, 48)
        rows = _log(rng, 64, 256) if dtype == "f32" else _log(rng, 64, 12288)
        row0 = 0 if rng.random() < 0.5 else rng.randrange(1, 257)
        return {"kind": kind, "dtype": dtype, "tokens": tokens, "in": in_dim, "rows": rows, "row0": row0}
    if kind == "heads":
        return {"kind": kind, "heads": _log(rng, 8, 128), "in": 256 * rng.randint(1, 3), "rows": 64 * rng.randint(2, 8)}
    if kind == "dense_mlp":
        return {"kind": kind, "hidden": 256 * _log(rng, 4, 32), "inter": 256 * _log(rng, 4, 48)}
    if kind == "mlp":
        extra = rng.choice(["", "576,1536", str(_log(rng, 64, 2048))])
        return {"kind": kind, "hidden": 256 * _log(rng, 4, 24), "inter": 256 * _log(rng, 4, 48),
                "tokens": _log(rng, 2, 512), "x": rng.choice(["f32", "bf16"]), "extra": extra}
    if kind == "gemm":
        return {"kind": kind, "tokens": _log(rng, 9, 2048), "in": 256 * _log(rng, 4, 24), "rows": _log(rng, 64, 12288)}
    experts = rng.choice([8, 16, 32, 64])
    return {"kind": "moe", "tokens": _log(rng, 1, 512), "experts": experts,
            "top_k": rng.randint(2, min(8, experts // 2)), "hidden": 256 * _log(rng, 4, 24),
            "inter": 256 * _log(rng, 2, 8), "shared": rng.random() < 0.7, "mode": rng.randint(0, 1)}


def _extra(case) -> list:
    return [int(v) for v in case["extra"].split(",") if v]


def _inputs(case, seed: int) -> dict:
    """The weights as GGUF rows and the activations, from the seed alone."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    k = case["kind"]
    if k == "product":
        dtype = DTYPES[case["dtype"]]
        return {"w": random_rows(gen, dtype, case["row0"] + case["rows"], case["in"]),
                "x": activations(gen, case["tokens"], case["in"])}
    if k == "heads":
        return {"w": random_rows(gen, IQ3_XXS, case["heads"] * case["rows"], case["in"]),
                "x": activations(gen, case["heads"], case["in"])}
    if k == "gemm":
        return {"w": random_rows(gen, IQ3_XXS, case["rows"], case["in"]),
                "x": activations(gen, case["tokens"], case["in"]).bfloat16()}
    if k in ("dense_mlp", "mlp"):
        h, i = case["hidden"], case["inter"]
        d = {"gate": random_rows(gen, IQ3_XXS, i, h), "up": random_rows(gen, IQ3_XXS, i, h),
             "down": random_rows(gen, IQ3_XXS, h, i)}
        if k == "dense_mlp":
            d["x"] = activations(gen, h)
            return d
        d["extra"] = [random_rows(gen, IQ3_XXS, r, h) for r in _extra(case)]
        x = activations(gen, case["tokens"], h)
        d["x"] = x.bfloat16() if case["x"] == "bf16" else x
        return d
    e, h, i = case["experts"], case["hidden"], case["inter"]
    d = {"gate": random_rows(gen, IQ3_XXS, e * i, h), "up": random_rows(gen, IQ3_XXS, e * i, h),
         "down": random_rows(gen, IQ3_XXS, e * h, i)}
    if case["shared"]:
        d["shared"] = [random_rows(gen, IQ3_XXS, r, c) for r, c in ((i, h), (i, h), (h, i))]
    d["x"] = activations(gen, case["tokens"], h)
    d["logits"] = torch.randn(case["tokens"], e, generator=gen, device="cuda")
    d["bias"] = 0.1 * torch.randn(e, generator=gen, device="cuda") if case["mode"] == 0 else None
    return d


def prepare(case, seed: int) -> dict:
    d = _inputs(case, seed)
    k, x = case["kind"], d["x"]
    s = {"case": case, "x": x}
    f32 = dict(dtype=torch.float32, device="cuda")
    if k == "product":
        s["store"] = G.WeightStore()
        s["store"].add("w", d["w"], case["in"], case["row0"] + case["rows"], DTYPES[case["dtype"]])
        if case["tokens"] == 1:
            s["x"] = x[0]
    elif k == "heads":
        n = case["heads"] * case["rows"]
        s["w"] = G.tile(d["w"], n, case["in"])
        s["out"] = torch.empty(case["heads"], case["rows"], **f32)
        s["ws"] = G.gemv_workspace(case["in"], n)
    elif k == "gemm":
        s["w"] = G.tile(d["w"], case["rows"], case["in"])
        s["out"] = torch.empty(case["tokens"], case["rows"], **f32)
        n = G.lib().gpeed_iq3xxs_gemm_ws_bytes(case["tokens"], case["in"], case["rows"], G.X_BF16)
        s["ws"] = G.ws_init(torch.empty(max(n, 256), dtype=torch.uint8, device="cuda"))
    elif k in ("dense_mlp", "mlp"):
        h, i = case["hidden"], case["inter"]
        s.update(gate=G.tile(d["gate"], i, h), up=G.tile(d["up"], i, h), down=G.tile(d["down"], h, i))
        if k == "dense_mlp":
            s["out"] = torch.empty(h, **f32)
            s["ws"] = G.dense_mlp_workspace(h, i)
        else:
            dims = _extra(case)
            s["extra"] = [(G.tile(w, r, h), r) for w, r in zip(d["extra"], dims)]
            s["out"] = torch.empty(case["tokens"], h, **f32)
            s["extra_out"] = [torch.empty(case["tokens"], r, **f32) for r in dims]
            s["ws"] = G.mlp_gemm_workspace(case["tokens"], h, i, G.X_BF16 if case["x"] == "bf16" else G.X_F32, dims)
    else:
        e, h, i = case["experts"], case["hidden"], case["inter"]
        s.update(gate=G.tile(d["gate"], e * i, h), up=G.tile(d["up"], e * i, h), down=G.tile(d["down"], e * h, i),
                 logits=d["logits"], bias=d["bias"], shared=None)
        if case["shared"]:
            g, u, dn = d["shared"]
            s["shared"] = (G.tile(g, i, h), G.tile(u, i, h), G.tile(dn, h, i))
        s["out"] = torch.empty(case["tokens"], h, **f32)
        s["ws"] = G.moe_batch_workspace(case["tokens"], e, case["top_k"], h, i, case["shared"])
    return s


def run(s):
    c = s["case"]
    k = c["kind"]
    if k == "product":
        if c["tokens"] == 1:
            return s["store"].matvec_quant("w", c["row0"], c["in"], c["rows"], s["x"])
        return s["store"].matmul_quant("w", c["row0"], c["in"], c["rows"], s["x"], c["tokens"])
    if k == "heads":
        return G.matvec_heads(s["w"], c["heads"] * c["rows"], 0, c["in"], c["rows"], s["x"], out=s["out"], ws=s["ws"])
    if k == "gemm":
        return G.gemm(s["w"], c["rows"], 0, c["in"], c["rows"], s["x"], out=s["out"], ws=s["ws"])
    if k == "dense_mlp":
        return G.dense_mlp(s["gate"], s["up"], s["down"], c["hidden"], c["inter"], s["x"], limit=LIMIT, out=s["out"],
                           ws=s["ws"])
    if k == "mlp":
        y, extra = G.mlp_gemm(s["gate"], s["up"], s["down"], c["hidden"], c["inter"], s["x"], limit=LIMIT,
                              extra=s["extra"], out=s["out"], extra_out=s["extra_out"], ws=s["ws"])
        return [y, *extra]
    return G.moe_batch(s["logits"], s["x"], s["gate"], s["up"], s["down"], c["experts"], c["hidden"], c["inter"],
                       c["top_k"], mode=c["mode"], bias=s["bias"], swiglu_limit=LIMIT, shared=s["shared"], out=s["out"],
                       ws=s["ws"])


def work(case) -> dict:
    k = case["kind"]
    if k == "product":
        t, n, m = case["tokens"], case["in"], case["rows"]
        return {"bytes": m * row_bytes(DTYPES[case["dtype"]], n) + 4 * t * (n + m), "flops": 2 * t * n * m}
    if k == "heads":
        h, n, m = case["heads"], case["in"], case["rows"]
        return {"bytes": h * (m * row_bytes(IQ3_XXS, n) + 4 * (n + m)), "flops": 2 * h * n * m}
    if k == "gemm":
        t, n, m = case["tokens"], case["in"], case["rows"]
        return {"bytes": m * row_bytes(IQ3_XXS, n) + t * (2 * n + 4 * m), "flops": 2 * t * n * m}
    h, i = case["hidden"], case["inter"]
    mlp_bytes = 2 * i * row_bytes(IQ3_XXS, h) + h * row_bytes(IQ3_XXS, i)
    if k == "dense_mlp":
        return {"bytes": mlp_bytes + 8 * h, "flops": 6 * h * i}
    t = case["tokens"]
    if k == "mlp":
        r = sum(_extra(case))
        x_bytes = (4 if case["x"] == "f32" else 2) * h
        return {"bytes": mlp_bytes + r * row_bytes(IQ3_XXS, h) + t * (x_bytes + 4 * (h + r)),
                "flops": 2 * t * h * (3 * i + r)}
    e, kk = case["experts"], case["top_k"]
    touched = e * (1.0 - (1.0 - kk / e) ** t)  # experts that get a token, on average
    sh = 1 if case["shared"] else 0
    return {"bytes": int((touched + sh) * mlp_bytes) + t * (8 * h + 4 * e), "flops": 6 * t * (kk + sh) * h * i}


def tolerance(case) -> dict:
    # float32 results against float64, measured over the listed and 100 drawn cases and stated about four
    # times over (weights and activations are exact operands; the float32 sums and the 22 bits that the
    # matrix path keeps of a float32 activation are what differs). Largest rel / max seen:
    k = case["kind"]
    if k == "heads":
        return {"rel": 4e-7, "max": 2e-6}  # 8.9e-8 / 4.9e-7
    if k == "dense_mlp":
        return {"rel": 8e-7, "max": 4e-6}  # 1.9e-7 / 7.7e-7
    if k == "gemm":
        return {"rel": 1.5e-6, "max": 1.5e-5}  # 3.4e-7 / 3.8e-6
    if k == "mlp":
        return {"rel": 2.5e-6, "max": 1.5e-5}  # 6.3e-7 / 3.3e-6
    if k == "moe":
        return {"rel": 3.5e-6, "max": 2.5e-5}  # 8.3e-7 / 5.6e-6
    if case["dtype"] == "iq3_xxs":
        return {"rel": 2e-6, "max": 2.5e-5}  # 5.2e-7 / 6.4e-6
    return {"rel": 7e-6, "max": 5e-5}  # 1.8e-6 / 1.2e-5


# ---- float64 ---------------------------------------------------------------------------------------


def _swiglu(g, u):
    g = torch.clamp(g, max=LIMIT)
    return g * torch.sigmoid(g) * torch.clamp(u, -LIMIT, LIMIT)


def _mlp64(gate, up, down, h: int, i: int, x):
    g = x @ decode_rows(IQ3_XXS, gate, h).T
    u = x @ decode_rows(IQ3_XXS, up, h).T
    return _swiglu(g, u) @ decode_rows(IQ3_XXS, down, i).T


def exact(case, seed: int):
    d = _inputs(case, seed)
    k, x = case["kind"], d["x"].double()
    if k in ("product", "gemm"):
        dtype = DTYPES[case["dtype"]] if k == "product" else IQ3_XXS
        rows = d["w"][case.get("row0", 0):]
        # (row slices: the float64 weights of the largest tensors a few hundred MB at a time)
        y = torch.cat([x @ decode_rows(dtype, r, case["in"]).T for r in rows.split(2048)], 1)
        return y[0] if k == "product" and case["tokens"] == 1 else y
    if k == "heads":
        w = decode_rows(IQ3_XXS, d["w"], case["in"]).reshape(case["heads"], case["rows"], case["in"])
        return (w * x.unsqueeze(1)).sum(2)
    h, i = case["hidden"], case["inter"]
    if k == "dense_mlp":
        return _mlp64(d["gate"], d["up"], d["down"], h, i, x.unsqueeze(0))[0]
    if k == "mlp":
        return [_mlp64(d["gate"], d["up"], d["down"], h, i, x)] + [x @ decode_rows(IQ3_XXS, w, h).T for w in d["extra"]]
    top_k, logits = case["top_k"], d["logits"]
    if case["mode"] == 0:
        # sigmoid router: ranked by score + bias, weights normalised over the selected scores
        score = torch.sigmoid(logits.double())
        sel = torch.topk(score + d["bias"].double(), top_k, dim=1).indices
        wt = torch.gather(score, 1, sel)
        wt = wt / (1e-20 + wt.sum(1, keepdim=True))
    else:
        top = torch.topk(logits.double(), top_k, dim=1)
        sel, wt = top.indices, torch.softmax(top.values, 1)
    y = torch.zeros(x.shape[0], h, dtype=torch.float64, device="cuda")
    for e in range(case["experts"]):
        t, slot = torch.nonzero(sel == e, as_tuple=True)
        if t.numel():
            out = _mlp64(*(d[n].chunk(case["experts"])[e] for n in ("gate", "up", "down")), h, i, x[t])
            y.index_add_(0, t, out * wt[t, slot].unsqueeze(1))
    if case["shared"]:
        y += _mlp64(*d["shared"], h, i, x)
    return y
