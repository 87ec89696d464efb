"""Performance cases: what a program that uses this library has it do.

listed() and draw() name the cases, prepare() makes a case's inputs on the GPU
from a seed, run() is one pass through the public entry points, work() the
bytes and operations a pass cannot do without, exact() the same result in
64 bits by plain torch, tolerance() what two correct implementations at the
same precision may differ by.

The inputs are synthetic and structured as a video model's K/V are: a row is a
shared center plus a decaying rank-64 residual plus noise.  The histories are
quantised here by plain torch, so a case's inputs do not depend on the
library's own encoder.
"""
from __future__ import annotations

import math

import torch

from nanokv_amd import codec_native, nanokv_codec, ops, synth

DEV = "cuda"
F64 = torch.float64
BF16 = torch.bfloat16
FRAME = 1560            # tokens per latent frame (a 30 x 52 grid)
GRID = (30, 52)


# ---------------------------------------------------------------- the cases
def listed() -> list:
    return [
        # config 0: one layer of a small 8-head model of 64-wide heads, a
        # short history: the smallest attention call a user makes
        dict(name="attend_d64_small", kind="attend", H=8, D=64, N=2048, Q=256, Nc=256, rK=64,
             rV=64, G=32, sdt="fp16", C=16, mean=False),
        # the payload-level call early in a rollout, through the cache a
        # backbone keeps: four committed segments (the last one ragged), each
        # with its own 64 centers, one bf16 scale per row
        dict(name="attend_segments", kind="segments", H=16, D=128, seglen=780, N=2757, Q=417,
             r=256, C=64),
        # config 1: one layer over 8 frames of history
        dict(name="attend_8_frames", kind="attend", H=24, D=128, N=12480, Q=1560, Nc=1560,
             rK=384, rV=384, G=32, sdt="fp16", C=256, mean=False),
        # config 2: the longest history, unequal ranks, 16-bit center ids
        dict(name="attend_long", kind="attend", H=24, D=128, N=49920, Q=780, Nc=780, rK=384,
             rV=256, G=32, sdt="fp16", C=1024, mean=False),
        # config 3: NanoKV-Fast with read-time RoPE and the camera
        dict(name="fast_rope_camera", kind="fast", H=24, D=128, N=12480, Q=1560, r=384, G=32,
             C=256, recent=2, d=32),
        # the commit of a chunk's K and V against shared centers, bf16 rows
        # read in place from the QKV projection's output (config 4's step)
        dict(name="encode_chunk", kind="encode_batch", HD=3072, rows=1560, r=384, G=32, C=256),
        # the commit as the codec API does it by default: centers fitted to
        # the chunk, bf16 quantiser, one scale per row
        dict(name="encode_fitted", kind="encode_tensor", B=1, HD=3072, rows=1560, r=384),
        # fp32 rows against a large shared table with 16-bit ids (config 2)
        dict(name="encode_1024_centers", kind="encode", HD=3072, rows=780, r=384, G=32, C=1024),
        # full decode of a segmented cache (the reference's own read path)
        dict(name="decode_cache", kind="decode_value", HD=3072, seglen=1560, N=12480, r=384, C=64),
        # decode of selected rows: a protected set, scattered, odd count
        dict(name="decode_rows", kind="decode_rows", HD=2048, N=6240, rows=1017, r=256, G=32,
             C=256),
        # a chunk's q, k and v before attention: RoPE on q and k, the camera
        # on all three
        dict(name="rope_camera_qkv", kind="transforms", H=24, S=1560),
        # the merge of a two-branch backbone: its low-dimensional history
        # output lifted to full width and merged by log-sum-exp
        dict(name="lift_merge", kind="lift", B=1, H=16, Q=1560, low=64),
    ]


def _logint(rng, lo: int, hi: int) -> int:
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng) -> dict:
    """One more case: the kinds above over the sizes, ranks, scale groups and
    center counts that their callers use, odd ones among them."""
    kind = rng.choice(["attend", "attend", "attend", "segments", "fast", "encode_batch",
                       "encode_tensor", "encode", "decode_value", "decode_rows", "transforms",
                       "lift"])
    ranks = [64, 128, 256, 384]             # the attention calls' ranks
    if kind == "attend":
        D = rng.choice([128, 128, 128, 64])
        H = rng.choice([8, 16, 24])
        rK, rV = rng.choice(ranks), rng.choice(ranks)
        # history and queries such that the call is no larger than attend_long
        N = _logint(rng, 64, 49920)
        Q = _logint(rng, 32, max(32, min(1560, int(780 * 49920 / N))))
        return dict(kind=kind, H=H, D=D, N=N, Q=Q, Nc=rng.choice([Q, 0]), rK=rK, rV=rV,
                    G=rng.choice([32, 64]), sdt=rng.choice(["fp16", "bf16"]),
                    C=rng.choice([16, 64, 256, 1024]), mean=rng.random() < 0.5)
    if kind == "segments":
        return dict(kind=kind, H=rng.choice([16, 24]), D=128, seglen=rng.choice([390, 780, 1560]),
                    N=_logint(rng, 390, 12480), Q=_logint(rng, 32, 1560), r=rng.choice(ranks),
                    C=rng.choice([64, 256]))
    if kind == "fast":
        frames = rng.randint(3, 8)
        return dict(kind=kind, H=24, D=128, N=FRAME * frames, Q=_logint(rng, 64, 1560), r=384,
                    G=32, C=256, recent=rng.randint(1, 2), d=rng.choice([32, 64]))
    HD = rng.choice([2048, 3072])
    r = rng.choice(ranks + [192, 320])      # the codec takes any multiple of 32
    if kind == "encode_batch":
        return dict(kind=kind, HD=HD, rows=_logint(rng, 32, 3120), r=r,
                    G=rng.choice([32, 64]), C=rng.choice([64, 256]))
    if kind == "encode_tensor":
        return dict(kind=kind, B=rng.choice([1, 1, 2]), HD=HD, rows=_logint(rng, 96, 3120), r=r)
    if kind == "encode":
        return dict(kind=kind, HD=HD, rows=_logint(rng, 32, 3120), r=r, G=rng.choice([32, 64]),
                    C=rng.choice([256, 512, 1024]))
    if kind == "decode_value":
        return dict(kind=kind, HD=HD, seglen=rng.choice([390, 780, 1560]),
                    N=_logint(rng, 100, 12480), r=r, C=rng.choice([64, 256]))
    if kind == "decode_rows":
        N = _logint(rng, 390, 12480)
        return dict(kind=kind, HD=HD, N=N, rows=_logint(rng, 16, N), r=r, G=rng.choice([32, 64]),
                    C=rng.choice([64, 256, 1024]))
    if kind == "transforms":
        return dict(kind=kind, H=rng.choice([16, 24]), S=_logint(rng, 32, 3120))
    return dict(kind="lift", B=rng.choice([1, 2]), H=rng.choice([8, 16, 24]),
                Q=_logint(rng, 32, 1560), low=rng.choice([32, 64, 96]))


# ---------------------------------------------------------------- inputs
class _Maker:
    """Seeded random tensors on the GPU, and the codec inputs made of them."""

    def __init__(self, seed: int):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(seed)

    def randn(self, *shape):
        return torch.randn(*shape, generator=self.g, device=DEV)

    def randint(self, hi, n):
        return torch.randint(0, hi, (n,), generator=self.g, device=DEV)

    def centers(self, C, HD):
        return self.randn(C, HD).to(BF16)

    def operator(self, HD, r):
        """(encoder [r, HD], decoder [HD, r]): a random decoder and its
        least-squares inverse."""
        dec = self.randn(HD, r) / r ** 0.5
        return ((dec.T * (r / HD)).to(BF16).contiguous(), dec.to(BF16).contiguous())

    def basis(self, HD):
        q, _ = torch.linalg.qr(self.randn(HD, 64).cpu())
        return q.T.contiguous().to(DEV)

    def residual(self, n, basis):
        decay = torch.arange(1, 65, device=DEV, dtype=torch.float32).rsqrt()
        return (self.randn(n, 64) * decay) @ basis

    def rows(self, n, centers):
        """n structured K or V rows [n, HD], bf16."""
        HD = centers.shape[1]
        x = self.residual(n, self.basis(HD)) + 0.05 * self.randn(n, HD)
        return (x + centers.float()[self.randint(centers.shape[0], n)]).to(BF16)

    def codes(self, n, enc, G, sdt):
        """Packed INT4 codes [n, r/2] and group scales [n, r/G] of n residual
        rows' coefficients: those of `residual` plus the noise through the
        encoder, formed at rank width."""
        r, HD = enc.shape
        e = enc.float()
        coeff = self.residual(n, self.basis(HD) @ e.T)
        coeff = coeff + 0.05 * self.randn(n, r) * e.square().sum(1).sqrt()
        x = coeff.view(n, r // G, G)
        s = x.abs().amax(-1, keepdim=True).clamp_min(2.0 ** -23) / 7
        q = (torch.round(x / s).clamp(-7, 7) + 7).to(torch.uint8).view(n, r)
        return ((q[:, 0::2] | (q[:, 1::2] << 4)).contiguous(),
                s.view(n, r // G).to(sdt).contiguous())

    def codec(self, N, HD, r, G, sdt, C, mean=False):
        cent = self.centers(C, HD)
        enc, dec = self.operator(HD, r)
        packed, scales = self.codes(N, enc, G, sdt)
        m = 0.1 * self.randn(HD) if mean else None
        ids = self.randint(C, N).to(ops.id_dtype_for(C))
        return ops.Codec(packed=packed[None], scales=scales[None], w_dec=dec, group=G,
                         ids=ids[None], centers=cent[None], mean=m)

    def bthd(self, n, H, D, centers):
        return self.rows(n, centers).view(1, n, H, D)

    def payload(self, kind, layer, n, HD, enc, C):
        """One committed segment as the codec API stores it: its own bf16
        centers, one bf16 scale per row."""
        r = enc.shape[0]
        packed, scales = self.codes(n, enc, r, BF16)
        return {"codec": nanokv_codec.CODEC, "kind": kind, "layer": layer, "shape": (1, n, HD),
                "latent_shape": (1, n, r), "latent_numel": n * r,
                "packed_codes": packed.reshape(-1), "scale": scales[None],
                "centers": self.centers(C, HD)[None], "ids": self.randint(C, n).to(torch.uint8)[None],
                "semantic": True, "source_dtype": "bfloat16", "scale_group": r,
                "scale_dtype": "bf16", "id_dtype": "uint8", "shared_centers": False}

    def cache(self, kind, layer, N, seglen, HD, r, C):
        enc, dec = self.operator(HD, r)
        mean = 0.1 * self.randn(HD)
        nanokv_codec.register_operator(kind, layer, encoder=enc, decoder=dec, mean=mean)
        value = None
        for s in range(0, N, seglen):
            value = nanokv_codec.concat_values(
                value, self.payload(kind, layer, min(seglen, N - s), HD, enc, C))
        return value


def _layer(seed: int) -> int:
    """The layer whose operators a state registers (one per seed, so that
    several states can be held at once)."""
    return int(seed) % 1000003


def _sdt(case):
    return torch.float16 if case["sdt"] == "fp16" else BF16


def prepare(case, seed):
    mk = _Maker(seed)
    k = case["kind"]
    st = {"kind": k, "case": case, "layer": _layer(seed)}
    if k == "attend":
        H, D, HD = case["H"], case["D"], case["H"] * case["D"]
        for w, r in (("key", case["rK"]), ("value", case["rV"])):
            st[w] = mk.codec(case["N"], HD, r, case["G"], _sdt(case), case["C"], case["mean"])
        st["q"] = (mk.randn(1, case["Q"], H, D) * (2.0 / D ** 0.5)).to(BF16)
        st["kc"] = st["vc"] = None
        if case["Nc"]:
            st["kc"] = mk.bthd(case["Nc"], H, D, st["key"].centers[0])
            st["vc"] = mk.bthd(case["Nc"], H, D, st["value"].centers[0])
        need = ops.attend_workspace_size(st["q"], case["N"], case["Nc"], st["key"], st["value"])
        st["ws"] = torch.empty(max(need, 1), device=DEV, dtype=torch.uint8)
    elif k == "segments":
        H, D, HD = case["H"], case["D"], case["H"] * case["D"]
        for w, kind in (("k", "k"), ("v", "v")):
            st[w] = mk.cache(kind, st["layer"], case["N"], case["seglen"], HD, case["r"], case["C"])
        st["q"] = (mk.randn(1, H, case["Q"], D) * (2.0 / D ** 0.5)).to(BF16)
        cent = mk.centers(case["C"], HD)
        # [B, T, H*D] projections viewed as [B, H, T, D], as a backbone has them
        st["kc"] = mk.bthd(case["Q"], H, D, cent).permute(0, 2, 1, 3)
        st["vc"] = mk.bthd(case["Q"], H, D, cent).permute(0, 2, 1, 3)
    elif k == "fast":
        _prepare_fast(case, mk, st)
    elif k == "encode_batch":
        qkv = torch.empty(case["rows"], 3 * case["HD"], device=DEV, dtype=BF16)
        qkv[:, :case["HD"]] = mk.randn(case["rows"], case["HD"]).to(BF16)
        st["p"] = []
        for i in (1, 2):
            cent = mk.centers(case["C"], case["HD"])
            sl = qkv[:, i * case["HD"]:(i + 1) * case["HD"]]
            sl.copy_(mk.rows(case["rows"], cent))
            st["p"].append({"x": sl, "w_enc": mk.operator(case["HD"], case["r"])[0],
                            "centers": cent})
    elif k == "encode_tensor":
        enc, dec = mk.operator(case["HD"], case["r"])
        st["mean"] = 0.1 * mk.randn(case["HD"])
        st["enc"] = enc
        nanokv_codec.register_operator("k", st["layer"], encoder=enc, decoder=dec, mean=st["mean"])
        x = mk.rows(case["B"] * case["rows"], mk.centers(48, case["HD"]))
        st["x"] = x.view(case["B"], case["rows"], case["HD"])
    elif k == "encode":
        st["cent"] = mk.centers(case["C"], case["HD"])
        st["x"] = mk.rows(case["rows"], st["cent"]).float()
        st["enc"] = mk.operator(case["HD"], case["r"])[0]
    elif k == "decode_value":
        st["v"] = mk.cache("v", st["layer"], case["N"], case["seglen"], case["HD"], case["r"],
                           case["C"])
    elif k == "decode_rows":
        st["codec"] = mk.codec(case["N"], case["HD"], case["r"], case["G"], torch.float16,
                               case["C"])
        perm = torch.randperm(case["N"], generator=mk.g, device=DEV)[:case["rows"]]
        st["rows"] = perm.sort().values.to(torch.int32)
    elif k == "transforms":
        H, S = case["H"], case["S"]
        frames = -(-S // FRAME)
        cent = mk.centers(64, H * 128)
        for w in ("q", "k", "v"):
            st[w] = mk.bthd(S, H, 128, cent)
        st["rope"] = ops.Rope.from_bands(ops.rope_bands(128), range(8, 8 + frames), *GRID,
                                         torch.device(DEV))
        P, P_T, P_inv = synth.camera_matrices(4, seed=seed)
        fm = (torch.arange(frames, dtype=torch.int32) % 4).to(DEV)
        st["P_T"] = ops.Camera(P_T.to(DEV), fm, FRAME)
        st["P_inv"] = ops.Camera(P_inv.to(DEV), fm, FRAME)
    elif k == "lift":
        B, H, Q, low = case["B"], case["H"], case["Q"], case["low"]
        st["native"] = mk.randn(2 * B, H, Q, 128).to(BF16)
        st["low"] = mk.randn(2 * B, H, Q, low).to(BF16)
        st["main"] = (mk.randn(H, low, 128) / low ** 0.5).to(BF16)
        st["mix"] = (mk.randn(H, low // 4, 32) / (low / 4) ** 0.5).to(BF16)
        st["nl"] = mk.randn(2 * B, H, Q) + 7
        st["hl"] = mk.randn(2 * B, H, Q) + 8
    torch.cuda.synchronize()
    return st


def _prepare_fast(case, mk, st):
    H, D, N, Q, r, d = (case[x] for x in ("H", "D", "N", "Q", "r", "d"))
    frames = N // FRAME
    key = mk.codec(N, H * D, r, case["G"], torch.float16, case["C"])
    val = mk.codec(N, H * D, r, case["G"], torch.float16, case["C"])
    sh = synth.Shape("fast", H=H, D=D, N=N, Q=Q, Nc=Q, rK=r, rV=r, G=case["G"], C=case["C"])
    lay = synth.Layer(key.centers[0], val.centers[0], None, key.w_dec, None, val.w_dec)
    payload = synth.make_readers(sh, lay, seed=_layer(st["layer"]), d=d)
    reader = codec_native.ReaderLayer(payload, torch.device(DEV))
    q_pre = (mk.randn(1, Q, H, D) * (2.0 / D ** 0.5)).to(BF16)
    kc, vc = mk.bthd(Q, H, D, key.centers[0]), mk.bthd(Q, H, D, val.centers[0])
    bands = ops.rope_bands(D)
    dev = torch.device(DEV)
    rope = ops.Rope.from_bands(bands, range(frames), *GRID, dev)
    q_rope = ops.Rope.from_bands(bands, [frames], *GRID, dev)
    P, P_T, P_inv = (m.to(DEV) for m in synth.camera_matrices(4, seed=7))
    fm = (torch.arange(frames, dtype=torch.int32) % 4).to(DEV)
    qf = torch.tensor([frames % 4], dtype=torch.int32, device=DEV)
    cam, q_cam, o_cam = (ops.Camera(P_inv, fm, FRAME), ops.Camera(P_T, qf, FRAME),
                         ops.Camera(P, qf, FRAME))
    c_cam = ops.Camera(P_inv, qf, FRAME)
    # the native partition's operands, transformed as the backbone hands them over
    q = ops.camera_apply(ops.rope_apply(q_pre, q_rope), q_cam)
    kc = ops.camera_apply(ops.rope_apply(kc, q_rope), c_cam)
    vc = ops.camera_apply(vc, c_cam)
    protect = synth.fast_protect_mask(sh, recent=case["recent"], device=DEV)
    st.update(key=key, value=val, payload=payload, q=q, kc=kc, vc=vc,
              groups=[g.tensors(rope=True, camera=True) for g in reader.groups],
              prot=torch.nonzero(protect).flatten().to(torch.int32),
              low=torch.nonzero(~protect).flatten().to(torch.int32),
              kw=dict(rope=rope, q_pre=q_pre, q_rope=q_rope, camera=cam, q_camera=q_cam,
                      out_camera=o_cam))
    need = ops.fast_attend_workspace_size(q, kc, vc, key, val, st["prot"], st["low"],
                                          st["groups"], **st["kw"])
    st["ws"] = torch.empty(max(need, 1), device=DEV, dtype=torch.uint8)


# ---------------------------------------------------------------- one pass
def run(st):
    k, case = st["kind"], st["case"]
    if k == "attend":
        return ops.attend(st["q"], st["kc"], st["vc"], st["key"], st["value"],
                          workspace=st["ws"])
    if k == "segments":
        return codec_native.codec_history_attention(st["q"], st["k"], st["v"], st["kc"],
                                                    st["vc"], return_lse=True)
    if k == "fast":
        return ops.fast_attend(st["q"], st["kc"], st["vc"], st["key"], st["value"], st["prot"],
                               st["low"], st["groups"], workspace=st["ws"], **st["kw"])
    if k == "encode_batch":
        out = ops.encode_batch(st["p"], group=case["G"], scale_dtype=torch.float16)
        return [e[n] for e in out for n in ("packed", "scales", "ids", "coeff")]
    if k == "encode_tensor":
        p = nanokv_codec.encode_tensor("k", st["layer"], st["x"])
        return [p["packed_codes"], p["scale"], p["centers"], p["ids"]]
    if k == "encode":
        e = ops.encode(st["x"], st["enc"], centers=st["cent"], group=case["G"],
                       scale_dtype=torch.float16)
        return [e[n] for n in ("packed", "scales", "ids", "coeff")]
    if k == "decode_value":
        return nanokv_codec.decode_value(st["v"], dtype=BF16, device=torch.device(DEV))
    if k == "decode_rows":
        return ops.decode(st["codec"], case["HD"], row_index=st["rows"])
    if k == "transforms":
        q = ops.camera_apply(ops.rope_apply(st["q"], st["rope"]), st["P_T"])
        kk = ops.camera_apply(ops.rope_apply(st["k"], st["rope"]), st["P_inv"])
        return q, kk, ops.camera_apply(st["v"], st["P_inv"])
    return ops.lift_lse_combine(st["native"], st["nl"], st["low"], st["main"], st["mix"],
                                st["hl"])


# ---------------------------------------------------------------- work
def work(case):
    k = case["kind"]
    if k in ("attend", "segments"):
        H, D, N, Q = case["H"], case["D"], case["N"], case["Q"]
        HD = H * D
        Nc = case.get("Nc", Q)
        rK, rV = case.get("rK", case.get("r")), case.get("rV", case.get("r"))
        tables = case["C"] * (1 if k == "attend" else -(-N // case["seglen"]))
        idb = 1 if case["C"] <= 256 else 2
        b = 2 * HD * 2 * Q + 4 * H * Q + 2 * 2 * HD * Nc + 4 * HD * min(tables, N)
        for r in (rK, rV):
            b += N * (r // 2 + 2 * (r // case.get("G", r)) + idb) + 2 * HD * r
        return {"bytes": b, "flops": 4 * Q * (N + Nc) * HD + 2 * N * (rK + rV) * HD}
    if k == "fast":
        H, D, N, Q, r, d, C = (case[x] for x in ("H", "D", "N", "Q", "r", "d", "C"))
        sh = synth.Shape("fast", H=H, D=D, N=N, Q=Q, Nc=Q, rK=r, rV=r, G=case["G"], C=C)
        f = sh.fast_flops(min(N, FRAME * case["recent"]), d=d)["total"]
        b = 3 * 2 * H * D * Q + 2 * 2 * H * D * Q + 4 * H * Q
        b += 2 * (N * (r // 2 + 2 * (r // case["G"]) + 1) + 2 * H * D * r + 2 * C * H * D)
        return {"bytes": b, "flops": int(f)}
    if k in ("encode_batch", "encode", "encode_tensor"):
        n, HD, r = case["rows"], case["HD"], case["r"]
        C, B = case.get("C", 64), case.get("B", 1)
        G = case.get("G", r)
        xb = 4 if k == "encode" else 2
        idb = 1 if C <= 256 else 2
        one = n * HD * xb + n * (r // 2 + 2 * (r // G) + idb) + 2 * C * HD
        if k != "encode_tensor":
            one += 4 * n * r
        flops = 2 * n * HD * (r + C)
        if k == "encode_tensor":
            # two search and two update rounds of the fit, then the projection
            flops = 2 * n * HD * r + 2 * (2 * n * HD * C + n * HD)
        times = 2 if k == "encode_batch" else B
        wts = 2 * r * HD * (2 if k == "encode_batch" else 1)
        return {"bytes": times * one + wts, "flops": times * flops}
    if k in ("decode_value", "decode_rows"):
        N, HD, r = case["N"], case["HD"], case["r"]
        n = case.get("rows", N)
        tables = case["C"] * (-(-N // case["seglen"]) if k == "decode_value" else 1)
        idb = 1 if case["C"] <= 256 else 2
        b = n * (r // 2 + 2 * (r // case.get("G", r)) + idb + 2 * HD) + 2 * HD * r
        return {"bytes": b + 2 * HD * min(tables, n), "flops": 2 * n * r * HD}
    if k == "transforms":
        elems = case["H"] * 128 * case["S"]
        return {"bytes": 6 * 2 * elems, "flops": 2 * 3 * elems + 3 * 7 * elems}
    rows = 2 * case["B"] * case["H"] * case["Q"]
    low = case["low"]
    return {"bytes": rows * (2 * 128 * 2 + 2 * low + 8) + 2 * case["H"] * low * (128 + 8),
            "flops": rows // 2 * (2 * low * 128 + 2 * (low // 4) * 128) + rows * 128 * 4}


# ---------------------------------------------------------------- tolerances
def tolerance(case):
    k = case["kind"]
    if k in ("attend", "segments", "fast"):
        return _TOL["attend"]
    if k in ("encode_batch", "encode"):
        return _TOL["encode"]
    return _TOL[k if k in _TOL else "decode"]


# About four times the difference between run() and exact() on the listed and
# drawn cases, whose size each comment gives.
_TOL = {
    # bf16 K, V and probabilities, fp32 sums, bf16 output: 1.8e-3 .. 2.4e-3
    "attend": {"rel": 1e-2},
    # fp16 scales 2.1e-4, fp32 coefficients 1.6e-7; a code differs only where
    # its fp32 value sits at a rounding tie
    "encode": {"rel": 8e-4, "differ": 1e-4},
    # bf16 scales of bf16-rounded coefficients 2.4e-3, bf16 centers 1.7e-3; a
    # tie moves a row's scale by 2^-8 and some of its codes with it
    "encode_tensor": {"rel": 1e-2, "differ": 2e-3},
    # bf16 rounding after the GEMM, after the mean and after the center: 1.7e-3
    "decode": {"rel": 7e-3},
    # two roundings to bf16: 2.3e-3
    "transforms": {"rel": 1e-2},
    # fp32 sums, one rounding to bf16: 1.7e-3
    "lift": {"rel": 7e-3},
}


# ---------------------------------------------------------------- 64 bits
def _latent64(packed, scales, r, G):
    """code * scale of [n, r/2] codes and [n, r/G] scales."""
    p = packed.reshape(-1, r // 2)
    q = torch.stack((p & 15, p >> 4), -1).reshape(-1, r).to(F64) - 7
    return (q.view(-1, r // G, G) * scales.reshape(-1, r // G, 1).to(F64)).view(-1, r)


def _decode64(c, rows=None, cols=slice(None), w=None):
    """K or V rows of a codec in 64 bits: latent W^T + mean + center."""
    r = c.w_dec.shape[1]
    sel = slice(None) if rows is None else rows.long()
    out = _latent64(c.packed[0][sel], c.scales[0][sel], r, c.group) @ c.w_dec[cols].to(F64).T
    if c.mean is not None:
        out += c.mean[cols].to(BF16).to(F64)
    return out + c.centers[0][:, cols].to(F64)[c.ids[0][sel].long()]


def _payload64(value, cols=slice(None)):
    outs = []
    for p in nanokv_codec.segments_of(value):
        op = nanokv_codec._operator(p["kind"], p["layer"], torch.device(DEV))
        r = p["latent_shape"][2]
        x = _latent64(p["packed_codes"], p["scale"], r, p["scale_group"])
        x = x @ op["decoder"][cols].to(F64).T + op["mean"][cols].to(BF16).to(F64)
        outs.append(x + p["centers"][0][:, cols].to(F64)[p["ids"][0].long()])
    return torch.cat(outs)


def _attend64(q, k, v, scale):
    """[Q, D] queries over [N, D] keys: (out, lse)."""
    s = (q.to(F64) @ k.to(F64).T) * scale
    lse = torch.logsumexp(s, 1)
    return torch.exp(s - lse[:, None]) @ v.to(F64), lse


def _rope64(x, freqs):
    """x [S, ..., 2P] rotated by freqs [S, P]."""
    c = torch.view_as_complex(x.to(F64).reshape(*x.shape[:-1], -1, 2).contiguous())
    f = freqs.view(freqs.shape[0], *([1] * (c.dim() - 2)), freqs.shape[1])
    return torch.view_as_real(c * f).flatten(-2)


def _freqs(rope, rows):
    """[rows, D/2] complex128 of codec rows 0 .. rows."""
    t, h, w = (torch.view_as_complex(x) for x in (rope.cs_t, rope.cs_h, rope.cs_w))
    n = torch.arange(rows, device=DEV)
    per = rope.grid_h * rope.grid_w
    return torch.cat([t[rope.frame_pos.long()[n // per]], h[n % per // rope.grid_w],
                      w[n % rope.grid_w]], 1)


def _mats64(cam, rows):
    """[rows, 4, 4, 4] bf16-rounded matrices of rows 0 .. rows."""
    f = torch.arange(rows, device=DEV) // cam.tokens_per_frame
    return cam.mats[0].to(BF16).to(F64)[cam.frame_mat.long()[f]]


def _cam64(x, mats, blocks=None):
    """x [S, ..., 8 nb]: block j's even and odd dims each a 4-vector times
    sub-frame blocks[j] (default j % 4) of mats [S, 4, 4, 4]."""
    nb = x.shape[-1] // 8
    sub = torch.arange(nb, device=DEV) % 4 if blocks is None else blocks.long()
    y = x.to(F64).reshape(x.shape[0], -1, nb, 4, 2)
    m = mats[:, sub]                                           # [S, nb, 4, 4]
    return (m[:, None, :, :, :, None] * y[:, :, :, None]).sum(4).reshape(x.shape)


def _fast64(st):
    case = st["case"]
    H, D, N, Q = case["H"], case["D"], case["N"], case["Q"]
    kw = st["kw"]
    kf, qf = _freqs(kw["rope"], N), _freqs(kw["q_rope"], Q)
    km, qm, om = _mats64(kw["camera"], N), _mats64(kw["q_camera"], Q), _mats64(kw["out_camera"], Q)
    scale = D ** -0.5
    prot, low = st["prot"].long(), st["low"].long()
    out = torch.empty(1, Q, H, D, device=DEV, dtype=F64)
    lse = torch.empty(1, H, Q, device=DEV, dtype=F64)
    for g in st["payload"]["groups"]:
        for i, h in enumerate(g["heads"].tolist()):
            cols = slice(h * D, (h + 1) * D)
            k = _cam64(_rope64(_decode64(st["key"], prot, cols), kf[prot]), km[prot])
            v = _cam64(_decode64(st["value"], prot, cols), km[prot])
            k = torch.cat([k, st["kc"][0, :, h].to(F64)])
            v = torch.cat([v, st["vc"][0, :, h].to(F64)])
            o1, l1 = _attend64(st["q"][0, :, h], k, v, scale)
            m = {n: g[n][i].to(DEV).to(BF16).to(F64)
                 for n in ("q_reduce", "k_read", "v_read", "k_affine", "v_affine")}
            pairs = g["indices"][i].to(DEV)[::2] // 2
            blocks = g["indices"][i].to(DEV)[::8] // 8 % 4
            ql = _rope64(kw["q_pre"][0, :, h].to(F64) @ m["q_reduce"], qf[:, pairs])
            ql = _cam64(ql, qm, blocks)

            def low_rows(c, read, affine):
                lat = _latent64(c.packed[0][low], c.scales[0][low], c.w_dec.shape[1], c.group)
                cent = c.centers[0][:, cols].to(F64) @ affine
                return lat @ read.T + cent[c.ids[0][low].long()]
            kl = _cam64(_rope64(low_rows(st["key"], m["k_read"], m["k_affine"]),
                                kf[low][:, pairs]), km[low], blocks)
            vl = _cam64(low_rows(st["value"], m["v_read"], m["v_affine"]), km[low])
            o2, l2 = _attend64(ql, kl, vl, scale)
            l = torch.logaddexp(l1, l2)
            o = o1 * torch.exp(l1 - l)[:, None] + o2 * torch.exp(l2 - l)[:, None]
            out[0, :, h] = _cam64(o, om)
            lse[0, h] = l
    return [out, lse]


def _residual64(x, cent, ids, mean=None):
    """The encoder's bf16 residual rows (the operand its operator is applied
    to), as 64-bit values."""
    res = x.float() - cent.float()[ids]
    if mean is not None:
        res = res - mean
    return res.to(BF16).to(F64)


def _scales64(coeff, G):
    s = coeff.view(-1, coeff.shape[-1] // G, G).abs().amax(-1) / 7
    return s.clamp_min(2.0 ** -23 / 7)


def _nearest64(x, cent):
    c = cent.to(F64)
    return (c.square().sum(1) - 2 * (x.to(F64) @ c.T)).argmin(1)


def _encode64(x, enc, cent, G):
    ids = _nearest64(x, cent)
    coeff = _residual64(x, cent, ids) @ enc.to(F64).T
    return [None, _scales64(coeff, G), ids, coeff]


def _fit64(x, layer):
    """Two rounds of labels and means from the API's seeded draw of rows."""
    S = x.shape[0]
    g = torch.Generator(device="cpu").manual_seed(20260804 + layer)
    cent = x[torch.randperm(S, generator=g)[:64].to(DEV)].float()
    for _ in range(2):
        ids = _nearest64(x, cent)
        n = torch.bincount(ids, minlength=64)
        total = torch.zeros(64, x.shape[1], device=DEV, dtype=F64).index_add_(0, ids, x.to(F64))
        mean = total / n.clamp_min(1)[:, None]
        cent = torch.where(n[:, None] > 0, mean.float(), cent)
    return cent, ids


def exact(case, seed):
    st = prepare(case, seed)
    k = case["kind"]
    if k in ("attend", "segments"):
        H, D, Q = case["H"], case["D"], case["Q"]
        seg = k == "segments"
        out = torch.empty(Q, H, D, device=DEV, dtype=F64)
        lse = torch.empty(1, H, Q, device=DEV, dtype=F64)
        for h in range(H):
            cols = slice(h * D, (h + 1) * D)
            if seg:
                kk, vv = _payload64(st["k"], cols), _payload64(st["v"], cols)
                q, kc, vc = st["q"][0, h], st["kc"][0, h], st["vc"][0, h]
            else:
                kk, vv = _decode64(st["key"], cols=cols), _decode64(st["value"], cols=cols)
                q = st["q"][0, :, h]
                kc = vc = None
                if st["kc"] is not None:
                    kc, vc = st["kc"][0, :, h], st["vc"][0, :, h]
            if kc is not None:
                kk, vv = torch.cat([kk, kc.to(F64)]), torch.cat([vv, vc.to(F64)])
            out[:, h], lse[0, h] = _attend64(q, kk, vv, D ** -0.5)
        return [(out.permute(1, 0, 2) if seg else out)[None], lse]
    if k == "fast":
        return _fast64(st)
    if k == "encode_batch":
        return [o for p in st["p"] for o in _encode64(p["x"], p["w_enc"], p["centers"], case["G"])]
    if k == "encode":
        return _encode64(st["x"], st["enc"], st["cent"], case["G"])
    if k == "encode_tensor":
        fits = [_fit64(x, st["layer"]) for x in st["x"]]
        scales = []
        for x, (cent, ids) in zip(st["x"], fits):
            res = _residual64(x, cent.to(BF16), ids, st["mean"])
            scales.append(_scales64(res @ st["enc"].to(F64).T, case["r"]))
        return [None, torch.stack(scales), torch.stack([c.to(F64) for c, _ in fits]),
                torch.stack([i for _, i in fits])]
    if k == "decode_value":
        return _payload64(st["v"])[None]
    if k == "decode_rows":
        return _decode64(st["codec"], st["rows"])[None]
    if k == "transforms":
        S = case["S"]
        f = _freqs(st["rope"], S)
        mt, mi = _mats64(st["P_T"], S), _mats64(st["P_inv"], S)
        return [_cam64(_rope64(st["q"][0], f), mt)[None], _cam64(_rope64(st["k"][0], f), mi)[None],
                _cam64(st["v"][0], mi)[None]]
    B, H, Q, low = case["B"], case["H"], case["Q"], case["low"]
    lo = st["low"].to(F64)
    main = lo[:B] @ st["main"].to(F64)
    quart = lo[B:].reshape(B, H, Q, low // 4, 4).transpose(-1, -2)          # [.., c, k]
    mixed = (quart @ st["mix"].to(F64)[:, None]).transpose(-1, -2).reshape(B, H, Q, 128)
    hist = torch.cat([main, mixed])
    w = torch.sigmoid(st["hl"].to(F64) - st["nl"].to(F64))[..., None]
    return st["native"].to(F64) * (1 - w) + hist * w
