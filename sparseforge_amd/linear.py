"""Masked linear + SLoRB as autograd functions over the sf_gemm MFMA engine.

Reference: legacy/sparse_modeling.py:56-132 (FusedMaskedLinearSTE) and
:737-796 (SparseLinear.forward with the SLoRB pair of F.linear).

    z  = x P^T                                    (SLoRB projection, [T, r])
    y  = x (W.E.s)^T + z S^T + b                  (one GEMM: the z S^T term is a second K segment)
    dz = dy S
    dx = dy (W.E) + dz P                          (one GEMM, two K segments; no s, as in :113-115)
    dW = dy^T x  (+ decay W [E < 0.5])            (STE: the mask does not enter dW, :120-125)
    db = sum_t dy,  dS = dy^T z,  dP = dz^T x

The backward is itself an autograd Function whose backward is written with
the same kernels, so torch.autograd.grad(..., create_graph=True) and the
Hutchinson Hessian-vector product (legacy/utils.py:772-795) work through it.
SLoRB ranks that are not a multiple of the 16-byte vector width are padded
with zero rows/columns of P and S, which leaves every product unchanged.
"""
from __future__ import annotations

import ctypes

import torch
from torch.autograd import forward_ad

from . import _lib as L
from . import kernels as K
from . import profiling as _prof


# ---------------------------------------------------------------------------
# GEMM front end
# ---------------------------------------------------------------------------
def _vec(dtype: torch.dtype) -> int:
    return 8 if dtype == torch.bfloat16 else 4


def gemm(M, N, A1, B1, K1, a_layout, b_layout, *, A2=None, B2=None, K2=0, bmask=None, bscale=1.0, bias=None,
         emask=None, dw=None, decay=0.0, out=None, out_dtype=None, accumulate=False, bmask_t=None) -> torch.Tensor:
    """C[M, N] = A1 . B1'^T (+ A2 . B2^T) on the device.

    a_layout: L.LAYOUT_K (A1 is [M, K]) or L.LAYOUT_MN (A1 is [K, M]);
    b_layout: L.LAYOUT_K (B1 is [N, K]) or L.LAYOUT_MN (B1 is [K, N]).
    bmask: effective mask of B1 in B1's dtype (multiplied in), or a uint8
    and-mask (0x00 / 0xFF per element) for a 0/1 mask.
    bmask_t: optional K-major copy [N, K] of a uint8 bmask of an N-contiguous
    B1 (transpose_u8(bmask)); the bf16 kernel then copies the mask with the
    weight tile instead of staging both through registers.
    """
    dev = L.require_device(A1, B1, A2, B2, bmask, bias, emask, dw, out, bmask_t)
    dt = A1.dtype
    # the checks run on every product of a step: inline comparisons, the message built only on a mismatch
    a_k, b_k = a_layout == L.LAYOUT_K, b_layout == L.LAYOUT_K
    b1_shape = (N, K1) if b_k else (K1, N)
    if A1.shape != ((M, K1) if a_k else (K1, M)):
        _bad_shape("A1", A1, (M, K1) if a_k else (K1, M))
    if B1.shape != b1_shape:
        _bad_shape("B1", B1, b1_shape)
    if bmask is not None and bmask.shape != b1_shape:
        _bad_shape("bmask", bmask, b1_shape)
    if K2:
        if A2 is None or B2 is None:
            raise ValueError("gemm: K2 > 0 needs A2 and B2")
        if A2.shape != ((M, K2) if a_k else (K2, M)):
            _bad_shape("A2", A2, (M, K2) if a_k else (K2, M))
        if B2.shape != ((N, K2) if b_k else (K2, N)):
            _bad_shape("B2", B2, (N, K2) if b_k else (K2, N))
    if bias is not None and bias.shape != (N,):
        _bad_shape("bias", bias, (N,))
    for t, name in ((emask, "emask"), (dw, "dw"), (out, "out")):
        if t is not None and t.shape != (M, N):
            _bad_shape(name, t, (M, N))
    bmask_bytes = bmask is not None and bmask.dtype == torch.uint8
    for t in (B1, A2, B2, None if bmask_bytes else bmask, emask, dw):
        if t is not None and t.dtype != dt:
            raise TypeError(f"gemm: operand dtype {t.dtype} != {dt}")
    if bmask_bytes and bscale != 1.0:
        raise ValueError("gemm: a byte and-mask cannot carry a weight-scaling factor")
    if out is None:
        out = torch.empty(M, N, dtype=out_dtype or dt, device=dev)
    d = L.GemmDesc()
    d.dtype = L.dtype_code(A1)
    d.a_layout, d.b_layout = a_layout, b_layout
    d.M, d.N, d.K1, d.K2 = M, N, K1, K2
    d.A1, d.B1 = A1.data_ptr(), B1.data_ptr()
    d.lda1 = K1 if a_k else M
    d.ldb1 = K1 if b_k else N
    if K2:
        d.A2, d.B2 = A2.data_ptr(), B2.data_ptr()
        d.lda2, d.ldb2 = (K2 if a_k else M), (K2 if b_k else N)
    if bmask is not None:
        d.bmask = bmask.data_ptr()
        d.bmask_bytes = int(bmask_bytes)
        if (bmask_t is not None and bmask_bytes and not b_k and dt == torch.bfloat16
                and K1 % 16 == 0 and bmask_t.data_ptr() % 16 == 0):
            if bmask_t.shape != (N, K1):
                _bad_shape("bmask_t", bmask_t, (N, K1))
            if bmask_t.dtype != torch.uint8:
                raise TypeError("gemm: bmask_t must be a uint8 and-mask")
            d.bmask, d.bmask_kmajor, d.ldbm = bmask_t.data_ptr(), 1, K1
    d.bscale = bscale
    d.C, d.ldc, d.c_dtype = out.data_ptr(), N, L.dtype_code(out)
    if bias is not None:
        d.bias, d.bias_dtype = bias.data_ptr(), L.dtype_code(bias)
    if emask is not None:
        d.emask = emask.data_ptr()
    if dw is not None:
        d.dw, d.decay = dw.data_ptr(), decay
    if accumulate:
        d.accumulate = 1
    ref, lib = ctypes.byref(d), L.lib()
    ws_bytes = lib.sf_gemm_workspace_size(ref)
    ws = None
    if ws_bytes:  # split-K scratch from torch's caching allocator; the library never allocates
        ws = torch.empty(ws_bytes, dtype=torch.uint8, device=dev)
        d.workspace, d.workspace_bytes = ws.data_ptr(), ws_bytes
    with _prof.region("sf_gemm", 2.0 * M * N * (K1 + K2), "FLOP", dev):
        rc = lib.sf_gemm(ref, L.stream(dev))
    if rc != L.SF_OK:
        L.check(rc, "sf_gemm")
    return out


def _bad_shape(name, t, want):
    raise ValueError(f"gemm: {name} has shape {tuple(t.shape)}, expected {tuple(want)}")


def mm_nt(A, B, **kw):
    """A [M, K] . B [N, K]^T"""
    return gemm(A.shape[0], B.shape[0], A, B, A.shape[1], L.LAYOUT_K, L.LAYOUT_K, **kw)


def mm_nn(A, B, **kw):
    """A [M, K] . B [K, N]"""
    return gemm(A.shape[0], B.shape[1], A, B, A.shape[1], L.LAYOUT_K, L.LAYOUT_MN, **kw)


def mm_tn(A, B, **kw):
    """A [K, M]^T . B [K, N]"""
    return gemm(A.shape[1], B.shape[1], A, B, A.shape[0], L.LAYOUT_MN, L.LAYOUT_MN, **kw)


def column_sum(A: torch.Tensor, out_dtype: torch.dtype) -> torch.Tensor:
    dev = L.require_device(A)
    out = torch.empty(A.shape[1], dtype=out_dtype, device=dev)
    L.check(L.lib().sf_column_sum(L.ptr(A), L.dtype_code(A), A.shape[0], A.shape[1], L.ptr(out),
                                  L.dtype_code(out), L.stream(dev)), "sf_column_sum")
    return out


def effective_mask(mask: torch.Tensor, dtype: torch.dtype, mode: str, hx: float, hard_kind: int, hard_n: int,
                   hard_m: int = 4) -> torch.Tensor:
    """E = mask.to(dtype) ('soft'), (hx*mask + (1-hx)*hard(mask)).to(dtype) ('mix') or hard(mask) ('hard').

    With mode 'hard' and dtype torch.uint8 the result is a byte and-mask
    (0xFF kept, 0x00 pruned) that the GEMMs apply while staging W.
    """
    dev = L.require_device(mask)
    eff = torch.empty(mask.shape, dtype=dtype, device=dev)
    m = {"mix": L.EFF_MIX, "hard": L.EFF_HARD}.get(mode, L.EFF_SOFT)
    code = L.DT_U8 if dtype == torch.uint8 else L.dtype_code(eff)
    nbytes = mask.numel() * (mask.element_size() + eff.element_size())
    with _prof.region("sf_effective_mask", nbytes, "B", dev):
        L.check(L.lib().sf_effective_mask(L.ptr(mask), L.dtype_code(mask), L.ptr(eff), code,
                                          mask.shape[0], mask.shape[1], m, float(hx), hard_kind, hard_n, hard_m,
                                          L.stream(dev)), "sf_effective_mask")
    return eff


def effective_mask_given(mask: torch.Tensor, hard: torch.Tensor, dtype: torch.dtype, mode: str,
                         hx: float) -> torch.Tensor:
    """effective_mask with the hard projection passed in (the block hard types)."""
    dev = L.require_device(mask, hard)
    if hard.shape != mask.shape:
        raise ValueError("hard mask shape differs from the soft mask")
    eff = torch.empty(mask.shape, dtype=dtype, device=dev)
    m = {"mix": L.EFF_MIX, "hard": L.EFF_HARD}.get(mode, L.EFF_SOFT)
    code = L.DT_U8 if dtype == torch.uint8 else L.dtype_code(eff)
    nbytes = mask.numel() * (mask.element_size() + hard.element_size() + eff.element_size())
    with _prof.region("sf_effective_mask", nbytes, "B", dev):
        L.check(L.lib().sf_effective_mask_given(L.ptr(mask), L.dtype_code(mask), L.ptr(hard), L.dtype_code(hard),
                                                L.ptr(eff), code, mask.shape[0], mask.shape[1], m, float(hx),
                                                L.stream(dev)), "sf_effective_mask_given")
    return eff


def apply_mask(W: torch.Tensor, E: torch.Tensor, scale: float = 1.0) -> torch.Tensor:
    """(W * E).to(W dtype) [* scale, rounded again]: the masked weight the unmasked GEMMs read."""
    dev = L.require_device(W, E)
    if E.shape != W.shape:
        raise ValueError(f"mask shape {tuple(E.shape)} != weight shape {tuple(W.shape)}")
    out = torch.empty_like(W)
    code = L.DT_U8 if E.dtype == torch.uint8 else L.dtype_code(E)
    with _prof.region("sf_apply_mask", W.numel() * (2 * W.element_size() + E.element_size()), "B", dev):
        L.check(L.lib().sf_apply_mask(L.ptr(W), L.dtype_code(W), L.ptr(E), code, float(scale), L.ptr(out),
                                      W.shape[0], W.shape[1], L.stream(dev)), "sf_apply_mask")
    return out


_BAD24: dict = {}


def apply_mask_2to4(W: torch.Tensor, E: torch.Tensor):
    """Wm = W * E for a bf16 W and a byte and-mask E that keeps two of every four columns, plus
    the packed 2:4 form of Wm (values, index words), in one pass (sf_apply_mask_2to4).  Groups
    keeping more than two columns are only counted in a per-device device counter, never read
    here: the N:M hard projection with N = 2, M = 4 produces none."""
    dev = L.require_device(W, E)
    out_f, in_f = W.shape
    Wm = torch.empty_like(W)
    vals = torch.empty(out_f, in_f // 2, dtype=torch.bfloat16, device=dev)
    idx = torch.empty(out_f * in_f // 8, dtype=torch.uint8, device=dev)
    key = dev.index if dev.index is not None else torch.cuda.current_device()
    bad = _BAD24.get(key)
    if bad is None:
        bad = _BAD24[key] = torch.zeros(1, dtype=torch.int64, device=dev)
    with _prof.region("sf_apply_mask_2to4", W.numel() * 5 + vals.numel() * 2 + idx.numel(), "B", dev):
        L.check(L.lib().sf_apply_mask_2to4(L.ptr(W), L.ptr(E), out_f, in_f, L.ptr(Wm), L.ptr(vals), L.ptr(idx),
                                           L.ptr(bad), L.stream(dev)), "sf_apply_mask_2to4")
    return Wm, vals, idx


def gemm_2to4(x2: torch.Tensor, vals: torch.Tensor, idx: torch.Tensor, out_features: int, z=None, S=None,
              bias=None) -> torch.Tensor:
    """y [T, out] bf16 = x2 Wm^T (+ z S^T) (+ bias) with Wm packed 2:4 (sf_gemm_2to4_lowrank)."""
    dev = L.require_device(x2, vals, idx, z, S, bias)
    T, in_f = x2.shape
    y = torch.empty(T, out_features, dtype=torch.bfloat16, device=dev)
    r = 0 if z is None else z.shape[1]
    flops = 2.0 * T * out_features * (in_f + r)
    with _prof.region("sf_gemm_2to4", flops, "FLOP", dev):
        L.check(L.lib().sf_gemm_2to4_lowrank(L.ptr(x2), x2.stride(0), T, L.ptr(vals), L.ptr(idx), out_features,
                                             in_f, L.ptr(z), 0 if z is None else z.stride(0), L.ptr(S),
                                             0 if S is None else S.stride(0), r, L.ptr(bias),
                                             L.dtype_code(bias) if bias is not None else 0, L.ptr(y),
                                             L.dtype_code(y), y.stride(0), L.stream(dev)), "sf_gemm_2to4_lowrank")
    return y


def transpose_u8(E: torch.Tensor) -> torch.Tensor:
    """[rows, cols] uint8 -> its transpose [cols, rows] (sf_transpose_u8)."""
    dev = L.require_device(E)
    if E.dtype != torch.uint8 or E.dim() != 2:
        raise TypeError("transpose_u8 expects a 2-D uint8 tensor")
    out = torch.empty(E.shape[1], E.shape[0], dtype=torch.uint8, device=dev)
    with _prof.region("sf_transpose_u8", 2 * E.numel(), "B", dev):
        L.check(L.lib().sf_transpose_u8(L.ptr(E), E.shape[0], E.shape[1], L.ptr(out), L.stream(dev)),
                "sf_transpose_u8")
    return out


def decay_term(G: torch.Tensor, E: torch.Tensor | None, decay: float, out: torch.Tensor | None = None) -> torch.Tensor:
    """out (+)= decay * G * [E < 0.5] in G's dtype (E = None: nothing is pruned and the term is 0).

    The derivative along G of the SR-STE term decay * W * [E < 0.5] of the weight
    gradient (legacy/sparse_modeling.py:123-125), which is elementwise in W.  Off
    the paper's path (its decay is 0), so it is two device elementwise ops.
    """
    L.require_device(G, E, out)
    if out is None:
        out = torch.zeros_like(G)
    if E is None:
        return out
    if E.shape != G.shape or out.shape != G.shape:
        raise ValueError("decay_term: G, E and out must have one shape")
    pruned = (E == 0) if E.dtype == torch.uint8 else (E < 0.5)
    out.add_(G * pruned.to(G.dtype), alpha=float(decay))
    return out


def _as_values(E: torch.Tensor | None, dt: torch.dtype) -> torch.Tensor | None:
    """A byte and-mask as 0/1 values of dtype dt (for epilogue products); other masks unchanged."""
    if E is not None and E.dtype == torch.uint8:
        return (E != 0).to(dt)
    return E


def _cat_k(parts, dim: int):
    """The operands of one K segment side by side (None when there are none)."""
    if not parts:
        return None
    return parts[0] if len(parts) == 1 else torch.cat(parts, dim).contiguous()


def _pad_rank(P: torch.Tensor, S: torch.Tensor):
    """Zero-pad the SLoRB rank to a multiple of the vector width."""
    r = P.shape[0]
    v = _vec(P.dtype)
    rp = (r + v - 1) // v * v
    if rp == r:
        return P.contiguous(), S.contiguous(), r
    Pp = torch.zeros(rp, P.shape[1], dtype=P.dtype, device=P.device)
    Pp[:r] = P
    Sp = torch.zeros(S.shape[0], rp, dtype=S.dtype, device=S.device)
    Sp[:, :r] = S
    return Pp, Sp, r


def _opt(t):
    return t.contiguous() if t is not None else None


class _Unrecorded:
    """Stands in for a Function's ctx when its forward runs outside a graph: nothing is kept."""

    def save_for_backward(self, *tensors):
        pass

    def set_materialize_grads(self, value):
        pass


def plain_backward() -> bool:
    """Whether a backward pass runs with nothing that looks into it: no create_graph (grad mode is on then), no
    functorch transform (torch.func, vmap) and no forward-mode level, which a direct call would pass by."""
    return not (torch.is_grad_enabled() or forward_ad._current_level >= 0
                or torch._C._are_functorch_transforms_active())


def apply_in_backward(fn, *args):
    """fn.apply(*args) for the gradient Functions (whose backward the Hutchinson probe takes).  In a plain
    backward pass nothing records them, so their forward runs as it is, without the 20 us that an autograd
    Function's apply costs; elsewhere apply records, transforms or refuses them."""
    return fn.forward(_Unrecorded(), *args) if plain_backward() else fn.apply(*args)


# ---------------------------------------------------------------------------
# autograd
# ---------------------------------------------------------------------------
class _MaskedLinearBackward(torch.autograd.Function):
    """(gy, x, W, P, S, b?) -> (dx, dW, db, dP, dS); differentiable for the HVP."""

    @staticmethod
    def forward(ctx, gy, x, W, P, S, E, decay, has_bias, z_fwd=None, wm_fwd=None):
        has_slorb = P is not None
        # z = x P^T is kept from the forward; its dependence on x and P is
        # written out explicitly in backward(), so the cached copy is detached.
        z = (z_fwd if z_fwd is not None else mm_nt(x, P)) if has_slorb else None
        dz = mm_nn(gy, S) if has_slorb else None
        # dx = gy (W.E): the forward's masked weight when it kept one (no weight-scaling factor),
        # else rebuilt with one elementwise pass
        Wm = wm_fwd if wm_fwd is not None else (apply_mask(W, E) if E is not None else W)
        if has_slorb:
            dx = mm_nn(gy, Wm, A2=dz, B2=P, K2=P.shape[0])
        else:
            dx = mm_nn(gy, Wm)
        if decay != 0.0:
            dW = mm_tn(gy, x, emask=_as_values(E, W.dtype), dw=W, decay=decay)
        else:
            dW = mm_tn(gy, x)
        dS = mm_tn(gy, z) if has_slorb else None
        db = column_sum(gy, W.dtype) if has_bias else None
        dP = mm_tn(dz, x) if has_slorb else None
        # outputs that no derivative reaches (a probe of the weight gradients leaves dP, dS and db out) come to
        # backward() as None and cost no product; zeros made for them were multiplied through six products
        ctx.set_materialize_grads(False)
        # W.E stays for the double backward's d/d gy (gdx (W.E)^T), so that product runs unmasked
        ctx.save_for_backward(gy, x, W, P, S, E, z, dz, Wm if E is not None else None)
        del Wm
        ctx.decay = decay
        ctx.has_slorb = has_slorb
        return dx, dW, db, dP, dS

    @staticmethod
    def backward(ctx, g_dx, g_dW, g_db, g_dP, g_dS):
        gy, x, W, P, S, E, z, dz, Wm = ctx.saved_tensors
        T, out = gy.shape
        dt = gy.dtype
        g_dx, g_dW, g_db, g_dP, g_dS = (_opt(t) for t in (g_dx, g_dW, g_db, g_dP, g_dS))
        if not ctx.has_slorb:
            g_dP = g_dS = None
        # d/d gy = gdx (W.E)^T + x gdW^T + u S^T + z gdS^T + gdb with u = gdx P^T + x gdP^T: the
        # low-rank terms ride as one second K segment [u | z] . [S | gdS]^T of the first full-size
        # product; the second full-size product accumulates into its output in the output dtype
        # (as autograd sums gradient contributions)
        u = None
        if ctx.has_slorb:
            if g_dx is not None:
                u = mm_nt(g_dx, P)
                if g_dP is not None:
                    mm_nt(x, g_dP, out=u, accumulate=True)
            elif g_dP is not None:
                u = mm_nt(x, g_dP)
        la = _cat_k([t for t in (u, z if g_dS is not None else None) if t is not None], 1)
        lb = _cat_k([t for t, a in ((S, u), (g_dS, g_dS)) if a is not None], 1)
        seg = {"A2": la, "B2": lb, "K2": la.shape[1]} if la is not None else {}
        ggy = None
        if g_dx is not None:
            ggy = mm_nt(g_dx, Wm if Wm is not None else W, bias=g_db, **seg)
            if g_dW is not None:
                mm_nt(x, g_dW, out=ggy, accumulate=True)
        elif g_dW is not None:
            ggy = mm_nt(x, g_dW, bias=g_db, **seg)
        elif la is not None:
            ggy = mm_nt(la, lb, bias=g_db)
        if ggy is None and g_db is not None:
            ggy = g_db.expand(T, out).to(dt).contiguous()
        # d/dx = gy gdW + [w | dz] . [P ; gdP] with w = gy gdS (one GEMM, the low-rank part its
        # second K segment)
        w = mm_nn(gy, g_dS) if ctx.has_slorb and g_dS is not None else None
        ra = _cat_k([t for t in (w, dz if g_dP is not None else None) if t is not None], 1)
        rb = _cat_k([t for t, a in ((P, w), (g_dP, g_dP)) if a is not None], 0)
        gx = None
        if g_dW is not None:
            gx = mm_nn(gy, g_dW, **({"A2": ra, "B2": rb, "K2": ra.shape[1]} if ra is not None else {}))
        elif ra is not None:
            gx = mm_nn(ra, rb)
        # d/dW = (gy^T gdx) . E  (+ decay gdW [E < 0.5]: the SR-STE term decay W [E < 0.5] of dW is
        # elementwise in W, legacy/sparse_modeling.py:123-125)
        gW = mm_tn(gy, g_dx, emask=_as_values(E, W.dtype)) if g_dx is not None else None
        if ctx.decay != 0.0 and g_dW is not None:
            gW = decay_term(g_dW, E, ctx.decay, out=gW)
        # d/dP = dz^T gdx + (gy gdS)^T x ;  d/dS = gy^T (gdx P^T + x gdP^T)
        gP = gS = None
        if ctx.has_slorb:
            if g_dx is not None and w is not None:  # two skinny products (K = tokens each)
                gP = mm_tn(dz, g_dx)
                mm_tn(w, x, out=gP, accumulate=True)
            elif g_dx is not None:
                gP = mm_tn(dz, g_dx)
            elif w is not None:
                gP = mm_tn(w, x)
            if u is not None:
                gS = mm_tn(gy, u)
            gP, gS = (torch.zeros_like(t) if g is None else g for g, t in ((gP, P), (gS, S)))
        # a derivative that is identically zero is still a tensor (callers without allow_unused)
        gx, gW = (torch.zeros_like(t) if g is None else g for g, t in ((gx, x), (gW, W)))
        return ggy, gx, gW, gP, gS, None, None, None, None, None


class _MaskedLinear(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x2, W, bias, P, S, E, scale, decay, nm24=False):
        z = None
        if nm24:
            # E is a 2:4 hard mask: the pass that writes W.E also packs it, and the product runs on
            # the sparse MFMA (the SLoRB term as a dense second segment of the same kernel)
            Wm, vals, idx = apply_mask_2to4(W, E)
            if P is not None:
                z = mm_nt(x2, P)
            y = gemm_2to4(x2, vals, idx, W.shape[0], z=z, S=S, bias=bias)
            del vals, idx
        else:
            # y = x (W.E.s)^T: one elementwise pass writes the masked weight, the GEMM runs unmasked
            Wm, s = (apply_mask(W, E, scale), 1.0) if E is not None else (W, scale)
            if P is not None:
                z = mm_nt(x2, P)
                y = mm_nt(x2, Wm, bscale=s, A2=z, B2=S, K2=P.shape[0], bias=bias)
            else:
                y = mm_nt(x2, Wm, bscale=s, bias=bias)
        # Without a weight-scaling factor the input gradient needs the same W.E: it is saved for the
        # backward (2 B/param of bf16 weight) instead of being rebuilt there by another pass.  It goes
        # through save_for_backward, so the version counters of W and E guard it like the rest.
        keep = E is not None and scale == 1.0
        ctx.save_for_backward(x2, W, P, S, E, z, Wm if keep else None)
        del Wm
        ctx.decay = decay
        ctx.has_bias = bias is not None
        return y

    @staticmethod
    def backward(ctx, gy):
        x2, W, P, S, E, z, wm = ctx.saved_tensors
        gy = gy.contiguous().to(W.dtype)
        dx, dW, db, dP, dS = apply_in_backward(_MaskedLinearBackward, gy, x2, W, P, S, E, ctx.decay, ctx.has_bias, z,
                                               wm)
        del wm
        return dx, dW, db, dP, dS, None, None, None, None


def _compute_dtype(x: torch.Tensor, W: torch.Tensor) -> torch.dtype:
    if torch.is_autocast_enabled("cuda"):
        return torch.get_autocast_dtype("cuda")
    return W.dtype


def masked_linear(x, weight, bias, mask, mask_mode, hx, hard_kind, hard_n, scale, P=None, S=None, decay=0.0,
                  eff=None, hard=None, hard_m=4, cache=None):
    """y = x (W.E.s)^T + (x P^T) S^T + b with STE gradients.

    mask_mode: 'none' (E = 1), 'soft' (E = mask) or 'mix' (E = hx*mask + (1-hx)*hard(mask)).
    eff: a precomputed E in the compute dtype (skips the mask pass).
    hard: a precomputed hard(mask) (block hard types); else hard_kind / hard_n / hard_m project
    per group of hard_m along the input dimension.
    cache: a dict owned by the caller (one per layer) that keeps the mixed-mode E between calls.
    The soft mask changes only when the mask update writes it, while the reference rebuilds
    hard(mask) on every forward (legacy/sparse_modeling.py:759-771); E is reused while the mask's
    storage, its version counter (bumped by every in-place write: torch ops, and the library's mask
    kernels explicitly) and the projection parameters are unchanged.
    Strided inputs are accepted (made contiguous before the kernels, as F.linear accepts them).
    """
    L.require_device_only(x, weight, bias, mask, P, S, eff, hard)
    dt = _compute_dtype(x, weight)
    if dt not in (torch.float32, torch.bfloat16):
        raise TypeError(f"sparseforge_amd: unsupported compute dtype {dt}")
    lead = x.shape[:-1]
    x2 = x.reshape(-1, x.shape[-1])
    if x2.dtype != dt:
        x2 = x2.to(dt)
    x2 = x2.contiguous()
    W = (weight if weight.dtype == dt else weight.to(dt)).contiguous()
    b = None if bias is None else (bias if bias.dtype == dt else bias.to(dt)).contiguous()
    mask = _opt(mask)
    hard = _opt(hard)
    own_hard_bytes = eff is None and hard is None and mask_mode == "mix" and hx <= 0.0 and scale == 1.0
    key = None
    if eff is None and cache is not None and mask_mode == "mix" and hard is None:
        key = (mask.data_ptr(), mask._version, tuple(mask.shape), mask.dtype, float(hx), float(scale), hard_kind,
               hard_n, hard_m, dt)
        if cache.get("key") == key:
            eff = cache["eff"]
        else:
            cache.clear()
    if eff is None and mask_mode != "none":
        if mask_mode == "mix" and hx <= 0.0 and scale == 1.0:
            # E = hard(mask) exactly: staged as a byte and-mask (W * 1 = W, W * 0 = 0)
            eff = (effective_mask_given(mask, hard, torch.uint8, "hard", 0.0) if hard is not None
                   else effective_mask(mask, torch.uint8, "hard", 0.0, hard_kind, hard_n, hard_m))
        elif hard is not None and mask_mode == "mix":
            eff = effective_mask_given(mask, hard, dt, mask_mode, hx)
        else:
            eff = effective_mask(mask, dt, mask_mode, hx, hard_kind, hard_n, hard_m)
        if key is not None:
            cache["key"], cache["eff"] = key, eff
    if mask_mode == "none":
        eff = None
    eff = _opt(eff)
    Pp = Sp = None
    r = 0
    if P is not None:
        Pp, Sp, r = (P, S, P.shape[0]) if P.dtype == dt else (P.to(dt), S.to(dt), P.shape[0])
        Pp, Sp = Pp.contiguous(), Sp.contiguous()
        if Pp.shape[0] % _vec(dt):
            Pp, Sp, r = _PadRank.apply(Pp, Sp)
    # A 2:4 hard mask along the input dimension (both N:M kinds keep exactly two of every four
    # columns when in % 4 == 0) runs the forward product on the sparse MFMA.
    nm24 = (own_hard_bytes and eff is not None and hard_kind in (L.HARD_NM_TAIL_KEEP, L.HARD_NM_STRICT)
            and hard_n == 2 and hard_m == 4 and dt == torch.bfloat16 and W.shape[0] % 32 == 0
            and W.shape[1] % 64 == 0 and x2.shape[0] * W.shape[1] * 2 < 2 ** 31
            and W.shape[0] * W.shape[1] < 2 ** 31)
    y = _MaskedLinear.apply(x2, W, b, Pp, Sp, eff, float(scale), float(decay), nm24)
    return y.view(*lead, y.shape[-1])


class _PadRank(torch.autograd.Function):
    """Zero-pad P [r, in] and S [out, r] to a rank multiple of the vector width (differentiable)."""

    @staticmethod
    def forward(ctx, P, S):
        Pp, Sp, r = _pad_rank(P, S)
        ctx.r = r
        return Pp, Sp, r

    @staticmethod
    def backward(ctx, gPp, gSp, _):
        r = ctx.r
        gP = gPp[:r] if gPp is not None else None
        gS = gSp[:, :r] if gSp is not None else None
        return gP, gS


class FusedMaskedLinearSTE(torch.autograd.Function):
    """Drop-in of legacy/sparse_modeling.py:56-132: apply(x, weight, bias, mask, decay, scale_factor).

    `mask` is the effective mask (any [out, in] float tensor); it is cast to the
    weight dtype as the reference's `mask_cast` and applied inside the GEMMs.
    """

    @staticmethod
    def apply(x, weight, bias, mask, decay: float, scale_factor: float = 1.0):  # noqa: D102
        m = mask.detach().contiguous()
        return masked_linear(x, weight, bias, m, "soft", 1.0, L.HARD_NONE, 2, scale_factor, decay=float(decay))
