"""MI355X launchers for the cuPOW NoisyGEMM hot path, on torch ROCm tensors and torch's current
stream: the call surface of the reference's miner/ampere/uwc_ampere/ops.py (same names,
argument meaning and error behaviour), over libuwc_hip.so's C-ABI (include/uwc.h).

Differences a caller can see:
  * two GEMM tilings, CONFIGS["256x256"] (the default; m and n multiples of 256) and
    CONFIGS["128x128"] (any m, n for plain GEMMs; m, n multiples of 128 with a transcript), with
    identical outputs and winners; a hashed GEMM therefore needs m, n % 128 == 0 where the
    reference needs m % 128 and n % BN;
  * gemm() can also dump every tile's message and digest (`dump`), and OUT_F32 is an extra output
    mode (the fused detrt dequant epilogue);
  * MinedWeight.forward_many runs a sweep of nonces with batched commitments, noise and GEMM
    launches, and sweep_winners() returns every nonce's winners.
"""
from __future__ import annotations

import contextlib
import ctypes
import functools
import gc
import sys
from dataclasses import dataclass, field

import numpy as np
import torch

from . import _lib

BM, BN, BK = 128, 128, 64

# L balanced base-128 limbs, each digit in [-64, 63], represent every |v| <= 63 (1 + 128 + ... +
# 128^(L-1)) = 63 (128^L - 1) / 127: 63, 8127, 1040319, ... (kernels.cu:357-360, 602-607).
LIMB_CAPS = tuple(63 * (128 ** L - 1) // 127 for L in range(1, 5))


def limbs_for_max(mx: int) -> int:
    """Limbs the denoise pass uses for a runtime max |projection| mx (kernels.cu:602-607); the
    kernels stop at 4."""
    return next((L for L, cap in enumerate(LIMB_CAPS[:3], 1) if mx <= cap), 4)


def limbs_for(k: int) -> int:
    """Limbs that cover any projection of k int8 values, |projection| <= 127 k (ops.py:18-24):
    the limb count the correction buffers are sized for."""
    return limbs_for_max(127 * k)


def bound_words(bound: int) -> np.ndarray:
    """A 256-bit difficulty bound as eight little-endian uint32 words (pearl_glue.py:65-66)."""
    return np.array([(bound >> (32 * i)) & 0xFFFFFFFF for i in range(8)], dtype=np.uint32)


WIN_WORDS = 10
DUMP_WORDS = 24
CHUNKS_PER_CTA = 64
FLAG_HASH, FLAG_DENOISE = 1, 2
FLAG_TILE128 = 0x100  # force the 128 x 128 tiling (identical results)
FLAG_PLAIN = 0x200  # force a configuration of the plain DMA kernel: plain_cfg(c) (identical results)


def plain_cfg(c: int) -> int:
    """Flags forcing configuration c of the plain DMA kernel (0: 128 x 128 tiles, 4-step ring;
    1: 128 x 256, 3 steps; 2: 128 x 128, 2 steps; 3: 128 x 256, 2 steps; c + 4: the same with
    each step's DMA spread over the next step's passes)."""
    return FLAG_PLAIN | (c << 12)
OUT_NONE, OUT_I32, OUT_BF16, OUT_F32 = 0, 1, 2, 3
# GEMM tilings: (tile M = N, pipeline stages, waves per SIMD). "256x256" serves m, n % 256 == 0
# and falls back to "128x128" otherwise; every tiling gives identical outputs and winners.
CONFIGS = {"256x256": (256, 4, 2), "128x128": (128, 2, 2)}
DEFAULT_CFG = "256x256"

# Pearl's v3 noise labels and salts (miner/ampere/uwc_ampere/reference.py:23-26):
# SEED_SALT_X = BLAKE3(b"pearl/cert-v3/noise-seed/X").
SEED_LABEL_A = b"A_tensor" + b"\x00" * 24
SEED_LABEL_B = b"B_tensor" + b"\x00" * 24
SEED_SALT_A = bytes.fromhex("8249406ca0ed15169616f692fcf076f892dbdb2a7023b852f0d47719c390017b")
SEED_SALT_B = bytes.fromhex("11300632ec6301ca2be2af718b3f4d4f1ae9c63988e8cc044844301d71b89aa9")


def _check(cond: bool, msg) -> None:
    # the reference asserts its preconditions; keep AssertionError, but independent of -O
    if not cond:
        raise AssertionError(msg)


def _p(t: torch.Tensor | None) -> int | None:
    return None if t is None else t.data_ptr()


_stream = _lib.stream


assert sys.byteorder == "little", "the 32-byte values are little-endian u32 words, as the host's int32"


def words(b: bytes, device="cuda") -> torch.Tensor:
    """A 32-byte value as the 8 int32 words the kernels take (little-endian u32, ops.py:73-78)."""
    _check(len(b) % 4 == 0, f"words: {len(b)} bytes is not a whole number of 32-bit words")
    return torch.frombuffer(bytearray(b), dtype=torch.int32).to(device)


def words_to_bytes(t: torch.Tensor) -> bytes:
    """The inverse of words(): the tensor's 32-bit words as little-endian bytes."""
    return t.detach().to("cpu", torch.int32).contiguous().numpy().tobytes()


LABEL_A = words(SEED_LABEL_A, "cpu")
LABEL_B = words(SEED_LABEL_B, "cpu")
SALT_A = words(SEED_SALT_A, "cpu")
SALT_B = words(SEED_SALT_B, "cpu")


@functools.lru_cache(maxsize=None)
def _consts_on(device: str) -> dict:
    return {"LABEL_A": LABEL_A.to(device), "LABEL_B": LABEL_B.to(device), "SALT_A": SALT_A.to(device),
            "SALT_B": SALT_B.to(device)}


def consts(device) -> dict:
    """The label and salt words resident on `device`, copied there once per device, so that a
    forward (and a graph capture of it) never copies host to device (ops.py:85-95)."""
    return _consts_on(str(torch.device(device)))


# ------------------------------------------------------------------ BLAKE3
def b3_scratch_words(nbytes: int) -> int:
    return _lib.lib().uwc_b3_scratch_words(nbytes)


def b3_root_and_seed(data: torch.Tensor, key: torch.Tensor, *, prefix=None, salt=None, dim: int = 0,
                     root_out=None, seed_out=None, scratch=None):
    """Keyed BLAKE3 of `data` (uint8/int8, length a multiple of 1024) -> root, optional salted seed."""
    nbytes = data.numel() * data.element_size()
    _check(nbytes % 1024 == 0 and nbytes > 0, f"b3_root_and_seed: {nbytes} bytes is not a positive multiple of 1024")
    _check(data.is_contiguous(), "b3_root_and_seed: data must be contiguous")
    need = b3_scratch_words(nbytes)
    if scratch is None or scratch.numel() < need:
        scratch = torch.empty(need, dtype=torch.int32, device=data.device)
    _lib.call("uwc_b3_root_and_seed", _p(data), nbytes, _p(key), _p(prefix), _p(salt), dim, _p(root_out), _p(seed_out),
              _p(scratch), scratch.numel(), _stream())
    return scratch


def _ptrs(ts) -> "ctypes.Array | None":
    """A host array of device pointers (None stays None: the C-ABI's absent array)."""
    if ts is None:
        return None
    return (ctypes.c_void_p * len(ts))(*[t.data_ptr() for t in ts])


MAX_BATCH = 32  # items per batched commitment / noise launch (the C-ABI's limit)


def b3_root_and_seed_many(datas, key: torch.Tensor, *, prefix=None, salt=None, dim: int = 0, root_outs=None,
                          seed_outs=None, scratch=None):
    """b3_root_and_seed of several equal-size inputs in one set of launches; item i's result equals
    b3_root_and_seed(datas[i], ...). Returns the scratch buffer (item i uses words
    [i * s, (i + 1) * s), s = b3_scratch_words(nbytes))."""
    count = len(datas)
    _check(1 <= count <= MAX_BATCH, f"b3_root_and_seed_many: {count} inputs, need 1..{MAX_BATCH}")
    nbytes = datas[0].numel() * datas[0].element_size()
    _check(nbytes % 1024 == 0 and nbytes > 0, f"b3_root_and_seed_many: {nbytes} bytes is not a positive multiple of 1024")
    for d in datas:
        _check(d.is_contiguous() and d.numel() * d.element_size() == nbytes,
               "b3_root_and_seed_many: inputs must be contiguous and of equal size")
    for outs in (root_outs, seed_outs):
        _check(outs is None or len(outs) == count, "b3_root_and_seed_many: one root / seed output per input")
    need = b3_scratch_words(nbytes) * count
    if scratch is None or scratch.numel() < need:
        scratch = torch.empty(need, dtype=torch.int32, device=datas[0].device)
    _lib.call("uwc_b3_root_and_seed_many", ctypes.cast(_ptrs(datas), ctypes.c_void_p), count, nbytes, _p(key),
              _p(prefix), _p(salt), dim, _arr(root_outs), _arr(seed_outs), _p(scratch), scratch.numel(), _stream())
    return scratch


def _arr(ts):
    a = _ptrs(ts)
    return None if a is None else ctypes.cast(a, ctypes.c_void_p)


def _ptr_array(addrs) -> ctypes.c_void_p:
    """A host array of device addresses (ints), as the void* the C-ABI's array arguments take
    (the cast keeps the array alive)."""
    return ctypes.cast((ctypes.c_void_p * len(addrs))(*addrs), ctypes.c_void_p)


# ------------------------------------------------------------------ noise
def noise_uniform(out: torch.Tensor, label: torch.Tensor, key: torch.Tensor, zero_me=None, zero_n: int = 0):
    _check(out.numel() % 32 == 0, "noise_uniform: out size must be a multiple of 32")
    _lib.call("uwc_noise_uniform", _p(out), out.numel() // 32, _p(label), _p(key), _p(zero_me), zero_n, _stream())


def noise_perm(out: torch.Tensor, k: int, r: int, label: torch.Tensor, key: torch.Tensor):
    _check(out.numel() >= k, "noise_perm: out too small")
    _lib.call("uwc_noise_perm", _p(out), k, r, _p(label), _p(key), _stream())


def nonce_noise(E: torch.Tensor, P: torch.Tensor, k: int, r: int, label: torch.Tensor, key: torch.Tensor,
                St: torch.Tensor | None = None, zero0=None, zero1=None, SpT: torch.Tensor | None = None):
    """noise_uniform(E) + noise_perm(P) + proj_matrix(P) -> St (and its transpose SpT, k x 64) in
    one launch; zeroes zero0 and zero1."""
    rows = E.shape[0]
    _check(E.shape[1] == r and P.numel() >= k, "nonce_noise: E must be rows x r and P hold k words")
    n0 = zero0.numel() if zero0 is not None else 0
    n1 = zero1.numel() if zero1 is not None else 0
    _lib.call("uwc_nonce_noise", _p(E), rows, r, _p(P), k, _p(St), _p(SpT), _p(label), _p(key), _p(zero0), n0,
              _p(zero1), n1, _stream())


def nonce_noise_many(Es, Ps, k: int, r: int, label: torch.Tensor, keys, Sts=None, zero0s=None, zero1s=None,
                     SpTs=None):
    """nonce_noise for several nonces in one launch (item i as nonce_noise(Es[i], Ps[i], k, r,
    label, keys[i], ...)). Every list has one entry per item or is None."""
    count = len(Es)
    _check(1 <= count <= MAX_BATCH, f"nonce_noise_many: {count} items, need 1..{MAX_BATCH}")
    rows = Es[0].shape[0]
    for E, P in zip(Es, Ps):
        _check(tuple(E.shape) == (rows, r) and P.numel() >= k, "nonce_noise_many: E must be rows x r and P hold k words")
    for xs in (Ps, keys, Sts, zero0s, zero1s, SpTs):
        _check(xs is None or len(xs) == count, "nonce_noise_many: one entry per item")
    n0 = zero0s[0].numel() if zero0s is not None else 0
    n1 = zero1s[0].numel() if zero1s is not None else 0
    for zs, nz in ((zero0s, n0), (zero1s, n1)):
        _check(zs is None or all(z.numel() == nz for z in zs), "nonce_noise_many: zero ranges must be of equal size")
    _lib.call("uwc_nonce_noise_many", count, _arr(Es), rows, r, _arr(Ps), k, _arr(Sts), _arr(SpTs), _p(label),
              _arr(keys), _arr(zero0s), n0, _arr(zero1s), n1, _stream())


def noise_rows(src, rows, k, r, *, E=None, Pn=None, dst=None, Pp=None, corr=None, corr_off=-1, ecopy_off=-1,
               maxabs=None, lmax=None):
    lmax = corr.shape[0] if corr is not None else 0
    _check(rows % 8 == 0 and k % 4 == 0, f"noise_rows: rows={rows} % 8 and k={k} % 4 must be 0")
    _lib.call("uwc_noise_rows", _p(src), rows, k, r, _p(E), _p(Pn), _p(dst), _p(Pp), _p(corr), corr_off, ecopy_off,
              _p(maxabs), lmax, _stream())


# ------------------------------------------------------------------ projections as int8 GEMMs
def proj_matrix(P: torch.Tensor, k: int, r: int, St: torch.Tensor | None = None) -> torch.Tensor:
    """S^T for a noise permutation P (k entries, +index in the low 16 bits, -index in the high 16):
    r x k int8 with S^T[lo(l), l] += 1 and S^T[hi(l), l] -= 1, so src @ S = noise_rows' projection."""
    St = torch.empty((r, k), dtype=torch.int8, device=P.device) if St is None else St
    _lib.call("uwc_proj_matrix", _p(P), k, r, _p(St), _stream())
    return St


def project(src: torch.Tensor, St: torch.Tensor, corr: torch.Tensor, corr_off: int, maxabs: torch.Tensor):
    """noise_rows' projection part (corr limbs at corr_off, maxabs) with the sum on the matrix cores:
    exact, since every term is an integer and int8 x int8 products accumulate exactly in int32."""
    rows, k = src.shape
    r = St.shape[0]
    _check(src.is_contiguous() and St.is_contiguous(), "project: src and St must be contiguous")
    _lib.call("uwc_project", _p(src), rows, k, r, _p(St), _p(corr), corr_off, _p(maxabs), corr.shape[0], _stream())


def noise_project(src, rows, k, r, *, E, Pn, dst, St=None, corr=None, corr_off=-1, ecopy_off=-1, maxabs=None):
    """One pass over src: noising (dst) + optional projection with St into limbs + optional E copy."""
    lmax = corr.shape[0] if corr is not None else 0
    _lib.call("uwc_noise_project", _p(src), rows, k, r, _p(E), _p(Pn), _p(dst), _p(St), _p(corr), corr_off, ecopy_off,
              _p(maxabs), lmax, _stream())


def side_ok(m: int, n: int, k: int, r: int) -> bool:
    """Shapes uwc_side_project takes."""
    return m % 32 == 0 and n % 32 == 0 and k % 256 == 0 and r in (16, 32, 64)


def side_project(A, EA, SpA, ApEA, StB, corrA, Bp, StA, corrB, *, maxabs, corr_a_off=0, ecopy_off=-1, corr_b_off=0):
    """One launch for a nonce's operand side (ops.py:331-336): ApEA = A noised with EA and the
    pairs whose transposed selection matrix is SpA (k x 64, nonce_noise's SpT), X = A StB^T and
    Y = Bp StA^T into their limbs (corrA / corrB), EA copied into corrA at ecopy_off,
    maxabs[0..1] = max(maxabs, max |X|), max(maxabs, max |Y|)."""
    m, k = A.shape
    n, r = Bp.shape[0], StA.shape[0]
    _check(side_ok(m, n, k, r), f"side_project: m={m} n={n} k={k} r={r} unsupported")
    _check(all(t.is_contiguous() for t in (A, EA, SpA, ApEA, StB, corrA, Bp, StA, corrB)),
           "side_project: tensors must be contiguous")
    _check(SpA.shape == (k, 64), "side_project: SpA must be k x 64")
    _check(corrA.shape[0] == corrB.shape[0], "side_project: corrA and corrB need the same limb count")
    _lib.call("uwc_side_project", _p(A), m, _p(EA), _p(SpA), _p(ApEA), _p(StB), _p(corrA), corr_a_off, ecopy_off,
              _p(Bp), n, _p(StA), _p(corrB), corr_b_off, k, r, _p(maxabs), corrA.shape[0], _stream())


def side_pairs_ok(m: int, n: int, k: int, r: int) -> bool:
    """Shapes uwc_side_project_pairs takes."""
    return m % 32 == 0 and n % 32 == 0 and k % 128 == 0 and r in (32, 64, 128)


def side_project_pairs(A, EA, PA, ApEA, StB, corrA, Bp, StA, corrB, *, maxabs, corr_a_off=0, ecopy_off=-1, corr_b_off=0):
    """side_project from the noise pairs PA (k words, nonce_noise's P) instead of their selection
    matrix SpA, for any rank up to 128."""
    m, k = A.shape
    n, r = Bp.shape[0], StA.shape[0]
    _check(side_pairs_ok(m, n, k, r), f"side_project_pairs: m={m} n={n} k={k} r={r} unsupported")
    _check(all(t.is_contiguous() for t in (A, EA, PA, ApEA, StB, corrA, Bp, StA, corrB)),
           "side_project_pairs: tensors must be contiguous")
    _check(PA.numel() >= k and tuple(EA.shape) == (m, r), "side_project_pairs: PA must hold k words and EA be m x r")
    _check(corrA.shape[0] == corrB.shape[0], "side_project_pairs: corrA and corrB need the same limb count")
    _lib.call("uwc_side_project_pairs", _p(A), m, _p(EA), _p(PA), _p(ApEA), _p(StB), _p(corrA), corr_a_off, ecopy_off,
              _p(Bp), n, _p(StA), _p(corrB), corr_b_off, k, r, _p(maxabs), corrA.shape[0], _stream())


def side_many_ok(m: int, n: int, k: int, r: int) -> bool:
    """Shapes uwc_side_project_many takes."""
    return m % 128 == 0 and n % 128 == 0 and k % 128 == 0 and r in (16, 32, 64)


def side_project_many(As, EAs, SpAs, ApEAs, StB, corrAs, Bp, StAs, corrBs, *, maxabss, corr_a_off=0, ecopy_off=-1,
                      corr_b_off=0):
    """side_project for a group of nonces sharing the block side (StB, Bp), one launch: item i as
    side_project(As[i], EAs[i], SpAs[i], ApEAs[i], StB, corrAs[i], Bp, StAs[i], corrBs[i],
    maxabs=maxabss[i], ...)."""
    count = len(As)
    _check(1 <= count <= MAX_BATCH, f"side_project_many: {count} items, need 1..{MAX_BATCH}")
    m, k = As[0].shape
    n, r = Bp.shape[0], StAs[0].shape[0]
    _check(side_many_ok(m, n, k, r), f"side_project_many: m={m} n={n} k={k} r={r} unsupported")
    for xs in (EAs, SpAs, ApEAs, corrAs, StAs, corrBs, maxabss):
        _check(len(xs) == count, "side_project_many: one entry per item")
    for A, SpA in zip(As, SpAs):
        _check(tuple(A.shape) == (m, k) and SpA.shape == (k, 64), "side_project_many: A must be m x k, SpA k x 64")
    _check(corrAs[0].shape[0] == corrBs[0].shape[0], "side_project_many: corrA and corrB need the same limb count")
    _lib.call("uwc_side_project_many", count, _arr(As), _arr(EAs), _arr(SpAs), _arr(ApEAs), _p(StB), _arr(corrAs),
              corr_a_off, ecopy_off, _p(Bp), _arr(StAs), _arr(corrBs), corr_b_off, m, n, k, r, _arr(maxabss),
              corrAs[0].shape[0], _stream())


# ------------------------------------------------------------------ activation quantizer
def quant_rows_had(x: torch.Tensor, bs: int, q: torch.Tensor | None = None, scale: torch.Tensor | None = None):
    """x: m x k bf16 (contiguous) -> (int8 q in [-64, 64], float32 per-row scale), block Hadamard of
    size bs (ops.py:172-181). Rows of any k % 8 == 0 when k % 512 == 0 and bs <= 512; else k <= 40960."""
    m, k = x.shape
    _check(x.dtype == torch.bfloat16 and x.is_contiguous() and k % 8 == 0 and (bs <= 1 or k % bs == 0),
           f"quant_rows_had: x must be contiguous bf16 with k % 8 == 0 and bs | k (k={k}, bs={bs})")
    q = torch.empty((m, k), dtype=torch.int8, device=x.device) if q is None else q
    scale = torch.empty(m, dtype=torch.float32, device=x.device) if scale is None else scale
    _lib.call("uwc_quant_rows_had", _p(x), m, k, bs, _p(q), _p(scale), _stream())
    return q, scale


# ------------------------------------------------------------------ GEMM
def gemm(A, B, *, r=128, flags=0, corrA=None, corrB=None, maxabs=None, key=None, target=None, wins=None,
         max_wins=0, a_scale=None, b_scale=None, out=None, out_mode=OUT_NONE, cfg=None, dump=None):
    """C = A @ B^T (int8, k contiguous) with the optional mining transcript / denoise / epilogue."""
    cfg = cfg or DEFAULT_CFG
    _check(cfg in CONFIGS, f"gemm: unknown cfg {cfg!r}")
    m, k = A.shape
    n = B.shape[0]
    if flags:
        _check(m % BM == 0 and n % BN == 0 and k % BK == 0 and r % BK == 0 and k % r == 0, (m, n, k, r))
    else:
        _check(k % BK == 0, (m, n, k))
    _check(A.dtype == torch.int8 and B.dtype == torch.int8 and A.is_contiguous() and B.is_contiguous(),
           "gemm: A and B must be contiguous int8")
    _lib.call("uwc_noisy_gemm", _p(A), _p(B), m, n, k, r, _p(corrA), _p(corrB), _p(maxabs),
              corrA.shape[0] if corrA is not None else 0, _p(key), _p(target), _p(wins), max_wins, _p(a_scale),
              _p(b_scale), _p(out), out_mode, flags | (FLAG_TILE128 if cfg == "128x128" else 0), _p(dump), _stream())


def gemm_many(As, B, *, r=128, flags=0, corrAs=None, corrBs=None, maxabss=None, keys=None, target=None, winss=None,
              max_wins=0, a_scale=None, b_scale=None, outs=None, out_mode=OUT_NONE, dumps=None):
    """gemm() of several operands As[i] against one B, item i with its own corrections, maxabs,
    seed, win buffer, output and optional tile dump. With FLAG_HASH | FLAG_DENOISE, OUT_I32 and
    m, n % 256 == 0 the items share launches (up to 32 per launch, output stores overlapping the
    next item); otherwise one launch per item. Results equal separate gemm() calls."""
    count = len(As)
    if count == 0:
        return
    m, k = As[0].shape
    n = B.shape[0]
    if flags:
        _check(m % BM == 0 and n % BN == 0 and k % BK == 0 and r % BK == 0 and k % r == 0, (m, n, k, r))
    for A in As:
        _check(tuple(A.shape) == (m, k) and A.dtype == torch.int8 and A.is_contiguous(),
               "gemm_many: every A must be a contiguous int8 m x k")
    _check(B.dtype == torch.int8 and B.is_contiguous(), "gemm_many: B must be contiguous int8")
    for xs in (corrAs, corrBs, maxabss, keys, winss, outs, dumps):
        _check(xs is None or len(xs) == count, "gemm_many: one entry per item")
    _check(outs is not None or out_mode == OUT_NONE, "gemm_many: outputs needed for this out_mode")
    lmax = corrAs[0].shape[0] if corrAs is not None else 0
    out_arr = _arr(outs) if outs is not None else ctypes.cast((ctypes.c_void_p * count)(), ctypes.c_void_p)
    _lib.call("uwc_noisy_gemm_many", count, _arr(As), _p(B), m, n, k, r, _arr(corrAs), _arr(corrBs), _arr(maxabss),
              lmax, _arr(keys), _p(target), _arr(winss), max_wins, _p(a_scale), _p(b_scale), out_arr, out_mode, flags,
              _arr(dumps), _stream())


def igemm_i32(A: torch.Tensor, B: torch.Tensor, out: torch.Tensor | None = None) -> torch.Tensor:
    """Exact int32 A @ B^T for any m, n (k % 64 == 0)."""
    m, k = A.shape
    n = B.shape[0]
    _check(A.is_contiguous() and B.is_contiguous() and A.dtype == torch.int8 and B.dtype == torch.int8,
           "igemm_i32: A and B must be contiguous int8")
    out = torch.empty((m, n), dtype=torch.int32, device=A.device) if out is None else out
    _lib.call("uwc_igemm_i32", _p(A), _p(B), m, n, k, _p(out), _stream())
    return out


# ------------------------------------------------------------------ one mined linear layer
_WORKSPACE: dict = {}
_SWEEP_SYNC: dict = {}
# nonces per batched commitment / noise launch and per batched GEMM launch in
# MinedWeight.forward_many: at most SWEEP_GROUP, the sweep split into equal groups (measured on
# warmed-up boxes, 4096^3 r = 64, 256 nonces: 0.1007 ms per nonce at 8, 0.0966-0.0984 at 16,
# 0.0973 at 24 and 32; 20 nonces: 0.1068 as one group, 0.1072 as 2 x 10, 0.1081 as 16 + 4)
SWEEP_GROUP = 32
GEMM_GROUP = 32


def sweep_group(n_items: int, most: int = SWEEP_GROUP) -> int:
    """The group size forward_many takes for n_items nonces: the fewest groups of at most `most`,
    as equal as possible (20 nonces: one group, 40: 2 x 20, 256: 8 x 32)."""
    ngroups = -(-n_items // most)
    return -(-n_items // ngroups)


@dataclass
class MinedWeight:
    """A weight B^T (n x k int8, values in [-64, 64]) prepared for mining under one block template.

    setup_block() runs once per (block header, k); forward() runs per call and needs no host sync.
    (miner/ampere/uwc_ampere/ops.py:205-371)
    """
    Bt: torch.Tensor
    b_scale: torch.Tensor
    r: int = 128
    max_wins: int = 64
    job_key: torch.Tensor | None = None
    b_seed: torch.Tensor | None = None
    target: torch.Tensor | None = None
    BpEBt: torch.Tensor | None = None
    PB: torch.Tensor | None = None
    EBRt: torch.Tensor | None = None
    corrB: torch.Tensor | None = None
    SBt: torch.Tensor | None = None
    _bufs: dict = field(default_factory=dict)
    _block_gen: int = 0  # bumped by every setup_block: per-slot copies of corrB made earlier are stale

    @property
    def n(self):
        return self.Bt.shape[0]

    @property
    def k(self):
        return self.Bt.shape[1]

    @property
    def device(self):
        return self.b_scale.device

    def setup_block(self, job_key: bytes, target_words: np.ndarray):
        dev = self.device
        n, k, r = self.n, self.k, self.r
        _check(n % BN == 0 and k % r == 0 and r % BK == 0, f"MinedWeight: n={n} k={k} r={r} unsupported")
        Bt = self.Bt if self.Bt.device == dev else self.Bt.to(dev, non_blocking=True)
        Bt = Bt.contiguous()
        self.job_key = words(job_key, dev)
        self.target = torch.from_numpy(np.asarray(target_words).astype(np.uint32).view(np.int32).copy()).to(dev)
        self.b_seed = torch.empty(8, dtype=torch.int32, device=dev)
        c = consts(dev)
        b3_root_and_seed(Bt.view(-1), self.job_key, prefix=self.job_key, salt=c["SALT_B"], dim=n, seed_out=self.b_seed)
        self.EBRt = torch.empty((n, r), dtype=torch.int8, device=dev)
        noise_uniform(self.EBRt, c["LABEL_B"], self.b_seed)
        self.PB = torch.empty(k, dtype=torch.int32, device=dev)
        noise_perm(self.PB, k, r, c["LABEL_B"], self.b_seed)
        if self.BpEBt is None:
            self.BpEBt = torch.empty((n, k), dtype=torch.int8, device=dev)
            self.corrB = torch.zeros((limbs_for(k), n, 2 * r), dtype=torch.int8, device=dev)
        if n % 16 == 0 and k % 64 == 0 and r <= 128:
            noise_project(Bt, n, k, r, E=self.EBRt, Pn=self.PB, dst=self.BpEBt, corr=self.corrB, ecopy_off=0)
        else:
            noise_rows(Bt, n, k, r, E=self.EBRt, Pn=self.PB, dst=self.BpEBt, corr=self.corrB, ecopy_off=0)
        self.SBt = proj_matrix(self.PB, k, r)
        self._block_gen += 1
        del Bt

    def _buf(self, m: int, slot: int = 0, wins: torch.Tensor | None = None):
        """Per-call buffers, a workspace shared by every weight with the same (m, k, r): layers run
        one after another on one stream (slot 0). forward_many gives each nonce of a group its own
        slot (1, 2, ...): noise, noised operand, corrections and commitment scratch, so that a
        group's projections all run before its GEMMs. Win records are per weight (or the caller's
        buffer); slots > 0 carry their own."""
        ws = self._ws(m, slot)
        if wins is None:
            wkey = (m, slot)
            wins = self._bufs.get(wkey)
            if wins is None:
                wins = self._bufs[wkey] = torch.zeros(1 + self.max_wins * WIN_WORDS, dtype=torch.int32,
                                                      device=self.device)
        return {**ws, "wins": wins}

    def _ws(self, m: int, slot: int) -> dict:
        """The (m, k, r, slot) workspace buffers (allocated on first use, then kept)."""
        dev, k, r = self.device, self.k, self.r
        key = (str(dev), m, k, r, slot)
        ws = _WORKSPACE.get(key)
        if ws is None:
            i8, i32 = torch.int8, torch.int32
            # buffer: (shape, dtype, starts zeroed)
            layout = {
                "a_seed": ((8,), i32, False),                     # the nonce's salted seed words
                "EAL": ((m, r), i8, False),                       # E_A
                "PA": ((k,), i32, False),                         # P_A: first | second << 16 per column
                "SA": ((r, k), i8, False),                        # S_A, the selection matrix of P_A
                "SpA": ((k, 64), i8, False) if r <= 64 else None,  # S_A transposed, zero past r
                "ApEA": ((m, k), i8, False),                      # A + E_A S_A
                "corrA": ((limbs_for(k), m, 2 * r), i8, True),    # [X limbs | E_A] per limb
                "maxabs": ((2,), i32, True),
                "scratch": ((max(8, b3_scratch_words(m * k)),), i32, False),  # commitment tree levels
            }
            ws = {name: None if spec is None else (torch.zeros if spec[2] else torch.empty)(spec[0], dtype=spec[1], device=dev)
                  for name, spec in layout.items()}
            _WORKSPACE[key] = ws
        return ws

    def _slot_set(self, m: int, parity: int, group: int, count: int) -> dict:
        """forward_many's workspace slots 1 + parity * group + j (j < count) as device-pointer
        arrays, one per buffer kind, built once per (m, slot set, count) and block template: the
        buffers stay where they are from sweep to sweep, so a group's launches only need the
        arrays of its operands, outputs and win rows. Building it refreshes the slots' corrB
        copies (on the current stream)."""
        key = ("slot_set", m, parity, group, count)
        ss = self._bufs.get(key)
        if ss is not None and ss["gen"] == self._block_gen:
            return ss
        slots = [1 + parity * group + j for j in range(count)]
        ws = [self._ws(m, sl) for sl in slots]
        ss = {"gen": self._block_gen, "limbs": ws[0]["corrA"].shape[0],
              "corrB": _ptr_array([self._slot_corrB(sl).data_ptr() for sl in slots])}
        for name in ("a_seed", "EAL", "PA", "SA", "SpA", "ApEA", "corrA", "maxabs"):
            ss[name] = _ptr_array([w[name].data_ptr() for w in ws])
        self._bufs[key] = ss
        return ss

    def _slot_corrB(self, slot: int) -> torch.Tensor:
        """A per-slot copy of corrB for forward_many: the E_B columns setup_block wrote, and room
        for the slot's nonce's Y limbs (the reference's single corrB serves one call at a time).
        The copy is refreshed (on the current stream) whenever setup_block has run since it was
        made: a new block template rewrites E_B in place."""
        gen, cb = self._bufs.get(("corrB", slot), (None, None))
        if cb is None or cb.shape != self.corrB.shape:
            cb = torch.empty_like(self.corrB)
            gen = None
        if gen != self._block_gen:
            cb.copy_(self.corrB)
            gen = self._block_gen
        self._bufs[("corrB", slot)] = (gen, cb)
        return cb

    def forward(self, A: torch.Tensor, a_scale: torch.Tensor, out: torch.Tensor | None = None,
                out_mode: int = OUT_BF16, hash_tiles: bool = True) -> torch.Tensor:
        """A: m x k int8 (values in [-64, 64]). Returns A @ Bt^T scaled (bf16/f32) or exact int32."""
        return self._forward(A, a_scale, out, out_mode, hash_tiles)

    def _check_a(self, A):
        m, k = A.shape
        _check(k == self.k and m % BM == 0, f"MinedWeight.forward: A is {tuple(A.shape)}, need m % {BM} == 0, k == {self.k}")
        _check(A.is_contiguous() and A.dtype == torch.int8, "MinedWeight.forward: A must be contiguous int8")

    def _commit(self, A, b):
        """1. commit to A, derive a_seed = H(b_seed || bind_a(root_A, m)) (ops.py:322-324)."""
        c = consts(A.device)
        b3_root_and_seed(A.view(-1), self.job_key, prefix=self.b_seed, salt=c["SALT_A"], dim=A.shape[0],
                         seed_out=b["a_seed"], scratch=b["scratch"])

    def _after_commit(self, A, b, a_scale, out, out_mode, hash_tiles, cfg=None, proj=True, dump=None):
        m, k = A.shape
        n, r = self.n, self.r
        c = consts(A.device)
        if proj:  # projections on the matrix cores (the reference's PROJ_GEMM path)
            side = side_ok(m, n, k, r)
            # 2. A-side noise E_AL, P_A (and its selection matrices); the same launch zeroes maxabs
            #    and the win counter
            nonce_noise(b["EAL"], b["PA"], k, r, c["LABEL_A"], b["a_seed"], St=b["SA"], zero0=b["maxabs"],
                        zero1=b["wins"][:1], SpT=b["SpA"] if side else None)
            return self._mine(A, b, a_scale, out, out_mode, hash_tiles, side, cfg=cfg, dump=dump)
        # projections by LDS atomics (noise_rows with Pp)
        noise_uniform(b["EAL"], c["LABEL_A"], b["a_seed"], zero_me=b["maxabs"], zero_n=2)
        b["wins"][:1].zero_()
        noise_perm(b["PA"], k, r, c["LABEL_A"], b["a_seed"])
        noise_rows(A, m, k, r, E=b["EAL"], Pn=b["PA"], dst=b["ApEA"], Pp=self.PB, corr=b["corrA"], corr_off=0,
                   ecopy_off=r, maxabs=b["maxabs"][0:1])
        noise_rows(self.BpEBt, n, k, r, Pp=b["PA"], corr=self.corrB, corr_off=r, maxabs=b["maxabs"][1:2])
        return self._gemm(b, a_scale, out, out_mode, hash_tiles, cfg=cfg, dump=dump)

    def _mine(self, A, b, a_scale, out, out_mode, hash_tiles, side, cfg=None, dump=None):
        """Steps 3-5 of a mined forward once the nonce's noise is drawn (ops.py:331-347)."""
        self._project(A, b, side, self.corrB)
        return self._gemm(b, a_scale, out, out_mode, hash_tiles, cfg=cfg, dump=dump)

    def _project(self, A, b, side, corrB):
        """3. ApEA = A + EAL*P_A ; X = A * P_B^T (limbs) ; EAL copy; 4. Y = BpEBt * P_A^T (limbs)
        into corrB."""
        m, k = A.shape
        r = self.r
        if side:
            side_project(A, b["EAL"], b["SpA"], b["ApEA"], self.SBt, b["corrA"], self.BpEBt, b["SA"], corrB,
                         maxabs=b["maxabs"], corr_a_off=0, ecopy_off=r, corr_b_off=r)
        elif side_pairs_ok(m, self.n, k, r):
            # r = 128 and k % 256 != 0: 4096^3 at r = 128 48.6 -> 27.8 us (one launch for two); at r =
            # 64 side_project's noise on the matrix cores is the faster there (17.2 against 19.7)
            side_project_pairs(A, b["EAL"], b["PA"], b["ApEA"], self.SBt, b["corrA"], self.BpEBt, b["SA"], corrB,
                               maxabs=b["maxabs"], corr_a_off=0, ecopy_off=r, corr_b_off=r)
        else:
            noise_project(A, m, k, r, E=b["EAL"], Pn=b["PA"], dst=b["ApEA"], St=self.SBt, corr=b["corrA"],
                          corr_off=0, ecopy_off=r, maxabs=b["maxabs"][0:1])
            project(self.BpEBt, b["SA"], corrB, r, b["maxabs"][1:2])

    def _gemm(self, b, a_scale, out, out_mode, hash_tiles, cfg=None, dump=None):
        # 5. noisy GEMM: hash every tile, denoise exactly, scale
        gemm(b["ApEA"], self.BpEBt, r=self.r, flags=(FLAG_HASH if hash_tiles else 0) | FLAG_DENOISE,
             corrA=b["corrA"], corrB=self.corrB, maxabs=b["maxabs"], key=b["a_seed"], target=self.target,
             wins=b["wins"], max_wins=self.max_wins, a_scale=a_scale, b_scale=self.b_scale, out=out, out_mode=out_mode,
             cfg=cfg, dump=dump)
        return out

    def _sweep_scratch(self, m: int, count: int) -> torch.Tensor:
        """Commitment scratch for `count` operands of m x k in one batched launch."""
        need = b3_scratch_words(m * self.k) * count
        key = (str(self.device), m, self.k, "sweep")
        t = _WORKSPACE.get(key)
        if t is None or t.numel() < need:
            t = _WORKSPACE[key] = torch.empty(need, dtype=torch.int32, device=self.device)
        return t

    def _out(self, m, out, out_mode):
        if out is None and out_mode != OUT_NONE:
            dt = {OUT_BF16: torch.bfloat16, OUT_I32: torch.int32, OUT_F32: torch.float32}[out_mode]
            out = torch.empty((m, self.n), dtype=dt, device=self.device)
        return out

    def _forward(self, A, a_scale, out, out_mode, hash_tiles, cfg=None, proj=True, dump=None):
        self._check_a(A)
        b = self._buf(A.shape[0])
        out = self._out(A.shape[0], out, out_mode)
        self._commit(A, b)
        return self._after_commit(A, b, a_scale, out, out_mode, hash_tiles, cfg=cfg, proj=proj, dump=dump)

    def forward_many(self, As, a_scale: torch.Tensor, outs=None, out_mode: int = OUT_BF16, hash_tiles: bool = True,
                     wins=None, group: int | None = None, gemm_group: int | None = None, dumps=None):
        """Mined forwards of a sequence of activations (the nonces of a sweep), each equal to
        forward(As[i]) bit for bit, winners included.

        The nonces go in groups of `group` (1..MAX_BATCH; by default sweep_group(len(As)), equal
        groups of at most SWEEP_GROUP): one set of launches commits the whole
        group (BLAKE3 trees and salted seeds) and one launch draws all of its noise, so those
        latency-bound chains run several waves per SIMD instead of one, on a second stream one
        group ahead, beside the previous group's projections (a sweep of one group queues them
        on the current stream); then the group's nonces run their
        projections and hashed GEMMs, `gemm_group` (by default the group) nonces per batched GEMM call (whose output
        stores overlap the next nonce's tiles). The work is queued behind the current stream,
        which then waits for all of it. Python's cyclic garbage collector is paused while the
        launches are queued (a full collection can stall the host for tens of milliseconds,
        longer than the GPU work already queued), and its previous state restored.

        Every nonce records its winners in its own buffer: the caller's `wins` (one int32 tensor
        of 1 + max_wins * WIN_WORDS words per item), or else a row of a device buffer that the
        weight keeps (reserve_sweep() allocates it ahead of time); sweep_winners() reads all rows
        back with one copy once the sweep is done. (Copying each group's rows to the host while
        the sweep runs, on a stream waiting for the group's GEMMs, stalled the host thread in the
        copy call and with it the queueing of the next groups.) winners(m) reports the last item,
        as after forward(). dumps: optional per-item tile dumps (gemm()'s `dump` layout).
        Returns the outputs."""
        n_items = len(As)
        if n_items == 0:
            return []
        if group is None:
            group = sweep_group(n_items)
        if gemm_group is None:
            gemm_group = min(group, GEMM_GROUP)
        _check(1 <= group <= MAX_BATCH, f"MinedWeight.forward_many: group={group}, need 1..{MAX_BATCH}")
        _check(gemm_group >= 1, f"MinedWeight.forward_many: gemm_group={gemm_group}")
        A0 = As[0]
        self._check_a(A0)
        m, k, r = A0.shape[0], self.k, self.r
        shape, i8 = A0.shape, torch.int8
        for A in As:  # the kernels assume every operand's shape, type and layout
            if A.shape != shape or A.dtype != i8 or not A.is_contiguous():
                self._check_a(A)
                _check(False, "MinedWeight.forward_many: every A needs the same shape")
        _check(wins is None or len(wins) == n_items, "MinedWeight.forward_many: one win buffer per item")
        _check(dumps is None or len(dumps) == n_items, "MinedWeight.forward_many: one tile dump per item")
        c = consts(A0.device)
        gc_on = gc.isenabled()
        gc.disable()
        try:
            if gemm_group >= group and side_many_ok(m, self.n, k, r):
                host = None
                if wins is None:  # row i of the sweep's win rows, by address
                    host = self.reserve_sweep(m, n_items)
                    base, pitch = host.data_ptr(), host.stride(0) * host.element_size()
                    win_ptrs = [base + i * pitch for i in range(n_items)]
                else:
                    win_ptrs = [wb.data_ptr() for wb in wins]
                self._sweep_host = (host, n_items) if host is not None else None
                outs = self._sweep_fast(As, a_scale, outs, out_mode, hash_tiles, win_ptrs, group, m, k, r, c, dumps,
                                        host)
            else:
                outs = [self._out(m, outs[i] if outs is not None else None, out_mode) for i in range(n_items)]
                side = side_ok(m, self.n, k, r)
                host = None
                if wins is None:
                    wins, host = self._sweep_win_rows(m, n_items)
                self._sweep_host = (host, n_items) if host is not None else None
                self._sweep(As, a_scale, outs, out_mode, hash_tiles, wins, group, gemm_group, m, k, r, c, side, host,
                            dumps)
        finally:
            if gc_on:
                gc.enable()
        return outs

    def reserve_sweep(self, m: int, n_items: int) -> torch.Tensor:
        """Allocate now the per-nonce win rows that forward_many of n_items nonces of m rows uses,
        so that the sweep itself allocates nothing."""
        words = 1 + self.max_wins * WIN_WORDS
        rows = self._bufs.get(("sweep_wins", m))
        if rows is None or rows.shape[0] < n_items:
            rows = self._bufs[("sweep_wins", m)] = torch.zeros((n_items, words), dtype=torch.int32, device=self.device)
        return rows

    def _sweep_win_rows(self, m: int, n_items: int):
        """Device win buffers for a sweep of n_items nonces: consecutive rows of one tensor."""
        rows = self.reserve_sweep(m, n_items)
        return [rows[i] for i in range(n_items)], rows

    def _sweep(self, As, a_scale, outs, out_mode, hash_tiles, wins, group, gemm_group, m, k, r, c, side, host=None,
               dumps=None):
        """Group g's commitment and noise go on a side stream, one group ahead, so that they run
        beside group g - 1's projections (the BLAKE3 chains are VALU-bound, the projections
        memory-bound, and a CU holds one workgroup of each); groups alternate between two sets of
        workspace slots, and a group's commitment waits until the GEMM of the group two back, the
        last user of its set, is done."""
        n_items = len(As)
        groups = [list(range(g0, min(g0 + group, n_items))) for g0 in range(0, n_items, group)]
        many = side_many_ok(m, self.n, k, r)  # one operand-side launch per GEMM batch
        cur = torch.cuda.current_stream(self.device)
        sc, committed, consumed = self._sweep_sync()
        sc.wait_stream(cur)

        def bufs_of(gi):
            out = []
            for j, i in enumerate(groups[gi]):
                out.append(self._buf(m, slot=1 + (gi % 2) * group + j, wins=wins[i]))
            return out

        def commit(gi):
            items, bufs = groups[gi], bufs_of(gi)
            with torch.cuda.stream(sc):
                if gi >= 2:
                    sc.wait_event(consumed[gi % 2])
                # 1. commit to every A of the group, a_seed_i = H(b_seed || bind_a(root_Ai, m))
                #    (ops.py:322-324)
                b3_root_and_seed_many([As[i].view(-1) for i in items], self.job_key, prefix=self.b_seed,
                                      salt=c["SALT_A"], dim=m, seed_outs=[b["a_seed"] for b in bufs],
                                      scratch=self._sweep_scratch(m, len(items)))
                # 2. every nonce's noise E_A, P_A and selection matrices; zeroes its maxabs and win
                #    count
                nonce_noise_many([b["EAL"] for b in bufs], [b["PA"] for b in bufs], k, r, c["LABEL_A"],
                                 [b["a_seed"] for b in bufs], Sts=[b["SA"] for b in bufs],
                                 zero0s=[b["maxabs"] for b in bufs], zero1s=[b["wins"][:1] for b in bufs],
                                 SpTs=[b["SpA"] for b in bufs] if side or many else None)
                committed[gi % 2].record(sc)

        commit(0)
        for gi, items in enumerate(groups):
            if gi + 1 < len(groups):
                commit(gi + 1)
            bufs = bufs_of(gi)
            cur.wait_event(committed[gi % 2])
            corrBs = [self._slot_corrB(1 + (gi % 2) * group + j) for j in range(len(items))]
            for s0 in range(0, len(items), gemm_group):
                sub = range(s0, min(s0 + gemm_group, len(items)))
                # 3.-4. the nonces' noised operands and projections (own slot and corrB copy): one
                # launch for the sub-batch, or one per nonce for shapes the batched form does not take
                if many:
                    side_project_many([As[items[j]] for j in sub], [bufs[j]["EAL"] for j in sub],
                                      [bufs[j]["SpA"] for j in sub], [bufs[j]["ApEA"] for j in sub], self.SBt,
                                      [bufs[j]["corrA"] for j in sub], self.BpEBt, [bufs[j]["SA"] for j in sub],
                                      [corrBs[j] for j in sub], maxabss=[bufs[j]["maxabs"] for j in sub],
                                      corr_a_off=0, ecopy_off=r, corr_b_off=r)
                else:
                    for j in sub:
                        self._project(As[items[j]], bufs[j], side, corrBs[j])
                # 5. their hashed GEMMs with exact denoise: one batched call
                gargs = ([bufs[j]["ApEA"] for j in sub], self.BpEBt)
                gkw = dict(r=r, flags=(FLAG_HASH if hash_tiles else 0) | FLAG_DENOISE,
                           corrAs=[bufs[j]["corrA"] for j in sub], corrBs=[corrBs[j] for j in sub],
                           maxabss=[bufs[j]["maxabs"] for j in sub], keys=[bufs[j]["a_seed"] for j in sub],
                           target=self.target, winss=[bufs[j]["wins"] for j in sub], max_wins=self.max_wins,
                           a_scale=a_scale, b_scale=self.b_scale,
                           outs=[outs[items[j]] for j in sub] if out_mode != OUT_NONE else None, out_mode=out_mode,
                           dumps=[dumps[items[j]] for j in sub] if dumps is not None else None)
                gemm_many(*gargs, **gkw)
                self._last_gemm = (len(sub), functools.partial(gemm_many, *gargs, **gkw))
            consumed[gi % 2].record(cur)
        if host is not None:  # winners(m) reports the sweep's last nonce, as after forward()
            self._buf(m)["wins"].copy_(host[n_items - 1])
        cur.wait_stream(sc)

    def last_gemm_launch(self):
        """(nonces, launch) of the last batched GEMM call forward_many queued: launch() queues the
        same call again on the current stream (same operands, corrections, seeds, target, win rows
        and outputs; the win rows then collect the repeats' records too). For timing the GEMM
        alone."""
        _check(getattr(self, "_last_gemm", None) is not None, "MinedWeight.last_gemm_launch: no forward_many has run")
        return self._last_gemm

    def _sweep_sync(self):
        """A default-priority side stream and four reusable events per device."""
        sync = _SWEEP_SYNC.get(str(self.device))
        if sync is None:
            sync = _SWEEP_SYNC[str(self.device)] = (torch.cuda.Stream(device=self.device),
                                                    [torch.cuda.Event() for _ in range(2)],
                                                    [torch.cuda.Event() for _ in range(2)])
        return sync

    def _sweep_fast(self, As, a_scale, outs, out_mode, hash_tiles, win_ptrs, group, m, k, r, c, dumps, host):
        """_sweep for the shapes the batched operand side takes, one GEMM launch per group, with
        the launches' array arguments passed as device addresses: the workspace slots' from
        _slot_set (built once), the group's operands, outputs and win rows per call. The first
        commitment is therefore queued after a few tens of microseconds of host work instead of
        after every nonce's bookkeeping (a 20-nonce sweep lost ~0.2 ms of GPU time to that).
        Same launches and order as _sweep; a sweep of one group, which has nothing to overlap its
        commitment with, queues everything on the current stream (no cross-stream waits, each of
        which left the GPU idle ~10 us). Returns the outputs."""
        n_items, n = len(As), self.n
        _check(m % BM == 0 and n % BN == 0 and k % BK == 0 and r % BK == 0 and k % r == 0, (m, n, k, r))
        bounds = [(g0, min(g0 + group, n_items)) for g0 in range(0, n_items, group)]
        cur = torch.cuda.current_stream(self.device)
        single = len(bounds) == 1
        sc, committed, consumed = self._sweep_sync()
        if single:
            sc = cur
        else:
            sc.wait_stream(cur)
        a_ptrs = [A.data_ptr() for A in As]
        scratch = self._sweep_scratch(m, group)
        key, prefix, salt, label = _p(self.job_key), _p(self.b_seed), _p(c["SALT_A"]), _p(c["LABEL_A"])

        def commit(gi):
            g0, g1 = bounds[gi]
            # the side stream current while the slot set may allocate (a one-group sweep has none)
            with contextlib.nullcontext() if single else torch.cuda.stream(sc):
                if gi >= 2:
                    sc.wait_event(consumed[gi % 2])
                ss = self._slot_set(m, gi % 2, group, g1 - g0)
                st = sc.cuda_stream
                # 1. commit to every A of the group, a_seed_i = H(b_seed || bind_a(root_Ai, m))
                #    (ops.py:322-324)
                _lib.call("uwc_b3_root_and_seed_many", _ptr_array(a_ptrs[g0:g1]), g1 - g0, m * k, key, prefix, salt, m,
                          None, ss["a_seed"], scratch.data_ptr(), scratch.numel(), st)
                # 2. every nonce's noise E_A, P_A and selection matrices; zeroes its maxabs (2
                #    words) and win count (1 word)
                _lib.call("uwc_nonce_noise_many", g1 - g0, ss["EAL"], m, r, ss["PA"], k, ss["SA"], ss["SpA"], label,
                          ss["a_seed"], ss["maxabs"], 2, _ptr_array(win_ptrs[g0:g1]), 1, st)
                if not single:
                    committed[gi % 2].record(sc)

        commit(0)
        outs = [self._out(m, outs[i] if outs is not None else None, out_mode) for i in range(n_items)]
        out_ptrs = [o.data_ptr() for o in outs] if out_mode != OUT_NONE else [0] * n_items
        dump_ptrs = [d.data_ptr() for d in dumps] if dumps is not None else None
        flags = (FLAG_HASH if hash_tiles else 0) | FLAG_DENOISE
        B, SBt, target = _p(self.BpEBt), _p(self.SBt), _p(self.target)
        asc, bsc = _p(a_scale), _p(self.b_scale)
        for gi, (g0, g1) in enumerate(bounds):
            if gi + 1 < len(bounds):
                commit(gi + 1)
            cnt = g1 - g0
            ss = self._slot_set(m, gi % 2, group, cnt)
            if not single:
                cur.wait_event(committed[gi % 2])
            st = cur.cuda_stream
            # 3.-4. the nonces' noised operands and projections (own slot and corrB copy), one launch
            _lib.call("uwc_side_project_many", cnt, _ptr_array(a_ptrs[g0:g1]), ss["EAL"], ss["SpA"], ss["ApEA"], SBt,
                      ss["corrA"], 0, r, B, ss["SA"], ss["corrB"], r, m, n, k, r, ss["maxabs"], ss["limbs"], st)
            # 5. their hashed GEMMs with exact denoise, one batched call
            gargs = (cnt, ss["ApEA"], B, m, n, k, r, ss["corrA"], ss["corrB"], ss["maxabs"], ss["limbs"], ss["a_seed"],
                     target, _ptr_array(win_ptrs[g0:g1]), self.max_wins, asc, bsc, _ptr_array(out_ptrs[g0:g1]),
                     out_mode, flags, _ptr_array(dump_ptrs[g0:g1]) if dump_ptrs is not None else None)
            _lib.call("uwc_noisy_gemm_many", *gargs, st)
            if not single:
                consumed[gi % 2].record(cur)
        self._last_gemm = (cnt, lambda: _lib.call("uwc_noisy_gemm_many", *gargs, _stream()))
        if host is not None:  # winners(m) reports the sweep's last nonce, as after forward()
            self._buf(m)["wins"].copy_(host[n_items - 1])
        if not single:
            cur.wait_stream(sc)
        return outs

    def noise_mine(self, A: torch.Tensor, dump=None):
        """One attempt of a miner that wants only tiles, not the product (ops.py:349-364): the
        commitment and noise of A, the noised operand, and the hashed GEMM with every tile
        digested. With no output there is nothing to denoise, so the projections X, Y are
        skipped too."""
        m, k = A.shape
        n, r = self.n, self.r
        _check(k == self.k and m % BM == 0, f"MinedWeight.noise_mine: A is {tuple(A.shape)}")
        dev = A.device
        b = self._buf(m)
        c = consts(dev)
        b3_root_and_seed(A.view(-1), self.job_key, prefix=self.b_seed, salt=c["SALT_A"], dim=m,
                         seed_out=b["a_seed"], scratch=b["scratch"])
        nonce_noise(b["EAL"], b["PA"], k, r, c["LABEL_A"], b["a_seed"], zero0=b["wins"][:1])
        if m % 16 == 0 and k % 64 == 0 and r <= 128:
            noise_project(A, m, k, r, E=b["EAL"], Pn=b["PA"], dst=b["ApEA"])
        else:
            noise_rows(A, m, k, r, E=b["EAL"], Pn=b["PA"], dst=b["ApEA"])
        gemm(b["ApEA"], self.BpEBt, r=r, flags=FLAG_HASH, key=b["a_seed"], target=self.target, wins=b["wins"],
             max_wins=self.max_wins, dump=dump)

    def winners(self, m: int) -> list[tuple[int, int, bytes]]:
        """(row_offset, col_offset, hash) for winning tiles of the last forward with this m
        (ops.py:366-371; reads the device buffer, so it waits for the work queued so far)."""
        return win_records(self._buf(m)["wins"], self.max_wins)

    def sweep_winners(self) -> list[list[tuple[int, int, bytes]]]:
        """Every nonce's winners of the last forward_many without caller win buffers, in item
        order (one device-to-host copy of the sweep's rows; waits for the work queued so far)."""
        _check(getattr(self, "_sweep_host", None) is not None,
               "MinedWeight.sweep_winners: no forward_many without caller win buffers has run")
        rows, n_items = self._sweep_host
        host = rows[:n_items].cpu()
        return [win_records(host[i], self.max_wins) for i in range(n_items)]


def win_records(buf: torch.Tensor, max_wins: int) -> list[tuple[int, int, bytes]]:
    """Parse a win buffer [count, (row, col, digest[8]) x max_wins] (kernels.cu:586-595): the
    first min(count, max_wins) records as (row_offset, col_offset, 32-byte digest)."""
    w = buf.detach().to("cpu").numpy().view(np.uint32)
    kept = min(int(w[0]), max_wins)
    out = []
    for rec in np.split(w[1:1 + kept * WIN_WORDS], kept) if kept else []:
        out.append((int(rec[0]), int(rec[1]), rec[2:].tobytes()))
    return out


class GraphedForward:
    """MinedWeight.forward at a fixed m replayed from one HIP graph (ops.py:374-396): the input,
    scale and output tensors are the graph's own (copy activations into .A, read .out).

    The captured forward records kernels only: the win counter and maxabs are cleared by the
    noise launch, never by a memset node. Before capture one eager forward on the capture stream
    allocates the workspace this (m, k, r) shares and sets the kernels' launch attributes, neither
    of which may happen inside a capture."""

    def __init__(self, w: MinedWeight, m: int, out_mode: int = OUT_BF16):
        self.w, self.m, self.out_mode = w, m, out_mode
        dev = w.device
        self.A = torch.zeros((m, w.k), dtype=torch.int8, device=dev)
        self.a_scale = torch.ones(m, dtype=torch.float32, device=dev)
        self.out = w._out(m, None, out_mode)
        self.graph = torch.cuda.CUDAGraph()
        self._record(torch.cuda.Stream(device=dev))

    def _forward(self):
        self.w.forward(self.A, self.a_scale, out=self.out, out_mode=self.out_mode)

    def _record(self, stream: torch.cuda.Stream):
        caller = torch.cuda.current_stream(self.w.device)
        stream.wait_stream(caller)
        with torch.cuda.stream(stream):
            self._forward()  # eager: workspace and attributes
            stream.synchronize()
            with torch.cuda.graph(self.graph, stream=stream):
                self._forward()
        caller.wait_stream(stream)

    def __call__(self) -> torch.Tensor:
        self.graph.replay()
        return self.out
