"""Host side of the flash-attention prefill example on the host-less route."""
from __future__ import annotations

import hashlib
import json
from pathlib import Path

import numpy as np

from ..pipec.launcher import HostlessSession, open_hostless
from ..stages.attention.params import params_blobs

HEAD_DIM = 128
Q_TILE = 128
K_BLOCK = 64
COMPUTE_UNITS = 256
HALF_TILES_UP_TO = 384


def _half_tiles_pay(heads: int, s: int, window: int | None) -> bool:
    """Whether tiles of 64 queries, twice as many workgroups with a wave per half of each key block, take less time than tiles
    of 128.  Half tiles shorten a tile's chain of key blocks, which is all a launch takes while compute units are left over;
    they cost a start and a merge per workgroup, which short chains do not earn back, and loads twice once every compute unit
    has two workgroups.  us half / us whole over 3700 random shapes (1 to 384 tiles, S 128 to 4096, causal and windows of 20
    keys up; a launch against itself: 0.95 .. 1.05), by the longest chain L of a whole tile in blocks, the average A and the load F = tiles * A / (256 L),
    with whole and half tiles that waited for the next block's loads in front of their V reads:
      up to 128 tiles    0.69 .. 0.98 whatever the chains
      129 to 256 tiles   L 2: 1.2, L 4: 0.97 to 1.04, L 6: 0.97 (up to 1.16), L 8: 0.93 (up to 1.08); from L 10 on and F up to 0.78:
                         0.79 .. 0.98, two shapes of 460 above 1 (1.01 and 1.03, L 10); beyond: up to 1.11
      257 to 384 tiles   from L 12 on and F up to 0.78: 0.81 .. 0.98; beyond: up to 1.26; L 10: 0.9 to 1.13, L 7 and
                         less: 1.03 to 1.37
      512 tiles          1.07 (S 2048), 1.16 (S 512)
    Without that wait half tiles are the shorter ones a little further; 260 shapes of 1 to 512 tiles:
      up to 128 tiles    0.67 .. 0.98
      129 to 256 tiles   L 3 and less: 0.92 to 1.13, L 4 and 5: 0.91 to 1.07, L 6 to 9: 0.76 to 0.92; from L 10 on 0.70 .. 0.87
      257 to 384 tiles   from L 12 on 0.76 .. 0.92, L 8 to 11: 0.93 to 1.16, less 1.06 to 1.24
      385 to 512 tiles   from L 20 on 0.79 .. 0.99, L 12 to 19: 0.98 to 1.06, less 1.11 to 1.20
    The line is the first table's still: 1.6 % above the better of the two on average, 1.32 at worst (1920 keys, a window of 443,
    135 tiles)."""
    tiles = heads * (s // Q_TILE)
    if tiles <= COMPUTE_UNITS // 2 or tiles > HALF_TILES_UP_TO:
        return tiles <= COMPUTE_UNITS // 2
    chains = [(q + Q_TILE) // K_BLOCK - (max(0, q - window + 1) // K_BLOCK if window else 0) for q in range(0, s, Q_TILE)]
    longest = max(chains)
    return longest >= (10 if tiles <= COMPUTE_UNITS else 12) and heads * sum(chains) <= 0.78 * COMPUTE_UNITS * longest


def _half_of(link_json: Path, link_bytes: bytes) -> tuple[dict, Path] | None:
    """The half-tile link that was made for exactly this link (``stages.attention.build.link_half``) and its folder, if there is
    one: a link redone since, with another mask for instance, has other bytes than the one recorded."""
    folder = link_json.parent.parent / "half"
    try:
        of = json.loads((folder / "of.json").read_text())
        if hashlib.sha256(link_bytes).hexdigest() != of["whole"]:
            return None
        half_bytes = (folder / "link" / "link.json").read_bytes()
        return (json.loads(half_bytes), folder / "link") if hashlib.sha256(half_bytes).hexdigest() == of["half"] else None
    except (OSError, ValueError, KeyError, TypeError):
        return None


def open_session(link_json: str | Path | dict, q_bits: np.ndarray, k_bits: np.ndarray, v_bits: np.ndarray, *, scale: float | None = None,
                 window: int | None = None, backend=None, image: str | Path | None = None) -> HostlessSession:
    """q_bits [B, Hq, S, 128], k_bits / v_bits [B, Hkv, S, 128]: bf16 bit patterns (uint16).  Buffers: q, k, v and
    o ([B, S, Hq * 128] uint16, zeroed).  `window`: for a link with fa.mask.window, the number of keys a query sees.
    (A link names one mask package; the params blob must be addressed to it.)"""
    if window is not None and window < 1:
        raise ValueError("a window is at least one key")
    if scale is not None and not (np.isfinite(scale) and scale > 0):
        raise ValueError("the softmax scale must be a positive finite number (masked scores are -1e30 times it)")
    if q_bits.ndim != 4 or k_bits.shape != v_bits.shape or k_bits.ndim != 4:
        raise ValueError("q is [B, Hq, S, D]; k and v are [B, Hkv, S, D]")
    b, hq, s, d = q_bits.shape
    b2, hkv, s2, d2 = k_bits.shape
    if (b, s, d) != (b2, s2, d2) or d != HEAD_DIM or s % Q_TILE or hkv <= 0 or hq % hkv:
        raise ValueError("head dimension must be 128, the sequence a multiple of 128, query heads a multiple of KV heads")
    if any(t.dtype != np.uint16 for t in (q_bits, k_bits, v_bits)):
        raise ValueError("operands are uint16 bf16 bit patterns")
    if s * d * 2 >= 1 << 31:
        raise ValueError("one head of K or V must stay below 2 GiB")
    buffers = {"q": q_bits, "k": k_bits, "v": v_bits, "o": ((b, s, hq * d), np.uint16)}
    if isinstance(link_json, dict):
        link = link_json
    else:
        link_bytes = Path(link_json).read_bytes()
        link, folder = json.loads(link_bytes), Path(link_json).parent
        if image is None:   # (an image of the caller's own, and a link handed over as an object, are run as they are)
            half = _half_of(Path(link_json), link_bytes) if _half_tiles_pay(b * hq, s, window) else None
            link, folder = half or (link, folder)
            image = folder / link["target"]["image"]
    grid = b * hq * (s // link.get("facts", {}).get("fa.core.tile_queries", Q_TILE))
    return open_hostless(link, buffers=buffers, params=lambda addr: params_blobs(addr, b, hq, hkv, s, scale, window),
                         grid=(grid,), backend=backend, image=image)
