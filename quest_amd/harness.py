"""Host-side counterparts of the reference's inference harness (gemm-quest/benchmarks/utils.py and
bench_e2e.py) on top of the HIP kernels: weight preparation, the W4A4 linear forward, the
`Linear4bit` module and the timing helpers.

Same function names, argument order and defaults as the reference.  The `backend` argument is
kept for call-site compatibility: 'hip' (default) and the reference's 'triton' / 'cuda' all run
the HIP kernels; 'pytorch' (the reference's eager-torch twin) is not part of this build.
"""
from __future__ import annotations

import torch
from torch import nn

from . import api as quest
from ._lib import host as native
from .api import HADAMARD_ENTRY

_HIP_BACKENDS = ('hip', 'triton', 'cuda')
WEIGHT_HADAMARD_SCALE = 2. ** -3.5      # utils.py:39

# Which matrix instructions the GEMM of `linear_forward` / `Linear4bit` runs on when the weight's E2M3 tiles are at
# hand: 'fp6' = the FP6 (E2M3) kernels where they are the faster ones, 'int8' = always the
# INT8 kernels on packed nibbles.  Both give the same bits.
MATRIX_PATH = 'fp6'
E2M3_MIN_TOKENS = 33                    # a fused block: from here on (see block_prefers_e2m3); a layer: see prefers_e2m3
E2M3_MIN_K = 1536                       # shortest rows that take them at more than E2M3_SHORT_ROWS_TOKENS tokens
E2M3_MIN_K_NARROW = 2048                # ... by a layer of fewer than E2M3_NARROW channels
E2M3_NARROW = 1536
E2M3_SHORT_ROWS_TOKENS = 4096
E2M3_RESIDENT_MAX_K = 1664              # longest rows of the FP6 kernel that keeps a channel tile's weights in LDS
E2M3_RESIDENT_WIDE = 16384              # ... which takes more channels only at more than
E2M3_RESIDENT_WIDE_TOKENS = 4864        # so many tokens (and, at fewer, some that the INT8 kernels keep)
# Whether a producer-fused block lets the FP6 GEMM of an output projection add into the residual stream itself
# (same bits as the addition inside the next norm kernel; one pass over the stream less).
GEMM_ADDS_RESIDUAL = True
GEMM_ADDS_RESIDUAL_PACKED = True       # ... also on packed nibbles, where the INT8 large-tile kernel takes the projection
# ... and the rotary embedding of q and k after the fused QKV projection (the FP6 GEMM's rotary epilogue)
GEMM_ROTATES_QK = True


def prefers_e2m3(m: int, k: int, n: int) -> bool:
    """Whether the FP6 kernels are the faster ones for an (m, k) x (n, k) layer on its own, quantiser included, with rows of whole 128s.  The rule
    is native code (csrc/host.cpp, with both sides of its lines, and what differs for other rows), for a layer's call asks it there: it was
    0.25 us of a call in Python."""
    return MATRIX_PATH == 'fp6' and native.prefers_e2m3(m, k, n, E2M3_MIN_K, E2M3_MIN_K_NARROW, E2M3_NARROW, E2M3_SHORT_ROWS_TOKENS)


def one_launch_on_tiles(m: int, k: int, n: int) -> bool:
    """Whether a layer on tiles is one launch at sizes where the INT8 kernels are the slower ones on the GPU too (csrc/host.cpp)."""
    return native.one_launch_on_tiles(m, k, n)


def block_prefers_e2m3(m: int, k: int, n: int) -> bool:
    """The same for a projection of a producer-fused block, where the FP6 kernels also save launches (the rotary embedding, the gated
    unit and both residual additions ride in their epilogues at every size).  Whole blocks, d = 256 to 4096, 33 to 4000 tokens,
    weights from HBM, INT8 / FP6 time: 0.97 to 1.18 ((d = 768, 1000 tokens) 0.97, (2560, 200) 0.99, (1024, 37) 1.08, (2560, 64)
    1.14, (4096, 500) 1.17).  Many tokens with short rows have a kernel of their own (gemm_e2m3_resident.hip), INT8 / FP6 time of
    the GEMM: (16384, 1024) x 1024 with the residual 1.28, x 3072 rotary 1.35, x 5632 gated 1.40; (16384, 768) x 1024 1.26; (8192,
    768) x 5632 1.45."""
    return (MATRIX_PATH == 'fp6' and m >= E2M3_MIN_TOKENS and k % 128 == 0 and native.tiles_addressable(m, k, n)
            and (m <= E2M3_SHORT_ROWS_TOKENS or _enough_per_row(k, n) or
                 (768 <= k <= E2M3_RESIDENT_MAX_K and n % 16 == 0 and (n <= E2M3_RESIDENT_WIDE or m > E2M3_RESIDENT_WIDE_TOKENS))))


def _enough_per_row(k: int, n: int) -> bool:
    # With short rows and many tokens the GEMM is mostly epilogue either way and the tile-writing activation kernels are a little
    # slower than the row-writing ones (12.0 against 10.2 us at [16384, 1024]).  Whole layers of 4097 to 16384 tokens, INT8 / FP6
    # time on the 256 x 256 tiles: K = 1792 1.14, K = 1920 1.16; K = 1024 0.85 to 1.18, K = 1152 to 1408 0.94 to 1.27.  Layers of 1024
    # channels lose 6 to 12 % at 8192 tokens up to K = 1920 (half a 256 x 256 tile per CU).  The resident channel tile has changed that up
    # to K = 1664 ((4097, 1536, 1536) 32.8 / 24.1 us, (8192, 1536, 8192) 120 / 78, (16384, 1536, 3072) 92 / 71): K = 640 to 1408 1.0 to 1.69 but for
    # less than 1024 channels ((16384, 1024, 8192) 164 / 117; (7883, 640, 904) 0.81).  Fused blocks follow it, layers on their own not yet.
    return k >= (E2M3_MIN_K if n >= E2M3_NARROW else E2M3_MIN_K_NARROW)


def e2m3_fits(k: int, rows: int) -> bool:
    """Whether codes of `rows` rows can be laid out as E2M3 tiles and multiplied by the FP6 kernels."""
    return k % 128 == 0 and 0 < k <= 65536 and rows <= 32 * 65535 and (rows + 287) // 32 * (k // 64) * 1536 < 1 << 31


def tiles_k(k: int, use_hadamard: bool) -> int:
    """The row length that a layer's tiles are laid out for: without the transform, rows of whole 32s get zeros up to a whole 128."""
    return k if use_hadamard or k % 32 else (k + 127) // 128 * 128


def _scales_in_pairs(scale) -> bool:
    """Whether the FP6 kernels can read a scale vector: two 16-bit values at a time."""
    return scale is None or scale.data_ptr() % 4 == 0


def weight_tiles(w_int_packed: torch.Tensor, out: torch.Tensor = None) -> torch.Tensor:
    """The E2M3 tiles of packed weight codes (N, K/2): the FP6 kernel's operand form (1.5 x the packed bytes)."""
    return quest.int4_to_e2m3_tiles(w_int_packed, out)


def _check_backend(backend: str) -> None:
    if backend not in _HIP_BACKENDS:
        raise NotImplementedError(
            f"backend {backend!r}: this build runs the HIP kernels only ('hip'; 'triton' and 'cuda' are aliases)")


def find_scale_int4(x: torch.Tensor, scale: torch.Tensor = None, backend: str = 'hip') -> torch.Tensor:
    """utils.py:114-159.  x: (..., K) -> scale (..., 1)."""
    _check_backend(backend)
    if scale is None:
        scale = torch.empty(*x.shape[:-1], 1, dtype=x.dtype, device=x.device)
    quest.find_scale_int4(x.view(-1, x.size(-1)), scale.view(-1, 1))
    return scale


def quantize_int4(x, scale, x_int=None, x_int_packed=None, x_int_row_sum=None, do_dequantize=False, backend='hip'):
    """utils.py:212-270."""
    _check_backend(backend)
    k = x.size(-1)
    quest.quantize_int4(
        x.view(-1, k), scale.view(-1, 1),
        None if x_int is None else x_int.view(-1, k),
        None if x_int_packed is None else x_int_packed.view(-1, k // 2),
        None if x_int_row_sum is None else x_int_row_sum.view(-1, 1),
        do_dequantize)
    return x, x_int, x_int_packed, x_int_row_sum


def add_mul_vv(vec_a_add, vec_a_mul, vec_b_add, vec_b_mul, mat_c, mat_d=None, backend='hip'):
    """utils.py:448-502."""
    _check_backend(backend)
    return quest.add_mul_vv(vec_a_add, vec_a_mul, vec_b_add, vec_b_mul, mat_c, mat_d)


def unpack_int4(x_int_packed: torch.Tensor, meta_e_no_reorder: torch.Tensor = None) -> torch.Tensor:
    """utils.py:420-445 (dense branch): uint8 (..., K/2) -> int8 (..., K), low nibble first."""
    if meta_e_no_reorder is not None:
        raise NotImplementedError('4:8-sparse weights are not part of this build')
    x_int = torch.empty(*x_int_packed.shape[:-1], x_int_packed.size(-1) * 2, dtype=torch.int8, device=x_int_packed.device)
    x_int[..., ::2] = x_int_packed & 0xF
    x_int[..., 1::2] = x_int_packed >> 4
    return torch.where(x_int >= 8, x_int - 16, x_int)


def fused_matmul_dequantize_int4_bf16(mat_a, mat_b, vec_a_add, vec_b_add, vec_a_mul, vec_b_mul, mat_d,
                                      _mat_c=None, debug_mode=True):
    """utils.py:548-587.  debug_mode=True runs the int32 GEMM and the scale epilogue as two
    launches, debug_mode=False the single fused kernel; both give the same bits here."""
    m, n = mat_a.size(0), mat_b.size(0)
    if mat_d is None:
        mat_d = torch.empty(m, n, dtype=vec_a_mul.dtype, device=mat_a.device)
    if debug_mode:
        mat_c = torch.empty(m, n, dtype=torch.int32, device=mat_a.device) if _mat_c is None else _mat_c
        quest.matmul_int4_int4t_int32(mat_a=mat_a, mat_b=mat_b, out=mat_c)
        quest.add_mul_vv(vec_a_add=vec_a_add, vec_a_mul=vec_a_mul, vec_b_add=vec_b_add, vec_b_mul=vec_b_mul,
                         mat_c=mat_c, mat_d=mat_d)
    else:
        quest.fused_matmul_dequantize_int4_int4t_bf16(mat_a=mat_a, mat_b=mat_b, vec_a_add=vec_a_add, vec_b_add=vec_b_add,
                                                      vec_a_mul=vec_a_mul, vec_b_mul=vec_b_mul, out=mat_d)
    return mat_d


def preprocess_weight(weight: torch.Tensor, use_sparse: bool = False, use_hadamard: bool = False, backend: str = 'hip',
                      w_scale_mode: str = 'rms', quantize_from_fp32: bool = False):
    """utils.py:20-53, dense branch: (N, K) float weight -> (w_int_packed (N, K/2) uint8,
    w_scale (N, 1), w_add (N, 1) int32 = row sum of the codes + K/2, None)."""
    _check_backend(backend)
    if use_sparse:
        raise NotImplementedError('4:8-sparse weights are not part of this build')
    weight = weight.contiguous()
    rule = {'rms': 'gaussian', 'absmax': 'absmax'}[w_scale_mode]
    done = quest.host.pack_weight(weight, WEIGHT_HADAMARD_SCALE if use_hadamard else 0., {'gaussian': 0, 'absmax': 1}[rule] | (4 if quantize_from_fp32 else 0))
    if done is not None:
        return *done, None
    n, k = weight.shape
    w_scale = torch.empty(n, 1, dtype=weight.dtype, device=weight.device)
    w_int_packed = torch.empty(n, k // 2, dtype=torch.uint8, device=weight.device)
    w_int_row_sum = torch.empty(n, 1, dtype=torch.int32, device=weight.device)
    # one pass: weight-side Hadamard (scale 2^-3.5) when asked, then scale, codes and row sums
    # (w_scale_mode: 'rms' is the reference's rule, 'absmax' puts the row's largest magnitude at the grid's edge)
    quest.hadamard_quantize_int4(weight, w_scale, w_int_packed, w_int_row_sum,
                                 hadamard_scale=WEIGHT_HADAMARD_SCALE if use_hadamard else 0.,
                                 scale_rule=rule, from_fp32=quantize_from_fp32)
    w_add = w_int_row_sum + k // 2
    return w_int_packed, w_scale, w_add, None


def linear_forward(activation, w_int_packed, w_scale, w_add, w_meta_e=None, out=None, _a_scale=None,
                   _a_int_packed=None, _a_int_row_sum=None, _c=None, use_hadamard=False, backend='hip', w_tiles=None,
                   _a_tiles=None, quantize_from_fp32=False):
    """utils.py:56-111, dense branch: out (M, N) = quantised activation @ quantised weight^T.
    Two launches: the fused Hadamard-scale-quantise-pack kernel, then the GEMM with the scale
    epilogue (the reference uses four).  With `w_tiles` (`weight_tiles(w_int_packed)`) and enough tokens the codes
    travel as E2M3 tiles and the GEMM runs on the FP6 matrix instructions: the same output bits, faster.
    quantize_from_fp32 (with use_hadamard): the activation codes come from the fp32 transform (factor 2^-3.5, the
    reference's evaluation-side arithmetic, src/eval_hswag.py:201-214) instead of from its 16-bit rounding."""
    _check_backend(backend)
    if w_meta_e is not None:
        raise NotImplementedError('4:8-sparse weights are not part of this build')
    m, k, n = activation.size(0), activation.size(1), w_int_packed.size(0)
    if w_tiles is not None and not prefers_e2m3(m, k, n):
        w_tiles = None
    if (_a_scale is None and _a_int_packed is None and _a_int_row_sum is None and _a_tiles is None
            and not (quantize_from_fp32 and use_hadamard) and activation.dim() == 2):
        done = quest.host.linear(activation, w_int_packed, w_scale, w_add, w_tiles, None, HADAMARD_ENTRY if use_hadamard else 0., out)
        if done is not None:
            return done
    dtype, device = activation.dtype, activation.device
    if out is None:
        out = torch.empty(m, n, dtype=dtype, device=device)
    if quantize_from_fp32 and use_hadamard:
        a_scale, a_int_packed, a_int_row_sum = quest.hadamard_quantize_int4(
            activation, _a_scale, _a_int_packed, _a_int_row_sum, hadamard_scale=WEIGHT_HADAMARD_SCALE, from_fp32=True)
        return quest.fused_matmul_dequantize_int4_int4t_bf16(mat_a=a_int_packed, mat_b=w_int_packed, vec_a_add=a_int_row_sum,
                                                             vec_b_add=w_add, vec_a_mul=a_scale, vec_b_mul=w_scale, out=out)
    if w_tiles is not None and _scales_in_pairs(w_scale) and _scales_in_pairs(_a_scale):
        a_scale, a_tiles = quest.hadamard_quantize_e2m3(activation, _a_scale, _a_tiles,
                                                        hadamard_scale=HADAMARD_ENTRY if use_hadamard else 0.)
        return quest.fused_matmul_dequantize_e2m3(a_tiles, w_tiles, a_scale, w_scale, k, out)
    a_scale = torch.empty(m, 1, dtype=dtype, device=device) if _a_scale is None else _a_scale
    a_int_packed = torch.empty(m, k // 2, dtype=torch.uint8, device=device) if _a_int_packed is None else _a_int_packed
    a_int_row_sum = torch.empty(m, 1, dtype=torch.int32, device=device) if _a_int_row_sum is None else _a_int_row_sum
    quest.hadamard_quantize_int4(activation, a_scale, a_int_packed, a_int_row_sum,
                                 hadamard_scale=HADAMARD_ENTRY if use_hadamard else 0.)
    quest.fused_matmul_dequantize_int4_int4t_bf16(mat_a=a_int_packed, mat_b=w_int_packed, vec_a_add=a_int_row_sum,
                                                  vec_b_add=w_add, vec_a_mul=a_scale, vec_b_mul=w_scale, out=out)
    return out


class Linear4bit(nn.Module):
    """bench_e2e.py:41-70: a linear layer that holds its weight as packed INT4 codes.

    Buffers, as in the reference: `w_int_packed` (N, K/2) uint8, `w_scale` (N, 1), `w_add` (N, 1) int32 and the
    unused `w_meta_e`; `weight` is a shape-only meta tensor; `bias` is a parameter or None.  The plain constructor
    packs the weight of a freshly initialised `nn.Linear` (the benchmarks never load trained weights),
    `from_weight` packs a given one and `empty` leaves the buffers to `load_state_dict`."""

    def __init__(self, in_features: int, out_features: int, bias: bool = True, device=None, dtype=None,
                 use_sparse: bool = False, use_hadamard: bool = False, use_noop: bool = False):
        super().__init__()
        if use_sparse:
            raise NotImplementedError('4:8-sparse weights are not part of this build')
        dense = nn.Linear(in_features, out_features, bias=bias, device=device, dtype=dtype)
        self._configure(use_hadamard, use_noop)
        self._install(dense.weight.data, dense.bias)

    def _configure(self, use_hadamard: bool, use_noop: bool) -> None:
        self.use_hadamard = use_hadamard
        self.use_noop = use_noop
        # codes from the fp32 transform instead of its 16-bit rounding (see linear_forward); set before packing a weight
        self.quantize_from_fp32 = getattr(self, 'quantize_from_fp32', False)

    def _install(self, weight: torch.Tensor, bias, lay_out: bool = True) -> None:
        """Pack `weight` (N, K) and keep `bias` (a tensor, a parameter or None) as a frozen parameter."""
        with torch.inference_mode(False), torch.no_grad():           # buffers with a version counter: see _kept_tiles
            packed, scale, add, _ = preprocess_weight(weight=weight, use_hadamard=self.use_hadamard,
                                                      quantize_from_fp32=self.quantize_from_fp32)
        self._set_buffers(weight.shape, weight.dtype, packed, scale, add)
        if lay_out:
            self.lay_out_tiles()
        if bias is None:
            self.bias = None
        else:
            self.bias = nn.Parameter(bias.detach().to(weight.dtype), requires_grad=False)

    def _set_buffers(self, shape, dtype, packed, scale, add) -> None:
        self.weight = torch.empty(shape, dtype=dtype, device='meta')
        for name, t in (('w_int_packed', packed), ('w_scale', scale), ('w_add', add), ('w_meta_e', None)):
            self.register_buffer(name, t)
        self._tiles = None               # (E2M3 tiles, of which tensor, its address, its version): derived, not in checkpoints

    def lay_out_tiles(self) -> None:
        """Keep the weight codes as E2M3 tiles as well, the FP6 kernels' operand form (1.5 x the packed bytes on top of them).
        Done where the buffers get their content -- packing, `load_state_dict`, a move to another device, a copy -- on the stream
        that writes them, so whoever may read the buffers may read the tiles, and no forward call, on whatever stream or
        under capture, has anything to build.  After writing into `w_int_packed` by hand, call it again: until then the layer runs on
        its packed codes (the same bits), but for a graph captured before, which reads the tiles.  They are rewritten in place while
        the buffer stays where it is, so that such a graph follows a reload as it does on packed codes.  Nothing is kept for a
        layer that the FP6 kernels do not take, or while MATRIX_PATH is 'int8'."""
        before, self._tiles = self._tiles, None
        with torch.inference_mode(False), torch.no_grad():
            for name, t in self._buffers.items():
                if type(t) is torch.Tensor and t.is_inference():     # (it would not show later writes)
                    self._buffers[name] = t.clone()
            w = self._buffers.get('w_int_packed')
            if type(w) is not torch.Tensor or not w.is_cuda or w.dim() != 2 or not w.is_contiguous():
                return
            k = w.size(1) * 2
            padded = tiles_k(k, self.use_hadamard)
            if MATRIX_PATH == 'fp6' and e2m3_fits(padded, w.size(0)) and (padded == k or 640 <= padded <= 32768):      # (others: see csrc/host.cpp)
                in_place = before is not None and before[1] is w and before[2] == w.data_ptr()
                lay = weight_tiles if padded == k else quest.int4_to_e2m3_tiles_padded
                self._tiles = (lay(w, before[0] if in_place else None), w, w.data_ptr(), w._version)

    def _kept_tiles(self):
        """The tiles of what `w_int_packed` holds now, or None."""
        kept = self._tiles
        if kept is None:
            return None
        tiles, source, address, version = kept                        # (what csrc/host.cpp asks as well: unchanged())
        w = self._buffers.get('w_int_packed')
        return tiles if w is source and w._version == version and w.data_ptr() == address else None

    def tiles_for(self, m: int):
        """The weight's E2M3 tiles where the FP6 kernels are the faster ones for m tokens, None where the packed codes serve."""
        n, k = self.weight.shape
        return self.readable_tiles() if prefers_e2m3(m, k, n) else None

    def readable_tiles(self):
        """The kept tiles, if the FP6 kernels can read the scales beside them and the rows are whole 128s."""
        return self._kept_tiles() if _scales_in_pairs(self.w_scale) and self.weight.size(1) % 128 == 0 else None

    def w_tiles(self) -> torch.Tensor:
        """The weight codes as E2M3 tiles: the kept ones, or a conversion of the buffer for this call."""
        tiles = self._kept_tiles() if self.weight.size(1) % 128 == 0 else None
        return weight_tiles(self.w_int_packed) if tiles is None else tiles

    def _load_from_state_dict(self, *args, **kwargs):
        super()._load_from_state_dict(*args, **kwargs)
        self.lay_out_tiles()

    def _apply(self, *args, **kwargs):
        super()._apply(*args, **kwargs)
        if self._kept_tiles() is None:
            self.lay_out_tiles()
        return self

    def __getstate__(self):
        return {**self.__dict__, '_tiles': None}

    def __setstate__(self, state):
        super().__setstate__(state)
        self.lay_out_tiles()

    @classmethod
    def from_weight(cls, weight: torch.Tensor, bias: torch.Tensor = None, use_hadamard: bool = False,
                    quantize_from_fp32: bool = False, lay_out: bool = True) -> 'Linear4bit':
        """Pack an existing (N, K) weight instead of a random one.  lay_out: keep its E2M3 tiles as well (`lay_out_tiles`)."""
        self = cls.__new__(cls)
        nn.Module.__init__(self)
        self.quantize_from_fp32 = bool(quantize_from_fp32)
        self._configure(use_hadamard, False)
        self._install(weight, bias, lay_out)
        return self

    @classmethod
    def empty(cls, in_features: int, out_features: int, bias: bool = False, device=None, dtype=None,
              use_hadamard: bool = False) -> 'Linear4bit':
        """A layer of the given shape with unset buffers, to be filled by `load_state_dict` from a packed checkpoint."""
        self = cls.__new__(cls)
        nn.Module.__init__(self)
        self._configure(use_hadamard, False)
        with torch.inference_mode(False):
            self._set_buffers((out_features, in_features), dtype,
                              torch.zeros(out_features, in_features // 2, dtype=torch.uint8, device=device),
                              torch.zeros(out_features, 1, dtype=dtype, device=device),
                              torch.zeros(out_features, 1, dtype=torch.int32, device=device))
        self.bias = nn.Parameter(torch.zeros(out_features, dtype=dtype, device=device), requires_grad=False) if bias else None
        return self

    def forward_quantized(self, a_scale, a_int_packed, a_int_row_sum, out=None, rope=None, add_to_out=False) -> torch.Tensor:
        """The GEMM half of `linear_forward` on activations some fused producer kernel has already quantised:
        (M, 1) scales, (M, K/2) codes, (M, 1) row sums -> (M, N).  In no-op mode the GEMM is skipped (zeros), which is
        what prices the GEMMs of a producer-fused model: everything else, the quantising producers included, still runs.
        rope = (freqs_cis, rot_cols, head_dim): the first rot_cols channels leave rotated (layers without a bias).
        add_to_out: the result is added to `out` (the residual stream), with the bits of `out + layer(x)` (layers without
        a bias; one launch where `quest.gemm_add_fuses` says so)."""
        if self.use_noop:
            return out if add_to_out else self._noop_output(a_scale)
        if add_to_out:
            assert self.bias is None and rope is None and out is not None
            return quest.fused_matmul_dequantize_add_int4_int4t(a_int_packed, self.w_int_packed, a_int_row_sum, self.w_add,
                                                                a_scale, self.w_scale, out)
        if rope is not None:
            assert self.bias is None
            return quest.fused_matmul_dequantize_rope_int4_int4t(a_int_packed, self.w_int_packed, a_int_row_sum, self.w_add,
                                                                 a_scale, self.w_scale, *rope, out=out)
        y = quest.fused_matmul_dequantize_int4_int4t_bf16(mat_a=a_int_packed, mat_b=self.w_int_packed,
                                                          vec_a_add=a_int_row_sum, vec_b_add=self.w_add,
                                                          vec_a_mul=a_scale, vec_b_mul=self.w_scale, out=out)
        if self.bias is not None:
            y += self.bias
        return y

    def _noop_output(self, a_scale) -> torch.Tensor:
        y = torch.zeros(a_scale.numel(), self.weight.size(0), dtype=a_scale.dtype, device=a_scale.device)
        if self.bias is not None:
            y += self.bias
        return y

    def forward_tiles(self, a_scale, a_tiles, out=None, add_to_out=False, rope=None) -> torch.Tensor:
        """The same for activations quantised to E2M3 tiles: the GEMM on the FP6 matrix instructions.  add_to_out: the
        result is added to `out` (the residual stream) inside the GEMM's launch, with the bits of `out + layer(x)`.
        rope = (freqs_cis, rot_cols, head_dim): the rotary embedding of the first rot_cols channels in the GEMM's launch
        (layers without a bias; the caller checks `quest.rope_gemm_fuses`)."""
        if self.use_noop:
            return out if add_to_out else self._noop_output(a_scale)
        if add_to_out and self.bias is not None:                     # out + (product + bias): the bias first, as torch would
            y = quest.fused_matmul_dequantize_e2m3(a_tiles, self.w_tiles(), a_scale, self.w_scale, self.weight.size(1))
            y += self.bias
            out += y
            return out
        assert rope is None or self.bias is None
        y = quest.fused_matmul_dequantize_e2m3(a_tiles, self.w_tiles(), a_scale, self.w_scale, self.weight.size(1), out,
                                               add_to_out=add_to_out, rope=rope)
        if self.bias is not None:
            y += self.bias
        return y

    def forward(self, x) -> torch.Tensor:
        if not self.use_noop and not self.quantize_from_fp32 and x.dim() > 0:
            held = self._buffers.get                  # (not there, e.g. made a parameter: the native call declines)
            if held('w_meta_e') is None:
                y = quest.host.linear(x, held('w_int_packed'), held('w_scale'), held('w_add'), self._tiles if MATRIX_PATH == 'fp6' else None, self.bias,
                                      HADAMARD_ENTRY if self.use_hadamard else 0., None,
                                      E2M3_MIN_K, E2M3_MIN_K_NARROW, E2M3_NARROW, E2M3_SHORT_ROWS_TOKENS)
                if y is not None:
                    return y
        lead, n = x.shape[:-1], self.weight.size(0)
        rows = x.contiguous().view(-1, x.size(-1))
        if self.use_noop:
            # the reference's no-op layer (bench_e2e.py:62-66) still rotates the activations, so that
            # "int4 minus noop" prices the quantiser and the GEMM only; the rotated tensor is dropped
            if self.use_hadamard:
                quest.hadamard128(rows)
            y = torch.zeros(rows.size(0), n, dtype=x.dtype, device=x.device)
        else:
            m, k = rows.shape
            y = linear_forward(rows, self.w_int_packed, self.w_scale, self.w_add, self.w_meta_e,
                               use_hadamard=self.use_hadamard, quantize_from_fp32=self.quantize_from_fp32,
                               w_tiles=None if self.quantize_from_fp32 else self.tiles_for(m))
        if self.bias is not None:
            y += self.bias
        return y.view(*lead, n)


def _elapsed_s(fn, n_iter: int) -> float:
    """Seconds per call of `fn`, from a pair of HIP events on the current stream around n_iter calls."""
    start, stop = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    start.record()
    for _ in range(n_iter):
        fn()
    stop.record()
    stop.synchronize()
    return start.elapsed_time(stop) * 1e-3 / n_iter


@torch.inference_mode()
def do_bench(f, n_iter: int = 100, n_warmup: int = 10) -> float:
    """utils.py:789-799: seconds per call of `f` after `n_warmup` untimed calls.  The reference brackets the timed
    calls with device synchronisations and the host clock; here the bracket is a pair of HIP events on the stream
    the calls go to, which leaves the host's launch jitter before the first call out of the figure."""
    for _ in range(n_warmup):
        f()
    torch.cuda.synchronize()
    return _elapsed_s(f, n_iter)


@torch.inference_mode()
def do_bench_network(f, M: int, K: int, N: int, dtype: torch.dtype, device: torch.device, n_layers: int = 20,
                     n_warmup: int = 3) -> float:
    """utils.py:802-835: `f(activation_in (M, K), activation_out (M, N))` called `n_layers` times back to back on
    two views of one buffer (so that no call finds a fresh output allocation), timed as plain launches and as one
    replayed HIP graph; returns the smaller of the two, in seconds per layer."""
    # Gaussian values, not the reference's uninitialised memory: the kernels' run time depends on the data (degenerate
    # rows take a slower quantiser path, the clock follows the operands' power), and garbage would time something else
    pool = torch.randn(M * max(K, N), dtype=torch.float32, device=device).to(dtype)
    a_in, a_out = pool[:M * K].view(M, K), pool[:M * N].view(M, N)

    def stack():
        for _ in range(n_layers):
            f(a_in, a_out)

    eager_s = do_bench(stack, n_iter=1, n_warmup=n_warmup)
    capture = torch.cuda.Stream(device=device)
    capture.wait_stream(torch.cuda.current_stream(device))
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(capture):
        for _ in range(n_warmup):
            stack()
        with torch.cuda.graph(graph, stream=capture):
            stack()
    torch.cuda.current_stream(device).wait_stream(capture)
    graph_s = do_bench(graph.replay, n_iter=1, n_warmup=n_warmup)
    return min(eager_s, graph_s) / n_layers
