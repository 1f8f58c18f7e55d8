"""Op dispatch: hand-written gfx950 HIP kernels on GPU, fp32 torch
references on CPU.

On a CUDA/ROCm device the HIP extension is REQUIRED — a missing .so
raises immediately rather than silently falling back to eager PyTorch
(the round-end check records which native libraries the GPU tests
actually loaded).  On CPU the ops/ref.py implementations run, which is
what the no-GPU plumbing tests and the gloo multi-process tests use.
"""

from __future__ import annotations

import functools
import os
import torch
from torch._C._functorch import peek_interpreter_stack
from torch.autograd import forward_ad

from . import ref  # noqa: F401

_HERE = os.path.dirname(os.path.abspath(__file__))
_SO_PATH = os.path.join(_HERE, "_rlli_hip.so")
_loaded = False
_loaded_libs: set = set()


class ExtensionMissing(RuntimeError):
    pass


def load_extension(required: bool = False) -> bool:
    """Load the in-tree .so (idempotent).  ``required=True`` (or any GPU
    call) raises if it is absent — no silent eager fallback on GPU."""
    global _loaded
    if _loaded:
        return True
    if os.path.exists(_SO_PATH):
        torch.ops.load_library(_SO_PATH)
        _loaded = True
        return True
    if required:
        raise ExtensionMissing(
            f"HIP extension not built: {_SO_PATH} missing. "
            f"Run `python -m resilient_llm_amd.ops.build`.")
    return False


def extension_loaded() -> bool:
    return _loaded


def _gpu() -> None:
    load_extension(required=True)


def load_libraries(libs) -> None:
    """Load kernel libraries by name (idempotent); raises if one is not
    built."""
    for lib in libs:
        if lib in _loaded_libs:
            continue
        if lib == "rlli_hip":
            _gpu()
            continue
        path = os.path.join(_HERE, f"_{lib}.so")
        if not os.path.exists(path):
            raise ExtensionMissing(
                f"HIP extension not built: {path} missing. "
                f"Run `python -m resilient_llm_amd.ops.build`.")
        torch.ops.load_library(path)
        _loaded_libs.add(lib)


# ------------------------------------------------------------------ ops
def rmsnorm(x: torch.Tensor, w: torch.Tensor, eps: float = 1e-5) -> torch.Tensor:
    if x.is_cuda:
        _gpu()
        return torch.ops.rlli.rmsnorm(x, w, eps)
    return ref.rmsnorm(x, w, eps)


def rmsnorm_residual_(x: torch.Tensor, residual: torch.Tensor, w: torch.Tensor,
                      eps: float = 1e-5) -> torch.Tensor:
    """``x`` may be the f32 parts of rows_linear_parts."""
    if x.is_cuda:
        _gpu()
        if x.dim() == 3 and x.dtype == torch.float32:
            return torch.ops.rlli.rmsnorm_residual_parts_(x, residual, w, eps)
        return torch.ops.rlli.rmsnorm_residual_(x, residual, w, eps)
    return ref.rmsnorm_residual_(x, residual, w, eps)


def rmsnorm_fp8(x, w, eps: float = 1e-5):
    """Fused rmsnorm + per-row fp8-e4m3 quantization -> (q, scales)."""
    if x.is_cuda:
        _gpu()
        return torch.ops.rlli.rmsnorm_fp8(x, w, eps)
    return ref.rmsnorm_fp8(x, w, eps)


def rmsnorm_residual_fp8(x, residual, w, eps: float = 1e-5):
    if x.is_cuda:
        _gpu()
        return torch.ops.rlli.rmsnorm_residual_fp8(x, residual, w, eps)
    return ref.rmsnorm_residual_fp8(x, residual, w, eps)


def silu_mul_fp8(gate_up):
    if gate_up.is_cuda:
        _gpu()
        return torch.ops.rlli.silu_mul_fp8(gate_up)
    return ref.silu_mul_fp8(gate_up)


def silu_mul(gate_up: torch.Tensor) -> torch.Tensor:
    if gate_up.is_cuda:
        _gpu()
        return torch.ops.rlli.silu_mul(gate_up)
    return ref.silu_mul(gate_up)


def rope_kv_append_(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor,
                    positions: torch.Tensor, cos_sin: torch.Tensor,
                    k_cache: torch.Tensor, v_cache: torch.Tensor,
                    slot_mapping: torch.Tensor) -> None:
    if q.is_cuda:
        _gpu()
        torch.ops.rlli.rope_kv_append_(q, k, v, positions, cos_sin,
                                       k_cache, v_cache, slot_mapping)
    else:
        ref.rope_kv_append_(q, k, v, positions, cos_sin, k_cache, v_cache,
                            slot_mapping)


def rope_kv_append_qkv_(qkv: torch.Tensor, positions: torch.Tensor,
                        cos_sin: torch.Tensor, k_cache: torch.Tensor,
                        v_cache: torch.Tensor, slot_mapping: torch.Tensor,
                        n_q: int) -> None:
    """Fused-QKV form: rope + cache append on strided views of the raw
    qkv GEMM output (no .contiguous() copies)."""
    if qkv.is_cuda:
        _gpu()
        torch.ops.rlli.rope_kv_append_qkv_(qkv, positions, cos_sin, k_cache,
                                           v_cache, slot_mapping, n_q)
        return
    T = qkv.shape[0]
    n_kv, _, D = k_cache.shape[1], k_cache.shape[2], k_cache.shape[3]
    q = qkv[:, :n_q * D].view(T, n_q, D)
    k = qkv[:, n_q * D:(n_q + n_kv) * D].view(T, n_kv, D)
    v = qkv[:, (n_q + n_kv) * D:].view(T, n_kv, D)
    ref.rope_kv_append_(q, k, v, positions, cos_sin, k_cache, v_cache,
                        slot_mapping)


def decode_attn_qkv(qkv: torch.Tensor, k_cache: torch.Tensor,
                    v_cache: torch.Tensor, block_table: torch.Tensor,
                    seq_lens: torch.Tensor, scale: float,
                    n_q: int) -> torch.Tensor:
    if qkv.is_cuda:
        _gpu()
        return torch.ops.rlli.decode_attn_qkv(qkv, k_cache, v_cache,
                                              block_table, seq_lens, scale, n_q)
    B = qkv.shape[0]
    D = k_cache.shape[3]
    q = qkv[:, :n_q * D].reshape(B, n_q, D)
    out = ref.decode_attn(q, k_cache, v_cache, block_table, seq_lens, scale)
    return out.reshape(B, n_q * D)


def decode_attn_qkv_out(qkv, k_cache, v_cache, block_table, seq_lens,
                        scale: float, n_q: int, out: torch.Tensor) -> None:
    """decode_attn_qkv to the first rows of ``out``."""
    if qkv.is_cuda:
        _gpu()
        torch.ops.rlli.decode_attn_qkv_out(qkv, k_cache, v_cache, block_table,
                                           seq_lens, scale, n_q, out)
        return
    out[:qkv.shape[0]] = decode_attn_qkv(qkv, k_cache, v_cache, block_table,
                                         seq_lens, scale, n_q)


def decode_attn_rope_qkv(qkv, positions, cos_sin, k_cache, v_cache,
                         slot_mapping, block_table, seq_lens, scale: float,
                         n_q: int) -> torch.Tensor:
    """Fused decode step: rope(q,k) + cache append + paged attention in
    one kernel on GPU; composed from the unfused reference ops on CPU.
    ``qkv`` may be the f32 parts of rows_linear_parts."""
    if qkv.is_cuda:
        _gpu()
        return torch.ops.rlli.decode_attn_rope_qkv(
            qkv, positions, cos_sin, k_cache, v_cache, slot_mapping,
            block_table, seq_lens, scale, n_q)
    rope_kv_append_qkv_(qkv, positions, cos_sin, k_cache, v_cache,
                        slot_mapping, n_q)
    return decode_attn_qkv(qkv, k_cache, v_cache, block_table, seq_lens,
                           scale, n_q)


def decode_attn_rope_linear(qkv, positions, cos_sin, k_cache, v_cache,
                            slot_mapping, block_table, seq_lens, scale: float,
                            n_q: int, w: torch.Tensor) -> torch.Tensor:
    """rows_linear_parts of decode_attn_rope_qkv's result with w.  Of one long
    sequence the product puts its parts together, without a launch for it."""
    _gpu()
    return torch.ops.rlli.decode_attn_rope_linear(
        qkv, positions, cos_sin, k_cache, v_cache, slot_mapping, block_table,
        seq_lens, scale, n_q, w)


def decode_attn_rows_qkv(qkv, positions, cos_sin, k_cache, v_cache,
                         slot_mapping, block_table, seq_lens, scale: float,
                         n_q: int) -> torch.Tensor:
    """decode_attn_rope_qkv for rows that may belong to one sequence: all
    keys and values are appended first."""
    if qkv.is_cuda:
        _gpu()
        torch.ops.rlli.kv_append_qkv_(qkv, positions, cos_sin, k_cache,
                                      v_cache, slot_mapping, n_q)
        return torch.ops.rlli.decode_attn_q_rope(
            qkv, positions, cos_sin, k_cache, v_cache, block_table, seq_lens,
            scale, n_q)
    rope_kv_append_qkv_(qkv, positions, cos_sin, k_cache, v_cache,
                        slot_mapping, n_q)
    return decode_attn_qkv(qkv, k_cache, v_cache, block_table, seq_lens,
                           scale, n_q)


def mixed_row_tables(rows: int, n_decode: int, tables_dec, lens_dec,
                     chunk_row0, chunk_pos0, chunk_nrows, chunk_btrow,
                     tables_pre) -> tuple[torch.Tensor, torch.Tensor]:
    """Block table and length of every row of a mixed step, for
    decode_attn_rows_qkv; rows of no tile see nothing."""
    if tables_pre.is_cuda:
        _gpu()
        return torch.ops.rlli.mixed_row_tables(
            rows, n_decode, tables_dec, lens_dec, chunk_row0, chunk_pos0,
            chunk_nrows, chunk_btrow, tables_pre)
    return ref.mixed_row_tables(rows, n_decode, tables_dec, lens_dec,
                                chunk_row0, chunk_pos0, chunk_nrows,
                                chunk_btrow, tables_pre)


def rows_faster(M: int, *shapes) -> bool:
    """Whether M rows' products with weights of these shapes are rows_linear's,
    as far as the shapes go."""
    return all(K % 64 == 0 and N % 16 == 0 and _rows_faster(M, N, K)
               for N, K in shapes)


def prompt_rows_layer(x, residual, ln1, w_qkv, w_o, ln2, w_gate_up, w_down,
                      positions, cos_sin, k_cache, v_cache, slot_mapping,
                      cu_seqlens, eps: float, scale: float,
                      n_q: int) -> tuple[torch.Tensor, torch.Tensor]:
    """A Llama layer behind the first for few rows of whole prompts on the GPU:
    x + residual, normed, ... the last product, which may come in parts, and
    the new residual (``residual`` is updated on the way).  The results are
    those of the ops one by one; of up to 64 rows attention rotates and appends
    in its own launch."""
    _gpu()
    return torch.ops.rlli.prompt_rows_layer(
        x, residual, ln1, w_qkv, w_o, ln2, w_gate_up, w_down, positions,
        cos_sin, k_cache, v_cache, slot_mapping, cu_seqlens, eps, scale, n_q)


def prefill_attn_qkv(qkv: torch.Tensor, cu_seqlens: torch.Tensor,
                     scale: float, n_q: int, n_kv: int,
                     head_dim: int) -> torch.Tensor:
    if qkv.is_cuda:
        _gpu()
        return torch.ops.rlli.prefill_attn_qkv(qkv, cu_seqlens, scale, n_q,
                                               n_kv, head_dim)
    T = qkv.shape[0]
    D = head_dim
    q = qkv[:, :n_q * D].reshape(T, n_q, D)
    k = qkv[:, n_q * D:(n_q + n_kv) * D].reshape(T, n_kv, D)
    v = qkv[:, (n_q + n_kv) * D:].reshape(T, n_kv, D)
    return ref.prefill_attn(q, k, v, cu_seqlens, scale).reshape(T, n_q * D)


def decode_attn(q: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor,
                block_table: torch.Tensor, seq_lens: torch.Tensor,
                scale: float) -> torch.Tensor:
    if q.is_cuda:
        _gpu()
        return torch.ops.rlli.decode_attn(q, k_cache, v_cache, block_table,
                                          seq_lens, scale)
    return ref.decode_attn(q, k_cache, v_cache, block_table, seq_lens, scale)


def prefill_attn(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor,
                 cu_seqlens: torch.Tensor, scale: float) -> torch.Tensor:
    if q.is_cuda:
        _gpu()
        return torch.ops.rlli.prefill_attn(q, k, v, cu_seqlens, scale)
    return ref.prefill_attn(q, k, v, cu_seqlens, scale)


def sample(logits: torch.Tensor, temperatures: torch.Tensor,
           seeds: torch.Tensor, step: int = 0) -> torch.Tensor:
    """Greedy argmax / Gumbel-max temperature sampling; ``seeds`` is a
    per-row int64 tensor (per-request reproducibility), ``step`` a
    uniform step offset mixed in-kernel."""
    if logits.is_cuda:
        _gpu()
        return torch.ops.rlli.sample(logits, temperatures, seeds, step)
    return ref.sample(logits, temperatures, seeds, step)


def decode_load(state, batch, bucket: int, scratch_block: int,
                scratch_slot: int) -> None:
    """The first ``bucket`` rows of a decode step's buffers ``state`` (ids,
    positions, tables, temperatures, seeds, state slots) from those of
    ``batch``, whose slots may be None; rows and pages that it does not have
    are the scratch block's and slot's.  One launch for tensors of the
    buffers' types on their GPU, a copy each for others."""
    ids, tables = batch[0], batch[2]
    B, W = ids.shape[0], tables.shape[1]
    if (B <= bucket and W <= state[2].shape[1] and state[0].is_cuda
            and all(t is None or (t.device == to.device and t.dtype == to.dtype
                                  and t.is_contiguous()
                                  and t.shape == ((B, W) if t is tables
                                                  else (B,)))
                    for t, to in zip(batch, state))):
        _gpu()
        torch.ops.rlli.decode_load(*state, *batch, bucket, scratch_block,
                                   scratch_slot)
        return
    for t, to in zip(batch, state):
        if t is tables:
            to[:B, :W].copy_(t)
            if W < to.shape[1]:          # stale tail from an earlier batch
                to[:B, W:].fill_(scratch_block)
        elif t is not None:
            to[:B].copy_(t)
    for to, fill in zip(state, (0, 0, scratch_block, 0, 0, scratch_slot)):
        to[B:bucket].fill_(fill)         # neutralize padded lanes


def decode_begin(positions: torch.Tensor, tables: torch.Tensor,
                 block_size: int) -> tuple[torch.Tensor, torch.Tensor]:
    """Of rows at ``positions``: the slots of their keys and values (in the
    table's last block beyond its end), and the tokens they see."""
    if positions.is_cuda:
        _gpu()
        return torch.ops.rlli.decode_begin(positions, tables, block_size)
    block = torch.clamp((positions // block_size).long(),
                        max=tables.shape[1] - 1)
    return (tables.gather(1, block.unsqueeze(1)).squeeze(1) * block_size
            + positions % block_size, positions + 1)


def decode_advance_(ids: torch.Tensor, positions: torch.Tensor,
                    seeds: torch.Tensor, tokens: torch.Tensor,
                    seed_step: int) -> None:
    """The next step's ids, positions and (mod 2^64) seeds."""
    if ids.is_cuda:
        _gpu()
        torch.ops.rlli.decode_advance_(ids, positions, seeds, tokens,
                                       seed_step)
        return
    ids.copy_(tokens)
    positions.add_(1)
    seeds.add_(seed_step)


def prefill_paged_attn(qkv, k_cache, v_cache, chunk_row0, chunk_pos0,
                       chunk_nrows, chunk_btrow, block_tables,
                       scale: float, n_q: int) -> torch.Tensor:
    if qkv.is_cuda:
        _gpu()
        return torch.ops.rlli.prefill_paged_attn(
            qkv, k_cache, v_cache, chunk_row0, chunk_pos0, chunk_nrows,
            chunk_btrow, block_tables, scale, n_q)
    return ref.prefill_paged_attn(qkv, k_cache, v_cache, chunk_row0,
                                  chunk_pos0, chunk_nrows, chunk_btrow,
                                  block_tables, scale, n_q)


def mixed_attn_qkv(qkv, k_cache, v_cache, chunk_row0, chunk_pos0, chunk_nrows,
                   chunk_btrow, tables_pre, tables_dec, lens_dec,
                   n_decode: int, scale: float, n_q: int) -> torch.Tensor:
    """Attention of a mixed step whose keys and values are in the cache:
    decode_attn_qkv for rows [0, n_decode), n_decode > 0, prefill_paged_attn for
    the tiles', at the same time where that is the faster way."""
    if qkv.is_cuda:
        _gpu()
        return torch.ops.rlli.mixed_attn_qkv(
            qkv, k_cache, v_cache, chunk_row0, chunk_pos0, chunk_nrows,
            chunk_btrow, tables_pre, tables_dec, lens_dec, n_decode, scale,
            n_q)
    out = prefill_paged_attn(qkv, k_cache, v_cache, chunk_row0, chunk_pos0,
                             chunk_nrows, chunk_btrow, tables_pre, scale, n_q)
    decode_attn_qkv_out(qkv[:n_decode], k_cache, v_cache, tables_dec,
                        lens_dec, scale, n_q, out)
    return out


def _rows_faster(M: int, N: int, K: int) -> bool:
    """Where rows_linear beats the library, with weights that no cache holds.
    Timed at 1 to 128 rows of 300 shapes from 16 to 128256 by 256 to 28672; by
    more than 7 % it is slower at K 8192 alone, for which the library is at its
    best (1 row, N 4096: 17.0 and 19.1 us)."""
    if M > 64:
        # rows of x cost too, and panels that leave CUs idle more so (128 rows,
        # us, the library first: 4096 x 4096 25.1 and 19.1, 4096 x 14336 77.5
        # and 40.9, 28672 x 4096 60.6 and 57.6, 16384 x 2048 with silu 26.6 and
        # 21.8; but 8192 x 2048 16.6 and 19.0, 12288 x 4096 34.3 and 37.0,
        # 20480 x 4096 47.9 and 61.4, 57344 x 5120 125 and 144)
        if N * K < 1 << 24:
            return False
        if N < 25600:
            return K >= 4096 if N <= 8192 else (12288 < N <= 16384
                                                and K <= 4096)
        return N <= 32768 or N >= 65536 or K >= 8192
    if N < 1024:
        # few panels: many parts to sum, or waves with long runs of K (256 x
        # 8192: 1 row 11.3 and 7.8, 64 rows 11.0 and 19.5; 64 x 14336, 1 row
        # 12.4 and 51; 512 x 14336, 64 rows 19.1 and 15.6)
        return K <= 4096 or (M <= 8 if K <= 8192 else N >= 512)
    if 16384 < N < 25600:
        # 64-row panels for more than one workgroup per CU and fewer than two
        # (20480 x 3072, 16 rows 58 and 30, 64 rows 33.9 and 38.6; 20480 x
        # 8192, 1 row 73.7 and 83.6)
        return K <= 1024 or K < 8192 and (M <= 16 or M <= 32 and K <= 4096)
    if 8192 < N <= 11520 and K <= 2048:
        # parts that cost as much as what they divide (10240 x 256, 16 rows
        # 6.3 and 6.2, 64 rows 6.7 and 10.2)
        return M <= 16
    return True


def _rows_take(M: int, N: int, K: int) -> bool:
    """Sizes that rows_linear takes faster than the library: as many rows as leave
    reading w what costs."""
    return (1 <= M <= 128 and K % 64 == 0 and K > 0 and N % 4 == 0 and N > 0
            and _rows_faster(M, N, K))


def rows_fit(x: torch.Tensor, w: torch.Tensor) -> bool:
    """Whether rows_linear takes x w^T and is the faster way.  (Sizes first: short
    prompts wait for the host, and what does not fit, as most of their products, is
    to cost it little.)"""
    return (x.dim() == w.dim() == 2 and x.is_cuda
            and _rows_take(x.shape[0], *w.shape) and product_operands(x, w))


def rows_linear(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """x w^T of few rows: a kernel that streams w once (rows_fit says
    whether it applies), F.linear on the CPU."""
    if x.is_cuda:
        _gpu()
        return torch.ops.rlli.rows_linear(x, w)
    return torch.nn.functional.linear(x, w)


def rows_linear_parts(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """rows_linear for readers that sum: f32 parts [n, rows, N] of the
    product, or all of it in bf16 [rows, N] where it was not divided."""
    if x.is_cuda:
        _gpu()
        return torch.ops.rlli.rows_linear_parts(x, w)
    return torch.nn.functional.linear(x, w)


def rows_linear_silu(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """silu_mul(x w^T) for the rows of rows_linear, without the product in
    between."""
    if x.is_cuda:
        _gpu()
        return torch.ops.rlli.rows_linear_silu(x, w)
    return silu_mul(torch.nn.functional.linear(x, w))


def rows_norm_fit(parts: torch.Tensor, residual: torch.Tensor,
                  w: torch.Tensor, silu: bool) -> bool:
    """Whether rows_norm_linear takes these."""
    if parts.dim() != 3 or parts.dtype != torch.float32 \
            or parts.shape[1] != 1 or not rows_fit(residual, w):
        return False
    _gpu()
    return torch.ops.rlli.rows_norm_ok(*w.shape, silu)


def rows_norm_linear(parts: torch.Tensor, residual: torch.Tensor,
                     gain: torch.Tensor, eps: float, w: torch.Tensor,
                     silu: bool) -> tuple[torch.Tensor, torch.Tensor]:
    """Of one row: rmsnorm_residual_ of rows_linear_parts's result and
    rows_linear_parts or rows_linear_silu of that, in one launch; the product
    and the new residual (``residual`` stays as it is)."""
    _gpu()
    return torch.ops.rlli.rows_norm_linear(parts, residual, gain, eps, w, silu)


def rows_whole(x: torch.Tensor, w: torch.Tensor) -> bool:
    """For x and w that rows_fit: whether rows_linear takes them without
    dividing K over workgroups; rows_linear_relu2 is for these."""
    _gpu()
    return torch.ops.rlli.rows_whole_ok(x.shape[0], *w.shape)


def rows_linear_relu2(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """relu2(x w^T), of the f32 sums."""
    _gpu()
    return torch.ops.rlli.rows_linear_relu2(x, w)


def rows_streams_fit(x: torch.Tensor, w: torch.Tensor, streams: torch.Tensor,
                     w_next: torch.Tensor) -> bool:
    """Whether rows_linear_streams_ and then rows_linear_scaled_relu2 take x, w and
    w_next."""
    if not rows_fit(x, w) or x.shape[0] > 32 \
            or not (w_next.dim() == 2 and w_next.shape[1] == w.shape[0]
                    and w_next.dtype == torch.bfloat16
                    and w_next.device == w.device and w_next.is_contiguous()
                    and w_next.data_ptr() % 16 == 0
                    and not w_next.requires_grad):
        return False
    _gpu()
    return torch.ops.rlli.rows_streams_ok(x.shape[0], *w.shape,
                                          streams.shape[1], w_next.shape[0])


def rows_linear_streams_(x, w, streams, mix, out_w, in_w, gain):
    """hyper_step of rows_linear, but for the norm's factor of a row: the next
    sublayer's input without it, and sums of squares for
    rows_linear_scaled_relu2."""
    _gpu()
    return torch.ops.rlli.rows_linear_streams_(x, w, streams, mix, out_w, in_w,
                                               gain)


def rows_linear_scaled_relu2(h, ss, eps: float, w):
    """rows_linear_relu2 of what rows_linear_streams_ left, normed."""
    _gpu()
    return torch.ops.rlli.rows_linear_scaled_relu2(h, ss, eps, w)


@functools.lru_cache(maxsize=4096)
def _tall_faster(M: int, N: int, K: int) -> bool:
    """Where rows_tall beats the other ways: rows_linear up to 128 rows, tiles and
    the library.  (As many times as fast, with the rows of x and w that one of its
    workgroups has where those decide: 2048 x 1024, 65 rows 1.90, 512 1.22; 1024 x
    2048, 768 1.05; 2048 x 2048, 320 1.02, 512 rows (128) 0.98, 3072 x 2048, 320
    rows (128) 0.93, but 4096 x 2048, 256 rows (128) 1.08; 256 x 2048, 96 rows
    0.85; 3072 x 3072, 65 1.57, 320 1.07; 8192 x 3072, 112 1.02; 2048 x 3072, 80
    1.00, 112 0.87; 2048 x 4096, 112 1.06, 448 1.09; 6144 x 4096, 65 1.09, 112
    1.02; 8192 x 4096, 65 0.94; 1536 x 4096, 128 0.90; 4096 x 5120, 128 1.02, 160
    0.82; 2048 x 6144, 65 1.06, 192 1.25, 320 1.07, 448 0.92; 1536 x 6144, 65
    1.02, 384 1.20, 512 1.01; 1536 x 4608, 65 1.14, 128 1.08, 320 1.15; 2048 x
    4608, 128 1.02, 384 1.22; 1536 x 5120, 129 1.01, 384 1.26; 2048 x 5120, 128
    0.98, 320 1.13; 2048 x 5632, 128 0.99, 384 1.01.  Of 5962 points that are
    taken, with weights that no cache holds, one is slower by more than 5 %: 4096 x
    4096, 144 0.94.)"""
    if not 64 < M <= 768 or K > 6144 or K % 64 or N < 256:
        return False
    _gpu()
    work = torch.ops.rlli.rows_tall_work(M, N)
    if work == 0:
        return False
    if K <= 1024:
        return True
    if K <= 2048:
        return N >= 512 and (work <= 112 or N >= 4096)
    if K <= 3072:
        return N >= 3072
    if K <= 4096:
        return 2048 <= N <= 6144
    return 1536 <= N <= 2048 and M <= 384


def rows_tall(x: torch.Tensor, w: torch.Tensor,
              relu2: bool = False) -> torch.Tensor:
    """x w^T of some hundred rows, or relu2 of that."""
    _gpu()
    return torch.ops.rlli.rows_tall(x, w, relu2)


def _tile_sizes(M: int, N: int, K: int) -> bool:
    """Sizes that the kernels of tiles and rows_tall take."""
    return N % 16 == 0 and K % 64 == 0 and max(M, N) * K < 1 << 31


def _tiles_take(x: torch.Tensor, w: torch.Tensor, faster) -> bool:
    """Whether the kernel of tiles takes x w^T and ``faster`` (rows, N, K)."""
    return (x.dim() == w.dim() == 2 and x.is_cuda
            and faster(x.shape[0], *w.shape)
            and _tile_sizes(x.shape[0], *w.shape) and product_operands(x, w))


def _tile_parts_faster(M: int, N: int, K: int) -> bool:
    """Where tile_linear_parts, with the pass that sums the parts, beats the other
    way.  Divided, K keeps all CUs busy where the library leaves some idle;
    parts cost the more the shorter K is.  (us with the norm behind it, the
    other way first.)"""
    if K < 4096 or not 1024 <= N <= 8192 or M <= 64:
        return False
    if M <= 128 and _rows_faster(M, N, K):
        # One row of tiles, divided by eight at most, leaves CUs idle below 4096
        # columns; rows_linear_parts does not (2048 x 8192, 65 rows 16 and 19;
        # 2048 x 14336, 65 rows 22 and 27; 1024 x 28672, 96 rows 24 and 42; 3072
        # x 14336, 96 rows 31 and 32; 4096 x 4096, 80 rows 16.6 and 18.0, but
        # 5120 x 4096 1.00, 4096 x 14336 34 and 31, 8192 x 14336 1.15 times as
        # fast).
        return N >= 4096 and N * K > 1 << 24
    if K < 6144:
        # (4096 x 4096, 129 rows 26 and 20, 192 37 and 21, 256 27 and 23, 320 29
        # and 27, but 384 30 and 31; 8192 x 4096, 129 rows 30 and 30, 256 49 and
        # 35, but 320 42 and 44; 2048 x 4096, 128 rows 16.0 and 16.9)
        return M <= 256
    if K < 8192:
        # parts of more than some 2 M elements cost what dividing gains (2048 x
        # 6144, 1024 rows 1.08 times as fast, 4096, 500 rows 1.13, but 768 55
        # and 67; 8192, 256 rows 1.44, but 384 60 and 72)
        return M <= 1280 and M * N <= 1 << 21
    # Beyond 2^23 elements the library has a tile of 256 x 128 for every CU (8192
    # x 14336, 1024 rows 1.10, but 1150 244 and 271, 2048 343 and 377; 5120 x
    # 14336, 1536 rows 1.16, but 2048 254 and 278; 4096 x 14336, 160 rows 89
    # and 41, 536 118 and 72, 1000 145 and 109, 2048 233 and 209, but 3072 297
    # and 299; 2048 x 8192, 536 rows 43 and 32, 1300 61 and 55, but 1536 60 and
    # 62).
    return M <= (1280 if K < 12288 else 2048) and M * N <= 1 << 23


def tile_parts_fit(x: torch.Tensor, w: torch.Tensor) -> bool:
    """Whether tile_linear_parts takes x w^T and is the faster way."""
    return _tiles_take(x, w, _tile_parts_faster)


def tile_linear_parts(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """rows_linear_parts for more rows."""
    _gpu()
    return torch.ops.rlli.tile_linear_parts(x, w)


def _tile_linear_faster(M: int, N: int, K: int) -> bool:
    """Where tile_linear beats the other way.  (us, that first, rows_linear up to
    128 rows and the library from there: 6144 x 4096, 65 rows 20 and 17, 129 39
    and 23, 160 25 and 24, but 200 23 and 25; 4096 x 4096, 96 rows 15.9 and
    16.7, 129 22 and 20, 160 28 and 19; 10240 x 8192, 65 rows 77 and 40, 129 57
    and 49, 256 88 and 56, 257 64 and 64; 5120 x 5120, 65 rows 20 and 18, 250 32
    and 28, 288 30 and 30; 12288 x 4096, 128 rows 32 and 35; 3072 x 2048, 128
    rows 12 and 14.  Slower by more than 5 % of 541 points timed: 8192 x 8192,
    65 to 96 rows 38 and 41, 8192 x 4096, 129 and 144 rows 27 and 29, and 6144 x
    5120, 208 and 240 rows 33 and 37, all beside rows where they gain more.)"""
    if K <= 2048 and N % 128 != 0:
        # The library is slow where rows of the result end amid its tiles (as
        # times as fast: 6160 x 2048, 1024 rows 1.11, 2048 1.20, 4000 1.05, 777
        # 0.91, 7613 0.96; 3088 x 2048, 1024 1.15, 2048 1.12, 5000 1.16; 8208 x
        # 2048, 1300 1.18, 3300 1.40, 5000 1.03; 10256 x 2048, 1024 1.15, 5000
        # 1.11; 6160 x 1024, 420 1.14, 1300 1.22, 5000 1.15; 2064 x 1024, 512
        # 0.93, 1024 1.12, 5000 1.21).  With long K, somewhat more tiles of 128 x
        # 128 than there are CUs take two rounds of them or of larger ones (3088 x
        # 2048, 1200 rows 1.18, 1300 0.95, 1600 0.94, 1800 1.02; 2064 x 2048, 1800
        # 1.14, 2048 0.93, 2300 0.92, 2600 1.00; 4112 x 2048, 1024 0.96, 1100 0.97,
        # 1200 1.05; 3088 x 1536, 1300 1.06), and just more of 256 x 256 than four
        # rounds have take a fifth (10256 x 2048, 6400 0.88; x 1536 0.92).
        def tiles(side):
            return -(-M // side) * -(-N // side)
        return ((1024 if K > 1024 else 600) <= M <= 6400 and 2048 <= N <= 10496
                and tiles(256) <= 1024
                and not (K > 1536 and 256 < tiles(128) < 328))
    return (64 < M <= (256 if K > 4096 else 160) and K >= 4096
            and 4096 <= N <= 10240 and (M > 128 or N * K > 1 << 24))


def tile_linear_fit(x: torch.Tensor, w: torch.Tensor) -> bool:
    """Whether tile_linear takes x w^T and is the faster way."""
    return _tiles_take(x, w, _tile_linear_faster)


def tile_linear(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """rows_linear for more rows."""
    _gpu()
    return torch.ops.rlli.tile_linear(x, w)


def _tile_silu_faster(M: int, N: int, K: int) -> bool:
    """Where tile_linear_silu beats the library and silu_mul (rows_linear_silu,
    where it applies, comes first).  K is not divided here, so a tile takes the
    longer, whatever the CUs that are left idle, the longer K is, while the pass
    for silu that is spared stays the same.  (us or times as fast, those first.)"""
    if K < 1024 or N < 4096:
        return False
    if K > 1536 and N < 5120:
        # 64 tiles of 128 x 128 at 256 rows (4096 x 2048, 256 rows 0.85, 512
        # 1.03, 600 1.32; 4096 x 4096, 256 rows 0.71, 600 1.08)
        if M < 600:
            return False
    if K >= 6144 and N < 7168:
        # (6144 x 6144, 192 rows 0.95, 300 0.89, 768 0.89, 1536 1.09)
        return False
    if K <= 1024 or K < 3072 and N > 8192:
        # (8192 x 1024, 65 rows 1.33; 12288 x 2048, 65 rows 20 and 17; but 8192
        # x 2048 0.93, 14336 x 5120 0.79)
        least = 65
    elif K < 3072 or N >= 11008:
        # (16384 x 2048, 160 rows 32 and 24; 28672 x 4096, 129 rows 68 and 68,
        # 160 68 and 66, 192 75 and 71; 28672 x 8192, 144 rows 117 and 118, 208
        # 140 and 128; 11008 x 4096, 129 rows 1.18; but 10240 x 4096 0.97)
        least = 129
    else:
        # (7168 x 4096, 192 rows 1.06, 160 0.94, 129 0.87)
        least = 192
    if N % 32768 == 0:
        # rows of the result are a multiple of 32 KB apart (see relu2: 32768 x
        # 4096, 1024 rows 1.04, 4096 0.93; 65536 x 4096, 4096 rows 1597 and
        # 1734)
        most = 1024
    elif K >= 8192:
        # (57344 x 8192, 2048 rows 1.02, 4096 2630 and 2760; 28672 x 8192, 2048
        # rows 0.97, 4096 0.96)
        most = 2048
    else:
        # The burst of 8192 rows gains nothing: 28672 x 4096, 1433 and 1428.
        # (28672 x 4096, 536 rows 147 and 113, 1024 222 and 190, 2048 416 and
        # 383, 8000 1412 and 1398; beyond, 10000 1908 and 1750, 16384 2829 and
        # 2797, and with 16384 x 2048, 8000 472 and 436, 16384 921 and 852, is
        # not taken so far.)
        most = 8000
    return least <= M <= most


def tile_silu_fit(x: torch.Tensor, w: torch.Tensor) -> bool:
    """Whether tile_linear_silu takes x w^T and is the faster way."""
    return _tiles_take(x, w, _tile_silu_faster)


def tile_linear_silu(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """rows_linear_silu for more rows."""
    _gpu()
    return torch.ops.rlli.tile_linear_silu(x, w)


def _tile_relu2_faster(M: int, N: int, K: int) -> bool:
    """Where tile_linear_relu2 beats the library and relu2; the same as with silu,
    but for how long a pass is spared and how wide the result is.  (us or times
    as fast, those first: 6144 x 2048, 128 rows 16 and 17, 192 21 and 18, 600 26
    and 20, 2048 53 and 41, 7613 170 and 149; 12288 x 4096, 192 rows 45 and 39,
    2048 174 and 164, 8000 613 and 608; 8192 x 4096, 160 rows 33 and 36.)"""
    if K < 1024 or N < 4096:
        return False
    if K > 1536 and N < (6144 if K >= 3072 else 5120) and M < 600:
        # (4096 x 2048, 192 rows 1.22, but 224 16.6 and 20.5, 256 0.78, 384 0.88,
        # 512 0.95, 600 1.27; 4096 x 4096, 256 rows 0.66, 600 1.06; 5120 x 4096,
        # 384 rows 0.82)
        return False
    if K >= 6144 and N < 7168:
        # (6144 x 6144, 300 rows 0.88, 600 1.12, 768 0.89)
        return False
    # Rows of the result that are a multiple of 32 KB apart are stored more
    # slowly (4096 rows of K 4096, N 16128, 16384 and 16640: 396, 448 and 456,
    # the others 418, 409 and 539; 32768 0.88, 24576 1.03).  With long K the
    # pass that is spared is a smaller part (14336 x 8192, 1024 rows 1.02, 4096
    # 0.95).
    return 192 <= M <= (1024 if N % 16384 == 0 or K >= 8192 else 8000)


def tile_relu2_fit(x: torch.Tensor, w: torch.Tensor) -> bool:
    """Whether tile_linear_relu2 takes x w^T and is the faster way."""
    return _tiles_take(x, w, _tile_relu2_faster)


def tile_linear_relu2(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """relu2(x w^T), of the 16-bit product."""
    _gpu()
    return torch.ops.rlli.tile_linear_relu2(x, w)


@functools.lru_cache(maxsize=8192)
def product_way(form: str, M: int, N: int, K: int) -> str | None:
    """Which kernel of ours takes M rows by w [N, K] for a reader of ``form``
    the fastest, of operands that product_operands: "rows", "tall" or "tile";
    None: none of them.  Forms: whole, parts, silu, relu2, and divided, which is
    parts where the kernel of few rows divides K and nothing else.  (Asked of
    the *_fit of one kernel after the other, a product cost the host 6 to 8 us
    ahead of its launch, and prompts of 12 mixed layers have 48.)"""
    if M < 1 or N < 1 or K < 1 or K % 64:
        return None
    rows, tiles = _rows_take(M, N, K), _tile_sizes(M, N, K)
    if form == "whole":
        if tiles and _tall_faster(M, N, K):
            return "tall"
        if tiles and _tile_linear_faster(M, N, K):
            return "tile"
        return "rows" if rows else None
    if form == "parts":
        if tiles and _tile_parts_faster(M, N, K):
            return "tile"
        return "rows" if rows else None
    if form == "divided":
        _gpu()
        return product_way("parts", M, N, K) if rows and not \
            torch.ops.rlli.rows_whole_ok(M, N, K) else None
    if form == "silu":
        if rows and N % 16 == 0:
            return "rows"
        return "tile" if tiles and _tile_silu_faster(M, N, K) else None
    if tiles and _tall_faster(M, N, K):
        return "tall"
    if tiles and _tile_relu2_faster(M, N, K):
        return "tile"
    if rows:
        _gpu()
        if torch.ops.rlli.rows_whole_ok(M, N, K):
            return "rows"
    return None


_STORED = frozenset((torch.Tensor, torch.nn.Parameter))


def _plain(x: torch.Tensor, w: torch.Tensor) -> bool:
    """Whether x and w are tensors with memory, which those of a trace and in
    vmap are not, and neither gradients nor tangents of x w^T are asked for."""
    return (type(x) in _STORED and type(w) in _STORED
            and not (x.requires_grad or w.requires_grad)
            and forward_ad._current_level < 0
            and peek_interpreter_stack() is None)


def product_operands(x: torch.Tensor, w: torch.Tensor) -> bool:
    """Whether x w^T is one that the kernels of product_way take."""
    return (x.is_cuda and x.dtype == w.dtype == torch.bfloat16
            and x.dim() == w.dim() == 2 and _plain(x, w)
            and x.is_contiguous() and w.is_contiguous()
            and (x.data_ptr() | w.data_ptr()) % 16 == 0)


def library_linear(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """F.linear(x, w), on the GPU in 16 bits without the library's search for
    its kernel at every call."""
    if (x.is_cuda and x.dim() == w.dim() == 2
            and x.dtype == w.dtype == torch.bfloat16
            and _plain(x, w) and not torch.is_autocast_enabled()
            and x.device == w.device and x.shape[1] == w.shape[1]
            and x.is_contiguous() and w.is_contiguous()):
        _gpu()
        return torch.ops.rlli.library_linear(x, w)
    return torch.nn.functional.linear(x, w)


def skinny_linear(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """rows_linear for K % 256 == 0 and N % 64 == 0."""
    if x.is_cuda:
        _gpu()
        return torch.ops.rlli.skinny_linear(x, w)
    return torch.nn.functional.linear(x, w)


def linear_auto(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """rows_linear for up to 64 rows, K % 256 == 0 and N % 64 == 0, whether it
    is the faster one or not; else hipBLASLt via F.linear."""
    if (x.is_cuda and x.dim() == 2 and 1 <= x.shape[0] <= 64
            and x.shape[1] % 256 == 0 and w.shape[0] % 64 == 0):
        _gpu()
        return torch.ops.rlli.skinny_linear(x, w)
    return torch.nn.functional.linear(x, w)


def skinny2_linear(x: torch.Tensor, w: torch.Tensor,
                   splitk: int = 0) -> torch.Tensor:
    """rows_linear for K % 256 == 0 and N % 64 == 0; ``splitk`` has no
    effect."""
    if x.is_cuda:
        _gpu()
        return torch.ops.rlli.skinny2_linear(x, w, splitk)
    return torch.nn.functional.linear(x, w)


def skinny2_silu_linear(gu: torch.Tensor, w: torch.Tensor,
                        splitk: int = 0) -> torch.Tensor:
    """SwiGLU + down-proj: (silu(gu[:, :K]) * gu[:, K:]) @ w^T."""
    if gu.is_cuda:
        _gpu()
        return torch.ops.rlli.skinny2_silu_linear(gu, w, splitk)
    return torch.nn.functional.linear(ref.silu_mul(gu), w)


build_cos_sin = ref.build_cos_sin
yarn_cos_sin = ref.yarn_cos_sin


# ----------------------------------------------- mixed-layer model ops
# f32 or bf16 activations.  On the GPU one namespace per kernel library
# (build.py), on the CPU one ref_*.py each.
from . import ref_attn, ref_blk, ref_lat, ref_mix, ref_rec  # noqa: E402
from .ref_rec import REC_CHUNK  # noqa: E402

_CPU_FORMS = {"rlli_attn": ref_attn, "rlli_mix": ref_mix,
              "rlli_blk": ref_blk, "rlli_rec": ref_rec, "rlli_lat": ref_lat}


_spaces: dict = {}       # of the libraries that are loaded


def _ns(lib: str, t: torch.Tensor):
    """The op namespace of ``lib`` for ``t``'s device."""
    if not t.is_cuda:
        return _CPU_FORMS[lib]
    space = _spaces.get(lib)
    if space is None:
        load_libraries((lib,))
        space = _spaces[lib] = getattr(torch.ops, lib)
    return space


def _mix(t: torch.Tensor):
    return _ns("rlli_mix", t)


def hyper_embed(ids, table, w_embed, x, in_w, gain, eps: float):
    """Fill the streams with the normed embedding; returns the normed
    input of the first sublayer.  Gains multiply (1 + w is folded in)."""
    return _mix(table).hyper_embed(ids, table, w_embed, x, in_w, gain, eps)


def hyper_step(x, y, mix, out_w, in_w, gain, eps: float, rows=None,
               keep: bool = True, split: bool = False):
    """Write one sublayer's output into the streams and return the normed
    input of the next (``in_w`` None: the plain stream sum).  ``y`` may be
    [T, parts, W], or with ``split`` the f32 parts [parts, T, W] of
    rows_linear_parts, the result then bf16; ``rows`` restricts the result
    (then keep=False)."""
    return _mix(y).hyper_step(x, y, mix, out_w, in_w, gain, eps, rows, keep,
                              split)


def relu2(x):
    return _mix(x).relu2(x)


def window_tile_rows(group: int, device) -> int:
    """Prompt-tile height that the tiled attention kernel wants."""
    if torch.device(device).type == "cuda":
        load_libraries(("rlli_mix",))
        return torch.ops.rlli_mix.window_tile_rows(group)
    return 32


def window_prefill(qkv, k_cache, v_cache, positions, cos_sin, slots,
                   block_tables, prompt, sink, scale: float, n_q: int,
                   window: int, keep_first: int, has_kv: bool):
    """Prompt rows: rotate, append to the cache (``has_kv``), attend."""
    if not qkv.is_cuda:
        return ref_attn.window_prefill(
            qkv, k_cache, v_cache, positions, cos_sin, slots, block_tables,
            prompt, sink, scale, n_q, window, keep_first, has_kv, None, None,
            0.0, 0, None)
    attn = _ns("rlli_attn", qkv)
    attn.window_append(qkv, k_cache, v_cache, positions, cos_sin, slots, n_q,
                       has_kv, None)
    mask = (sink, scale, n_q, window, keep_first, has_kv)
    if attn.window_fast(k_cache, v_cache, qkv.dtype == torch.float32):
        h = window_tile_rows(n_q // k_cache.shape[1], qkv.device)
        return _mix(qkv).window_tiled(qkv, k_cache, v_cache, block_tables,
                                      prompt.tiles(h), h, *mask)
    return attn.window_rows(qkv, k_cache, v_cache, block_tables,
                            prompt.tiles(32), 32, *mask, None, None, 0.0, 0)


def window_decode(qkv, k_cache, v_cache, positions, cos_sin, slots,
                  block_tables, sink, scale: float, n_q: int, window: int,
                  keep_first: int, has_kv: bool):
    """One new token per sequence: rotation, append and attention fused."""
    return _ns("rlli_attn", qkv).window_decode(
        qkv, k_cache, v_cache, positions, cos_sin, slots, block_tables, sink,
        scale, n_q, window, keep_first, has_kv, None, None, 0.0, 0, None)


FULL = 1 << 30        # a window that never ends


def biased_decode(qkv, k_cache, v_cache, positions, slots, block_tables,
                  scale: float, n_q: int, r1, r2, temp_coef: float,
                  temp_every: int, v_eps=None):
    """Causal attention without rotation: a score loses r1 ln(1 + r2
    distance), queries are multiplied by 1 + temp_coef ln((p + 1) //
    temp_every + 1), values cached over their root mean square (``v_eps``).
    One new token per sequence, append included."""
    return _ns("rlli_attn", qkv).window_decode(
        qkv, k_cache, v_cache, positions, None, slots, block_tables, None,
        scale, n_q, FULL, 0, True, r1, r2, temp_coef, temp_every, v_eps)


def biased_prefill(qkv, k_cache, v_cache, positions, slots, block_tables,
                   prompt, scale: float, n_q: int, r1, r2, temp_coef: float,
                   temp_every: int, v_eps=None):
    """The same for prompt rows: append, then attend over the sequence's
    gathered keys and values (sizes that the tiled kernel does not take:
    over the pages, row by row)."""
    score = (r1, r2, temp_coef, temp_every)
    if not qkv.is_cuda:
        return ref_attn.window_prefill(
            qkv, k_cache, v_cache, positions, None, slots, block_tables,
            prompt, None, scale, n_q, FULL, 0, True, *score, v_eps)
    attn = _ns("rlli_attn", qkv)
    attn.window_append(qkv, k_cache, v_cache, positions, None, slots, n_q,
                       True, v_eps)
    _, n_kv, _, dim = k_cache.shape
    vdim = v_cache.shape[3]
    if qkv.dtype == torch.float32 or not attn.expanded_ok(dim, vdim):
        return attn.window_rows(qkv, k_cache, v_cache, block_tables,
                                prompt.tiles(32), 32, None, scale, n_q, FULL,
                                0, True, *score)
    blocks, kv_off, tokens = prompt.gathered(64)
    k, vt = attn.kv_gather(k_cache, v_cache, block_tables, blocks, tokens)
    out = torch.empty((qkv.shape[0], n_q * vdim), dtype=qkv.dtype,
                      device=qkv.device)
    attn.expanded_attn(qkv[:, :n_q * dim], k, vt, None, prompt.tiles(128),
                       kv_off, n_q, n_kv, scale, out, *score)
    return out


def diff_decode(qkv, gate, k_cache, v_cache, positions, cos_sin, slots,
                block_tables, n_q: int, bias, q_norm, k_norm, scale: float,
                chunk: int, cap: float, lam: float, out_scale: float,
                eps: float):
    """Differential attention, one new token per sequence, append included.
    ``qkv``: q | k | v | .., ``bias`` added to the three; a head's query and
    key are two maps side by side, each normed and rotated (pairs i, i + rot
    / 2); scores capped; a query sees its chunk of positions; the maps'
    outputs a1 - lam a2 over their root mean square, times out_scale and the
    sigmoid of ``gate`` [rows, n_q]."""
    return _ns("rlli_attn", qkv).diff_decode(
        qkv, k_cache, v_cache, positions, cos_sin, slots, block_tables, gate,
        scale, n_q, bias, q_norm, k_norm, chunk, cap, lam, out_scale, eps)


def diff_prefill(qkv, gate, k_cache, v_cache, positions, cos_sin, slots,
                 block_tables, prompt, n_q: int, bias, q_norm, k_norm,
                 scale: float, chunk: int, cap: float, lam: float,
                 out_scale: float, eps: float):
    """The same for prompt rows: append, then attend over what the rows'
    chunks hold, gathered (sizes that the tiled kernel does not take: over
    the pages, row by row)."""
    if not qkv.is_cuda:
        return ref_attn.diff_prefill(
            qkv, gate, k_cache, v_cache, positions, cos_sin, slots,
            block_tables, prompt, n_q, bias, q_norm, k_norm, scale, chunk,
            cap, lam, out_scale, eps)
    attn = _ns("rlli_attn", qkv)
    attn.diff_append(qkv, k_cache, v_cache, positions, cos_sin, slots, n_q,
                     bias, q_norm, k_norm, eps)
    tail = (chunk, cap, lam, out_scale, eps)
    _, n_kv, _, width = k_cache.shape
    vdim = v_cache.shape[3]
    if (qkv.dtype == torch.float32 or qkv.shape[1] % 8
            or not attn.expanded_ok(width // 2, vdim, 2)):
        return attn.diff_rows(qkv, k_cache, v_cache, block_tables,
                              prompt.tiles(32), 32, gate, scale, n_q, *tail)
    blocks, kv_off, tokens = prompt.gathered(64, chunk)
    k, vt = attn.kv_gather(k_cache, v_cache, block_tables, blocks, tokens)
    out = torch.empty((qkv.shape[0], n_q * vdim), dtype=qkv.dtype,
                      device=qkv.device)
    attn.diff_expanded(qkv[:, :n_q * width], k, vt, gate, prompt.tiles(128),
                       kv_off, n_q, n_kv, scale, out, *tail)
    return out


def _out(proj, state, vdim, out):
    if out is not None:
        return out
    return torch.empty((proj.shape[0], state.shape[1] * vdim),
                       dtype=proj.dtype, device=proj.device)


def gla_decode(proj, a2, a2_bias, norm, state, slots, positions, vdim: int,
               tau: float, eps: float, out=None):
    """Gated linear attention, one new token per sequence.  ``out`` may be
    a column range of a wider matrix."""
    out = _out(proj, state, vdim, out)
    _ns("rlli_rec", proj).gla_decode(proj, a2, a2_bias, norm, state, slots,
                                     positions, vdim, tau, eps, out)
    return out


def gla_prefill(proj, a2, a2_bias, norm, state, prompt, vdim: int,
                tau: float, eps: float, out=None):
    out = _out(proj, state, vdim, out)
    _ns("rlli_rec", proj).gla_prefill(
        proj, a2, a2_bias, norm, state, prompt.tiles(REC_CHUNK),
        prompt.seqs(REC_CHUNK), vdim, tau, eps, out)
    return out


def hgrn2_decode(proj, bias, lower, norm, state, slots, positions, vdim: int,
                 eps: float, out=None):
    """HGRN2: the same recurrence with k = 1 - decay, silu queries and a
    lower-bounded decay; ``proj`` is q | forget logit | v."""
    out = _out(proj, state, vdim, out)
    _ns("rlli_rec", proj).hgrn2_decode(proj, bias, lower, norm, state, slots,
                                       positions, vdim, eps, out)
    return out


def hgrn2_prefill(proj, bias, lower, norm, state, prompt, vdim: int,
                  eps: float, out=None):
    out = _out(proj, state, vdim, out)
    _ns("rlli_rec", proj).hgrn2_prefill(
        proj, bias, lower, norm, state, prompt.tiles(REC_CHUNK),
        prompt.seqs(REC_CHUNK), vdim, eps, out)
    return out


def rwkv_decode(rkvg, low, w2, w0, bonus, norm, state, slots, positions,
                eps: float, out):
    """RWKV-style recurrence, one new token per sequence: ``rkvg`` [4, rows,
    heads * dim], decay e^(-e^(w2 tanh(low) + w0)), bonus for the present
    token, norm over a head, silu gate."""
    _ns("rlli_rec", rkvg).rwkv_decode(rkvg, low, w2, w0, bonus, norm, state,
                                      slots, positions, eps, out)
    return out


def rwkv_prefill(rkvg, low, w2, w0, bonus, norm, state, prompt, eps: float,
                 out):
    _ns("rlli_rec", rkvg).rwkv_prefill(
        rkvg, low, w2, w0, bonus, norm, state, prompt.tiles(REC_CHUNK),
        prompt.seqs(REC_CHUNK), eps, out)
    return out


def delta_decode(proj, taps, tail, a_rate, dt_bias, norm, state, slots,
                 positions, kv_heads: int, vdim: int, eps: float, out):
    """Gated delta rule, one new token per sequence, convolution of
    q | k | v included.  ``proj``: q | k | v | gate | beta | decay."""
    _ns("rlli_rec", proj).delta_decode(
        proj, taps, tail, a_rate, dt_bias, norm, state, slots, positions,
        kv_heads, vdim, eps, out)
    return out


def delta_prefill(proj, taps, tail, a_rate, dt_bias, norm, state, prompt,
                  kv_heads: int, vdim: int, eps: float, out):
    x = torch.empty((proj.shape[0], taps.shape[1]), dtype=proj.dtype,
                    device=proj.device)
    conv_prompt(proj[:, :taps.shape[1]], taps, tail, prompt, x, silu=True)
    _ns("rlli_rec", proj).delta_prefill(
        proj, x, a_rate, dt_bias, norm, state, prompt.tiles(REC_CHUNK),
        prompt.seqs(REC_CHUNK), kv_heads, vdim, eps, out)
    return out


def mlstm_decode(proj, i_bias, f_bias, norm, state, m, slots, positions,
                 vdim: int, cap: float, eps: float, out):
    """mLSTM, one new token per sequence.  ``proj``: q | k | v | gate | i |
    f; the state's last column is the normalizer, ``m`` the running
    maximum."""
    _ns("rlli_rec", proj).mlstm_decode(proj, i_bias, f_bias, norm, state, m,
                                       slots, positions, vdim, cap, eps, out)
    return out


def mlstm_prefill(proj, i_bias, f_bias, norm, state, m, prompt, vdim: int,
                  cap: float, eps: float, out):
    _ns("rlli_rec", proj).mlstm_prefill(
        proj, i_bias, f_bias, norm, state, m, prompt.tiles(REC_CHUNK),
        prompt.seqs(REC_CHUNK), vdim, cap, eps, out)
    return out


def moe_route(h, router, top: int):
    return _mix(h).moe_route(h, router, top)


def moe_experts(h, router, w_up, w_down, top: int, limit: float):
    """[T, top, W]: one row per chosen expert; the consumer sums them."""
    return _mix(h).moe_experts(h, router, w_up, w_down, top, limit)


def moe_route_softmax(h, router, correction, top: int, groups: int,
                      keep: int):
    return _mix(h).moe_route_softmax(h, router, correction, top, groups, keep)


def moe_relu2(h, router, correction, w_up, w_down, top: int, groups: int,
              keep: int):
    """Squared-relu experts.  Softmax over all routes; ``correction`` shifts
    the choice, which the best ``keep`` of ``groups`` groups of neighbours
    hold; weights sum to one.  Returns (y [T, top, W], ids, weights); routes
    past the experts are identities, whose rows of y are not written."""
    return _mix(h).moe_relu2(h, router, correction, w_up, w_down, top, groups,
                             keep)


# --------------------------------------------------- residual blocks
CONV_SPAN = 16        # prompt rows that one convolution workgroup walks


def block_embed(ids, table, pos_table, positions, x, gain, groups: int,
                eps: float, taps=None, tail=None, slots=None,
                n_decode: int = 0, scale: float = 1.0):
    """Fill the f32 residual with scaled embedding + position and return its
    grouped norm h and, for the first ``n_decode`` rows (one token per
    sequence), h + conv(h) from the sequences' tails.  ``taps`` [branches,
    taps, width] makes that [branches, rows, width]."""
    return _ns("rlli_blk", table).block_embed(
        ids, table, pos_table, positions, x, gain, groups, eps, taps, tail,
        slots, n_decode, scale)


def block_step(x, y, gain, groups: int, eps: float, positions, taps=None,
               tail=None, slots=None, n_decode: int = 0, rows=None,
               keep: bool = True, y2=None, gain1=None, gain2=None,
               part_ids=None, part_w=None, part_h=None, part_limit: int = 0,
               y_bias=None):
    """Add a block's output to the residual; then as block_embed.  ``rows``
    restricts the result (then keep=False).  With ``y2`` half the sum of
    both outputs is added, each normed first (``gain1``, ``gain2``).  With
    ``part_ids`` [T, parts] the sum over y [T, parts, W] is added, where a
    part whose id is ``part_limit`` or more is part_w part_h instead.
    ``y_bias`` [W] goes with a single output."""
    return _ns("rlli_blk", y).block_step(x, y, gain, groups, eps, positions,
                                         taps, tail, slots, n_decode, rows,
                                         keep, y2, gain1, gain2, part_ids,
                                         part_w, part_h, part_limit, y_bias)


def conv_prompt(h, taps, tail, prompt, out, silu: bool = False):
    """out = h + conv(h), or silu(conv(h)), for prompt rows, and their
    sequences' tails.  Branches as in block_embed."""
    _ns("rlli_blk", h).conv_prompt(h, taps, tail, prompt.spans(CONV_SPAN),
                                   prompt.spans(1 << 30), out, silu)


def gate_act(gate_up, out, act: str, limit: float = 0.0):
    """out = act(gate) * up of [rows, gate | up]; act 'clamp_glu': g
    sigmoid(1.702 g) (u + 1) with g <= limit, |u| <= limit."""
    _ns("rlli_blk", gate_up).gate_act(gate_up, out, act, limit)
    return out


def soft_cap(x, cap: float):
    """cap * tanh(x / cap), 32-bit."""
    return _ns("rlli_blk", x).soft_cap(x, cap)


# ------------------------------------------------------------- latents
LATENT_VECTORS = 32   # (row, head) queries of one absorbed prompt tile


def latent_prep(proj, q_norm, kv_norm, eps: float, cache, slots):
    """Norm both latents of ``proj`` (query | key/value | ...), cache the
    second, return the first."""
    return _ns("rlli_lat", proj).latent_prep(proj, q_norm, kv_norm, eps,
                                             cache, slots)


def head_linear(x, w, gate=None, out=None):
    """out[t, h] = w[h] x[t, h] (times sigmoid(gate)); w [heads, n, k]."""
    if out is None:
        out = torch.empty((x.shape[0], w.shape[0] * w.shape[1]),
                          dtype=x.dtype, device=x.device)
    _ns("rlli_lat", w).head_linear(x, w, gate, out)
    return out


def latent_decode(q, gate, cache, positions, block_tables, scale: float,
                  w_uk, w_uv, out):
    """One new token per sequence: absorbed queries over the cached
    latents.  w_uk [heads, rank, dim], w_uv [heads, vdim, rank]."""
    heads = w_uk.shape[0]
    ns = _ns("rlli_lat", q)
    c = ns.latent_attn(head_linear(q, w_uk), cache, block_tables, scale,
                       heads, positions, None, None)
    return head_linear(c, w_uv, gate, out)


def expands(prompt, rank: int, dim: int, vdim: int) -> bool:
    """Whether a step's prompt rows are cheaper with expanded keys and
    values: rebuilding them costs a fixed amount per cached token, a score
    and value row of latent width costs more per (row, token)."""
    absorbed = expanded = 0
    for p in prompt.portions:
        ctx = p.pos0 + p.n
        absorbed += p.n * ctx * 2 * rank
        expanded += ctx * (dim + vdim) * (rank + p.n)
    # the absorbed kernel reaches about half the expanded one's rate
    return 2 * absorbed > expanded


def latent_prefill(q, gate, cache, block_tables, prompt, scale: float, w_uk,
                   w_uv, w_k, w_v, out, expand=None):
    """Prompt rows over the cached latents, their own included: with keys
    and values expanded from the latents (w_k [heads * dim, rank], w_v
    [heads * vdim, rank]) or with absorbed queries, whichever is cheaper
    (``expand`` forces one)."""
    heads, rank, dim = w_uk.shape
    vdim = w_uv.shape[1]
    ns = _ns("rlli_lat", q)
    fast = q.is_cuda and ns.latent_fast(cache, q.dtype == torch.float32)
    attn = _ns("rlli_attn", q) if fast else None
    ok = fast and attn.expanded_ok(dim, vdim) and all(
        t.stride(0) % 4 == 0 and t.data_ptr() % 8 == 0 for t in (gate, out))
    if expand is None:
        expand = ok and expands(prompt, rank, dim, vdim)
    if expand and ok:
        blocks, kv_off, tokens = prompt.gathered(64)
        c = ns.latent_gather(cache, block_tables, blocks, tokens)
        k = torch.nn.functional.linear(c, w_k)
        vt = torch.nn.functional.linear(w_v, c)      # already transposed
        attn.expanded_attn(q, k, vt, gate, prompt.tiles(128), kv_off, heads,
                           heads, scale, out, None, None, 0.0, 0)
        return out
    tiles = prompt.vectors(LATENT_VECTORS, heads) if fast else prompt.tiles(32)
    c = ns.latent_attn(head_linear(q, w_uk), cache, block_tables, scale,
                       heads, None, tiles, prompt.pos0())
    return head_linear(c, w_uv, gate, out)
