"""The row counts and sizes at which the kernel provider changes from one kernel to
another, in one table, each entry with what it was measured on.

None of these decides what is computed, only by which kernel; every one was found by
timing captured steps on an MI355X at the shapes named below.  A model of other shapes
runs correctly with them and may be faster with others: `HipOps.dispatch` is an ordinary
attribute, `dataclasses.replace(ops.dispatch, decode_items=...)` gives a changed copy, and
`MEASURED` is where a table measured on other shapes is added.
"""

from __future__ import annotations

from dataclasses import dataclass


@dataclass(frozen=True)
class Dispatch:
    # ---- the product behind a norm whose rows the weight-streaming kernel in front has prepared: the
    # same kernels', or in captured steps from `tiled_scaled_rows` rows (gate/up products of more than
    # `tiled_scaled_pair_columns` columns from `tiled_scaled_pair_rows`) the LDS-tiled kernel's in tiles of 64
    # rows, whose workgroups read the rows once in 32 or 64 columns, not in 16.  The one and the other, us,
    # weights from memory, launch after launch in a graph, 17, 32 and 48 rows: 3,072 x 1,024 6.5 / 6.9, 7.5 /
    # 7.1, 9.7 / 7.4; 1,536 x 1,536 6.6 / 9.0, 7.9 / 9.2, 10.3 / 9.5; gate/up 2 x 3,072 x 1,024 9.1 / 7.2,
    # 10.0 / 7.5, 12.9 / 7.7; 2 x 2,048 x 1,024 6.8 / 7.0, 6.7 / 7.3, 9.9 / 7.4.  Captured steps with the
    # streaming kernels alone and so: 0.6B 17 rows 1,404 / 1,351, 32 1,535 / 1,461, 33 1,635 / 1,513, 64
    # 2,078 / 1,911 (the tiled kernel for both from 17 rows on: 1,388 and 1,480); its layers with an inner size of
    # 2,048 17 rows 1,285 / 1,287 (1,336), 33 1,520 / 1,458.
    # K = 512 gains nothing (1,024 columns 3.4 / 4.2, 3.5 / 4.3, 4.7 / 4.4), K = 2,048 as much as it loses
    # (4,096 columns 17 rows 8.9 / 10.7, 33 rows 11.9 / 10.9).
    # Results that leave in float32 stay with the weight-streaming kernel, whose short runs of K round
    # less: K = 1,024 1.1e-7 against 3.2e-7 of float64, 1,536 1.2e-7 and 4.3e-7.  In bfloat16 both are off by
    # its rounding, 1.6556e-3 and 1.6556e-3 (gate/up 3.040e-3 and 3.040e-3); 2 to 4 values in 10,000 differ.
    tiled_scaled_rows: int = 33
    tiled_scaled_pair_rows: int = 17
    tiled_scaled_pair_columns: int = 2048
    tiled_scaled_k: tuple[int, int] = (1024, 1536)

    # ---- plain bfloat16 products: from how many rows the vendor library (hipBLASLt)
    # takes them, as the reference sends every linear layer to its vendor library
    # (engine/nn/base_layers.py:7-10).  Measured inside captured graphs at the Qwen3-0.6B
    # layer shapes (K = 1,024 to 3,072, N = 1,024 to 6,144).
    #: up to 64 rows the weight-streaming kernels here are faster at the layer products
    #: and fuse the norm before and the SwiGLU after
    library_rows: int = 65
    #: in the wide layout (a short K: four waves along N) the library is ahead from 17 rows
    library_rows_wide: int = 17
    #: at the output head (N from `head_columns`: every one of thousands of workgroups
    #: reads all rows of x) from 9 rows: float32 logits of 8 and 9 rows here, of the time of the
    #: library's first algorithm, N = 151,936 and K = 1,024 0.98 and 1.02, K = 4,096 0.89 and 0.96,
    #: K = 5,120 1.00 and 1.09; 128,256 x 4,096 1.00 and 1.09; 32,000 x 2,048 0.85 and 0.90.  Steps that
    #: are captured, or run to be, have the algorithm that is fastest with the weights in memory:
    #: there from 7 rows with K above 2,048 (K = 4,096 6 rows 0.97, 7 rows 1.00, 8 rows 1.02) and from
    #: 5 above 4,096 (K = 5,120 4 rows 0.99, 5 rows 1.01; 8,192 6 rows 0.99, 7 rows 1.01), below as
    #: before (K = 2,048 8 rows 0.95, 9 rows 1.01)
    library_rows_head: int = 9
    library_rows_long_head: int = 7
    library_rows_longest_head: int = 5
    head_columns: int = 16384
    #: a gate/up product, whose SiLU-multiply is then a kernel of its own, goes there only where
    #: its weight is above `pair_head_weight` elements, from 5 rows: 8 rows, here and with the
    #: library, 16,384 x 2,048 15.3 / 20.5 us, 24,576 x 4,096 38.3 / 46.2, 51,200 x 5,120 108 / 93
    library_rows_pair: int = 5
    pair_head_weight: int = 1 << 27
    #: weights above `large_weight` elements (the layer shapes of the 8B and 32B models:
    #: products bound by bandwidth, not latency): every workgroup's reading of the rows of
    #: x costs as much as the weights from 16 rows on, and the library is ahead from there
    #: (a decode step of the 8B shape with 12 requests 4.13 ms here against 4.37 with the
    #: library, with 16 requests 4.47 against 4.43, with 32 5.59 against 4.92); whether it
    #: also takes the rows below is decided per weight shape by the warm-up
    library_rows_large: int = 16
    large_weight: int = 1 << 23

    # ---- products of many rows (from `library_rows`), the LDS-tiled kernel or the library.
    #: A gate/up product with the SiLU-multiply in its epilogue is the tiled kernel's: neither
    #: is the [M, 2 I] intermediate written nor read.  Against the library's product and the
    #: SiLU-multiply kernel, 65 to 8,192 rows: 2 x 3,072 x 1,024 0.46 to 0.80 of their time,
    #: 2 x 8,192 x 2,048 0.71 to 0.93, 2 x 12,288 x 4,096 0.80 to 0.98 (from `library_rows_large`
    #: rows already: 24 to 64 rows 17.6 to 17.9 / 21.2 to 22.1 and 43.4 to 45.4 / 49.6 us); only
    #: the largest weights (2 x 25,600 x 5,120: 0.83 to 0.94 from 512 rows on, 0.85 to 1.12 below)
    #: wait for `tiled_pair_rows_large` rows.
    tiled_pair_weight: int = 1 << 27
    tiled_pair_rows_large: int = 512
    #: From `tiled_fill_rows` rows of weights above `large_weight` elements, gate/up products
    #: also have to fill so many per cent of their tiles' rounds
    #: (`ts_gemm_tiled_fill`): gate/up products at 46 row counts from 260 to 6,400 take 0.79 to 1.04
    #: of the library's and the SiLU kernel's time from 65 per cent on, 0.92 in the mean, and 1.04
    #: below, up to 1.14; the largest weights (above `tiled_pair_weight`) 0.85 to 0.87 at 650 to 750
    #: rows, above `tiled_fill_large_rows` 0.80 to 0.95 from 75 per cent on, and 1.00 to 1.04 from 65 to
    #: 75, in a step of 900 rows of the 32B shape 1.10.
    tiled_fill: int = 65
    tiled_fill_large: int = 75
    tiled_fill_large_rows: int = 768
    tiled_fill_rows: int = 256
    #: rows from which, and elements of a weight [N, K] up to which, the product that ends a
    #: sub-layer is the LDS-tiled kernel's tail form (it adds itself into the float32 stream
    #: and prepares the rows for the norm behind it, whose product then takes the scaled
    #: form) instead of the library's product and a norm kernel.
    tiled_stream_rows: int = 512
    #: Larger weights keep the separate kernels, whose products are each the faster one's: a layer's
    #: products and norms at 26 row counts from 512 to 8,192 take 1.00 to 1.11 of their time in
    #: these forms at the 8B shape, 0.98 to 1.06 at the 32B shape.
    tiled_stream_weight: int = 1 << 23
    #: Weights of `tiled_stream_few_weight` to `large_weight` elements take it from fewer rows in
    #: an eager step (captured ones, of up to 256 single tokens, do not: 4.99 against 4.77 ms), where
    #: two norm kernels and three library calls a layer hold the host up: a step of the 0.6B shape
    #: with 300 tokens 3,400 -> 2,050 us when it had tiles of 128 rows only (N = 1,024 fills few units
    #: with them), 1,740 with tiles of 64 and a sub-layer a call.  Fewer rows were measured in
    #: tiles of 128, nearly half empty.  The lower line of weights is none of speed: below it the forms are ahead as well
    #: (products and norms of a layer of hidden size 512, 72 to 511 rows, 76 -> 35 us eager and 30 to 33
    #: -> 27 to 31 on the GPU), but portions below 512 rows of such models have had the separate kernels,
    #: and their sums in another order, all along.
    tiled_stream_few_rows: int = 72
    tiled_stream_few_weight: int = 1 << 20
    #: Plain products: from `tiled_stream_rows` rows and up to so many elements the tiled
    #: kernel's (the same time on the GPU, 22.5 against 22.4 us for the 0.6B model's qkv at 2,048
    #: rows, and a fifth of the library call's 20 to 30 us on the host, which the GPU waits for
    #: at a step's start); others where `ts_gemm_tiled_ahead` says so.
    tiled_plain_weight: int = 1 << 23

    #: Second steps of two low-rank projections: one launch, whose wavefronts read their operands
    #: from memory, for ranks up to `low_rank_most` and rows x ranks x columns (of both) up to
    #: `low_rank_work`; above, two products.  One launch of the two's time: rank 64, 512 + 1,024
    #: columns, 8 rows 0.51, 1,000 0.67, 2,048 0.95, 4,096 1.37; 2,048 + 2,048 columns 512 rows 0.74,
    #: 1,000 1.09; rank 128, 4,096 + 4,096 200 rows 0.77, 512 1.29; rank 512, 65 rows 0.63, 200 1.29,
    #: 16,384 7.5; rank 1,024 8 rows 1.18
    low_rank_most: int = 512
    low_rank_work: int = 3 << 26

    # ---- attention.  Measured at 16 query / 8 key-value heads of 128, page size 16.
    #: workgroups (entries x key/value heads) up to which a decode step takes the decode
    #: kernel; with more, the chip is full anyway and the smaller workgroups of the
    #: general kernel do better
    decode_items: int = 512
    #: a step that holds a portion of at least `portion_tokens` tokens takes the kernel
    #: for long portions from this many 16-row wave tiles (one portion of 256 tokens 11.0
    #: against the general kernel's 16.6 us in tiles of 16 rows, and since in tiles of 32
    #: 1,024 tokens 18.7 against 34.4, 1,536 tokens 25.5 against 96.8; below that the two
    #: are equal)
    portion_tiles: int = 256
    portion_tokens: int = 32
    #: a step of single tokens only takes it where the chip is full without splitting
    #: keys: from 1,024 wave tiles (128 entries at 8 key/value heads) it is ahead of the
    #: general kernel at every context length tried (136 entries: 34 against 41 us at 300
    #: tokens each, 130 against 150 at 100 to 2,000, 426 against 445 at 4,000; 200
    #: entries: 46 / 51, 180 / 223, 608 / 653), at 576 to 768 it is level or behind
    single_token_tiles: int = 1024
    #: the general kernel: up to this many tiles a workgroup per tile and chunk whose
    #: waves share the chunk (decode), above it a wavefront per tile walks its keys
    #: (prompts); and the workgroups each mode spreads a tile's key chunks over
    cooperative_items: int = 1024
    cooperative_workgroups: int = 512
    per_wave_workgroups: int = 4096

    # ---- recurrences.  A step whose longest portion has more tokens than this runs in chunks of
    # 64 tokens as products of matrices, below it every entry is walked whole by one launch.
    # Three launches have a length of their own, a walked token costs 0.24 to 0.28 us (16 heads
    # of 128 x 128, a decay per head: 128 tokens 38 us walked, 40 in chunks; 144 tokens 42 / 41;
    # 512 tokens 130 / 45).
    scan_whole_tokens: int = 128
    #: so many more for the delta rule, whose launches take longer: 16 heads of 128 x 128, 128
    #: tokens 43 us walked, 52 in chunks; 160 tokens 53 / 54; 192 tokens 62 / 54; 512 tokens
    #: 153 / 69.  8 heads of 64 x 128, a decay per row: 35 / 39, 42 / 40, 49 / 41, 121 / 46.
    delta_whole_more: int = 32
    #: the state-space scan, whose workgroup walks 64 columns: 1.45 us a token at 64 heads of
    #: 128 x 64 (64 tokens 96 us walked, 33 in chunks), 1.05 at 32 heads of 64 x 64 (68 / 23).
    #: The line lies higher than that says because a step that short is eager and mostly as long
    #: as its launches: two more a layer cost it more on the host than the walk does on the GPU.
    #: Steps of one portion, six such layers, walked and in chunks: the smaller size 45 tokens
    #: 1.12 / 1.21 ms, 64 tokens 1.12 / 1.21, 96 tokens 1.34 / 1.44; the larger 45 tokens
    #: 1.30 / 1.39, 64 tokens 1.48 / 1.39, 96 tokens 1.77 / 1.44 (beside 11 single tokens, 64:
    #: 1.55 / 1.61).  One line for both sizes: what is lost at the larger, up to a third of a
    #: millisecond at 96, is won back at smaller ones, which would rather have it higher.
    state_space_whole_tokens: int = 96

    # ---- latent attention on the matrix cores: a wavefront per tile of 16 (token, head)
    # rows.  A step with fewer tiles than `latent_full_tiles` gives every tile a workgroup
    # whose four wavefronts share its keys out, in runs of a multiple of `latent_split_keys`
    # keys (a block of 32 for each wavefront) over up to about `latent_workgroups` workgroups.
    latent_full_tiles: int = 1024
    latent_split_keys: int = 128
    latent_workgroups: int = 512


#: what each table was measured on -> the table
MEASURED: dict[str, Dispatch] = {
    "gfx950 (MI355X, 256 compute units); Qwen3 dense at the 0.6B, 8B and 32B layer shapes: "
    "16 to 64 query heads over 8 key/value heads of 128, page size 16": Dispatch(),
}


def default_dispatch() -> Dispatch:
    """The table for this build's one target."""
    return next(iter(MEASURED.values()))
