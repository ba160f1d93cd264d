"""Shared case tables for the parity tests."""

# The reference's pytest matrix (libs/moda_triton/tests/ops/test_moda.py:95-198):
# (B, T_kv, H, L, G, dtype 'h'=fp16 | 'b'=bf16, scale or None for D**-0.5); D = 64.
REFERENCE_MATRIX = [
    (1, 63, 1, 0, 1, "h", 1.0), (2, 128, 2, 0, 2, "h", 1.0), (2, 111, 2, 4, 1, "h", 1.0), (2, 256, 4, 4, 2, "h", 1.0),
    (2, 192, 4, 0, 4, "h", 0.1), (1, 160, 2, 8, 2, "b", 0.1), (1, 128, 2, 8, 4, "b", 0.1), (1, 1, 1, 0, 1, "h", None),
    (1, 2, 2, 0, 2, "h", None), (2, 3, 2, 0, 2, "h", 1.0), (1, 63, 1, 0, 1, "h", 1.0), (1, 64, 2, 0, 2, "h", None),
    (1, 65, 2, 0, 4, "h", None), (2, 47, 3, 0, 4, "h", 0.5), (2, 95, 4, 0, 4, "h", None), (3, 80, 3, 0, 2, "h", None),
    (2, 111, 5, 0, 2, "h", 1.0), (1, 32, 2, 0, 8, "h", None), (1, 40, 2, 0, 8, "h", 0.25), (1, 64, 2, 1, 1, "h", None),
    (1, 63, 2, 1, 2, "h", 1.0), (2, 65, 2, 2, 1, "h", None), (2, 47, 3, 2, 2, "h", None), (1, 64, 2, 3, 2, "h", None),
    (1, 63, 2, 3, 4, "h", 0.1), (2, 80, 2, 4, 2, "h", None), (2, 95, 4, 4, 1, "h", None), (1, 64, 2, 5, 2, "h", None),
    (1, 63, 2, 5, 2, "h", 0.2), (2, 47, 2, 7, 2, "h", None), (1, 32, 2, 8, 2, "h", None), (1, 40, 2, 8, 4, "h", None),
    (1, 64, 2, 0, 2, "b", None), (1, 63, 2, 4, 2, "b", None), (2, 80, 3, 4, 4, "b", 0.1), (2, 95, 4, 8, 2, "b", None),
    (1, 64, 2, 0, 1, "h", 1.0), (1, 64, 2, 0, 1, "h", 0.03125), (1, 127, 2, 0, 1, "h", None),
    (1, 128, 2, 0, 2, "h", None), (1, 129, 2, 0, 4, "h", None), (2, 191, 4, 0, 2, "h", None),
    (2, 192, 4, 0, 4, "h", None), (2, 193, 4, 0, 8, "h", None), (1, 128, 2, 4, 2, "h", None),
    (1, 128, 2, 7, 2, "h", None), (1, 129, 2, 5, 2, "h", None), (2, 192, 4, 4, 2, "h", 0.1),
    (2, 192, 4, 8, 2, "h", None), (4, 64, 8, 4, 2, "h", None), (4, 63, 8, 5, 2, "h", None), (4, 95, 8, 7, 2, "h", None),
    (3, 111, 3, 3, 2, "h", None), (3, 111, 3, 5, 2, "h", None), (3, 111, 3, 7, 2, "h", None),
    (1, 48, 2, 4, 8, "h", None), (1, 48, 2, 5, 8, "h", None), (2, 128, 4, 4, 2, "b", None),
    (2, 128, 4, 7, 2, "b", None), (2, 128, 4, 8, 2, "b", 0.05), (2, 192, 4, 8, 2, "b", None),
    (3, 97, 3, 5, 2, "h", None), (3, 97, 3, 7, 2, "h", None), (3, 129, 5, 5, 2, "h", None), (2, 256, 8, 4, 2, "h", None),
    (2, 256, 8, 8, 2, "h", None), (1, 96, 6, 9, 2, "h", None), (2, 96, 6, 12, 4, "h", None),
    (2, 96, 7, 13, 2, "h", 0.5), (3, 96, 7, 15, 2, "h", None), (3, 96, 7, 16, 2, "h", None),
    (4, 160, 6, 9, 2, "h", None), (4, 160, 6, 12, 2, "h", None), (4, 160, 6, 13, 4, "h", None),
    (5, 160, 6, 15, 2, "h", None), (5, 160, 6, 16, 2, "h", 0.1), (6, 128, 5, 9, 4, "h", None),
    (6, 128, 5, 12, 4, "h", None), (6, 128, 5, 13, 2, "b", None), (6, 128, 5, 15, 4, "b", None),
    (6, 128, 5, 16, 4, "b", 0.2), (2, 48, 4, 9, 8, "h", None), (2, 48, 4, 12, 8, "h", None),
    (2, 48, 4, 13, 8, "h", 0.25), (5, 72, 5, 0, 8, "h", None), (6, 72, 5, 0, 8, "b", None),
    (1, 64, 4, 0, 1, "h", 0.015625), (1, 64, 4, 0, 1, "h", 2.0), (2, 80, 4, 8, 2, "b", 2.0),
    (2, 256, 8, 0, 2, "h", None), (2, 256, 8, 8, 2, "h", None), (2, 256, 8, 16, 2, "h", None),
    (1, 224, 8, 12, 2, "h", None), (1, 224, 8, 15, 2, "h", None), (1, 224, 8, 16, 2, "b", None),
    (1, 128, 6, 9, 8, "h", None), (1, 128, 6, 12, 8, "h", None), (1, 128, 6, 16, 8, "h", None),
    (5, 96, 7, 16, 4, "h", None), (5, 96, 7, 15, 4, "b", None), (2, 191, 6, 16, 2, "h", None),
    (2, 193, 6, 16, 2, "h", None),
]
assert len(REFERENCE_MATRIX) == 102

# Backward passes at the edges of what dQ and sequence dK/dV take as one launch (256 compute units):
# (B, T, H, G, D, L, L_valid, mode, dtype), one launch or not
ONE_LAUNCH = [
    # one workgroup; ragged tiles with four row waves; more than 1024 query rows; head dims below the tile width; a partial
    # stream; no stream; depth gradients of their own launch (G 3); chunk-visible
    ((1, 1, 1, 1, 64, 1, 1, "CAUSAL", "fp16"), True),
    ((2, 95, 4, 2, 64, 8, 8, "CAUSAL", "fp16"), True),
    ((3, 257, 1, 4, 64, 3, 3, "NONCAUSAL", "bf16"), False),
    ((2, 130, 2, 1, 40, 5, 2, "NONCAUSAL", "bf16"), True),
    ((2, 77, 3, 2, 64, 0, 0, "CAUSAL", "bf16"), True),
    ((1, 70, 2, 3, 48, 4, 4, "CAUSAL", "fp16"), True),
    ((1, 100, 2, 4, 64, 3, 3, "CHUNK_VISIBLE", "bf16"), True),
    # more than twice the compute units, then the last size in one launch and the first one in two: 510 and 515 workgroups; as
    # many query rows as row waves take, and one token more
    ((32, 127, 4, 1, 64, 2, 2, "CAUSAL", "bf16"), False),
    ((32, 129, 4, 1, 64, 2, 2, "CAUSAL", "bf16"), False),
    ((51, 127, 2, 1, 64, 2, 2, "CAUSAL", "bf16"), True),
    ((103, 127, 1, 1, 64, 2, 2, "NONCAUSAL", "bf16"), False),
    ((3, 256, 4, 4, 64, 2, 2, "CAUSAL", "fp16"), True),
    ((4, 1024, 3, 1, 64, 1, 1, "NONCAUSAL", "bf16"), True),
    ((3, 1025, 1, 1, 64, 1, 1, "NONCAUSAL", "bf16"), False),
    # fp32: both instantiations, one row, an empty and a partial stream, chunk-visible, the last size in one launch and the
    # first one in two (256 and 260 workgroups)
    ((1, 1, 1, 1, 64, 1, 1, "CAUSAL", "fp32"), True),
    ((1, 256, 4, 1, 64, 4, 4, "CAUSAL", "fp32"), True),
    ((2, 61, 2, 2, 36, 3, 2, "NONCAUSAL", "fp32"), True),
    ((1, 90, 2, 3, 64, 0, 0, "CAUSAL", "fp32"), True),
    ((1, 70, 2, 4, 20, 3, 3, "CHUNK_VISIBLE", "fp32"), True),
    ((1, 1024, 1, 2, 64, 8, 8, "CAUSAL", "fp32"), True),
    ((1, 1025, 1, 2, 64, 8, 8, "CAUSAL", "fp32"), False),
]

# Small shapes used to cross-check the oracle's forms on the CPU:
# (B, T, H, D, L, G, mode, chunk_tokens)
ORACLE_SMALL = [
    (1, 1, 1, 8, 0, 1, "causal", 0),
    (1, 1, 1, 8, 3, 2, "causal", 0),
    (2, 7, 2, 8, 0, 1, "causal", 0),
    (2, 7, 2, 8, 3, 1, "causal", 0),
    (1, 9, 2, 16, 5, 2, "causal", 0),
    (1, 9, 2, 16, 5, 2, "noncausal", 0),
    (2, 6, 1, 8, 0, 4, "noncausal", 0),
    (1, 13, 2, 8, 3, 2, "chunk_visible", 4),
    (1, 13, 2, 8, 3, 1, "chunk_visible", 1),
    (1, 16, 1, 8, 2, 4, "chunk_visible", 16),
    (2, 5, 2, 8, 4, 1, "depth_only", 0),
    (1, 6, 2, 16, 7, 4, "depth_only", 0),
]
