"""Engine settings.

``default_dtype``: coefficient dtype of new sectors.  complex128 runs the
FP64 engine; complex64 runs the mixed-precision engine (complex FP32
storage, BF16 hi/lo split matrix-core GEMM with FP32 accumulation, FP64
norms and Taylor accumulation).

``contraction``: arithmetic of the complex128 split apply's alpha-row
contraction.  "fp64" multiplies on the FP64 matrix cores; "ozaki" forms
the same products exactly from 8-bit digits on the int8 matrix cores
(complex128 storage kept), about 1e-11 from the FP64 result.
"""

import numpy

default_dtype = numpy.complex128

# Maximum number of orbitals of the GPU string tables (uint64 strings,
# int32-addressed tables).
max_norb = 32

# Use the fused gather + GEMM + scatter kernels for real operators when the
# sector fits them (else, and for complex operators, the unfused kernels).
fused = True

# complex64 applies of a pair-symmetric real operator: beta-beta block as
# one BF16x3 GEMM and an alpha-only row kernel (no beta scatter).  Off, or
# for other operators, the row kernel also scatters beta excitations.
split = True

# complex128 applies of a pair-symmetric real operator: beta-beta block as
# one FP64 matrix-core GEMM and an FP64 row kernel over the live alpha pair
# rows.  Off, the FP64 row kernel also scatters beta excitations.
split_fp64 = True

# Kernel of the split row pass: 0 = MFMAs over the live pair rows of each
# alpha string only (excitations to another string plus the folded
# diagonal row); 16 = MFMAs over all npair + 1 pair rows.
split_tile = 0

# Kernel of complex128 two-body applies (with split_fp64): None = the pull
# form (alpha rows of C contracted with the opposite-spin coupling, beta
# excitations accumulated within the row), for real, complex and
# spin-orbital operators; a number = the split row pass of real
# pair-symmetric operators, 0 with column-owned waves (the D' values of a
# wave's columns gathered into its MFMA registers, A' in LDS), 32 with a
# shared, double-buffered D tile, other operators on the unfused kernels.
split_tile_fp64 = None

# Arithmetic of complex128 applies of pair-symmetric real operators: "fp64"
# (FP64 matrix cores) or "ozaki" (exact int8 digit products, FP64 assembly).
contraction = "fp64"

# With contraction = "ozaki": the same-spin products as digit products too
# (else FP64 matrix cores for those).
ozaki_beta = True

# With contraction = "ozaki": sectors below this many determinants run in
# FP64, where the digit kernels' extra launches (maxima, digits) cost more
# than the faster products save; 0: digits wherever the kernels take them.
# It is the size of a sector of as many alpha as beta strings; of others the
# work of the same-spin products is compared with that one's (runs_digits).
ozaki_min_determinants = 385000

# Largest apply workspace (bytes) allocated at once: a complex128 sector
# whose unfused dvec + Y would need more runs the apply in panels of
# orbital pairs within this budget (fqehip_apply_panels).
max_workspace_bytes = 96 << 30

# Single-sector time evolution: record the whole Taylor series once into a
# HIP graph (fqehip_taylor_graph_create) and replay it with one launch per
# time_evolve; the graph and its buffers are cached on the operator for the
# last (sector, time, accuracy, expansion) it ran.
taylor_graph = False


def kernel_choice():
    """Every setting that picks an apply's kernels."""
    return (fused, split, split_fp64, split_tile, split_tile_fp64, contraction,
            ozaki_beta, ozaki_min_determinants)


def runs_digits(lena, lenb):
    """Whether a sector runs on digits with contraction = "ozaki".
    Measured, FP64 / digits in us (strings alpha x beta):
    - by the work of the same-spin products: 462 x 462 91 / 132, 220 x 924
      106 / 130, 495 x 792 180 / 175, 364 x 1001 231 / 217, 495 x 924 199 /
      192, 792 x 792 316 / 266, 1001 x 1001 519 / 381;
    - FP64 rows of few alpha strings leave the chip idle, digit rows are
      shared out: 13 x 1716 120 / 92, 78 x 1716 163 / 136, 91 x 2002 245 /
      170, 14 x 3432 356 / 152, but 66 x 924 80 / 93;
    - a digit row costs its set-up, whatever its length: 6435 x 15 359 / 605,
      3003 x 91 302 / 311, 3432 x 91 359 / 351 (first apply 803 / 1300),
      6435 x 105 961 / 688."""
    least = ozaki_min_determinants
    if least == 0:
        return True
    if lena <= 128 and lenb * lenb >= 4 * least:
        return True
    work = lena * lenb * (lena + lenb) / (2 * least**1.5)
    return work >= (1 if lenb >= 128 else 4)
