// cluster_words.h — the geometry of a clustered launch (norm_cluster.h) in two words, and back.  Plain C++, which the host and the
// device compile alike.
//
// With the operands of the tile the words are the arguments that the waves find in their registers when they start (14 dwords of
// them): what has to be loaded is not waited for until the rows have been asked for.  The number of strips comes with its reciprocal.
#pragma once

constexpr int CL_NBLK_BITS = 12, CL_SPLIT_BITS = 2, CL_STRIP_BITS = 11, CL_RECIP = 20;

// csplit: a power of two
constexpr unsigned cluster_word_a(int nblk, int csplit, int rows_pm) {
    return (unsigned)nblk | (unsigned)__builtin_ctz((unsigned)csplit) << CL_NBLK_BITS | (unsigned)rows_pm << (CL_NBLK_BITS + CL_SPLIT_BITS);
}
constexpr unsigned cluster_word_b(int strips) {
    return (unsigned)strips | (unsigned)(((1 << CL_RECIP) + strips - 1) / strips) << CL_STRIP_BITS;
}
constexpr int cluster_nblk(unsigned wa) { return (int)(wa & ((1u << CL_NBLK_BITS) - 1)); }

// Workgroup number -> (slab, strip, member), the members of a cluster and the first of them, the rows of a member.
struct ClusterGeo {
    int blk, first, csplit, member, slab, strip, rows_pm;
};
constexpr ClusterGeo cluster_of(unsigned wa, unsigned wb, int blk) {
    const int shift = (int)(wa >> CL_NBLK_BITS & ((1u << CL_SPLIT_BITS) - 1));
    const unsigned cluster = (unsigned)blk >> shift;
    const int first = (int)(cluster << shift);
    const int slab = (int)(cluster * (wb >> CL_STRIP_BITS) >> CL_RECIP);
    const int strip = (int)cluster - slab * (int)(wb & ((1u << CL_STRIP_BITS) - 1));
    return {blk, first, 1 << shift, blk - first, slab, strip, (int)(wa >> (CL_NBLK_BITS + CL_SPLIT_BITS))};
}
