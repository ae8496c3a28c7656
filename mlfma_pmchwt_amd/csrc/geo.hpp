// Plain-old-data records shared by host setup code and device kernels.
#pragma once

namespace mlfma {

// Geometry of one RWG function, in the loop order of the reference's near-field
// operators: side 0 = negative face, side 1 = positive face
// (Code/Operator.h:727-776).
struct RwgGeo {
    double tri[2][9];    // v1, v2, v3 (xyz) of each face, file vertex order
    double vf[2][3];     // free vertex of each face
    double nrm[2][3];    // unit normal (snapped, Code/NASReader.cpp:52-56)
    double area[2];
    double len;          // common edge length
};

struct GaussRule {       // Dunavant rule, weights sum to 0.5
    int n;
    double l1[16], l2[16], l3[16], w[16];
};

// One face, for the near-field set-up (area and unit normal as in RwgGeo).
struct FaceGeo {
    double tri[9], nrm[3], area;
    int id;                  // face id, for the identical-triangle test
};

// A block of the near field being filled: rows of target group gt x columns of
// source group gs (groups: at most kFillRows RWG of one leaf, with the faces
// they touch), entry (row, col) of plane p at out + p * plane + col * ld + row.
struct FillBlock {
    int gt, gs, ld;
    long long out, plane;
    long long slot0;         // its first face pair in the batch's scratch (source face * target faces + target face)
};

struct NearFill {
    const FaceGeo* faces;
    const int* face_ptr;     // per group, its faces in face_idx
    const int* face_idx;
    const int* row_ptr;      // first internal RWG of each group
    const int2* side;        // per RWG: (face within its group) * 4 + free vertex, of the negative and positive half
    const double* len;       // edge lengths, internal order
    const FillBlock* blocks;
};

// Near field of one target leaf t: `planes` dense column-major matrices of
// nt rows and C_t = sum of its source leaves' sizes columns, one after the
// other from tgt_off[t]; the columns are the source leaves in pair order (near
// neighbours, then t itself) and pair p starts at column pair_col[p].
// PEC: 1 plane; PMCHWT: z11, zK, z22 (z12 = -zK, z21 = zK).
struct NearDev {
    int planes, nleaf, N;
    const int* leaf_ptr;
    const int* perm;
    const int* order;         // target leaves by decreasing nt * C_t (launch order)
    const long long* tgt_off; // first entry of each target's plane 0
    const int* tgt_cols;      // C_t
    const int* col_ptr;       // per target, first entry in colref
    const int* colref;        // caller-order index of x for every column
    int nitem;                // matrix-core work items: (target, first 16-row tile), <= 4 tiles each,
    const int2* items;        // by decreasing rows * C_t
    int nsplit;               // column-range items of the single-vector product (0: one workgroup per leaf)
    int nsplit32;             // the same for entries stored in FP32: nsplit or 0
    const int4* split;        // items: (target, first column, end column, index among the target's items), largest first
    const long long* part_ptr;   // per target, first of its items' partial sums in part: [item][current][row]
    double2* part;
    const int* leaf_of;       // leaf of every internal row
};

}  // namespace mlfma
