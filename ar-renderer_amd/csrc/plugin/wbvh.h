// 8-wide quantised BVH for the MI355X traversal kernels.
//
// The node follows the published compressed wide BVH (Ylitie, Karras, Laine, "Efficient Incoherent Ray
// Traversal on GPUs Through Compressed Wide BVHs", HPG 2017): a local grid of 8-bit planes, and children
// addressed by two bases and a byte each. The byte's meaning and the order of traversal are this file's
// and trace_dev.h's own.
//
// Layout in HBM:
//   WNode[]  80 bytes of node in a 128-byte line. Child boxes are quantised to 8 bits per axis
//            against the node's origin and power-of-two scale, rounded outwards so every decoded
//            child box contains its primitives. A node's internal children are consecutive nodes
//            and its leaf children's records are consecutive records, so a child is one byte.
//   TriRec[] 48-byte leaf records in leaf order: a triangle's p0, e1 = p1 - p0, e2 = p2 - p0
//            (the exact float operands of the reference's Moller-Trumbore test) and its
//            original primitive index; a sphere stores its centre and radius. The last record of
//            a leaf is marked.
#pragma once

#include <cstdint>
#include <vector>

#include "prender_gpu.h"

#ifndef PG_NODE_ALIGN
#define PG_NODE_ALIGN 128
#endif

namespace pgpu {

constexpr uint32_t kLeafBit = 0x80000000u;
constexpr int kMaxLeafPrims = 8;  // primitives per leaf child (count - 1 in 3 bits)
constexpr uint32_t kSphereBit = 0x80000000u;  // TriRec::prim flag: a sphere
constexpr uint32_t kLastBit = 0x40000000u;    // TriRec::prim flag: the last record of its leaf
constexpr uint32_t kPrimMask = 0x3fffffffu;

// A child's meta byte and the node's two bases give its reference in one addition: internal child
// k of the node is childBase + k (meta k, 0 .. 7); a leaf child whose first record is record o of
// the node's is recBase + (0x80 + o), with kLeafBit and -0x80 folded into recBase. A slot without
// a child has an inverted box (lower planes 255, upper 0), which no ray enters, and the meta byte
// of a leaf, so that even a distance so large that its planes coincide only tests a record twice.
struct alignas(PG_NODE_ALIGN) WNode {
    float ox, oy, oz;            // quantisation origin
    uint8_t ex, ey, ez;          // scale = 2^(e - 127) per axis: the exponent field of the float
    uint8_t pad;
    uint32_t childBase, recBase;
    uint8_t meta[8];
    uint8_t qlo[3][8];           // [axis][child]
    uint8_t qhi[3][8];
};
static_assert(sizeof(WNode) == (PG_NODE_ALIGN > 80 ? PG_NODE_ALIGN : 80), "WNode");

struct alignas(16) TriRec {
    float p0x, p0y, p0z;
    float e1x, e1y, e1z;
    float e2x, e2y, e2z;
    uint32_t prim;  // original primitive index | kSphereBit for spheres (p0 = centre, e1x = radius) | kLastBit
    uint32_t pad[2];
};
static_assert(sizeof(TriRec) == 48, "TriRec is 48 bytes");

struct WideBVH {
    std::vector<WNode> nodes;
    std::vector<TriRec> recs;  // in leaf order, then one record that no ray hits (never empty)
    int depth = 0;         // maximum node depth (root = 1)
    float lo[3], hi[3];    // scene bounds
};

// Builds the wide BVH over the scene's primitives (binned SAH binary build, collapsed to 8-wide).
void BuildWideBVH(const prgpu::Primitive *prims, int count, WideBVH *out);

}  // namespace pgpu
