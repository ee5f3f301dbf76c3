// Octree traversal state machine shared by the raymarch kernels.
//
// Restates VoxelOctree::raymarch (src/VoxelOctree.cpp:207-346) in FP32 with
// the reference's operation order; ray_init is the set-up before the loop
// (:216-250), ray_step one pass of the loop body (:252-338), walk the whole
// loop for finite rays in fewer, larger passes. Splitting the loop into
// resumable steps lets a persistent wave hand a finished lane a new ray while
// the other lanes keep walking; the other kernels use walk.
//
// The same source also compiles for the host (single-ray calls, where a
// device round trip costs far more than the walk itself): every operation is
// a correctly rounded FP32 add, multiply or divide, a comparison or integer
// bit work, so host and device give the same bits.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace svo {
namespace march {

#define SVO_HD __host__ __device__ __forceinline__

constexpr int kMaxScale = 23;  // VoxelOctree::MaxScale, src/VoxelOctree.hpp:38

SVO_HD float smin(float a, float b) { return (b < a) ? b : a; }  // std::min
SVO_HD float smax(float a, float b) { return (a < b) ? b : a; }  // std::max
SVO_HD uint32_t f2u(float f) { return __builtin_bit_cast(uint32_t, f); }
SVO_HD float u2f(uint32_t u) { return __builtin_bit_cast(float, u); }
SVO_HD int popc32(uint32_t x) { return __builtin_popcount(x); }
// bit 0 of x (a v_bfe_u32 on the device)
SVO_HD uint32_t bit0(uint32_t x) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_ubfe(x, 0, 1);
#else
    return x & 1u;
#endif
}

SVO_HD int umax(int a, int b) { return uint32_t(a) > uint32_t(b) ? a : b; }
// bit k of x
SVO_HD uint32_t bit_at(uint32_t x, int k) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_ubfe(x, uint32_t(k), 1);
#else
    return (x >> k) & 1u;
#endif
}

// All ones where a < b (finite), else 0: the sign of the difference, which is
// zero only for equal values.
SVO_HD uint32_t lt_bits(float a, float b) { return uint32_t(int32_t(f2u(a - b)) >> 31); }
// Bitwise function of three words by its truth table (a = 0xF0, b = 0xCC, c = 0xAA).
template <int Table>
SVO_HD uint32_t bitop(uint32_t a, uint32_t b, uint32_t c) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_bitop3_b32(a, b, c, Table);
#else
    uint32_t r = 0;
    for (int k = 0; k < 8; ++k)
        if (Table >> k & 1) r |= (k & 4 ? a : ~a) & (k & 2 ? b : ~b) & (k & 1 ? c : ~c);
    return r;
#endif
}
// invSqrt, src/Util.hpp:47-58
SVO_HD float quake_rsqrt(float x) {
    float half = x * 0.5f;
    float y = u2f(0x5f3759dfu - (f2u(x) >> 1));
    return y * (1.5f - half * y * y);
}

// The restart stack has one entry per scale a ray can push from: depth - 1
// for a tree of `depth` (descriptor levels + 1). The top `reg` entries live in
// registers instead of LDS: entry 0, the root's, is always (word 0, the ray's
// initial maxT: nothing changes maxT while the ray is at the root), entries 1
// and 2 are register pairs. 160 KiB of LDS holds 32 waves' stacks of 10
// entries (8 bytes per lane), so trees up to depth 12 keep one entry in
// registers and deeper ones three (the 8192^3 terrain, depth 14: 26 -> 32
// waves per CU).
__host__ __device__ inline int reg_entries(int depth) { return depth > 12 ? 3 : 1; }
__host__ __device__ inline int lds_slots(int depth, int reg) { return depth - 1 - reg > 0 ? depth - 1 - reg : 1; }

// Per-lane restart stack in LDS, one entry per scale below the root's children.
// 64-bit word indices: [slot][stride] indices then [slot][stride] maxT.
template <typename Idx>
struct Stack {
    Idx *off;
    float *tmax;
    int stride;
    int slots;
    int lane;
    SVO_HD Stack(void *base, int stride_, int slots_, int lane_)
        : off(reinterpret_cast<Idx *>(base)),
          tmax(reinterpret_cast<float *>(reinterpret_cast<Idx *>(base) + size_t(slots_) * stride_)),
          stride(stride_), slots(slots_), lane(lane_) {}
    SVO_HD void push(int slot, Idx parent, float t) const {
        off[slot * stride + lane] = parent;
        tmax[slot * stride + lane] = t;
    }
    SVO_HD void pop(int slot, Idx &parent, float &t) const {
        parent = off[slot * stride + lane];
        t = tmax[slot * stride + lane];
    }
};

// 32-bit word indices: one 8-byte {index, maxT} entry per [slot][stride], so a
// push or pop is a single 64-bit LDS access (same 8 bytes per entry).
template <>
struct Stack<uint32_t> {
    uint2 *e;
    int stride;
    int slots;
    SVO_HD Stack(void *base, int stride_, int slots_, int lane_)
        : e(reinterpret_cast<uint2 *>(base) + lane_), stride(stride_), slots(slots_) {}
    SVO_HD void push(int slot, uint32_t parent, float t) const { e[slot * stride] = make_uint2(parent, f2u(t)); }
    SVO_HD void pop(int slot, uint32_t &parent, float &t) const {
        const uint2 v = e[slot * stride];
        parent = v.x;
        t = u2f(v.y);
    }
};

template <typename Idx>
struct Ray {
    float dTx, dTy, dTz, bTx, bTy, bTz;
    float minT, maxT, maxT0, posX, posY, posZ, scaleExp2, rayScale;  // maxT0: the root's maxT
    Idx parent1, parent2;  // stack entries 1 and 2 when they are held in registers
    float maxT1, maxT2;
    uint32_t current;
    Idx parent;
    int octantMask, idx, scale;
};

// Outcome of a finished ray.
enum : int { kRunning = -1, kMiss = 0, kLeaf = 1, kLod = 2 };

// Set-up before the loop (:216-250). The root descriptor is read here, the
// read the first loop pass makes (:254).
template <typename Idx>
SVO_HD void ray_init(Ray<Idx> &r, const uint32_t *__restrict__ tree, float ox, float oy, float oz, float dx, float dy,
                     float dz, float rayScale) {
    if (fabsf(dx) < 1e-4f) dx = 1e-4f;
    if (fabsf(dy) < 1e-4f) dy = 1e-4f;
    if (fabsf(dz) < 1e-4f) dz = 1e-4f;
    r.dTx = 1.0f / -fabsf(dx);
    r.dTy = 1.0f / -fabsf(dy);
    r.dTz = 1.0f / -fabsf(dz);
    r.bTx = r.dTx * ox;
    r.bTy = r.dTy * oy;
    r.bTz = r.dTz * oz;
    r.octantMask = 7;
    if (dx > 0.0f) { r.octantMask ^= 1; r.bTx = 3.0f * r.dTx - r.bTx; }
    if (dy > 0.0f) { r.octantMask ^= 2; r.bTy = 3.0f * r.dTy - r.bTy; }
    if (dz > 0.0f) { r.octantMask ^= 4; r.bTz = 3.0f * r.dTz - r.bTz; }
    float minT = smax(2.0f * r.dTx - r.bTx, smax(2.0f * r.dTy - r.bTy, 2.0f * r.dTz - r.bTz));
    r.maxT = smin(r.dTx - r.bTx, smin(r.dTy - r.bTy, r.dTz - r.bTz));
    minT = smax(minT, 0.0f);
    r.minT = minT;
    r.maxT0 = r.maxT;
    r.current = tree[0];
    r.parent = 0;
    r.idx = 0;
    r.posX = 1.0f;
    r.posY = 1.0f;
    r.posZ = 1.0f;
    r.scale = kMaxScale - 1;
    r.scaleExp2 = 0.5f;
    r.rayScale = rayScale;
    if (1.5f * r.dTx - r.bTx > minT) { r.idx ^= 1; r.posX = 1.5f; }
    if (1.5f * r.dTy - r.bTy > minT) { r.idx ^= 2; r.posY = 1.5f; }
    if (1.5f * r.dTz - r.bTz > minT) { r.idx ^= 4; r.posZ = 1.5f; }
}

// False when a ray coefficient is NaN (a NaN origin or direction component, or
// an infinite origin on an axis whose direction is infinite: -0 * inf). Every
// corner time is then NaN, no axis ever steps and the reference's loop does not
// end. For all other rays some axis steps on every advance (the minimum corner
// time equals at least one corner time), each node is entered at most once and
// the walk ends.
template <typename Idx>
SVO_HD bool ray_defined(const Ray<Idx> &r) {
    return r.dTx == r.dTx && r.dTy == r.dTy && r.dTz == r.dTz && r.bTx == r.bTx && r.bTy == r.bTy &&
           r.bTz == r.bTz;
}

// Origin and direction finite, origin below 2^100: every corner time is finite
// and never -0 (see ray_step).
SVO_HD bool ray_finite(float ox, float oy, float oz, float dx, float dy, float dz) {
    constexpr float kOrigin = 1.2676506e30f, kFloatMax = 3.4028234663852886e38f;
    return fabsf(ox) < kOrigin && fabsf(oy) < kOrigin && fabsf(oz) < kOrigin && fabsf(dx) <= kFloatMax &&
           fabsf(dy) <= kFloatMax && fabsf(dz) <= kFloatMax;
}

// One pass of the loop body. Returns kRunning, or the outcome with tOut /
// normal / leaf set as the reference sets them. The descriptor of the node
// the ray is in (`current`) is read as soon as its index is known (init,
// push, pop) rather than at the top of the next pass; the value is the same.
//
//  Lod = false: the ray's rayScale is 0 (+0 or -0). maxTC is finite, so
//    maxTC * rayScale >= scaleExp2 (> 0) never holds and the test is dropped.
//  Normal = false: the caller needs only the hit code and t; a leaf hit
//    leaves `leaf` and `normal` unset and reads no leaf word.
//  Reg: how many top stack entries are held in registers (1 or 3); the LDS
//    stack holds the others, entry e at LDS slot e - Reg.
//  Finite = true: the ray's origin and direction are finite (|origin| below
//    2^100). Then every corner t is finite and never -0 (pos*dT is a nonzero
//    product; a difference of equal nonzero values is +0), so the minimum of
//    the three corner times does not depend on the order of ties or on NaN
//    handling and one hardware min3 returns the reference's std::min result.
template <bool Lod, bool Finite, typename Idx, bool Normal = true, int Reg = 1>
SVO_HD int ray_step(Ray<Idx> &r, const uint32_t *__restrict__ tree, const Stack<Idx> &stk,
                                        uint32_t &normal, float &tOut, Idx &leaf) {
    const float cornerTX = r.posX * r.dTx - r.bTx;
    const float cornerTY = r.posY * r.dTy - r.bTy;
    const float cornerTZ = r.posZ * r.dTz - r.bTz;
    const float maxTC = Finite ? fminf(cornerTX, fminf(cornerTY, cornerTZ)) : smin(cornerTX, smin(cornerTY, cornerTZ));

    const int childShift = r.idx ^ r.octantMask;
    const uint32_t childMasks = r.current << childShift;

    if ((childMasks & 0x8000u) && r.minT <= r.maxT) {
        if (Lod && maxTC * r.rayScale >= r.scaleExp2) {
            tOut = maxTC;
            return kLod;
        }
        const float maxTV = smin(r.maxT, maxTC);
        const float half = r.scaleExp2 * 0.5f;
        const float centerTX = half * r.dTx + cornerTX;
        const float centerTY = half * r.dTy + cornerTY;
        const float centerTZ = half * r.dTz + cornerTZ;

        if (r.minT <= maxTV) {
            Idx childOffset = Idx(r.current >> 18);
            if (r.current & 0x20000u)
                childOffset = Idx((uint64_t(r.current >> 18) << 32) | uint64_t(tree[r.parent + 1]));
            if (!(childMasks & 0x80u)) {
                if (Normal) {
                    leaf = childOffset + r.parent +
                           Idx(popc32((((childMasks >> (8 + childShift)) << childShift) & 127u)));
                    normal = tree[leaf];
                }
                tOut = r.minT;
                return kLeaf;
            }
            // slot - Reg < stk.slots: a node at level L (slot L) pushes only when
            // it has a non-leaf child, and octree_validate then counted depth >=
            // L + 2 (every loaded or built tree is validated); the root's entry
            // (slot 0) is (0, maxT0) and is not stored
            const int slot = (kMaxScale - 1) - r.scale;
            static_assert(Reg == 1 || Reg == 3, "register-held stack entries: 1 or 3");
            if (slot >= Reg) {
                stk.push(slot - Reg, r.parent, r.maxT);
            } else if (Reg == 3 && slot == 1) {
                r.parent1 = r.parent;
                r.maxT1 = r.maxT;
            } else if (Reg == 3 && slot == 2) {
                r.parent2 = r.parent;
                r.maxT2 = r.maxT;
            }

            const Idx siblingCount = Idx(popc32(childMasks & 127u));
            r.parent += childOffset + siblingCount;
            if (r.current & 0x10000u) r.parent += siblingCount;
            r.current = tree[r.parent];

            r.scale--;
            r.scaleExp2 = half;
            const bool cx = centerTX > r.minT, cy = centerTY > r.minT, cz = centerTZ > r.minT;
            if (cx) r.posX += r.scaleExp2;
            if (cy) r.posY += r.scaleExp2;
            if (cz) r.posZ += r.scaleExp2;
            r.idx = (cx ? 1 : 0) | (cy ? 2 : 0) | (cz ? 4 : 0);
            r.maxT = maxTV;
            return kRunning;
        }
    }

    const bool sx = cornerTX <= maxTC, sy = cornerTY <= maxTC, sz = cornerTZ <= maxTC;
    if (sx) r.posX -= r.scaleExp2;
    if (sy) r.posY -= r.scaleExp2;
    if (sz) r.posZ -= r.scaleExp2;
    const int stepMask = (sx ? 1 : 0) | (sy ? 2 : 0) | (sz ? 4 : 0);

    r.minT = maxTC;
    r.idx ^= stepMask;

    if ((r.idx & stepMask) != 0) {
        uint32_t diff = 0;
        if (stepMask & 1) diff |= f2u(r.posX) ^ f2u(r.posX + r.scaleExp2);
        if (stepMask & 2) diff |= f2u(r.posY) ^ f2u(r.posY + r.scaleExp2);
        if (stepMask & 4) diff |= f2u(r.posZ) ^ f2u(r.posZ + r.scaleExp2);
        // The reference takes the highest differing bit from the exponent of
        // float(int(diff)) (src/VoxelOctree.cpp:318-325). diff is non-zero (a
        // stepped coordinate in [1,2) changes by at least its ulp); below 2^23
        // the conversion is exact, so the exponent is 31 - clz(diff); from 2^23
        // up both forms give a scale >= 23 and the ray leaves the octree. The
        // reference then reads rayStack[scale] and leaves the loop; that read
        // cannot reach the result.
        if (diff >= (1u << kMaxScale)) return kMiss;
        r.scale = 31 - __builtin_clz(diff);
        r.scaleExp2 = u2f(uint32_t(r.scale - kMaxScale + 127) << 23);
        const int slot = (kMaxScale - 1) - r.scale;  // a slot pushed earlier: the new scale is above the current one
        if (slot >= Reg) {
            stk.pop(slot - Reg, r.parent, r.maxT);
        } else if (slot == 0) {
            r.parent = 0;
            r.maxT = r.maxT0;
        } else if (Reg == 3 && slot == 1) {
            r.parent = r.parent1;
            r.maxT = r.maxT1;
        } else if (Reg == 3) {
            r.parent = r.parent2;
            r.maxT = r.maxT2;
        }
        r.current = tree[r.parent];

        const uint32_t shX = f2u(r.posX) >> r.scale;
        const uint32_t shY = f2u(r.posY) >> r.scale;
        const uint32_t shZ = f2u(r.posZ) >> r.scale;
        r.posX = u2f(shX << r.scale);
        r.posY = u2f(shY << r.scale);
        r.posZ = u2f(shZ << r.scale);
        r.idx = int(bit0(shX) | (bit0(shY) << 1) | (bit0(shZ) << 2));
    }
    return kRunning;
}

// ---- whole-ray walk of finite rays ------------------------------------------
//
// The same outcome as ray_step taken to its end, for rays ray_finite accepts,
// from two properties of finite rays:
//  - a node's maxT is its own exit time, the smallest of its corner times: a
//    child's corner times are no later than its parent's, since a corner
//    coordinate grows from parent to child, dT is negative and a rounded
//    product and difference are monotone. So `minT <= maxT && minT <= maxTV`
//    is `minT <= maxTC`, and neither a ray nor a stack entry holds a maxT.
//  - every advance leaves the ray at the scale of the highest position bit
//    it changed, the current scale when it stays in the node: one piece of
//    code serves an advance inside the node and a pop, if the stack holds an
//    entry for the current node too.
// A pass takes an advance (or pop) where the cell cannot be entered and then,
// in the same pass, the descent into the cell it reached where that can be
// entered. A pop reads its node from LDS, so a pass waits for the tree's
// memory once, for the descriptor it descended into (and its far word, which
// travels with it). The next cell and its corner times are computed while that
// read is under way and carried to the next pass.
//
// What bounds it: while all wave slots are busy VALU issue and the waits for
// descriptors about equally (a wave executes nearly every pass's advance and
// descent, 41 of 64 lanes active on average); at a launch's end the dependent
// descriptor reads of the slowest tile. Against one step per pass through
// ray_step (2048^3 mesh octree, 1920x1080, outputs equal): 8 views in one
// launch 1,375 -> 858 us, one planned view 246 -> 146 us; 3840x2160 with
// shadows over an 8192^3 terrain 1,515 -> 985 us. Of that, the corner times
// carried over and computed behind the read (they were computed again at the
// top of each pass, after the wait) gave 1,064 -> 978, 221 -> 191 and 1,267 ->
// 1,179 us, the far word read beside its descriptor instead of after it 982 ->
// 964, 181 -> 157 and 1,182 -> 1,104 us, a far test only in two-word slots, one
// loop exit (the outcome read off the position afterwards) and the values
// pinned by SVO_HOLD 945 -> 896, 154 -> 152 and 1,087 -> 1,030 us. A second
// advance per pass was slower (982 -> 1,046 us: fewer passes, but more of them
// executed for few lanes).
//
// The loop prefers instructions that issue two per four cycles on a SIMD
// (measured on this card with all wave slots busy: f32 add, subtract, multiply,
// and/or/xor, right shifts, u32 add and subtract, bitop3) over those that issue
// one (compares, selects, min/max, left shifts, bit-field extracts, shift-adds,
// anything with a scalar operand): a selection is a sign mask and an `and`
// (lt_bits, bitop) where that takes no more instructions. 45 of the pass's 86
// instructions were of the slower kind, 26 of 87 now: 893 -> 858, 151 -> 146
// and 1,029 -> 985 us. Trading the position bits' three extracts for six
// faster instructions gave nothing more.

// The nodes on a ray's path, one entry per scale of their children: a node's
// child block (a byte address from the tree's first word whose low two bits
// hold the descriptor's large and far flags) and its two masks, 6 bytes per
// entry and lane (10 for 64-bit addresses). `levels` entries, for scales
// kMaxScale - levels and up; laid out [scale][lane], addresses then masks.
template <typename Addr>
struct PathStack {
    Addr *a;
    uint16_t *m;
    int stride;
    SVO_HD PathStack(void *base, int stride_, int levels, int lane)
        : a(reinterpret_cast<Addr *>(base) + (lane - (kMaxScale - levels) * stride_)),
          m(reinterpret_cast<uint16_t *>(reinterpret_cast<Addr *>(base) + levels * stride_) +
            (lane - (kMaxScale - levels) * stride_)),
          stride(stride_) {}
    SVO_HD void put(int scale, Addr addr, uint32_t masks) const {
        a[scale * stride] = addr;
        m[scale * stride] = uint16_t(masks);
    }
    SVO_HD void get(int scale, Addr &addr, uint32_t &masks) const {
        addr = a[scale * stride];
        masks = m[scale * stride];
    }
};
template <typename Addr>
__host__ __device__ inline size_t path_bytes(int levels) {
    return size_t(levels) * 64 * (sizeof(Addr) + sizeof(uint16_t));
}

template <typename Addr>
SVO_HD uint32_t tree_word(const uint32_t *__restrict__ tree, Addr byte) {
    return *reinterpret_cast<const uint32_t *>(reinterpret_cast<const char *>(tree) + byte);
}

// The child block of the node whose descriptor `d` lies at byte p: bits 31..18
// are words, shifted to bytes above the two flag bits; with the far flag they
// are the high bits of a word offset whose low 32 bits are farWord.
template <typename Addr>
SVO_HD Addr near_block(Addr p, uint32_t d) { return p + Addr(d >> 16); }
template <typename Addr>
SVO_HD Addr far_block(Addr p, uint32_t d, uint32_t farWord) {
    return p + Addr(((uint64_t(d >> 18) << 32) | farWord) << 2) + Addr((d >> 16) & 3u);
}

// Where a walk ended: the cell's child slot in the node `block`/`masks`.
template <typename Addr>
struct WalkEnd {
    Addr block;
    uint32_t masks, slot;
    // word index of the leaf the walk ended in
    SVO_HD Addr leaf() const { return (block >> 2) + Addr(popc32(((masks >> 8) << slot) & 127u)); }
};

// Work between a load and its first use: SVO_ISSUED keeps the code after it
// behind the load, SVO_HOLD makes its values exist where it stands (ahead of
// a later use of the loaded value).
#if defined(__HIP_DEVICE_COMPILE__)
#define SVO_ISSUED() __builtin_amdgcn_sched_barrier(0)
#define SVO_HOLD(...) asm volatile("" : __VA_ARGS__)
#else
#define SVO_ISSUED()
#define SVO_HOLD(...)
#endif

// Walks one ray (r from ray_init) to its end: kMiss, kLeaf (tOut, end) or, with
// Lod, kLod (tOut). With Count, *passes counts the passes.
template <bool Lod, bool Count, typename Addr>
SVO_HD int walk(const Ray<Addr> &r, const uint32_t *__restrict__ tree, const PathStack<Addr> &path, float &tOut,
                WalkEnd<Addr> &end, uint32_t *passes = nullptr) {
    // only descriptors in two-word slots have far words (the others, which no
    // builder writes, take the 64-bit walk: path_launch)
    constexpr bool Tight = sizeof(Addr) == 4;
    // a cell's mask bits are shifted by its slot + 16: valid in bit 31,
    // non-leaf in bit 23, its earlier siblings' non-leaf bits in 22..16
    const uint32_t oct = uint32_t(r.octantMask) | 16u;
    float px = r.posX, py = r.posY, pz = r.posZ, minT = r.minT, e = 0.5f;
    int scale = kMaxScale - 1;
    uint32_t cs = uint32_t(r.idx) ^ oct, m = r.current;
    Addr block = near_block<Addr>(0, m);
    if (m & 0x20000u) block = far_block<Addr>(0, m, tree[1]);
    path.put(scale, block, m);
    float tx = px * r.dTx - r.bTx, ty = py * r.dTy - r.bTy, tz = pz * r.dTz - r.bTz;
    float tc = fminf(tx, fminf(ty, tz));
    bool stop;
    do {
        if (Count) ++*passes;
        uint32_t w = m << cs;
        bool in = int32_t(bitop<0x30>(w, f2u(tc - minT), 0u)) < 0;
        if (Lod && int32_t(w) < 0 && minT > tc) {
            // the reference's cut-off asks for minT <= the parent's exit only
            const uint32_t up = ~1u << scale;
            const float qx = u2f(f2u(px) & up) * r.dTx - r.bTx, qy = u2f(f2u(py) & up) * r.dTy - r.bTy,
                        qz = u2f(f2u(pz) & up) * r.dTz - r.bTz;
            if (minT <= fminf(qx, fminf(qy, qz)) && tc * r.rayScale >= e) {
                tOut = tc;
                return kLod;
            }
        }
        if (!in) {
            const uint32_t ox = f2u(px), oy = f2u(py), oz = f2u(pz);
            px -= u2f(bitop<0x30>(f2u(e), lt_bits(tc, tx), 0u));  // e where the axis's corner time is the smallest
            py -= u2f(bitop<0x30>(f2u(e), lt_bits(tc, ty), 0u));
            pz -= u2f(bitop<0x30>(f2u(e), lt_bits(tc, tz), 0u));
            minT = tc;
            SVO_HOLD("+v"(minT));
            const uint32_t diff = bitop<0xBE>(f2u(pz), oz, bitop<0xBE>(f2u(py), oy, f2u(px) ^ ox));
            const bool out = diff >= (1u << kMaxScale);
            // a ray that left the tree reads the root's entry and stops below
            scale = 31 - umax(__builtin_clz(diff), 32 - kMaxScale);
            SVO_HOLD("+v"(scale));
            e = u2f(uint32_t(scale - kMaxScale + 127) << 23);
            path.get(scale, block, m);
            const uint32_t keep = ~0u << scale;
            px = u2f(f2u(px) & keep);
            py = u2f(f2u(py) & keep);
            pz = u2f(f2u(pz) & keep);
            cs = (bit_at(f2u(px), scale) | (bit_at(f2u(py), scale) << 1) | (bit_at(f2u(pz), scale) << 2)) ^ oct;
            tx = px * r.dTx - r.bTx;
            ty = py * r.dTy - r.bTy;
            tz = pz * r.dTz - r.bTz;
            tc = fminf(tx, fminf(ty, tz));
            w = m << cs;
            in = int32_t(bitop<0x30>(w, f2u(tc - minT), 0u)) < 0;
            if (out) {  // stops like a leaf
                in = true;
                w = 0;
            }
        }
        if (Lod && in && w && tc * r.rayScale >= e) {
            tOut = tc;
            return kLod;
        }
        const bool down = in && (w & 0x800000u);
        stop = in && !down;
        if (down) {
            const uint32_t sib = uint32_t(popc32(w & 0x7F0000u));
            uint32_t width = bitop<0xEA>(uint32_t(block), 1u, 2u);  // log2 of a slot's bytes
            SVO_HOLD("+v"(width));
            const Addr p = ((Addr(sib) << width) + block) & ~Addr(3);
            // a two-word slot's far word travels with its descriptor (device
            // arrays have a word to spare after the last, kSpareWords)
            const bool two = width == 3;
            uint32_t farWord;
            m = tree_word<Addr>(tree, p);
            if (two) farWord = tree_word<Addr>(tree, p + 4);
            SVO_ISSUED();
            --scale;
            e *= 0.5f;
            const uint32_t mx = lt_bits(minT, e * r.dTx + tx), my = lt_bits(minT, e * r.dTy + ty),
                           mz = lt_bits(minT, e * r.dTz + tz);
            px += u2f(bitop<0xC0>(f2u(e), mx, 0u));
            py += u2f(bitop<0xC0>(f2u(e), my, 0u));
            pz += u2f(bitop<0xC0>(f2u(e), mz, 0u));
            cs = bitop<0x78>(bitop<0x78>(bitop<0x78>(oct, mx, 1u), my, 2u), mz, 4u);  // oct ^ (mx & 1) ^ ...
            tx = px * r.dTx - r.bTx;
            ty = py * r.dTy - r.bTy;
            tz = pz * r.dTz - r.bTz;
            tc = fminf(tx, fminf(ty, tz));
            SVO_HOLD("+v"(cs), "+v"(tx), "+v"(ty), "+v"(tz), "+v"(tc));
            SVO_HOLD("+v"(m));
            block = near_block<Addr>(p, m);
            if (Tight) {
                if (two) {
                    SVO_HOLD("+v"(farWord));  // not shifted before the wait
                    if (m & 0x20000u) block = far_block<Addr>(p, m, farWord);
                }
            } else if (m & 0x20000u) {
                block = far_block<Addr>(p, m, two ? farWord : tree_word<Addr>(tree, p + 4));
            }
            path.put(scale, block, m);
        }
    } while (!stop);
    tOut = minT;
    end.block = block;
    end.masks = m;
    end.slot = cs & 7u;
    // outside the tree a coordinate is below 1 (bit 23 of its float clear)
    return (f2u(px) & f2u(py) & f2u(pz) & (1u << kMaxScale)) ? kLeaf : kMiss;
}

}  // namespace march
}  // namespace svo
