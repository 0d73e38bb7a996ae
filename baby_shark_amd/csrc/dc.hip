// Dual contouring on the device (DualContouringMesher::mesh,
// src/voxel/meshing/dual_contouring.rs:23-83).
//
// The reference runs three visitor passes and keeps the edge crossings and
// the cell points in sparse trees behind locks.  Here:
//   * cell pass: one wavefront per leaf stages the leaf and a one-to-two voxel
//     halo (an 11^3 block from the 27 surrounding leaves) in LDS, one z-row per
//     lane, with a word of activity and sign bits per row.  Bit operations on
//     those words find the rows' crossing edges without all six gradients (the
//     reference's unreachable!() case), the crossing edges and the fully
//     active sign-changing cubes.  Then a lane takes an edge each (its crossing
//     and normal, to LDS) and after that a cube each (the damped particle
//     iteration over its listed edges).  Cell points go to the leaf's compact
//     list, in cell order, with a 512-bit presence mask and the leaf's signs.
//   * triangle pass: from the presence masks and signs alone, each row's
//     sign-changing edges whose four cells exist; a lane per such edge fetches
//     the four points and emits two triangles, scaled by the voxel size,
//     degenerate ones dropped.  A counting launch, a scan and a writing
//     launch give the sequential order: leaves by origin, voxels x-y-z, edges
//     X-Y-Z.
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <cmath>
#include <mutex>
#include <string>

#include "common.hpp"
#include "leafmap.hpp"

namespace bs {

Topology& ensure_topology(bs_ctx* ctx, bs_volume* v);

namespace {

constexpr int HB = 11;  // staged block edge: leaf-local -1 .. 9
constexpr int HR = HB * HB;
constexpr int CB = 9;    // rows of corners that the leaf's cells touch: 0 .. 8
constexpr int CR = CB * CB;
constexpr int EDGE_LDS = 192;  // crossing edges kept in LDS per leaf (about 45 on a smooth surface)

struct DcArgs {
    LeafMap map;
    const int4* origins;
    const uint64_t* masks;
    const float* values;
    float* cell_pts;        // per leaf 512 * 3: the points of its cells, in cell order, from its start
    uint64_t* cell_mask;    // n_leaves * 8
    uint64_t* neg_mask;     // n_leaves * 8: active voxels with the sign bit set
    float voxel_size;
    uint32_t* fail;         // bit 0: gradient without neighbours
};

struct Block {
    float val[HB * HR];
    uint32_t row[HR];        // z-row (x, y): bit z + 1 active, bit z + 17 active with the sign bit set
    uint32_t edge_row[CR];   // crossing edges from row (x, y), bit 9 * axis + z
    uint32_t edge_pre[CR];   // edges of the rows before
    float4 edge[EDGE_LDS];   // crossing coordinate along the edge, unit normal
    uint16_t list[EDGE_LDS > 512 ? EDGE_LDS : 512];  // edges, then cells
    int32_t nb[27];
};

__device__ inline int ridx(int x, int y) { return (x + 1) * HB + (y + 1); }

// Row r of the staged block: its eight own voxels in two 16-byte loads, one
// voxel of the leaf below and two of the leaf above, and the rows' mask bytes
// (byte y of word x holds row (x, y)).  A missing leaf's loads go to leaf 0 and
// are masked off, so all of a row's loads travel together.
struct RowLoads {
    float4 v0, v1;
    float2 up;
    float down;
    uint32_t m0, m1, m2;
};
__device__ inline void row_issue(const Block& B, const DcArgs& a, int r, RowLoads& q) {
    const int x = r / HB - 1, y = r % HB - 1;
    const int32_t* nb = B.nb + ((x >> 3) + 1) * 9 + ((y >> 3) + 1) * 3;
    const int32_t s0 = nb[0], s1 = nb[1], s2 = nb[2];
    const uint64_t t0 = s0 >= 0 ? s0 : 0, t1 = s1 >= 0 ? s1 : 0, t2 = s2 >= 0 ? s2 : 0;
    const int ro = ((x & 7) << 6) | ((y & 7) << 3), mo = ((x & 7) << 3) | (y & 7);
    const uint8_t* mb = reinterpret_cast<const uint8_t*>(a.masks);
    q.m0 = mb[t0 * 64 + mo];
    q.m1 = mb[t1 * 64 + mo];
    q.m2 = mb[t2 * 64 + mo];
    const float4* p = reinterpret_cast<const float4*>(a.values + t1 * 512 + ro);
    q.v0 = p[0];
    q.v1 = p[1];
    q.down = a.values[t0 * 512 + ro + 7];
    q.up = *reinterpret_cast<const float2*>(a.values + t2 * 512 + ro);
    if (s0 < 0) q.m0 = 0;
    if (s1 < 0) q.m1 = 0;
    if (s2 < 0) q.m2 = 0;
}
__device__ inline void row_store(Block& B, int r, const RowLoads& q) {
    const float v[HB] = {q.down, q.v0.x, q.v0.y, q.v0.z, q.v0.w, q.v1.x, q.v1.y, q.v1.z, q.v1.w, q.up.x, q.up.y};
    const uint32_t act = (q.m0 >> 7) | (q.m1 << 1) | ((q.m2 & 3u) << 9);
    uint32_t neg = 0;
#pragma unroll
    for (int k = 0; k < HB; ++k) {
        B.val[r * HB + k] = v[k];
        neg |= (__float_as_uint(v[k]) >> 31) << k;
    }
    B.row[r] = act | ((neg & act) << 16);
}

// Stages the values and the activity and sign bits of leaf-local voxels -1..9.
__device__ inline void stage_block(Block& B, const DcArgs& a, int4 org, int lane) {
    if (lane < 27) {
        const int dx = lane / 9 - 1, dy = (lane / 3) % 3 - 1, dz = lane % 3 - 1;
        B.nb[lane] = a.map.find((org.x >> 3) + dx, (org.y >> 3) + dy, (org.z >> 3) + dz);
    }
    __syncthreads();
    const int r1 = min(lane + 64, HR - 1);
    RowLoads q0, q1;
    row_issue(B, a, lane, q0);
    row_issue(B, a, r1, q1);
    row_store(B, lane, q0);
    if (lane + 64 < HR) row_store(B, lane + 64, q1);
    __syncthreads();
}

// Crossing edge (v, v + e_d), v = (x, y, z) leaf-local, both ends active and of
// different sign (dual_contouring.rs:257-349): the crossing's coordinate along
// the edge in voxel units of the global grid, and the unit normal.  A gradient
// without both neighbours is one-sided; one without any is the reference's
// unreachable!(), reported before this is used.
__device__ inline float4 edge_crossing(const Block& B, int4 org, int x, int y, int z, int d) {
    const int step = d == 0 ? HR : (d == 1 ? HB : 1);
    const int rstep = d == 0 ? HB : (d == 1 ? 1 : 0);
    const int r1 = ridx(x, y), c1 = r1 * HB + z + 1;
    const float v1 = B.val[c1], v2 = B.val[c1 + step];
    const float t = (v1 == v2) ? 0.5f : v1 / (v1 - v2);
    float g[2][3];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        const int r = r1 + e * rstep, c = c1 + e * step, b = z + 1 + (d == 2 ? e : 0);
        const float vc = e ? v2 : v1;
#pragma unroll
        for (int ax = 0; ax < 3; ++ax) {
            const int s = ax == 0 ? HR : (ax == 1 ? HB : 1), rs = ax == 0 ? HB : (ax == 1 ? 1 : 0);
            const float l = B.val[c - s], h = B.val[c + s];
            const bool hl = (B.row[r - rs] >> (ax == 2 ? b - 1 : b)) & 1u, hr = (B.row[r + rs] >> (ax == 2 ? b + 1 : b)) & 1u;
            g[e][ax] = (hl && hr) ? (h - l) * 0.5f : (hr ? h - vc : vc - l);
        }
    }
    float n[3];
#pragma unroll
    for (int ax = 0; ax < 3; ++ax) n[ax] = (1.0f - t) * g[0][ax] + t * g[1][ax];
    const float len = sqrt_rn((n[0] * n[0] + n[1] * n[1]) + n[2] * n[2]);
    const float base = (float)(d == 0 ? org.x + x : (d == 1 ? org.y + y : org.z + z));
    return make_float4(base + t, n[0] / len, n[1] / len, n[2] / len);
}

// EDGE_OFFSETS (dual_contouring.rs:410-423): edge e's base offset and axis,
// five bits each (dx, dy, dz, axis).
constexpr uint64_t edge_code(int dx, int dy, int dz, int d) { return (uint64_t)(dx | dy << 1 | dz << 2 | d << 3); }
constexpr uint64_t EDGE_CODES =
    edge_code(0, 0, 0, 0) | edge_code(0, 0, 0, 1) << 5 | edge_code(0, 0, 0, 2) << 10 | edge_code(1, 0, 0, 1) << 15 |
    edge_code(1, 0, 0, 2) << 20 | edge_code(0, 0, 1, 0) << 25 | edge_code(0, 0, 1, 1) << 30 |
    edge_code(0, 1, 0, 0) << 35 | edge_code(0, 1, 0, 2) << 40 | edge_code(1, 0, 1, 1) << 45 |
    edge_code(0, 1, 1, 0) << 50 | edge_code(1, 1, 0, 2) << 55;

// Opt-in vertex placement (BS_DC_VERTEX_QEF_F64; the reference has only the
// particle iteration): the point minimising sum_i (n_i . (x - p_i))^2 over the
// cell's edge crossings p_i with unit normals n_i, in FP64.  Relative to the
// mass point m (the crossings' mean), A = sum n n^T and b = sum n (n . (p - m));
// A's eigenvectors come from cyclic Jacobi rotations and x = m + sum_k
// (v_k . b / l_k) v_k over the eigenvalues l_k > QEF_TRUNC * l_max (a plane
// fixes one direction, an edge two, a corner three; the rest stays at m).
// The point is clamped to the cell.
constexpr double QEF_TRUNC = 0.1;

// One Jacobi rotation zeroing A[p][q] of the symmetric A (Numerical Recipes'
// form: theta = (A_qq - A_pp) / (2 A_pq), t = sgn(theta) / (|theta| +
// sqrt(theta^2 + 1))), accumulated into the eigenvector columns of V.
template <int P, int Q>
__device__ inline void jacobi_rotate(double (&A)[3][3], double (&V)[3][3]) {
    const double apq = A[P][Q];
    if (apq == 0.0) return;
    const double theta = (A[Q][Q] - A[P][P]) / (2.0 * apq);
    const double t = (theta >= 0.0 ? 1.0 : -1.0) / (fabs(theta) + sqrt(theta * theta + 1.0));
    const double c = 1.0 / sqrt(t * t + 1.0), s = t * c;
    constexpr int R = 3 - P - Q;  // the third index
    const double arp = A[R][P], arq = A[R][Q];
    A[P][P] -= t * apq;
    A[Q][Q] += t * apq;
    A[P][Q] = A[Q][P] = 0.0;
    A[R][P] = A[P][R] = c * arp - s * arq;
    A[R][Q] = A[Q][R] = s * arp + c * arq;
#pragma unroll
    for (int r = 0; r < 3; ++r) {
        const double vp = V[r][P], vq = V[r][Q];
        V[r][P] = c * vp - s * vq;
        V[r][Q] = s * vp + c * vq;
    }
}

__device__ inline void qef_point(const float (&P)[12][3], const float (&N)[12][3], uint32_t valid, float cx0,
                                 float cy0, float cz0, float out[3]) {
    double m[3] = {0.0, 0.0, 0.0};
    const double cnt = (double)__popc(valid);
#pragma unroll
    for (int e = 0; e < 12; ++e)
        if (valid & (1u << e))
#pragma unroll
            for (int k = 0; k < 3; ++k) m[k] += (double)P[e][k];
#pragma unroll
    for (int k = 0; k < 3; ++k) m[k] /= cnt;
    double A[3][3] = {{0.0, 0.0, 0.0}, {0.0, 0.0, 0.0}, {0.0, 0.0, 0.0}}, b[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int e = 0; e < 12; ++e) {
        if (!(valid & (1u << e))) continue;
        const double n0 = N[e][0], n1 = N[e][1], n2 = N[e][2];
        const double d = n0 * ((double)P[e][0] - m[0]) + n1 * ((double)P[e][1] - m[1]) + n2 * ((double)P[e][2] - m[2]);
        A[0][0] += n0 * n0, A[0][1] += n0 * n1, A[0][2] += n0 * n2;
        A[1][1] += n1 * n1, A[1][2] += n1 * n2, A[2][2] += n2 * n2;
        b[0] += n0 * d, b[1] += n1 * d, b[2] += n2 * d;
    }
    A[1][0] = A[0][1], A[2][0] = A[0][2], A[2][1] = A[1][2];
    double V[3][3] = {{1.0, 0.0, 0.0}, {0.0, 1.0, 0.0}, {0.0, 0.0, 1.0}};
    for (int sweep = 0; sweep < 8; ++sweep) {
        jacobi_rotate<0, 1>(A, V);
        jacobi_rotate<0, 2>(A, V);
        jacobi_rotate<1, 2>(A, V);
    }
    const double lmax = fmax(fmax(A[0][0], A[1][1]), A[2][2]);
    double x[3] = {m[0], m[1], m[2]};
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const double l = A[k][k];
        if (!(l > QEF_TRUNC * lmax)) continue;
        const double w = (V[0][k] * b[0] + V[1][k] * b[1] + V[2][k] * b[2]) / l;
#pragma unroll
        for (int r = 0; r < 3; ++r) x[r] += w * V[r][k];
    }
    // the cell spans [c0, c0 + 1] on each axis (voxel units)
    out[0] = (float)fmin(fmax(x[0], (double)cx0), (double)cx0 + 1.0);
    out[1] = (float)fmin(fmax(x[1], (double)cy0), (double)cy0 + 1.0);
    out[2] = (float)fmin(fmax(x[2], (double)cz0), (double)cz0 + 1.0);
}

// Bound by latency at 12 to 15 waves per CU (120 VGPRs, 10.7 KB of LDS), the
// staging loads first.  The bit words replace per-voxel scans, a shared edge is
// computed once instead of by its four cells, and a cell's loop runs over its
// own edges instead of all twelve: 1.45 ms for 571 k leaves with 12.8 M cells
// (9.07 ms with those scans and per-cell edges, 3200 vector instructions a
// leaf), 0.84 TB/s of leaf data.
template <bool QEF>
__global__ __launch_bounds__(64) void k_dc_cells(uint64_t n_leaves, DcArgs a) {
    __shared__ Block B;
    const int lane = threadIdx.x;
    const int x = lane >> 3, y = lane & 7;
    const uint64_t span = xcd_span(n_leaves);
    for (uint64_t v = blockIdx.x; v < span; v += gridDim.x) {
        const uint64_t leaf = xcd_item(v);
        if (leaf >= n_leaves) continue;
        const int4 org = a.origins[leaf];
        stage_block(B, a, org, lane);
        uint32_t cells;
        {
            // the words of rows (x - 1 .. x + 2, y - 1 .. y + 2) that the row's own edges and cells meet
            const int r = ridx(x, y);
            const uint32_t w00 = B.row[r], w10 = B.row[r + HB], w01 = B.row[r + 1], w11 = B.row[r + HB + 1];
            const uint32_t wm0 = B.row[r - HB], w20 = B.row[r + 2 * HB], w0m = B.row[r - 1], w02 = B.row[r + 2];
            const uint32_t w1m = B.row[r + HB - 1], wm1 = B.row[r - HB + 1];
            // edge sweep (dual_contouring.rs:352-387): every crossing edge from a voxel of this leaf needs
            // all six gradients; bit z + 1 of g** says that voxel z of that row has its three
            const uint32_t g00 = w00 & (w00 << 1 | w00 >> 1) & (wm0 | w10) & (w0m | w01);
            const uint32_t g10 = w10 & (w10 << 1 | w10 >> 1) & (w00 | w20) & (w1m | w11);
            const uint32_t g01 = w01 & (w01 << 1 | w01 >> 1) & (wm1 | w11) & (w00 | w02);
            const uint32_t n00 = w00 >> 16, n10 = w10 >> 16, n01 = w01 >> 16, n11 = w11 >> 16;
            const uint32_t bad = (w00 & w10 & (n00 ^ n10) & ~(g00 & g10)) | (w00 & w01 & (n00 ^ n01) & ~(g00 & g01)) |
                                 (w00 & w00 >> 1 & (n00 ^ n00 >> 1) & ~(g00 & g00 >> 1));
            if (__ballot((bad & 0x1FEu) != 0) && lane == 0) atomicOr(a.fail, 1u);
            // cells with all eight corners active and mixed signs (dual_contouring.rs:176-247)
            const uint32_t all = w00 & w10 & w01 & w11, some = n00 | n10 | n01 | n11, every = n00 & n10 & n01 & n11;
            cells = ((all & all >> 1 & (some | some >> 1) & ~(every & every >> 1)) >> 1) & 0xFFu;
            const uint64_t cw = gather_word(cells, y), nw = gather_word((n00 >> 1) & 0xFFu, y);
            if (y == 0) {
                a.cell_mask[leaf * 8 + x] = cw;
                a.neg_mask[leaf * 8 + x] = nw;
            }
        }
        if (!__ballot(cells != 0)) {
            __syncthreads();
            continue;
        }
        // the crossing edges between corners 0..8, counted per row and listed (row-major, axis, z)
        uint32_t n_edges = 0;
        for (int r0 = 0; r0 < CR; r0 += 64) {
            const int r = r0 + lane, rx = r / CB, ry = r % CB;
            uint32_t e = 0;
            if (r < CR) {
                const uint32_t w = B.row[ridx(rx, ry)], wx = B.row[ridx(rx, ry) + HB], wy = B.row[ridx(rx, ry) + 1];
                const uint32_t ex = rx < 8 ? (w & wx & (w ^ wx) >> 16) >> 1 & 0x1FFu : 0;
                const uint32_t ey = ry < 8 ? (w & wy & (w ^ wy) >> 16) >> 1 & 0x1FFu : 0;
                const uint32_t ez = (w & w >> 1 & (w ^ w >> 1) >> 16) >> 1 & 0xFFu;
                e = ex | ey << 9 | ez << 18;
            }
            uint32_t total;
            uint32_t at = n_edges + wave_prefix((uint32_t)__popc(e), lane, total);
            if (r < CR) {
                B.edge_row[r] = e;
                B.edge_pre[r] = at;
            }
            for (; e && at < EDGE_LDS; e &= e - 1, ++at) B.list[at] = (uint16_t)(r << 5 | (__ffs((int)e) - 1));
            n_edges += total;
        }
        __syncthreads();
        // one lane per listed edge (past EDGE_LDS each cell computes its own)
        for (uint32_t k = lane; k < min(n_edges, (uint32_t)EDGE_LDS); k += 64) {
            const int code = B.list[k], r = code >> 5, bit = code & 31, d = bit >= 18 ? 2 : (bit >= 9 ? 1 : 0);
            B.edge[k] = edge_crossing(B, org, r / CB, r % CB, bit - 9 * d, d);
        }
        __syncthreads();
        uint32_t n_cells;
        {
            uint32_t at = wave_prefix((uint32_t)__popc(cells), lane, n_cells);
            for (uint32_t c = cells; c; c &= c - 1, ++at) B.list[at] = (uint16_t)((lane << 3) | (__ffs((int)c) - 1));
        }
        __syncthreads();
        for (uint32_t k0 = 0; k0 < n_cells; k0 += 64) {
            const uint32_t k = k0 + lane;
            const bool on = k < n_cells;
            const int cell = B.list[on ? k : 0];
            const int cx0 = cell >> 6, cy0 = (cell >> 3) & 7, cz0 = cell & 7;
            // the cell's crossing edges in EDGE_OFFSETS order, packed to the front
            uint32_t valid = 0;
#pragma unroll
            for (int e = 0; e < 12; ++e) {
                constexpr uint64_t codes = EDGE_CODES;
                const int code = (int)(codes >> (5 * e)) & 31, d = code >> 3;
                const uint32_t w = B.edge_row[(cx0 + (code & 1)) * CB + cy0 + ((code >> 1) & 1)];
                valid |= ((w >> (9 * d + cz0 + ((code >> 2) & 1))) & 1u) << e;
            }
            const int cnt = __popc(valid);
            int most = on ? cnt : 0;
#pragma unroll
            for (int s = 32; s >= 1; s >>= 1) most = max(most, __shfl_xor(most, s));
            most = __builtin_amdgcn_readfirstlane(most);
            // point and normal of the lane's edge e: from the list, or past it computed here
            auto fetch = [&](int e, float (&p)[3], float (&n)[3]) {
                const int code = (int)(EDGE_CODES >> (5 * e)) & 31, d = code >> 3;
                const int ex = cx0 + (code & 1), ey = cy0 + ((code >> 1) & 1), ez = cz0 + ((code >> 2) & 1);
                const uint32_t w = B.edge_row[ex * CB + ey];
                const uint32_t at = B.edge_pre[ex * CB + ey] + __popc(w & ((1u << (9 * d + ez)) - 1u));
                const float4 q = at < EDGE_LDS ? B.edge[at] : edge_crossing(B, org, ex, ey, ez, d);
                p[0] = d == 0 ? q.x : (float)(org.x + ex);
                p[1] = d == 1 ? q.x : (float)(org.y + ey);
                p[2] = d == 2 ? q.x : (float)(org.z + ez);
                n[0] = q.y, n[1] = q.z, n[2] = q.w;
            };
            // the first KEEP stay in registers (a smooth surface crosses 3 to 6 of a cell's edges)
            constexpr int KEEP = QEF ? 12 : 6;
            float P[KEEP][3], N[KEEP][3];
#pragma unroll
            for (int j = 0; j < KEEP; ++j) {
                P[j][0] = P[j][1] = P[j][2] = N[j][0] = N[j][1] = N[j][2] = 0.0f;
                if (j >= most || !valid) continue;
                fetch(__ffs((int)valid) - 1, P[j], N[j]);
                valid &= valid - 1;
            }
            if (!on) continue;
            float* out = a.cell_pts + (leaf * 512 + (uint64_t)k) * 3;
            if constexpr (QEF) {
                qef_point(P, N, (1u << cnt) - 1u, (float)(org.x + cx0), (float)(org.y + cy0), (float)(org.z + cz0), out);
                continue;
            } else {
                // find_feature_point (dual_contouring.rs:433-458)
                const float fc = (float)cnt;
                float cx = 0.0f, cy = 0.0f, cz = 0.0f;
#pragma unroll
                for (int j = 0; j < KEEP; ++j)
                    if (j < most && j < cnt) cx = cx + P[j][0], cy = cy + P[j][1], cz = cz + P[j][2];
                for (uint32_t rest = valid; rest; rest &= rest - 1) {
                    float p[3], n[3];
                    fetch(__ffs((int)rest) - 1, p, n);
                    cx = cx + p[0], cy = cy + p[1], cz = cz + p[2];
                }
                cx = cx / fc, cy = cy / fc, cz = cz / fc;
                for (int it = 0; it < 50; ++it) {
                    float fx = 0.0f, fy = 0.0f, fz = 0.0f;
                    auto pull = [&](const float (&p)[3], const float (&n)[3]) {
                        const float d = (n[0] * (cx - p[0]) + n[1] * (cy - p[1])) + n[2] * (cz - p[2]);
                        fx = fx + (n[0] * -1.0f) * d;
                        fy = fy + (n[1] * -1.0f) * d;
                        fz = fz + (n[2] * -1.0f) * d;
                    };
#pragma unroll
                    for (int j = 0; j < KEEP; ++j)
                        if (j < most && j < cnt) pull(P[j], N[j]);
                    for (uint32_t rest = valid; rest; rest &= rest - 1) {
                        float p[3], n[3];
                        fetch(__ffs((int)rest) - 1, p, n);
                        pull(p, n);
                    }
                    const float damping = 1.0f - (float)it / 50.0f;
                    cx = cx + (fx * damping) / fc;
                    cy = cy + (fy * damping) / fc;
                    cz = cz + (fz * damping) / fc;
                    if ((fx * fx + fy * fy) + fz * fz < 1e-6f) break;
                }
                out[0] = cx;
                out[1] = cy;
                out[2] = cz;
            }
        }
        __syncthreads();
    }
}

// Triangle3::is_degenerate (triangle3.rs:272-275) of the scaled corners
__device__ inline bool degenerate(const float a[3], const float b[3], const float c[3]) {
    const float ux = b[0] - a[0], uy = b[1] - a[1], uz = b[2] - a[2];
    const float vx = c[0] - a[0], vy = c[1] - a[1], vz = c[2] - a[2];
    const float cx = uy * vz - uz * vy, cy = uz * vx - ux * vz, cz = ux * vy - uy * vx;
    return (cx * cx + cy * cy) + cz * cz == 0.0f;
}

// dual_contouring.rs:389-408: the four cells around an edge, as offsets 0 or
// -1 on the two other axes, in three bits per cell (x, y, z; set = -1).
constexpr uint32_t cell_codes(uint32_t c0, uint32_t c1, uint32_t c2, uint32_t c3) { return c0 | c1 << 3 | c2 << 6 | c3 << 9; }
constexpr uint32_t CELLS_X = cell_codes(0, 4, 6, 2), CELLS_Y = cell_codes(0, 1, 5, 4), CELLS_Z = cell_codes(2, 3, 1, 0);

// WRITE = false: triangles per leaf into tri_count.  WRITE = true: the
// triangles at tri_off[leaf].  Everything but the points comes from the
// presence masks of the leaf and its seven neighbours towards -x, -y, -z and
// the sign masks of the leaf and its three neighbours towards +x, +y, +z
// (704 B a leaf).  A leaf's quads (crossing edges whose four cells exist, so
// whose ends are active) are listed in the sequential order (z-rows = lanes,
// then z, then axis) and taken 64 at a time, one per lane; each lane's
// triangles go after those of the quads before it (two ballots give the
// prefix), assembled in LDS and written coalesced, so the soup keeps that
// order (dual_contouring.rs:93-174, :62-79).  At 571 k leaves and 38.4 M
// triangles counting takes 0.35 ms and writing 0.73 ms (1.9 TB/s of soup; the
// scattered point fetches bound it); 5.45 and 7.18 ms when both staged the
// leaf's values again and looked each cell up in memory.
template <bool WRITE>
__global__ __launch_bounds__(64) void k_dc_triangles(uint64_t n_leaves, DcArgs a, uint32_t* __restrict__ tri_count,
                                                     const uint64_t* __restrict__ tri_off, float* __restrict__ out) {
    __shared__ int32_t slot[8];        // leaves at offsets 0 or -1 (bit 0 x, bit 1 y, bit 2 z set = -1)
    __shared__ uint64_t word[64];      // their presence words
    __shared__ uint16_t before[64];    // cells of the leaf's words before
    __shared__ uint16_t quads[512 * 3];  // lane << 5 | z << 2 | axis, sign in bit 15
    __shared__ float tri[WRITE ? 64 * 18 : 1];
    const int lane = threadIdx.x;
    const int x = lane >> 3, y = lane & 7;
    const unsigned long long lt = (1ull << lane) - 1;
    const uint64_t span = xcd_span(n_leaves);
    for (uint64_t v = blockIdx.x; v < span; v += gridDim.x) {
        const uint64_t leaf = xcd_item(v);
        if (leaf >= n_leaves) continue;
        const int4 org = a.origins[leaf];
        int32_t s = (int32_t)leaf;
        if (lane >= 1 && lane < 11) {
            const int k = lane;  // 1..7: towards -, 8..10: towards + on one axis
            const int dx = k < 8 ? -(k & 1) : k == 8, dy = k < 8 ? -((k >> 1) & 1) : k == 9,
                      dz = k < 8 ? -((k >> 2) & 1) : k == 10;
            s = a.map.find((org.x >> 3) + dx, (org.y >> 3) + dy, (org.z >> 3) + dz);
        }
        if (lane < 8) slot[lane] = s;
        const int32_t sx = __builtin_amdgcn_readlane(s, 8), sy = __builtin_amdgcn_readlane(s, 9),
                      sz = __builtin_amdgcn_readlane(s, 10);
        const int32_t sq = __shfl(s, lane >> 3);
        const uint64_t w = sq >= 0 ? a.cell_mask[(uint64_t)sq * 8 + (lane & 7)] : 0;
        const uint8_t* nb = reinterpret_cast<const uint8_t*>(a.neg_mask);  // byte y of word x is row (x, y)
        const uint32_t n0 = nb[leaf * 64 + lane];
        const int32_t lx = x < 7 ? (int32_t)leaf : sx, ly = y < 7 ? (int32_t)leaf : sy;
        const uint32_t nx = lx >= 0 ? nb[(uint64_t)lx * 64 + (((x + 1) & 7) << 3 | y)] : 0;
        const uint32_t ny = ly >= 0 ? nb[(uint64_t)ly * 64 + (x << 3 | ((y + 1) & 7))] : 0;
        const uint32_t nz = sz >= 0 ? nb[(uint64_t)sz * 64 + lane] : 0;
        word[lane] = w;
        uint32_t pre = (uint32_t)__popcll(w);
        const uint32_t own = pre;
#pragma unroll
        for (int d = 1; d < 8; d <<= 1) {
            const uint32_t u = (uint32_t)__shfl_up((int)pre, d, 64);
            if ((lane & 7) >= d) pre += u;
        }
        before[lane] = (uint16_t)(pre - own);
        __syncthreads();
        // presence bits z - 1 .. 7 of the cell rows (x, y), (x - 1, y), (x, y - 1), (x - 1, y - 1): bit z + 1
        auto cell_row = [&](int mx, int my) {
            const int cx = x - mx, cy = y - my, q = (cx < 0) | (cy < 0) << 1, wi = cx & 7, sh = (cy & 7) * 8;
            return (uint32_t)((word[q * 8 + wi] >> sh) & 0xFFu) << 1 | (uint32_t)((word[(q | 4) * 8 + wi] >> (sh + 7)) & 1u);
        };
        const uint32_t c00 = cell_row(0, 0), cm0 = cell_row(1, 0), c0m = cell_row(0, 1), cmm = cell_row(1, 1);
        const uint32_t ax = c00 & c0m, ay = c00 & cm0, az = ax & cm0 & cmm;
        const uint32_t qx = ax >> 1 & ax & (n0 ^ nx), qy = ay >> 1 & ay & (n0 ^ ny),
                       qz = az >> 1 & (n0 ^ (n0 >> 1 | (nz & 1u) << 7)) & 0xFFu;
        uint32_t n_quads;
        uint32_t at = wave_prefix((uint32_t)(__popc(qx) + __popc(qy) + __popc(qz)), lane, n_quads);
        for (uint32_t any = qx | qy | qz; any; any &= any - 1) {
            const int z = __ffs((int)any) - 1;
            const uint32_t code = (uint32_t)(lane << 5 | z << 2) | ((n0 >> z) & 1u) << 15;
            if (qx >> z & 1u) quads[at++] = (uint16_t)code;
            if (qy >> z & 1u) quads[at++] = (uint16_t)(code | 1u);
            if (qz >> z & 1u) quads[at++] = (uint16_t)(code | 2u);
        }
        __syncthreads();
        const uint64_t base = WRITE ? tri_off[leaf] : 0;
        uint32_t done = 0;
        for (uint32_t k0 = 0; k0 < n_quads; k0 += 64) {
            const uint32_t k = k0 + (uint32_t)lane;
            float q[6][3];
            bool keep[2] = {false, false};
            if (k < n_quads) {
                const uint32_t e = quads[k];
                const int el = (e >> 5) & 63, ex = el >> 3, ey = el & 7, ez = (e >> 2) & 7, d = e & 3;
                const bool s1 = e >> 15;
                const uint32_t codes = d == 0 ? CELLS_X : (d == 1 ? CELLS_Y : CELLS_Z);
                float p[4][3];
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const uint32_t m = codes >> (3 * c);
                    const int cx = ex - (int)(m & 1), cy = ey - (int)(m >> 1 & 1), cz = ez - (int)(m >> 2 & 1);
                    const int lq = (cx < 0) | (cy < 0) << 1 | (cz < 0) << 2, wi = lq * 8 + (cx & 7);
                    const int bit = (cy & 7) * 8 + (cz & 7);
                    const uint32_t rank = before[wi] + (uint32_t)__popcll(word[wi] & ((1ull << bit) - 1));
                    const float* src = a.cell_pts + ((uint64_t)(uint32_t)slot[lq] * 512 + rank) * 3;
                    p[c][0] = src[0];
                    p[c][1] = src[1];
                    p[c][2] = src[2];
                }
                // [p0, p1, p2, p2, p3, p0], with 1<->2 and 4<->5 swapped when v is negative
                const int f1 = s1 ? 2 : 1, f2 = s1 ? 1 : 2, f4 = s1 ? 0 : 3, f5 = s1 ? 3 : 0;
                const int f[6] = {0, f1, f2, 2, f4, f5};
#pragma unroll
                for (int c = 0; c < 6; ++c) {
                    const int src = f[c];
#pragma unroll
                    for (int j = 0; j < 3; ++j)
                        q[c][j] = (src == 0 ? p[0][j] : src == 1 ? p[1][j] : src == 2 ? p[2][j] : p[3][j]) * a.voxel_size;
                }
                keep[0] = !degenerate(q[0], q[1], q[2]);
                keep[1] = !degenerate(q[3], q[4], q[5]);
            }
            const unsigned long long b0 = __ballot(keep[0]), b1 = __ballot(keep[1]);
            const uint32_t n_tri = (uint32_t)(__popcll(b0) + __popcll(b1));
            if (WRITE) {
                uint32_t to = (uint32_t)(__popcll(b0 & lt) + __popcll(b1 & lt));
#pragma unroll
                for (int tr = 0; tr < 2; ++tr) {
                    if (!keep[tr]) continue;
#pragma unroll
                    for (int kk = 0; kk < 3; ++kk)
#pragma unroll
                        for (int j = 0; j < 3; ++j) tri[to * 9 + kk * 3 + j] = q[3 * tr + kk][j];
                    ++to;
                }
                __syncthreads();
                float* o = out + 9 * (base + done);
                for (uint32_t i = lane; i < 9 * n_tri; i += 64) o[i] = tri[i];
                __syncthreads();
            }
            done += n_tri;
        }
        if (!WRITE && lane == 0) tri_count[leaf] = done;
        __syncthreads();
    }
}

__global__ void k_fill_u32(uint32_t* __restrict__ p, uint64_t n, uint32_t v) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
        p[i] = v;
}

// Fills n 32-bit words with a kernel (not hipMemsetAsync, so that the call
// stays valid inside a caller's graph capture).
void fill_u32(hipStream_t st, void* p, uint64_t n, uint32_t v) {
    k_fill_u32<<<(unsigned)std::min<uint64_t>(div_up(n, 256), 2048), 256, 0, st>>>(static_cast<uint32_t*>(p), n, v);
    BS_HIP(hipGetLastError());
}

// Device buffers of one dual-contouring call.  The usual entry point takes
// them from the context's scratch arena; bs_dual_contour_into from the
// per-device static workspace below.
struct DcWork {
    LeafMap map;
    uint32_t* fail;
    float* cell_pts;
    uint64_t* cell_mask;
    uint64_t* neg_mask;
    uint32_t* tri_count;
    uint64_t* tri_off;
    void* scan_tmp;
    size_t scan_bytes;
};

uint64_t hash_capacity(uint64_t n) {
    uint64_t cap = 1024;
    while (cap < 2 * n) cap <<= 1;
    return cap;
}

// Everything up to the triangle count: leaf map, cell points, per-leaf
// triangle counts and their scan.  Returns the soup's triangle count.
uint64_t dc_count(hipStream_t st, const bs_volume* vol, float voxel_size, bool qef, DcWork& w, DcArgs& a) {
    const uint64_t n = vol->n_leaves;
    if (w.map.dense) {
        fill_u32(st, w.map.cells, (uint64_t)w.map.nx * w.map.ny * w.map.nz, 0xFFFFFFFFu);
    } else {
        const uint64_t cap = (uint64_t)w.map.cap_mask + 1;
        fill_u32(st, w.map.keys, 2 * cap, 0xFFFFFFFFu);
        fill_u32(st, w.map.cells, cap, 0xFFFFFFFFu);
    }
    fill_u32(st, w.fail, 1, 0);
    k_leafmap_insert<<<div_up(n, 256), 256, 0, st>>>(n, reinterpret_cast<const int4*>(vol->origins), w.map, w.fail);
    BS_HIP(hipGetLastError());

    a = DcArgs{};
    a.map = w.map;
    a.origins = reinterpret_cast<const int4*>(vol->origins);
    a.masks = vol->masks;
    a.values = vol->values;
    a.cell_pts = w.cell_pts;
    a.cell_mask = w.cell_mask;
    a.neg_mask = w.neg_mask;
    a.voxel_size = voxel_size;
    a.fail = w.fail;
    const unsigned grid = xcd_grid(n);
    if (qef)
        k_dc_cells<true><<<grid, 64, 0, st>>>(n, a);
    else
        k_dc_cells<false><<<grid, 64, 0, st>>>(n, a);
    BS_HIP(hipGetLastError());
    k_dc_triangles<false><<<grid, 64, 0, st>>>(n, a, w.tri_count, nullptr, nullptr);
    BS_HIP(hipGetLastError());
    size_t bytes = w.scan_bytes;
    BS_HIP(hipcub::DeviceScan::ExclusiveSum(w.scan_tmp, bytes, w.tri_count, w.tri_off, (int)n, st));
    uint32_t h_fail = 0, last_cnt = 0;
    uint64_t last_off = 0;
    BS_HIP(hipMemcpyAsync(&h_fail, w.fail, sizeof(uint32_t), hipMemcpyDeviceToHost, st));
    BS_HIP(hipMemcpyAsync(&last_cnt, w.tri_count + n - 1, sizeof(uint32_t), hipMemcpyDeviceToHost, st));
    BS_HIP(hipMemcpyAsync(&last_off, w.tri_off + n - 1, sizeof(uint64_t), hipMemcpyDeviceToHost, st));
    BS_HIP(hipStreamSynchronize(st));
    BS_REQUIRE(!(h_fail & 1u), BS_ERR_INTERNAL,
               "dual contouring: a crossing voxel has no neighbour along an axis; the reference reaches "
               "unreachable!() (dual_contouring.rs:347)");
    return last_off + last_cnt;
}

void dc_write(hipStream_t st, uint64_t n, const DcArgs& a, const DcWork& w, float* out) {
    const unsigned grid = xcd_grid(n);
    k_dc_triangles<true><<<grid, 64, 0, st>>>(n, a, nullptr, w.tri_off, out);
    BS_HIP(hipGetLastError());
}

void check_meshable(bs_ctx* ctx, const bs_volume* vol) {
    BS_REQUIRE(vol->device == ctx->device, BS_ERR_INVALID_ARG, "volume lives on another device");
    // visit_leafs_par meets every active tile: todo!() (dual_contouring.rs:146,181,354)
    BS_REQUIRE(vol->tiles.empty(), BS_ERR_UNSUPPORTED_TILE,
               "dual contouring of a volume with active tiles: the reference stops at todo!()");
}

// ---------------------------------------------------------------- workspace of bs_dual_contour_into
// bs_dual_contour_into allocates nothing: its buffers live in this array,
// which each device holds from the library's load until the process ends.
// Sized for DC_NOALLOC_MAX_LEAVES leaves with the hash leaf map.
constexpr uint64_t DC_NOALLOC_MAX_LEAVES = BS_DC_INTO_MAX_LEAVES;
constexpr uint64_t DC_NOALLOC_HASH_CAP = 2 * DC_NOALLOC_MAX_LEAVES;  // power of two >= 1024
constexpr uint64_t DC_NOALLOC_SCAN_BYTES = 1ull << 20;
constexpr uint64_t al256(uint64_t b) { return (b + 255) & ~255ull; }
constexpr uint64_t NA_KEYS = 0;
constexpr uint64_t NA_CELLS = NA_KEYS + al256(8 * DC_NOALLOC_HASH_CAP);
constexpr uint64_t NA_FAIL = NA_CELLS + al256(4 * DC_NOALLOC_HASH_CAP);
constexpr uint64_t NA_PTS = NA_FAIL + 256;
constexpr uint64_t NA_CMASK = NA_PTS + al256(4ull * 512 * 3 * DC_NOALLOC_MAX_LEAVES);
constexpr uint64_t NA_NMASK = NA_CMASK + al256(64ull * DC_NOALLOC_MAX_LEAVES);
constexpr uint64_t NA_TCNT = NA_NMASK + al256(64ull * DC_NOALLOC_MAX_LEAVES);
constexpr uint64_t NA_TOFF = NA_TCNT + al256(4ull * DC_NOALLOC_MAX_LEAVES);
constexpr uint64_t NA_SCAN = NA_TOFF + al256(8ull * (DC_NOALLOC_MAX_LEAVES + 1));
constexpr uint64_t NA_BYTES = NA_SCAN + DC_NOALLOC_SCAN_BYTES;
static_assert(DC_NOALLOC_HASH_CAP >= 1024 && (DC_NOALLOC_HASH_CAP & (DC_NOALLOC_HASH_CAP - 1)) == 0, "hash capacity");

}  // namespace

// The array itself.  In host code this name is a stand-in, not a device
// address: host code uses the address hipGetSymbolAddress returned for the
// device (dc_noalloc_ptr), never the name.
static __device__ __align__(256) unsigned char scratch[NA_BYTES];

namespace {
constexpr int NA_MAX_DEVICES = 64;
std::mutex g_na_mutex;
unsigned char* g_na_ptr[NA_MAX_DEVICES] = {};
}  // namespace

// Looks up this device's copy of the workspace once, with `device` current.
// Called by bs_ctx_create, so the entry point itself needs no set-up call.
void dc_noalloc_init(int device) {
    BS_REQUIRE(device >= 0 && device < NA_MAX_DEVICES, BS_ERR_INVALID_ARG, "device ordinal out of range");
    std::lock_guard<std::mutex> lock(g_na_mutex);
    if (g_na_ptr[device]) return;
    void* p = nullptr;
    BS_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    BS_REQUIRE(p != nullptr, BS_ERR_HIP, "hipGetSymbolAddress returned no address for the DC workspace");
    g_na_ptr[device] = static_cast<unsigned char*>(p);
}

static unsigned char* dc_noalloc_ptr(int device) {
    std::lock_guard<std::mutex> lock(g_na_mutex);
    BS_REQUIRE(device >= 0 && device < NA_MAX_DEVICES && g_na_ptr[device], BS_ERR_INTERNAL,
               "the DC workspace of this device was not set up (bs_ctx_create does it)");
    return g_na_ptr[device];
}

// DualContouringMesher::default().with_voxel_size(h).mesh(volume): the
// triangle soup (n_tris * 9 floats) in device memory owned by the caller
// (free_block), or nullptr for no triangle.
void dual_contour_device(bs_ctx* ctx, bs_volume* vol, float voxel_size, float** out_dev, uint64_t* n_tris,
                         bs_dc_stats* stats) {
    hipStream_t st = ctx->stream;
    *out_dev = nullptr;
    *n_tris = 0;
    check_meshable(ctx, vol);
    const uint64_t n = vol->n_leaves;
    if (stats) *stats = bs_dc_stats{};
    if (!n) return;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    if (stats) {
        BS_HIP(hipEventCreate(&e0));
        BS_HIP(hipEventCreate(&e1));
        BS_HIP(hipEventRecord(e0, st));
    }

    // leaf map over the leaves' box (one leaf of margin for the halo lookups)
    int32_t lo[3], hi[3];
    leaf_box(ctx, vol->origins, n, lo, hi);
    DcWork w{};
    uint64_t cells = 1;
    for (int k = 0; k < 3; ++k) cells *= (uint64_t)(hi[k] - lo[k] + 1);
    w.map.dense = !(ctx->paths & BS_PATH_FORCE_HASH) && cells <= (1ull << 28);
    if (w.map.dense) {
        w.map.x0 = lo[0], w.map.y0 = lo[1], w.map.z0 = lo[2];
        w.map.nx = hi[0] - lo[0] + 1, w.map.ny = hi[1] - lo[1] + 1, w.map.nz = hi[2] - lo[2] + 1;
        w.map.cells = ctx->scratch.as<int32_t>(S_DC_MAP, cells);
    } else {
        const uint64_t cap = hash_capacity(n);
        w.map.cap_mask = (uint32_t)(cap - 1);
        w.map.keys = ctx->scratch.as<uint64_t>(S_DC_KEYS, cap);
        w.map.cells = ctx->scratch.as<int32_t>(S_DC_MAP, cap);
    }
    w.fail = ctx->scratch.as<uint32_t>(S_DC_FAIL, 1);
    w.cell_pts = ctx->scratch.as<float>(S_DC_CELLS, n * 512 * 3);
    w.cell_mask = ctx->scratch.as<uint64_t>(S_DC_CELLMASK, n * 8);
    w.neg_mask = ctx->scratch.as<uint64_t>(S_DC_NEGMASK, n * 8);
    w.tri_count = ctx->scratch.as<uint32_t>(S_DC_TRICNT, n);
    w.tri_off = ctx->scratch.as<uint64_t>(S_DC_TRIOFF, n + 1);
    BS_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, w.scan_bytes, w.tri_count, w.tri_off, (int)n, st));
    w.scan_tmp = ctx->scratch.get(S_CUB, w.scan_bytes);

    DcArgs a{};
    const uint64_t total = dc_count(st, vol, voxel_size, ctx->dc_vertex == BS_DC_VERTEX_QEF_F64, w, a);
    if (total) {
        float* out = static_cast<float*>(alloc_block(sizeof(float) * 9 * total));
        try {
            dc_write(st, n, a, w, out);
            BS_HIP(hipStreamSynchronize(st));
        } catch (...) {
            free_block(out);
            throw;
        }
        *out_dev = out;
    }
    *n_tris = total;
    if (stats) {
        BS_HIP(hipEventRecord(e1, st));
        BS_HIP(hipEventSynchronize(e1));
        float ms = 0.0f;
        BS_HIP(hipEventElapsedTime(&ms, e0, e1));
        stats->ms_total = ms;
        stats->n_leaves = n;
        stats->n_tris = total;
        stats->used_hash = !w.map.dense;
        (void)hipEventDestroy(e0);
        (void)hipEventDestroy(e1);
    }
}

// bs_dual_contour_into: the same soup written to the caller's device buffer
// of capacity_tris triangles, with every intermediate buffer in this
// device's static workspace and no device or host allocation.  *n_tris is
// the soup's triangle count; a soup larger than the capacity writes nothing
// and reports BS_ERR_CAPACITY.  Calls that overlap on one device race on the
// shared workspace.
void dual_contour_into(bs_ctx* ctx, const bs_volume* vol, float voxel_size, float* out_dev, uint64_t capacity_tris,
                       uint64_t* n_tris) {
    hipStream_t st = ctx->stream;
    *n_tris = 0;
    check_meshable(ctx, vol);
    const uint64_t n = vol->n_leaves;
    BS_REQUIRE(n <= DC_NOALLOC_MAX_LEAVES, BS_ERR_CAPACITY,
               "bs_dual_contour_into: the volume has more leaves than the workspace holds (" +
                   std::to_string(n) + " > " + std::to_string(DC_NOALLOC_MAX_LEAVES) + ")");
    if (!n) return;
    unsigned char* base = dc_noalloc_ptr(ctx->device);
    DcWork w{};
    const uint64_t cap = hash_capacity(n);
    w.map.dense = 0;
    w.map.cap_mask = (uint32_t)(cap - 1);
    w.map.keys = reinterpret_cast<uint64_t*>(base + NA_KEYS);
    w.map.cells = reinterpret_cast<int32_t*>(base + NA_CELLS);
    w.fail = reinterpret_cast<uint32_t*>(base + NA_FAIL);
    w.cell_pts = reinterpret_cast<float*>(base + NA_PTS);
    w.cell_mask = reinterpret_cast<uint64_t*>(base + NA_CMASK);
    w.neg_mask = reinterpret_cast<uint64_t*>(base + NA_NMASK);
    w.tri_count = reinterpret_cast<uint32_t*>(base + NA_TCNT);
    w.tri_off = reinterpret_cast<uint64_t*>(base + NA_TOFF);
    w.scan_tmp = base + NA_SCAN;
    size_t need = 0;
    BS_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, need, w.tri_count, w.tri_off, (int)n, st));
    BS_REQUIRE(need <= DC_NOALLOC_SCAN_BYTES, BS_ERR_INTERNAL, "scan workspace too small");
    w.scan_bytes = need;

    DcArgs a{};
    const uint64_t total = dc_count(st, vol, voxel_size, ctx->dc_vertex == BS_DC_VERTEX_QEF_F64, w, a);
    *n_tris = total;
    BS_REQUIRE(total <= capacity_tris, BS_ERR_CAPACITY,
               "bs_dual_contour_into: the soup has " + std::to_string(total) +
                   " triangles, more than the output capacity of " + std::to_string(capacity_tris));
    if (total) {
        BS_REQUIRE(out_dev != nullptr, BS_ERR_INVALID_ARG, "null output buffer");
        dc_write(st, n, a, w, out_dev);
        BS_HIP(hipStreamSynchronize(st));
    }
}

}  // namespace bs
