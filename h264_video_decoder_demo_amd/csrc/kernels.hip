// kernels.hip -- gfx950 kernels of the H.264 picture-reconstruction engine.
//
// One wavefront (64 lanes) reconstructs one macroblock.  Three stages per picture,
// in the reference's order (inter MBs never read the current picture, intra MBs read
// unfiltered neighbours, deblocking runs after the whole picture is built,
// H264PictureBase.cpp:707):
//   inter   -- fully parallel over inter (and I_PCM) MBs: fractional-sample MC from
//              the device-resident DPB + weighted prediction + residual.
//              The same launch derives the boundary strengths of deblocking.
//   intra   -- bands of MB rows, a wave per row and plane type, walking its intra MBs
//              behind the row above.
//   deblock -- bands likewise, over all MBs, with the raster-order edge filter.
// Before them a staging kernel, a lane per MB, checks a picture's records and expands them.
// The per-MB wavefront and row schedules (queues ordered by t = x + 2y, progress words in
// device memory) are alternatives.  A launch holds the pictures of any number of streams.
#include <hip/hip_runtime.h>

#include <mutex>

#include "h264g_dev.h"

// Device memory seen through global-address-space pointers: loads and stores through
// them are global_* instructions, which count on the vector-memory counter only.  Through
// generic pointers they would be flat_* instructions, which also count on the LDS counter,
// so every LDS wait would wait for them too (a prefetch from HBM would stall the next LDS
// access).
// (The host pass of this file parses the device code too; it sees plain pointers.)
#if defined(__HIP_DEVICE_COMPILE__)
#define GAS __attribute__((address_space(1)))
#else
#define GAS
#endif
typedef GAS uint8_t gu8;
template <typename T>
__device__ __forceinline__ GAS T *G(T *p) { return (GAS T *)p; }
template <typename T>
__device__ __forceinline__ const GAS T *G(const T *p) { return (const GAS T *)p; }


namespace {

constexpr int WAVE = 64;

// ------------------------------------------------------------------ tables
// Table 8-13 / 8-14 zig-zag (scan position -> raster index), H264PictureBase.cpp:4542-4744
// (constexpr so that fully unrolled loops index register arrays with constants)
__device__ constexpr uint8_t c_zz4[16] = {0, 1, 4, 8, 5, 2, 3, 6, 9, 12, 13, 10, 7, 11, 14, 15};
// the field scan of Table 8-13 (field MBs of MBAFF frames)
__device__ constexpr uint8_t c_fld4[16] = {0, 4, 1, 8, 12, 5, 9, 13, 2, 6, 10, 14, 3, 7, 11, 15};
__constant__ uint8_t c_zz8[64] = {
    0, 1, 8, 16, 9, 2, 3, 10, 17, 24, 32, 25, 18, 11, 4, 5, 12, 19, 26, 33, 40, 48, 41, 34, 27, 20, 13, 6, 7, 14, 21, 28,
    35, 42, 49, 56, 57, 50, 43, 36, 29, 22, 15, 23, 30, 37, 44, 51, 58, 59, 52, 45, 38, 31, 39, 46, 53, 60, 61, 54, 47, 55, 62, 63};
// raster position -> 8x8 zig-zag scan index (inverse of c_zz8)
__constant__ uint8_t c_izz8[64] = {
    0, 1, 5, 6, 14, 15, 27, 28, 2, 4, 7, 13, 16, 26, 29, 42, 3, 8, 12, 17, 25, 30, 41, 43, 9, 11, 18, 24, 31, 40, 44, 53,
    10, 19, 23, 32, 39, 45, 52, 54, 20, 22, 33, 38, 46, 51, 55, 60, 21, 34, 37, 47, 50, 56, 59, 61, 35, 36, 48, 49, 57, 58, 62, 63};
// raster position -> 8x8 field scan index (inverse of Table 8-14's field scan)
__constant__ uint8_t c_ifld8[64] = {
    0, 3, 8, 15, 22, 30, 38, 52, 1, 4, 14, 21, 29, 37, 45, 53, 2, 7, 16, 23, 31, 39, 46, 58, 5, 9, 20, 28, 36, 44, 51, 59,
    6, 13, 24, 32, 40, 47, 54, 60, 10, 17, 25, 33, 41, 48, 55, 61, 11, 18, 26, 34, 42, 49, 56, 62, 12, 19, 27, 35, 43, 50, 57, 63};
// normAdjust values v (8-315, 8-318), H264PictureBase.cpp:4900-4950
__constant__ uint8_t c_v4[6][3] = {{10, 16, 13}, {11, 18, 14}, {13, 20, 16}, {14, 23, 18}, {16, 25, 20}, {18, 29, 23}};
__constant__ uint8_t c_v8[6][6] = {{20, 18, 32, 19, 25, 24}, {22, 19, 35, 21, 28, 26}, {26, 23, 42, 24, 33, 31},
                                   {28, 25, 45, 26, 35, 33}, {32, 28, 51, 30, 40, 38}, {36, 32, 58, 34, 46, 43}};
// Tables 8-16 / 8-17, Deblock.cpp:1330-1409
__constant__ uint8_t c_alpha[52] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 4, 4, 5, 6, 7, 8, 9, 10, 12, 13,
                                    15, 17, 20, 22, 25, 28, 32, 36, 40, 45, 50, 56, 63, 71, 80, 90, 101, 113, 127, 144, 162, 182, 203, 226, 255, 255};
__constant__ uint8_t c_beta[52] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 2, 2, 2, 3, 3, 3, 3, 4, 4, 4,
                                   6, 6, 7, 7, 8, 8, 9, 9, 10, 10, 11, 11, 12, 12, 13, 13, 14, 14, 15, 15, 16, 16, 17, 17, 18, 18};
__constant__ uint8_t c_tc0[3][52] = {
    {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 2, 2, 2, 2, 3, 3, 3, 4, 4, 4, 5, 6, 6, 7, 8, 9, 10, 11, 13},
    {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 2, 2, 2, 2, 3, 3, 3, 4, 4, 5, 5, 6, 7, 8, 8, 10, 11, 12, 13, 15, 17},
    {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 2, 2, 2, 2, 3, 3, 3, 4, 4, 4, 5, 6, 6, 7, 8, 9, 10, 11, 13, 14, 16, 18, 20, 23, 25}};

__device__ __forceinline__ int clip3(int lo, int hi, int v) { return v < lo ? lo : (v > hi ? hi : v); }
__device__ __forceinline__ int clip1(int v) { return clip3(0, 255, v); }
__device__ __forceinline__ int iabs(int v) { return v < 0 ? -v : v; }

__device__ __forceinline__ int ls4(int m, int i, int j) {
    int cls = ((i | j) & 1) == 0 ? 0 : (((i & j) & 1) ? 1 : 2);
    return 16 * c_v4[m][cls];
}

// luma4x4BlkIdx -> (x, y) in the MB (6.4.3)
__device__ __forceinline__ int blk_x(int b) { return ((b >> 2) & 1) * 8 + (b & 1) * 4; }
__device__ __forceinline__ int blk_y(int b) { return ((b >> 3) & 1) * 8 + ((b >> 1) & 1) * 4; }

__device__ __forceinline__ int wave_lane() { return threadIdx.x & (WAVE - 1); }

// Orders the LDS accesses of the lanes of one wave (LDS instructions of a wave execute in
// order; the fences keep the compiler from moving memory operations across).  Every
// LDS working set below belongs to one wave, so this is the only barrier the per-MB code
// needs, also when several waves share a workgroup.
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// ------------------------------------------------------------ residuals
// LDS scratch of one wave: the MB's levels as they arrive -- per slot (0 = Intra16x16
// DC, 1 + luma4x4BlkIdx (8x8 block q = slots 1+4q..4+4q), 17/18 = chroma DC Cb/Cr,
// 19 + 4c + b = chroma AC) its 16-bit mask of non-zero scan positions and the index of
// its first value, and the values in stream order -- then the residual planes.
// Luma interpolation of one list (inter MBs, after the residual is built).  Window row rr
// of 4x4 block b holds reference row y0 - 2 + rr at columns x0 - 2 .. x0 + 5, where
// (x0, y0) is the block's integer sample position; b1 is the unrounded horizontal 6-tap
// value between columns x0 + i and x0 + i + 1 (8-241).
struct WaveMc {
    uint32_t raw[16][9][2];   // window columns 0..7, packed bytes
    uint32_t hb[16][5];       // b = Clip1((b1 + 16) >> 5), i = 0..3, of window rows 2..6
    int16_t b1t[16][4][10];   // b1 of column i, window rows 0..8 (+ one pad row): [b][i][rr]
};

struct alignas(16) WaveRes {
    union {
        struct {
            uint32_t sm[28];          // slot: mask (bits 0..15) | index of its first value << 16
            int16_t vals[7 * WAVE];   // level values in stream order (at most 27 * 16)
            int32_t dense[4][64];     // the 8x8 blocks dequantised, raster order, or [0] = the
                                      // Intra16x16 DC block in scan order
            int32_t cdc[2][4];        // scan-order levels: chroma DC
            int32_t t8[4][64];        // 8x8 transform: rows after the horizontal pass
        };
        WaveMc mc;                    // live only after the residual planes are built
    };
    int16_t rl[256];      // luma residual, raster 16x16
    int16_t rc[2][64];    // chroma residual, raster 8x8
};

// Slot (see WaveRes) of the MB's i-th level mask, in the order of the level stream: the
// Intra16x16 DC block, the four 4x4 blocks (or 16-level chunks of the 8x8 block) of each
// 8x8 quadrant whose cbp bit is set, the chroma DC blocks, the chroma AC blocks; -1 past
// the end.
__device__ __forceinline__ int level_slot(int i, int i16, int cbp) {
    if (i16) {
        if (i == 0) return 0;
        i--;
    }
    const int lm = cbp & 15, nl = 4 * __popc(lm);
    if (i < nl) {
        int c = i >> 2, q = 0;  // q: the (i >> 2)-th set bit of lm
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const int set = (lm >> t) & 1;
            if (set && c == 0) q = t;
            c -= set;
        }
        return 1 + 4 * q + (i & 3);
    }
    i -= nl;
    const int cc = cbp >> 4;
    if (cc >= 1) {
        if (i < 2) return 17 + i;
        i -= 2;
    }
    if (cc == 2 && i < 8) return 19 + i;
    return -1;
}

// Scan positions of the samples (r, 0..3) of a 4x4 block, 4 bits each: the inverse of c_zz4
// (IZZ4) and of c_fld4 (IFLD4).
constexpr uint64_t iscan4_table(const uint8_t (&scan)[16]) {
    uint64_t v = 0;
    for (int k = 0; k < 16; k++) v |= (uint64_t)k << (4 * scan[k]);
    return v;
}
constexpr uint64_t IZZ4 = iscan4_table(c_zz4);
constexpr uint64_t IFLD4 = iscan4_table(c_fld4);

// The value of the lane's neighbour in its quad, lane ^ 1 / lane ^ 2.
__device__ __forceinline__ int dpp_xor1(int v) { return __builtin_amdgcn_mov_dpp(v, 0xB1, 0xF, 0xF, true); }  // [1,0,3,2]
__device__ __forceinline__ int dpp_xor2(int v) { return __builtin_amdgcn_mov_dpp(v, 0x4E, 0xF, 0xF, true); }  // [2,3,0,1]

// 4x4 byte transpose over the four lanes of a quad: lane j holds row j of a block of bytes
// (byte c = column c) and gets column j (byte r = row r).  Two exchange stages, each a DPP
// quad permutation and one byte permute with a lane-dependent selector; applied twice it
// gives the rows back.
__device__ __forceinline__ uint32_t quad_transpose_bytes(uint32_t v, int j) {
    // even j: (own c0, partner c0, own c2, partner c2); odd j: (partner c1, own c1, partner c3, own c3)
    const uint32_t x = (uint32_t)dpp_xor1((int)v);
    const uint32_t t = __builtin_amdgcn_perm(x, v, (j & 1) ? 0x03070105u : 0x06020400u);
    // j < 2: own low half, then the low half of lane j + 2; j >= 2: the high half of lane j - 2, then own
    const uint32_t y = (uint32_t)dpp_xor2((int)t);
    return __builtin_amdgcn_perm(y, t, (j & 2) ? 0x03020706u : 0x05040100u);
}

// Level at scan position k (< 16) of the block with slot entry e: 0 unless mask bit k is
// set, else the value at the block's first index plus the number of mask bits below k.
__device__ __forceinline__ int32_t level_at(uint32_t e, const int16_t *vals, int k) {
    const uint32_t below = __popc(e & ((1u << k) - 1u));
    return ((e >> k) & 1u) ? (int32_t)vals[(e >> 16) + below] : 0;
}

// 8.5.12 for row r of a 4x4 block on the quad that holds the block (lane r of the quad):
// dequantise the row's levels (slot entry e), horizontal pass, vertical pass; returns row
// quad_row(r) of the residual, four 16-bit values.  dc_pass: sample (0, 0) is
// `dc` as it stands (Intra16x16 and chroma DC).  field: the levels follow the field scan
// (field MBs, H264PictureBase.cpp:3419).
__device__ __forceinline__ int quad_row(int r) { return (0x2130 >> (4 * r)) & 3; }
template <bool SCALED = false>
__device__ __forceinline__ uint2 residual4x4_quad(uint32_t se, const int16_t *vals, int qp, bool dc_pass, int dc, int r,
                                                 bool field, const GAS uint16_t *lsm = nullptr) {
    const int m = qp % 6, e = qp / 6;
    // LevelScale4x4 of row r: with flat lists 16 v0 at (even, even), 16 v1 at (odd, odd),
    // 16 v2 elsewhere; with scaling matrices (SCALED) lsm holds LevelScale4x4(qP % 6, i, j),
    // raster
    int ls[4];
    if (SCALED) {
        const uint2 t = *(const GAS uint2 *)(lsm + 4 * r);
        ls[0] = (int)(t.x & 0xFFFFu); ls[1] = (int)(t.x >> 16); ls[2] = (int)(t.y & 0xFFFFu); ls[3] = (int)(t.y >> 16);
    } else {
        const int s0 = 16 * c_v4[m][0], s1 = 16 * c_v4[m][1], s2 = 16 * c_v4[m][2];
        ls[0] = ls[2] = (r & 1) ? s2 : s0;
        ls[1] = ls[3] = (r & 1) ? s1 : s2;
    }
    // 8-336 / 8-337 as one expression: qP / 6 >= 4 shifts left, else rounds and shifts right
    const int lsh = e >= 4 ? e - 4 : 0, rsh = e >= 4 ? 0 : 4 - e, rnd = e >= 4 ? 0 : 1 << (3 - e);
    const uint32_t iz = (uint32_t)((field ? IFLD4 : IZZ4) >> (16 * r)) & 0xFFFFu;
    int32_t d[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int32_t v = level_at(se, vals, (int)((iz >> (4 * j)) & 15u));
        d[j] = (int32_t)(((uint32_t)(v * ls[j]) << lsh) + (uint32_t)rnd) >> rsh;
    }
    if (dc_pass && r == 0) d[0] = dc;
    int32_t f[4];
    {
        const int32_t e0 = d[0] + d[2], e1 = d[0] - d[2], e2 = (d[1] >> 1) - d[3], e3 = d[1] + (d[3] >> 1);
        f[0] = e0 + e3; f[1] = e1 + e2; f[2] = e1 - e2; f[3] = e0 - e3;
    }
    // Vertical pass across the quad, for every column: with f_r lane r's value, lanes 0..3 first
    // hold f0 + f2, f1 + (f3 >> 1), f0 - f2 - 1, (f1 >> 1) - f3 - 1 (x ^ -1 is -x - 1), then, from
    // their neighbours', rows 0, 3, 1 and 2 but for constants that join the rounding's 32.  Half the
    // instructions of a 4x4 transpose and a pass in each lane, and a lane's results lie together.
    const uint32_t neg1 = (r & 1) ? ~0u : 0u, neg2 = (r & 2) ? ~0u : 0u, add = r == 0 ? 32u : r == 2 ? 34u : 33u;
    uint32_t o[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const uint32_t t = ((uint32_t)f[j] ^ neg2) + (uint32_t)(dpp_xor2(f[j]) >> (r & 1));
        o[j] = (uint32_t)((int32_t)((t ^ neg1) + (uint32_t)dpp_xor1((int)t) + add) >> 6);
    }
    return make_uint2(__builtin_amdgcn_perm(o[1], o[0], 0x05040100u), __builtin_amdgcn_perm(o[3], o[2], 0x05040100u));
}

__device__ __forceinline__ void idct8(int32_t *v, int s) {  // 8.5.13.2, in place, stride s
    int32_t d0 = v[0], d1 = v[s], d2 = v[2 * s], d3 = v[3 * s], d4 = v[4 * s], d5 = v[5 * s], d6 = v[6 * s], d7 = v[7 * s];
    int32_t e0 = d0 + d4, e1 = -d3 + d5 - d7 - (d7 >> 1), e2 = d0 - d4, e3 = d1 + d7 - d3 - (d3 >> 1);
    int32_t e4 = (d2 >> 1) - d6, e5 = -d1 + d7 + d5 + (d5 >> 1), e6 = d2 + (d6 >> 1), e7 = d3 + d5 + d1 + (d1 >> 1);
    int32_t f0 = e0 + e6, f1 = e1 + (e7 >> 2), f2 = e2 + e4, f3 = e3 + (e5 >> 2);
    int32_t f4 = e2 - e4, f5 = (e3 >> 2) - e5, f6 = e0 - e6, f7 = e7 - (e1 >> 2);
    v[0] = f0 + f7; v[s] = f2 + f5; v[2 * s] = f4 + f3; v[3 * s] = f6 + f1;
    v[4 * s] = f6 - f1; v[5 * s] = f4 - f3; v[6 * s] = f2 - f5; v[7 * s] = f0 - f7;
}

// Places the MB's levels in LDS and computes all residual blocks into ws->rl / ws->rc.  Must be called by the whole wave.  Returns false when the MB has no levels.
// Bound: vector instructions (the kernel's time follows their number).  The vertical pass of a 4x4
// block across its quad, 8x8 blocks dequantised where a lane has one scale, values two per lane
// and residuals added in pairs: three 1920x1088 B pictures 58.6 to 56.1 us, the 64-stream pass
// 24.0 to 23.3 ms.
// Field MBs of MBAFF frames take the field scans.  lstab: the picture's LevelScale tables
// when it has scaling matrices (DevPic::ls), else null (flat lists).
template <bool MBAFF, bool SCALED>
__device__ __forceinline__ bool build_residual(const h264g_mb *mb, const DevAux &ax, const int16_t *levels, WaveRes *ws,
                                               const GAS uint16_t *lstab) {
    const int lane = wave_lane();
    if (!(ax.kind & AUX_RESID)) return false;
    const bool field = MBAFF && (mb->flags & H264G_MBF_FIELD) != 0;
    const int cbp = mb->cbp;
    const int i16 = mb->mb_type == H264G_MB_I16x16;
    const int t8 = (ax.kind & AUX_T8) ? 1 : 0;
    const int qp = (int)__builtin_amdgcn_readfirstlane((uint32_t)mb->qp_y);
    // the MB's luma lists (intra or inter), which serve its chroma blocks too (quirk Q13)
    const bool inter = !(ax.kind & AUX_INTRA);
    const GAS uint16_t *ls4t = SCALED ? lstab + (inter ? LS4_LIST : 0) : nullptr;
    const GAS uint16_t *ls8t = SCALED ? lstab + LS8_AT + (inter ? LS8_LIST : 0) : nullptr;
    const int16_t *lv = levels + mb->level_offset;
    // <= 27 masks of 16 bits, so at most 432 values; staging counted them, so the masks
    // and the values load together (coalesced, all in flight at once), two values per lane and
    // only as many rounds as the MB has values for (mostly two of the four)
    const int nmask = ax.nmask, total = (int)__builtin_amdgcn_readfirstlane(ax.ires >> AUX_NVALS_SHIFT);
    const int mask = lane < nmask ? (uint16_t)lv[lane] : 0;
    typedef uint32_t __attribute__((aligned(2), may_alias)) u32_a2;
    uint32_t v[4];
#pragma unroll
    for (int t = 0; t < 4; t++) {
        const int k = 2 * (lane + t * WAVE);
        if (2 * t * WAVE < total) v[t] = *(const GAS u32_a2 *)(lv + nmask + min(k, total - 1));
    }
    const int cnt = __popc(mask);
    // exclusive prefix sum of cnt (0..16) over the lanes, bit plane by bit plane (ballot +
    // mbcnt, no cross-lane shuffles)
    int pre = 0;
#pragma unroll
    for (int bit = 0; bit < 5; bit++) {
        const uint64_t bl = __builtin_amdgcn_ballot_w64((cnt >> bit) & 1);
        pre += (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(bl >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)bl, 0u)) << bit;
    }
    // slot entries (absent slots 0; the wave's LDS writes land in program order) and values
    if (lane < 28) ws->sm[lane] = 0u;
    if (lane < nmask) ws->sm[level_slot(lane, i16, cbp)] = (uint32_t)mask | (uint32_t)pre << 16;
#pragma unroll
    for (int t = 0; t < 4; t++)
        if (2 * t * WAVE < total && lane + t * WAVE < 7 * WAVE / 2) ((uint32_t *)ws->vals)[lane + t * WAVE] = v[t];
    wave_sync();
    // dense levels where a pass reads positions of other rows: the 8x8 blocks, the
    // Intra16x16 DC block (lanes 0..15) and the chroma DC blocks (lanes 56..63)
    if (t8) {  // lane = raster position in the 8x8 blocks, p its scan position
        const int p = field ? c_ifld8[lane] : c_izz8[lane];
        // 8.5.13.1: dequantised here, where every lane has one position and so one LevelScale8x8:
        // that of its class among the six of 8-318, by row and column mod 4, or the matrix's
        const int m = qp % 6, e = qp / 6;
        int ls;
        if (SCALED) {
            ls = ls8t[64 * m + lane];
        } else {
            const uint32_t cls = (uint32_t)(0x1513525415133430ull >> (16 * ((lane >> 3) & 3) + 4 * (lane & 3))) & 15u;
            const uint32_t lo = (uint32_t)c_v8[m][0] | (uint32_t)c_v8[m][1] << 8 | (uint32_t)c_v8[m][2] << 16 | (uint32_t)c_v8[m][3] << 24,
                           hi = (uint32_t)c_v8[m][4] | (uint32_t)c_v8[m][5] << 8;
            ls = (int)__builtin_amdgcn_perm(hi, lo, cls | 0x0c0c0c00u) << 4;
        }
        // 8-338 / 8-339 as one expression (qP / 6 >= 6 shifts left)
        const int lsh = e >= 6 ? e - 6 : 0, rsh = e >= 6 ? 0 : 6 - e, rnd = e >= 6 ? 0 : 1 << (5 - e);
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int v = level_at(ws->sm[1 + 4 * q + (p >> 4)], ws->vals, p & 15);
            ws->dense[q][lane] = (int32_t)(((uint32_t)(v * ls) << lsh) + (uint32_t)rnd) >> rsh;
        }
    } else if (i16 && lane < 16) {
        ws->dense[0][lane] = level_at(ws->sm[0], ws->vals, lane);
    }
    if ((cbp >> 4) && lane >= 56) ws->cdc[(lane - 56) >> 2][lane & 3] = level_at(ws->sm[17 + ((lane - 56) >> 2)], ws->vals, lane & 3);
    if (t8 || i16 || (cbp >> 4)) wave_sync();
    if (t8) {
        // 8.5.13: lanes 0-31 = (8x8 block q, row i): horizontal pass ...
        if (lane < 32) {
            const int q = lane >> 3, i = lane & 7;
            int32_t d[8];
#pragma unroll
            for (int j = 0; j < 8; j++) d[j] = ws->dense[q][i * 8 + j];
            idct8(d, 1);
#pragma unroll
            for (int j = 0; j < 8; j++) ws->t8[q][i * 8 + j] = d[j];
        }
    } else if (i16 || (cbp & 15)) {
        // 4x4 luma blocks: the quad of lanes 4b..4b+3 takes block luma4x4BlkIdx b, lane 4b + r
        // its row r (then column r)
        const int b = lane >> 2, r = lane & 3;
        int dc = 0;
        if (i16) {  // 8.5.10: f = (H c H)[row][col] with H the 4x4 Hadamard, then scaling
            const int row = blk_y(b) >> 2, col = blk_x(b) >> 2;
            // H[r][i] is -1 where: r = 1, i >= 2; r = 2, i in {1, 2}; r = 3, i odd
            auto hneg = [](int r, int i) { return r == 1 ? (i >> 1) : r == 2 ? ((i == 1) | (i == 2)) : r == 3 ? (i & 1) : 0; };
            int32_t f = 0;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                int32_t acc = 0;
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    int32_t vz = 0, vf = 0;
#pragma unroll
                    for (int k = 0; k < 16; k++) {  // resolved at compile time
                        if (c_zz4[k] == i * 4 + j) vz = ws->dense[0][k];
                        if (c_fld4[k] == i * 4 + j) vf = ws->dense[0][k];
                    }
                    const int32_t v = field ? vf : vz;
                    acc += hneg(col, j) ? -v : v;
                }
                f += hneg(row, i) ? -acc : acc;
            }
            const int sc = SCALED ? ls4t[16 * (qp % 6)] : ls4(qp % 6, 0, 0);
            dc = qp >= 36 ? (f * sc) << (qp / 6 - 6) : (f * sc + (1 << (5 - qp / 6))) >> (6 - qp / 6);
        }
        const uint2 o = residual4x4_quad<SCALED>(ws->sm[1 + b], ws->vals, qp, i16, dc, r, field, ls4t + 16 * (qp % 6));
        *(uint2 *)&ws->rl[(blk_y(b) + quad_row(r)) * 16 + blk_x(b)] = o;
    } else {  // no luma levels
        ((uint2 *)ws->rl)[lane] = make_uint2(0u, 0u);
    }
    if (!(cbp >> 4)) {  // no chroma levels
        ((uint32_t *)ws->rc)[lane] = 0u;
    } else if (lane < 32) {  // chroma: 8.5.11 DC then 8.5.12 per 4x4 block, a quad per block
        const int c = lane >> 4, b = (lane >> 2) & 3, r = lane & 3;
        const int qpc = ax.qpc[c];
        const int32_t *dcv = ws->cdc[c];
        const int32_t e00 = dcv[0] + dcv[2], e01 = dcv[1] + dcv[3], e10 = dcv[0] - dcv[2], e11 = dcv[1] - dcv[3];
        const int32_t f = b == 0 ? e00 + e01 : b == 1 ? e00 - e01 : b == 2 ? e10 + e11 : e10 - e11;
        const int dc = ((f * (SCALED ? ls4t[16 * (qpc % 6)] : ls4(qpc % 6, 0, 0))) << (qpc / 6)) >> 5;
        const uint2 o = residual4x4_quad<SCALED>(ws->sm[19 + 4 * c + b], ws->vals, qpc, true, dc, r, field, ls4t + 16 * (qpc % 6));
        *(uint2 *)&ws->rc[c][((b >> 1) * 4 + quad_row(r)) * 8 + (b & 1) * 4] = o;
    }
    if (t8) {
        wave_sync();
        // ... then lanes 0-31 = (block q, column j): vertical pass and (x + 32) >> 6
        if (lane < 32) {
            const int q = lane >> 3, j = lane & 7;
            int32_t d[8];
#pragma unroll
            for (int i = 0; i < 8; i++) d[i] = ws->t8[q][i * 8 + j];
            idct8(d, 1);
            const int x0 = (q & 1) * 8, y0 = (q >> 1) * 8;
#pragma unroll
            for (int i = 0; i < 8; i++) ws->rl[(y0 + i) * 16 + x0 + j] = (int16_t)((d[i] + 32) >> 6);
        }
    }
    wave_sync();
    return true;
}

// ------------------------------------------------------------ inter MC
__device__ __forceinline__ gu8 *slot_base(const DevPic &P, int s) { return G(P.dpb) + (uint64_t)s * P.slot_bytes; }

// Where an MB's samples lie (6.4.1, H264PictureBase.cpp:2503-2530): the picture row of its
// first luma / chroma sample and the row step (2 for field MBs of MBAFF frames, whose rows
// are every other picture row, 8.5.14), and its row origin in the coordinates of the
// pictures it predicts from (frame rows, or field rows for field MBs,
// H264InterPrediction.cpp:553-557).
struct MbGeo {
    int mbx, ly, cy, step, mcy, bot;
    bool field;
};
template <bool MBAFF>
__device__ __forceinline__ MbGeo mb_geo(const DevPic &P, int addr) {
    MbGeo g;
    if (!MBAFF || !P.mbaff) {
        const int y = addr / P.W;
        g.mbx = addr % P.W;
        g.ly = y * 16;
        g.cy = y * 8;
        g.step = 1;
        g.mcy = g.ly;
        g.bot = 0;
        g.field = false;
        return g;
    }
    const int pair = addr >> 1, py = pair / P.W;
    g.mbx = pair % P.W;
    g.bot = addr & 1;
    g.field = (G(P.mbs)[addr].flags & H264G_MBF_FIELD) != 0;
    g.step = g.field ? 2 : 1;
    g.ly = py * 32 + (g.field ? g.bot : 16 * g.bot);
    g.cy = py * 16 + (g.field ? g.bot : 8 * g.bot);
    g.mcy = g.field ? py * 16 : g.ly;
    return g;
}

// (P1 + P2 + 1) >> 1 of every luma position (xF, yF), 8.4.2.2.1 (H264InterPrediction.cpp:2344-2480),
// with P1, P2 among 0 = G (integer sample), 1 = b (horizontal half sample), 2 = h
// (vertical half sample), 3 = j: 4 bits (P1 | P2 << 2) at bit 4 * (4 * yF + xF).  The
// quarter positions right of or below the half samples read them one column right
// (m instead of h, G at x + 1) or one row down (s instead of b, G at y + 1).
constexpr uint64_t mc_sel_table() {
    const int t[16][2] = {{0, 0}, {0, 1}, {1, 1}, {0, 1}, {0, 2}, {1, 2}, {1, 3}, {1, 2},
                          {2, 2}, {2, 3}, {3, 3}, {2, 3}, {0, 2}, {1, 2}, {1, 3}, {1, 2}};
    uint64_t v = 0;
    for (int i = 0; i < 16; i++) v |= (uint64_t)(t[i][0] | t[i][1] << 2) << (4 * i);
    return v;
}
constexpr uint64_t MC_SEL = mc_sel_table();
// 6-tap (1, -5, 20, 20, -5, 1) as signed byte weights for v_dot4: samples s..s+3 and
// s+4, s+5 (bytes 0-1; bytes 2-3 for the second column of a pair).  The samples enter
// as x ^ 0x80 = x - 128, so every tap sum is short by 128 * 32 = 4096.
constexpr int TAP_LO = 0x1414fb01, TAP_HI = 0x000001fb, TAP_HI2 = 0x01fb0000, TAP_BIAS = 4096;

__device__ __forceinline__ uint32_t align8(uint32_t hi, uint32_t lo, uint32_t bytes) {
    return __builtin_amdgcn_alignbyte(hi, lo, bytes);
}
__device__ __forceinline__ int sdot4(uint32_t a, int w, int acc) { return __builtin_amdgcn_sdot4((int)a, w, acc, false); }
__device__ __forceinline__ int sdot2(uint32_t a, short w0, short w1, int acc) {
    typedef short short2_t __attribute__((ext_vector_type(2)));
    return __builtin_amdgcn_sdot2(__builtin_bit_cast(short2_t, a), (short2_t){w0, w1}, acc, false);
}
// Low bytes of v0..v3 as one dword, through v_perm.  Written with shifts and ORs, hipcc
// fuses Clip1(x >> n) of two values into v_ashr_pk_u8_i32 and ORs the other two bytes
// onto its destination, whose upper half then still holds the register's old contents
// on gfx950; the permutes keep that instruction out.
__device__ __forceinline__ uint32_t pack4(int v0, int v1, int v2, int v3) {
    const uint32_t lo = __builtin_amdgcn_perm((uint32_t)v1, (uint32_t)v0, 0x0c0c0400u);
    const uint32_t hi = __builtin_amdgcn_perm((uint32_t)v3, (uint32_t)v2, 0x0c0c0400u);
    return __builtin_amdgcn_perm(hi, lo, 0x05040100u);
}
// Per-byte (a + b + 1) >> 1.
__device__ __forceinline__ uint32_t avg4(uint32_t a, uint32_t b) { return (a | b) - (((a ^ b) >> 1) & 0x7f7f7f7fu); }

// Luma prediction samples of list l: lane = (4x4 block b = lane & 15, row r = lane >> 4),
// four samples packed in a dword (0 where the lane's quadrant does not use list l).
// Stage 1 (lane = block b, window rows r, r + 4, r + 8): dword loads of the window row,
// the horizontal 6-tap values b1 of its four columns (v_dot4), all into LDS.  Stage 2:
// the lane's vertical 6-taps on window bytes (h, or m) and on b1 (j), and the pair of
// the position's inputs.  Both stages are the same for every (xF, yF), so lanes with
// different quarter-sample positions do not diverge; the wave skips what no lane uses.
// A field MB of an MBAFF frame predicts from one field of the reference frame: its rows
// are every other frame row from row `parity`, and the reference's field view reports
// that row pitch, twice the width, as its width, which is also where it clamps x
// (H264InterPrediction.cpp:2363 with H264PictureBase.cpp:209-210): right of the picture
// the samples come from the next frame row, on the bottom field's last row from the next
// plane (the DPB slots of MBAFF streams end in a zeroed tail for the Cr plane).
__device__ __forceinline__ uint32_t luma_list(const DevPic &P, const h264g_mb *mb, const DevAux &ax, int l, const MbGeo &g,
                                              WaveRes *ws) {
    const int lane = wave_lane();
    const int W = P.W, wl = W * 16 * g.step, hl = P.H * 16 / g.step;  // row pitch / clamp width, clamp height
    const int bx0 = g.mbx * 16, by0 = g.mcy;
    const int b = lane & 15, r = lane >> 4, bx = b & 3, by = b >> 2, q = ((by >> 1) << 1) | (bx >> 1);
    const bool use = (ax.pf >> (4 * l + q)) & 1;
    const int mvx = mb->mv[l][b][0], mvy = mb->mv[l][b][1];
    const int xF = mvx & 3, yF = mvy & 3;
    const int sel = (int)((MC_SEL >> (4 * (4 * yF + xF))) & 15), s1 = sel & 3, s2 = sel >> 2;
    const uint32_t uses = use ? (1u << s1) | (1u << s2) : 0u;
    const bool need_b = __ballot(uses & 2) != 0, need_h = __ballot(uses & 4) != 0, need_j = __ballot(uses & 8) != 0;
    const int x0 = bx0 + bx * 4 + (mvx >> 2), y0 = by0 + by * 4 + (mvy >> 2);
    WaveMc &mc = ws->mc;
    if (use) {
        const uint8_t *ref = slot_base(P, ax.refid[l][q]) + (g.field && ((ax.fpar >> (4 * l + q)) & 1) ? wl / 2 : 0);
        const int xs = x0 - 2, xa = xs & ~3, off = xs & 3;
        const bool inside = xa >= 0 && xa + 12 <= wl;
#pragma unroll
        for (int k = 0; k < 3; k++) {
            const int rr = r + 4 * k;
            if (rr < 9) {
                const uint8_t *row = ref + (uint64_t)clip3(0, hl - 1, y0 - 2 + rr) * wl;
                uint32_t w0, w1, w2;
                if (inside) {
                    const uint32_t *p = (const uint32_t *)(row + xa);
                    const uint32_t d0 = p[0], d1 = p[1], d2 = p[2];
                    w0 = align8(d1, d0, off); w1 = align8(d2, d1, off); w2 = d2 >> (8 * off);
                } else {  // the window leaves the picture: clamped columns (8.4.2.2.1)
                    int v[9];
#pragma unroll
                    for (int t = 0; t < 9; t++) v[t] = row[clip3(0, wl - 1, xs + t)];
                    w0 = pack4(v[0], v[1], v[2], v[3]); w1 = pack4(v[4], v[5], v[6], v[7]); w2 = (uint32_t)v[8];
                }
                mc.raw[b][rr][0] = w0;
                mc.raw[b][rr][1] = w1;
                if (need_b || need_j) {
                    const uint32_t s0 = w0 ^ 0x80808080u, sx = w1 ^ 0x80808080u, sy = w2 ^ 0x80u;
                    int hv[4];
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const uint32_t lo = i ? align8(sx, s0, i) : s0, hi = i ? align8(sy, sx, i) : sx;
                        hv[i] = sdot4(hi, TAP_HI, sdot4(lo, TAP_LO, TAP_BIAS));
                        mc.b1t[b][i][rr] = (int16_t)hv[i];
                    }
                    if (rr >= 2 && rr <= 6)
                        mc.hb[b][rr - 2] = pack4(clip1((hv[0] + 16) >> 5), clip1((hv[1] + 16) >> 5), clip1((hv[2] + 16) >> 5),
                                                 clip1((hv[3] + 16) >> 5));
                }
            }
        }
    }
    wave_sync();
    uint32_t out = 0;
    if (use) {
        const int dx = xF == 3, dy = yF == 3;
        uint32_t R[6];
#pragma unroll
        for (int k = 0; k < 6; k++) R[k] = align8(mc.raw[b][r + k][1], mc.raw[b][r + k][0], 2 + dx);
        uint32_t cand[4];
        cand[0] = dy ? R[3] : R[2];
        cand[1] = need_b ? mc.hb[b][r + dy] : 0u;
        cand[2] = 0;
        if (need_h) {  // vertical 6-tap of the four columns: byte transpose, then v_dot4
            const uint32_t t0 = __builtin_amdgcn_perm(R[1], R[0], 0x05010400u), t1 = __builtin_amdgcn_perm(R[1], R[0], 0x07030602u);
            const uint32_t t2 = __builtin_amdgcn_perm(R[3], R[2], 0x05010400u), t3 = __builtin_amdgcn_perm(R[3], R[2], 0x07030602u);
            const uint32_t c0 = __builtin_amdgcn_perm(t2, t0, 0x05040100u) ^ 0x80808080u;
            const uint32_t c1 = __builtin_amdgcn_perm(t2, t0, 0x07060302u) ^ 0x80808080u;
            const uint32_t c2 = __builtin_amdgcn_perm(t3, t1, 0x05040100u) ^ 0x80808080u;
            const uint32_t c3 = __builtin_amdgcn_perm(t3, t1, 0x07060302u) ^ 0x80808080u;
            const uint32_t e01 = __builtin_amdgcn_perm(R[5], R[4], 0x05010400u) ^ 0x80808080u;
            const uint32_t e23 = __builtin_amdgcn_perm(R[5], R[4], 0x07030602u) ^ 0x80808080u;
            const int h0 = sdot4(e01, TAP_HI, sdot4(c0, TAP_LO, TAP_BIAS + 16));
            const int h1 = sdot4(e01, TAP_HI2, sdot4(c1, TAP_LO, TAP_BIAS + 16));
            const int h2 = sdot4(e23, TAP_HI, sdot4(c2, TAP_LO, TAP_BIAS + 16));
            const int h3 = sdot4(e23, TAP_HI2, sdot4(c3, TAP_LO, TAP_BIAS + 16));
            cand[2] = pack4(clip1(h0 >> 5), clip1(h1 >> 5), clip1(h2 >> 5), clip1(h3 >> 5));
        }
        cand[3] = 0;
        if (need_j) {  // vertical 6-tap over b1 (8-243) with v_dot2 on row pairs
            const uint32_t sh = 2 * (r & 1);
            int jv[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const uint32_t *c = (const uint32_t *)&mc.b1t[b][i][r & ~1];
                const uint32_t d0 = c[0], d1 = c[1], d2 = c[2], d3 = c[3];
                const uint32_t p0 = align8(d1, d0, sh), p1 = align8(d2, d1, sh), p2 = align8(d3, d2, sh);
                jv[i] = clip1(sdot2(p2, -5, 1, sdot2(p1, 20, 20, sdot2(p0, 1, -5, 512))) >> 10);
            }
            cand[3] = pack4(jv[0], jv[1], jv[2], jv[3]);
        }
        const uint32_t a = s1 == 0 ? cand[0] : s1 == 1 ? cand[1] : s1 == 2 ? cand[2] : cand[3];
        const uint32_t c = s2 == 0 ? cand[0] : s2 == 1 ? cand[1] : s2 == 2 ? cand[2] : cand[3];
        out = avg4(a, c);
    }
    wave_sync();  // the buffer is reused by the next list
    return out;
}

// Two horizontally adjacent chroma prediction samples at (xC, yC) with a 1/8-sample
// MV, 8.4.2.2.2 (H264InterPrediction.cpp:2485-2522), coordinates clamped: samples
// A, B (row yi) and C, D (row yi + 1) weighted (8 - xF)(8 - yF), xF(8 - yF), (8 - xF)yF,
// xF yF.  The three columns of each row arrive as one dword (two aligned dword loads
// where the columns lie inside the row, clamped byte loads at the picture's edges), and
// each output is one v_dot4 of the bytes (A, B, C, D) with the four weights.
__device__ __forceinline__ void chroma2(const gu8 *ref, int wc, int hc, int xC, int yC, int mvx, int mvy, int &o0, int &o1) {
    const int xi = xC + (mvx >> 3), yi = yC + (mvy >> 3), xF = mvx & 7, yF = mvy & 7;
    const gu8 *r0 = ref + (uint64_t)clip3(0, hc - 1, yi) * wc, *r1 = ref + (uint64_t)clip3(0, hc - 1, yi + 1) * wc;
    const int xa = xi & ~3;
    uint32_t a, b;  // bytes 0..2: columns xi .. xi + 2 of rows yi, yi + 1
    if (xa >= 0 && xa + 8 <= wc) {
        const GAS uint32_t *p0 = (const GAS uint32_t *)(r0 + xa), *p1 = (const GAS uint32_t *)(r1 + xa);
        a = align8(p0[1], p0[0], (uint32_t)(xi & 3));
        b = align8(p1[1], p1[0], (uint32_t)(xi & 3));
    } else {
        const int x0 = clip3(0, wc - 1, xi), x1 = clip3(0, wc - 1, xi + 1), x2 = clip3(0, wc - 1, xi + 2);
        a = pack4(r0[x0], r0[x1], r0[x2], 0);
        b = pack4(r1[x0], r1[x1], r1[x2], 0);
    }
    const uint32_t w = (uint32_t)((8 - xF) * (8 - yF)) | (uint32_t)(xF * (8 - yF)) << 8 | (uint32_t)((8 - xF) * yF) << 16 |
                       (uint32_t)(xF * yF) << 24;
    o0 = (int)(__builtin_amdgcn_udot4(__builtin_amdgcn_perm(b, a, 0x05040100u), w, 32u, false) >> 6);
    o1 = (int)(__builtin_amdgcn_udot4(__builtin_amdgcn_perm(b, a, 0x06050201u), w, 32u, false) >> 6);
}

// Explicit weighted prediction, 8.4.2.3.2 (H264InterPrediction.cpp:2526-2829), as one
// v_dot2 per sample: the two lists' samples as the 16-bit halves of a dword (list 0
// low), weighted (w0, w1) -- one of them 0 for a single list -- plus the rounding term,
// then shifted, offset and clipped.  The host resolved the weights, including the
// L1-only luma entries of quirk Q2, into w0 / o0.  (Default weighting, 8.4.2.3.1, is
// the rounded average and stays outside.)
struct WpTerms {
    uint32_t w;          // (w0, w1) as 16-bit halves
    int rnd, sh, off;
};
__device__ __forceinline__ WpTerms wp_terms(const DevWeight &w, int c, int pf0, int pf1) {
    const int lw = w.logWD[c];
    WpTerms t;
    if (pf0 && pf1) {
        t.w = (uint16_t)w.w0[c] | (uint32_t)(uint16_t)w.w1[c] << 16;
        t.rnd = 1 << lw;
        t.sh = lw + 1;
        t.off = (w.o0[c] + w.o1[c] + 1) >> 1;
    } else {
        const int ww = (pf0 || c == 0) ? w.w0[c] : w.w1[c];
        t.w = pf0 ? (uint32_t)(uint16_t)ww : (uint32_t)(uint16_t)ww << 16;
        t.rnd = lw >= 1 ? 1 << (lw - 1) : 0;
        t.sh = lw;
        t.off = (pf0 || c == 0) ? w.o0[c] : w.o1[c];
    }
    return t;
}
__device__ __forceinline__ int wp_apply(const WpTerms &t, uint32_t pair) {
    typedef short short2_t __attribute__((ext_vector_type(2)));
    const int v = __builtin_amdgcn_sdot2(__builtin_bit_cast(short2_t, pair), __builtin_bit_cast(short2_t, t.w), t.rnd, false);
    return clip1((v >> t.sh) + t.off);
}

// Clip1 of the sums of two samples and two residual values, 16 bits each (the sums saturate).
__device__ __forceinline__ uint32_t add_clip1(uint32_t samples, uint32_t res) {
    typedef short short2_t __attribute__((ext_vector_type(2)));
    const short2_t v = __builtin_elementwise_add_sat(__builtin_bit_cast(short2_t, samples), __builtin_bit_cast(short2_t, res));
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_min(__builtin_elementwise_max(v, (short2_t){0, 0}), (short2_t){255, 255}));
}

// Inter MB (or I_PCM copy): prediction + residual, written to the destination slot.
// SCALED: the launch holds pictures with scaling matrices (their residual code reads the
// LevelScale tables; the other pictures' the flat one).
template <bool MBAFF, bool SCALED>
__device__ void inter_mb(const DevPic &P, int addr, WaveRes *ws) {
    const int lane = wave_lane();
    const h264g_mb *mb = &G(P.mbs)[addr];
    const DevAux &ax = G(P.aux)[addr];  // per-lane fields (refid[q], wp[q]) are read from memory
    const int W = P.W, H = P.H, wl = W * 16, hl = H * 16, wc = W * 8, hc = H * 8;
    const MbGeo g = mb_geo<MBAFF>(P, addr);
    const int mbx = g.mbx;
    uint8_t *dst = slot_base(P, P.dst);
    uint8_t *dy = dst, *dcb = dst + (uint64_t)wl * hl, *dcr = dcb + (uint64_t)wc * hc;
    if (ax.kind & AUX_PCM) {  // 8.3.5 (H264PictureBase.cpp:2449-2499)
        const int16_t *pcm = G(P.levels) + mb->level_offset;
        for (int i = lane; i < 256; i += WAVE) dy[(g.ly + (i >> 4) * g.step) * wl + mbx * 16 + (i & 15)] = (uint8_t)pcm[i];
        dcb[(g.cy + (lane >> 3) * g.step) * wc + mbx * 8 + (lane & 7)] = (uint8_t)pcm[256 + lane];
        dcr[(g.cy + (lane >> 3) * g.step) * wc + mbx * 8 + (lane & 7)] = (uint8_t)pcm[320 + lane];
        return;
    }
    const bool res = SCALED && P.ls ? build_residual<MBAFF, SCALED>(mb, ax, G(P.levels), ws, G(P.ls))
                                    : build_residual<MBAFF, false>(mb, ax, G(P.levels), ws, nullptr);
    // ---- luma: lane -> 4x4 block b = lane & 15 (raster), row r = lane >> 4
    {
        const int b = lane & 15, r = lane >> 4, bx = b & 3, by = b >> 2, q = (by >> 1) * 2 + (bx >> 1);
        const int pf0 = (ax.pf >> q) & 1, pf1 = (ax.pf >> (4 + q)) & 1;
        uint32_t p0 = 0, p1 = 0;
#pragma nounroll
        for (int l = 0; l < 2; l++) {  // one inlined copy of the interpolation for both lists
            if (!(ax.pf & (0x0F << (4 * l)))) continue;  // MB-uniform
            const uint32_t v = luma_list(P, mb, ax, l, g, ws);
            if (l) p1 = v; else p0 = v;
        }
        const DevWeight &w = G(P.wt)[ax.wp[q]];
        uint32_t packed;
        if (!w.mode) {
            packed = pf0 && pf1 ? avg4(p0, p1) : (pf0 ? p0 : p1);
        } else {  // byte i of p0 / p1 as the 16-bit halves of one dword (v_perm, 0x0c = zero)
            const WpTerms t = wp_terms(w, 0, pf0, pf1);
            packed = pack4(wp_apply(t, __builtin_amdgcn_perm(p1, p0, 0x0c040c00u)),
                           wp_apply(t, __builtin_amdgcn_perm(p1, p0, 0x0c050c01u)),
                           wp_apply(t, __builtin_amdgcn_perm(p1, p0, 0x0c060c02u)),
                           wp_apply(t, __builtin_amdgcn_perm(p1, p0, 0x0c070c03u)));
        }
        if (res) {
            const uint2 rl = *(const uint2 *)&ws->rl[(by * 4 + r) * 16 + bx * 4];
            packed = __builtin_amdgcn_perm(add_clip1(__builtin_amdgcn_perm(0u, packed, 0x0c030c02u), rl.y),
                                           add_clip1(__builtin_amdgcn_perm(0u, packed, 0x0c010c00u), rl.x), 0x06040200u);
        }
        *(uint32_t *)&dy[(uint64_t)(g.ly + (by * 4 + r) * g.step) * wl + mbx * 16 + bx * 4] = packed;
    }
    // ---- chroma: lane -> component c, 4x4 luma block b, chroma row r (2 samples)
    {
        int c = lane >> 5, i = lane & 31, b = i >> 1, r = i & 1, bx = b & 3, by = b >> 2, q = (by >> 1) * 2 + (bx >> 1);
        int pf0 = (ax.pf >> q) & 1, pf1 = (ax.pf >> (4 + q)) & 1;
        int xC = mbx * 8 + bx * 2, yC = g.mcy / 2 + by * 2 + r;
        int c00 = 0, c01 = 0, c10 = 0, c11 = 0;
        const uint64_t coff = (uint64_t)wl * hl + (uint64_t)c * wc * hc;
        // field MBs: the parity's field of the reference (row pitch and clamp width 2 wc,
        // see luma_list) and the vertical chroma vector offset of Table 8-10
        // (H264InterPrediction.cpp:2024-2043)
        const int fw = wc * g.step, fh = hc / g.step;
        int mvy0 = mb->mv[0][b][1], mvy1 = mb->mv[1][b][1];
        uint64_t o0 = coff, o1 = coff;
        if (g.field) {
            const int par0 = (ax.fpar >> q) & 1, par1 = (ax.fpar >> (4 + q)) & 1;
            o0 += par0 ? wc : 0;
            o1 += par1 ? wc : 0;
            mvy0 += par0 == g.bot ? 0 : (par0 ? -2 : 2);
            mvy1 += par1 == g.bot ? 0 : (par1 ? -2 : 2);
        }
        if (pf0) chroma2(slot_base(P, ax.refid[0][q]) + o0, fw, fh, xC, yC, mb->mv[0][b][0], mvy0, c00, c01);
        if (pf1) chroma2(slot_base(P, ax.refid[1][q]) + o1, fw, fh, xC, yC, mb->mv[1][b][0], mvy1, c10, c11);
        const DevWeight &w = G(P.wt)[ax.wp[q]];
        uint8_t *plane = c == 0 ? dcb : dcr;
        int v0, v1;
        if (!w.mode) {
            v0 = pf0 && pf1 ? (c00 + c10 + 1) >> 1 : (pf0 ? c00 : c10);
            v1 = pf0 && pf1 ? (c01 + c11 + 1) >> 1 : (pf0 ? c01 : c11);
        } else {
            const WpTerms t = wp_terms(w, 1 + c, pf0, pf1);
            v0 = wp_apply(t, (uint32_t)c00 | (uint32_t)c10 << 16);
            v1 = wp_apply(t, (uint32_t)c01 | (uint32_t)c11 << 16);
        }
        uint32_t v = (uint32_t)v0 | (uint32_t)v1 << 16;
        if (res) v = add_clip1(v, *(const uint32_t *)&ws->rc[c][(by * 2 + r) * 8 + bx * 2]);
        *(uint16_t *)&plane[(uint64_t)(g.cy + (by * 2 + r) * g.step) * wc + xC] = (uint16_t)(v | v >> 8);
    }
    (void)H;
}

// ------------------------------------------------------------ wavefront helpers
__device__ __forceinline__ uint32_t ld_acquire(const uint32_t *p) {
    return __hip_atomic_load(p, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_release(uint32_t *p, uint32_t v) {
    __hip_atomic_store(p, v, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
}

constexpr uint32_t SPIN_LIMIT = 1u << 20;

// The persistent loops below keep all control flow around the ticket, the waits and
// the publication wave-uniform: every lane executes the same atomics, loads and stores
// (lane-identical addresses and values), and each value a branch depends on is made
// scalar with readfirstlane.  Lane-conditional regions here (e.g. "lane 0 publishes,
// then lane 0 takes the next ticket") let the compiler thread the two regions together
// across the loop latch; its CFG structurizer then leaves lanes 1..63 iterating on
// their own, which never terminates.
__device__ __forceinline__ uint32_t uniform(uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }

// Sets the device error word (polled by the other waits, so it is device memory) and its copy in
// pinned memory that the host reads.
__device__ __forceinline__ void report_timeout(uint32_t *err) {
    atomicOr(err, DEVERR_TIMEOUT);
    __hip_atomic_store(G(G((const DevErr *)err)->host), DEVERR_TIMEOUT, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Waits until flags[i] == epoch for each listed neighbour.  Bounded: after SPIN_LIMIT
// polls, or once another wave has raised the error word, the wave stops waiting (its
// output is then wrong, and h264g_sync reports the error).
// One of them (d < 0: none); the caller issues the acquire fence.
__device__ __forceinline__ void wait_dep(const uint32_t *flags, int dep, uint32_t epoch, uint32_t *err) {
    const int d = (int)uniform((uint32_t)dep);
    if (d < 0) return;
    for (uint32_t it = 0;; ++it) {
        if (uniform(ld_acquire(&flags[d])) == epoch) break;
        if (it >= SPIN_LIMIT) {
            report_timeout(err);
            break;
        }
        if ((it & 255u) == 255u && uniform(__hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) != 0u) break;
        __builtin_amdgcn_s_sleep(1);
    }
}
__device__ void wait_deps(const uint32_t *flags, const int *deps, int nd, uint32_t epoch, uint32_t *err) {
    for (int k = 0; k < nd; k++) wait_dep(flags, deps[k], epoch, err);
    __atomic_thread_fence(__ATOMIC_ACQUIRE);
}

// The barrier orders every lane's stores before the (wave-wide) release store.
__device__ void publish(uint32_t *flag, uint32_t epoch) {
    wave_sync();
    st_release(flag, epoch);
}

// Next ticket of a persistent launch (same value in every lane), or -1.  Only lane 0
// adds 1; the compiler's wave-level atomic combining issues one atomic for the wave.
__device__ int next_ticket(DevCtl *ctl, uint32_t n) {
    const uint32_t t = uniform(atomicAdd(&ctl->ticket, wave_lane() == 0 ? 1u : 0u));
    return t < n ? (int)t : -1;
}

// The launch's epoch: progress words equal to it are this launch's.  Read once at
// kernel start; it only changes when the launch's last wave retires, after every
// wave of the launch has read it.
__device__ __forceinline__ uint32_t launch_epoch(const uint32_t *epoch) {
    return uniform(__hip_atomic_load(epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}

// The last wave of a launch resets the control block for the next launch on the stream
// and advances the shared epoch, so the next wavefront launch (of either kind) uses a
// value no progress word holds yet.  Launch arguments therefore stay identical from one
// launch to the next (a caller may capture them).
__device__ void retire(DevCtl *ctl, uint32_t total_waves, uint32_t *epoch, uint32_t cur) {
    const uint32_t d = uniform(atomicAdd(&ctl->done, wave_lane() == 0 ? 1u : 0u));
    if (d == total_waves - 1) {
        __hip_atomic_store(&ctl->ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(&ctl->done, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(epoch, cur + 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

__device__ __forceinline__ bool cls_inter(int c) { return c == H264G_MB_P || c == H264G_MB_P_SKIP || c == H264G_MB_B; }
// An MB that constrained intra prediction hides from intra MBs: the reference tests
// IS_INTER_Prediction_Mode(m_mb_pred_mode) (H264PictureBase.cpp:1129; H264CommonFunc.h:273),
// false for P_8x8 / B_8x8 (Pred_NA, H264MacroBlock.cpp:99-100, 142), which stay available.
__device__ __forceinline__ bool cip_hides(const h264g_mb &m) {
    return m.mb_type == H264G_MB_P_SKIP ||
           ((m.mb_type == H264G_MB_P || m.mb_type == H264G_MB_B) && m.part_shape != H264G_PART_8x8);
}
__device__ __forceinline__ bool cls_intra(int c) { return c == H264G_MB_I4x4 || c == H264G_MB_I8x8 || c == H264G_MB_I16x16; }

// ------------------------------------------------------------ intra (8.3)
// LDS tile of one wave: luma T[y+1][x+1] for x in [-1, 23], y in [-1, 15] (row -1 holds
// the top and top-right neighbours, column -1 the left ones), chroma C[c][y+1][x+1] for
// x, y in [-1, 7]; availability of the neighbouring MBs A, B, C, D.
struct WaveIntra {
    WaveRes res;
    uint8_t T[17][25];
    uint8_t C[2][9][9];
    int16_t pf[25];        // filtered 8x8 reference samples p'[-1,-1..7] then p'[0..15,-1]
    int16_t U[25];         // the same samples before filtering (-1: not available)
    int16_t X[2][16];      // neighbour lines of two 4x4 blocks (see pred4x4)
    union {
        uint32_t p4[10][WAVE];  // Intra_4x4 wavefront step t, lane: see intra4_prep
        struct {
            int32_t ua[4][32];      // Intra_8x8 block, reference sample: see intra8_prep
            uint32_t tp[4][WAVE];   // Intra_8x8 block, pixel: taps on the filtered samples
        } p8;
    };
};

// Availability of the neighbouring MBs A, B, C, D for intra prediction as bits 0..3 of
// one word (a struct of four fields selected per lane would be indexed in scratch).
struct Avail {
    uint32_t m;
    __device__ bool A() const { return m & 1u; }
    __device__ bool B() const { return m & 2u; }
    __device__ bool C() const { return m & 4u; }
    __device__ bool D() const { return m & 8u; }
};

// Flat index into the tile WaveIntra::T (T[0][0] = p[-1, -1] of the MB, T[1 + y][1 + x] =
// sample (x, y)) of sample p[x, y] relative to the 4x4 / 8x8 block at (xO, yO) of the
// current MB, or -1 when it is not available for intra prediction (6.4.12.1,
// H264PictureBase.cpp:1099-1155; blk4: the 4x4 block, whose top-right samples inside the
// MB are not available for blocks 3 and 11, H264PictureBase.cpp:1131).
__device__ __forceinline__ int tile_a(const Avail &av, int xO, int yO, int x, int y, int blk4) {
    const int xx = xO + x, yy = yO + y;
    if (yy < 0) {
        if (xx < 0) return av.D() ? 0 : -1;
        if (xx < 16) return av.B() ? xx + 1 : -1;
        return av.C() ? xx + 1 : -1;
    }
    if (xx < 0) return av.A() ? (yy + 1) * 25 : -1;
    if (xx >= 16) return -1;
    if (blk4 >= 0 && x > 3 && (blk4 == 3 || blk4 == 11)) return -1;
    return (yy + 1) * 25 + xx + 1;
}

// 8.3.1.2 for pixel (x, y) of a 4x4 block (H264PictureBase.cpp:1062-1419), from the
// block's neighbour line X[0..14] = L3 L3 L2 L1 L0 TL T0 .. T7 T7 (L = p[-1, y],
// T = p[x, -1], TL = p[-1, -1]; T4..T7 already substituted by T3 when unavailable;
// -1 = not available).  Every directional mode reads a copy X[i], a 2-tap
// (X[i] + X[i+1] + 1) >> 1 or a 3-tap (X[c-1] + 2 X[c] + X[c+1] + 2) >> 2 of this line:
// the equations of 8.3.1.2.4 - 8.3.1.2.9 with p[-1, y] and p[x, -1] mapped to their X
// positions (the duplicated end samples give the corner cases, e.g. Diagonal_Down_Left
// at (3, 3) and Horizontal_Up at zHU = 5).  All three are (X[i0] + X[i1] + X[i2] + X[i3]
// + 2) >> 2: a copy repeats one index four times, a 2-tap equals (2 X[i] + 2 X[i+1] + 2)
// >> 2 and a 3-tap repeats its middle index.  i4_taps gives the four indices (4 bits each,
// i0 lowest) of sample (x, y) in mode m; DC (mode 2) is 0xFFFF.
constexpr uint16_t i4_copy(int i) { return (uint16_t)(i | i << 4 | i << 8 | i << 12); }
constexpr uint16_t i4_tap2(int i) { return (uint16_t)(i | i << 4 | (i + 1) << 8 | (i + 1) << 12); }
constexpr uint16_t i4_tap3(int c) { return (uint16_t)((c - 1) | c << 4 | c << 8 | (c + 1) << 12); }
constexpr uint16_t i4_taps(int mode, int x, int y) {
    switch (mode) {
    case 0: return i4_copy(6 + x);
    case 1: return i4_copy(4 - y);
    case 2: return 0xFFFF;
    case 3: return i4_tap3(7 + x + y);
    case 4: return i4_tap3(5 + x - y);
    case 5: {
        const int z = 2 * x - y;
        if (z >= 0) return (z & 1) ? i4_tap3(5 + x - (y >> 1)) : i4_tap2(5 + x - (y >> 1));
        return z == -1 ? i4_tap3(5) : i4_tap3(6 - y);
    }
    case 6: {
        const int z = 2 * y - x;
        if (z >= 0) return (z & 1) ? i4_tap3(5 - y + (x >> 1)) : i4_tap2(4 - y + (x >> 1));
        return z == -1 ? i4_tap3(5) : i4_tap3(4 + x);
    }
    case 7: return (y & 1) ? i4_tap3(7 + x + (y >> 1)) : i4_tap2(6 + x + (y >> 1));
    default: {
        const int z = x + 2 * y;
        if (z < 5) return (z & 1) ? i4_tap3(3 - y - (x >> 1)) : i4_tap2(3 - y - (x >> 1));
        return z == 5 ? i4_tap3(1) : i4_copy(1);
    }
    }
}
struct I4Taps {
    uint16_t v[9][16];
};
constexpr I4Taps make_i4taps() {
    I4Taps t{};
    for (int m = 0; m < 9; m++)
        for (int k = 0; k < 16; k++) t.v[m][k] = i4_taps(m, k & 3, k >> 2);
    return t;
}
__constant__ I4Taps c_i4taps = make_i4taps();

// What an Intra_4x4 MB's wavefront steps need that does not depend on samples, gathered
// into wi->p4 before the MB waits for its neighbours: per step t and lane the flat tile
// index of neighbour-line sample j (lanes j < 15 of each 16-lane group; -1: not
// available, T4..T7 already substituted by T3) in the low half and the taps of pixel j of
// the lane's block (c_i4taps) in the high half.  The LDS writes are ordered before the
// MB's first wave barrier in intra_mb.
__device__ __forceinline__ void intra4_prep(const h264g_mb *mb, const Avail &av, WaveIntra *wi) {
    const int lane = wave_lane(), g = lane >> 4, j = lane & 15;
#pragma unroll  // (the loads of a step's modes and taps beside those of the others)
    for (int t = 0; t < 10; t++) {
        const int by = (t < 2 ? 0 : (t - 2) >> 1) + g, bx = t - 2 * by;
        const bool has = lane < 32 && bx >= 0 && by < 4;
        const int blk = 8 * (by >> 1) + 4 * (bx >> 1) + 2 * (by & 1) + (bx & 1), xO = bx * 4, yO = by * 4;
        int a = -1;
        uint32_t tp = 0;
        if (has) {
            if (j < 5) a = tile_a(av, xO, yO, -1, j == 0 ? 3 : 4 - j, blk);
            else if (j == 5) a = tile_a(av, xO, yO, -1, -1, blk);
            else if (j < 15) {
                const int tx = j == 14 ? 7 : j - 6;
                a = tile_a(av, xO, yO, tx, -1, blk);
                if (tx >= 4 && a < 0) {  // p[4..7, -1] <- p[3, -1] (H264PictureBase.cpp:1161-1167)
                    const int a3 = tile_a(av, xO, yO, 3, -1, blk);
                    if (a3 >= 0) a = a3;
                }
            }
            tp = c_i4taps.v[mb->intra_pred_modes[blk]][j];
        }
        wi->p4[t][lane] = ((uint32_t)a & 0xFFFFu) | tp << 16;
    }
}

// Intra_8x8 sample (x, y) of mode m (8.3.2.2.2 - 8.3.2.2.10, H264PictureBase.cpp:1601-1843)
// as (pf[i0] + pf[i1] + pf[i2] + pf[i3] + 2) >> 2 on the filtered reference samples
// pf[0] = p'[-1, -1], pf[1 + y] = p'[-1, y], pf[9 + x] = p'[x, -1], like i4_taps (copy =
// one index four times, 2-tap = both twice, 3-tap = middle twice; a weight 3 repeats an
// index three times); 5 bits each, i0 lowest; DC (mode 2) is 0xFFFFFFFF.
constexpr int i8_ft(int i) { return i < 0 ? 0 : 9 + i; }
constexpr int i8_fl(int i) { return i < 0 ? 0 : 1 + i; }
constexpr uint32_t i8_pack(int a, int b, int c, int d) { return (uint32_t)(a | b << 5 | c << 10 | d << 15); }
constexpr uint32_t i8_tap2(int a, int b) { return i8_pack(a, a, b, b); }
constexpr uint32_t i8_tap3(int a, int c, int b) { return i8_pack(a, c, c, b); }
constexpr uint32_t i8_taps(int mode, int x, int y) {
    switch (mode) {
    case 0: return i8_pack(i8_ft(x), i8_ft(x), i8_ft(x), i8_ft(x));
    case 1: return i8_pack(i8_fl(y), i8_fl(y), i8_fl(y), i8_fl(y));
    case 2: return 0xFFFFFFFFu;
    case 3:
        if (x == 7 && y == 7) return i8_pack(i8_ft(14), i8_ft(15), i8_ft(15), i8_ft(15));
        return i8_tap3(i8_ft(x + y), i8_ft(x + y + 1), i8_ft(x + y + 2));
    case 4:
        if (x > y) return i8_tap3(i8_ft(x - y - 2), i8_ft(x - y - 1), i8_ft(x - y));
        if (x < y) return i8_tap3(i8_fl(y - x - 2), i8_fl(y - x - 1), i8_fl(y - x));
        return i8_tap3(i8_ft(0), 0, i8_fl(0));
    case 5: {
        const int z = 2 * x - y;
        if (z >= 0 && !(z & 1)) return i8_tap2(i8_ft(x - (y >> 1) - 1), i8_ft(x - (y >> 1)));
        if (z >= 0) return i8_tap3(i8_ft(x - (y >> 1) - 2), i8_ft(x - (y >> 1) - 1), i8_ft(x - (y >> 1)));
        if (z == -1) return i8_tap3(i8_fl(0), 0, i8_ft(0));
        return i8_tap3(i8_fl(y - 2 * x - 1), i8_fl(y - 2 * x - 2), i8_fl(y - 2 * x - 3));
    }
    case 6: {
        const int z = 2 * y - x;
        if (z >= 0 && !(z & 1)) return i8_tap2(i8_fl(y - (x >> 1) - 1), i8_fl(y - (x >> 1)));
        if (z >= 0) return i8_tap3(i8_fl(y - (x >> 1) - 2), i8_fl(y - (x >> 1) - 1), i8_fl(y - (x >> 1)));
        if (z == -1) return i8_tap3(i8_fl(0), 0, i8_ft(0));
        return i8_tap3(i8_ft(x - 2 * y - 1), i8_ft(x - 2 * y - 2), i8_ft(x - 2 * y - 3));
    }
    case 7:
        if (!(y & 1)) return i8_tap2(i8_ft(x + (y >> 1)), i8_ft(x + (y >> 1) + 1));
        return i8_tap3(i8_ft(x + (y >> 1)), i8_ft(x + (y >> 1) + 1), i8_ft(x + (y >> 1) + 2));
    default: {
        const int z = x + 2 * y;
        if (z < 13 && !(z & 1)) return i8_tap2(i8_fl(y + (x >> 1)), i8_fl(y + (x >> 1) + 1));
        if (z < 13) return i8_tap3(i8_fl(y + (x >> 1)), i8_fl(y + (x >> 1) + 1), i8_fl(y + (x >> 1) + 2));
        if (z == 13) return i8_pack(i8_fl(6), i8_fl(7), i8_fl(7), i8_fl(7));
        return i8_pack(i8_fl(7), i8_fl(7), i8_fl(7), i8_fl(7));
    }
    }
}
struct I8Taps {
    uint32_t v[9][64];
};
constexpr I8Taps make_i8taps() {
    I8Taps t{};
    for (int m = 0; m < 9; m++)
        for (int k = 0; k < 64; k++) t.v[m][k] = i8_taps(m, k & 7, k >> 3);
    return t;
}
__constant__ I8Taps c_i8taps = make_i8taps();

// What an Intra_8x8 MB's four blocks need that does not depend on samples, gathered into
// wi->p8 before the MB waits for its neighbours: per block the flat tile index of each of
// the 25 reference samples before filtering (U[0] = p[-1, -1], U[1 + y] = p[-1, y],
// U[9 + x] = p[x, -1] with p[8..15, -1] <- p[7, -1] when not available; -1: not
// available) and each pixel's taps (c_i8taps).
__device__ __forceinline__ void intra8_prep(const h264g_mb *mb, const Avail &av, WaveIntra *wi) {
    const int lane = wave_lane();
#pragma unroll 1
    for (int blk = 0; blk < 4; blk++) {
        const int xO = (blk & 1) * 8, yO = (blk >> 1) * 8;
        if (lane < 25) {
            int a;
            if (lane == 0) a = tile_a(av, xO, yO, -1, -1, -1);
            else if (lane < 9) a = tile_a(av, xO, yO, -1, lane - 1, -1);
            else {
                const int x = lane - 9;
                a = tile_a(av, xO, yO, x, -1, -1);
                if (x >= 8 && a < 0) {
                    const int a7 = tile_a(av, xO, yO, 7, -1, -1);
                    if (a7 >= 0) a = a7;
                }
            }
            wi->p8.ua[blk][lane] = a;
        }
        wi->p8.tp[blk][lane] = c_i8taps.v[mb->intra_pred_modes[blk]][lane];
    }
}

// Residuals of intra MBs.  They need no neighbour samples, so the inter stage, which is
// parallel over MBs, builds them (intra_res_build) and leaves them in G(P.ires); the intra
// schedules load an MB's residual (intra_res_fetch, lanes 0-47 one 16-byte piece each)
// before they wait for its neighbours and put it in the tile after the wait
// (intra_res_place).
static_assert(offsetof(WaveRes, rc) == offsetof(WaveRes, rl) + 512 && offsetof(WaveRes, rl) % 16 == 0,
              "luma and chroma residual planes are one 768-byte run");
template <bool MBAFF, bool SCALED>
__device__ __forceinline__ void intra_res_build(const DevPic &P, int addr, WaveRes *ws) {
    const DevAux &ax = G(P.aux)[addr];
    if (!MBAFF) {  // the MB's entry for the band schedule: its ICOL word, types and modes
        const GAS h264g_mb *const mb = &G(P.mbs)[addr];
        const uint32_t idx = ax.ires & AUX_IRES_MASK, icol = G(P.irow)[P.H + 1 + idx];
        const uint32_t type = mb->mb_type == H264G_MB_I4x4 ? 0u : mb->mb_type == H264G_MB_I8x8 ? 1u : 2u;
        const GAS uint32_t *const m = (const GAS uint32_t *)mb->intra_pred_modes;
        auto nibbles = [](uint32_t v) {  // the low nibbles of four bytes
            v &= 0x0F0F0F0Fu;
            v = (v | v >> 4) & 0x00FF00FFu;
            return (v | v >> 8) & 0xFFFFu;
        };
        if (wave_lane() == 0)
            G((uint4 *)P.imeta)[idx] = make_uint4(icol | type << IMETA_TYPE_SHIFT | (uint32_t)mb->intra16x16_pred_mode << IMETA_I16_SHIFT |
                                                      (uint32_t)mb->intra_chroma_pred_mode << IMETA_CHROMA_SHIFT,
                                                  nibbles(m[0]) | nibbles(m[1]) << 16, nibbles(m[2]) | nibbles(m[3]) << 16, 0u);
    }
    if (!(SCALED && P.ls ? build_residual<MBAFF, SCALED>(&G(P.mbs)[addr], ax, G(P.levels), ws, G(P.ls))
                         : build_residual<MBAFF, false>(&G(P.mbs)[addr], ax, G(P.levels), ws, nullptr)))
        return;
    const int lane = wave_lane();
    if (lane < 48) ((uint4 *)(G(P.ires) + (size_t)(ax.ires & AUX_IRES_MASK) * 384))[lane] = ((const uint4 *)ws->rl)[lane];
}
struct IntraRes {
    uint4 v;
    bool res;
};
__device__ __forceinline__ IntraRes intra_res_fetch(const DevPic &P, int addr) {
    const DevAux &ax = G(P.aux)[addr];
    IntraRes r;
    r.res = (ax.kind & AUX_RESID) != 0;
    r.v = make_uint4(0, 0, 0, 0);
    if (r.res && wave_lane() < 48) r.v = ((const uint4 *)(G(P.ires) + (size_t)(ax.ires & AUX_IRES_MASK) * 384))[wave_lane()];
    return r;
}
__device__ __forceinline__ void intra_res_place(const IntraRes &r, WaveIntra *wi) {
    if (r.res && wave_lane() < 48) ((uint4 *)wi->res.rl)[wave_lane()] = r.v;
}

// Prediction and reconstruction of an intra MB whose residual intra_res_place left in
// wi->res (res: the MB has levels); the neighbours it reads are final.  The LDS writes of
// the residual are ordered before its first wave barrier.
// An Intra_4x4 MB has run intra4_prep, an Intra_8x8 MB intra8_prep.  PLANES: 1 luma, 2 chroma
// (which share nothing that either writes), 3 both.
struct IntraHdr {
    int type, i16, chroma;     // mb_type, Intra16x16 and chroma prediction modes
};
template <int PLANES>
__device__ __forceinline__ void intra_mb(const DevPic &P, const MbGeo &g, const IntraHdr &mb, WaveIntra *wi, const Avail &av, bool res) {
    constexpr bool LUMA = PLANES & 1, CHROMA = PLANES & 2;
    const int lane = wave_lane();
    const int W = P.W, H = P.H, wl = W * 16, hl = H * 16, wc = W * 8, hc = H * 8;
    // In an MBAFF frame every neighbouring sample that 6.4.12.2 (Table 6-4) gives an MB lies
    // in the MB's own view of the picture: frame rows for frame MBs, the rows of its parity
    // for field MBs (rows step apart from its first row), at the same columns; Table 6-4
    // only decides availability (the caller's av).
    const int mbx = g.mbx, st = g.step;
    uint8_t *dst = slot_base(P, P.dst);
    uint8_t *dy = dst, *dcb = dst + (uint64_t)wl * hl, *dcr = dcb + (uint64_t)wc * hc;
    // ---- neighbours into the tile
    if (lane < 25) {  // row -1, x = lane - 1
        int x = lane - 1;
        bool ok = x < 0 ? av.D() : (x < 16 ? av.B() : av.C());
        if (LUMA && ok) wi->T[0][lane] = dy[(uint64_t)(g.ly - st) * wl + mbx * 16 + x];
    } else if (lane < 41) {  // column -1
        int y = lane - 25;
        if (LUMA && av.A()) wi->T[y + 1][0] = dy[(uint64_t)(g.ly + y * st) * wl + mbx * 16 - 1];
    } else if (lane < 59) {  // chroma row -1 (x = -1..7) for both planes
        int k = lane - 41, c = k / 9, x = k % 9 - 1;
        bool ok = x < 0 ? av.D() : av.B();
        const uint8_t *pl = c == 0 ? dcb : dcr;
        if (CHROMA && ok) wi->C[c][0][x + 1] = pl[(uint64_t)(g.cy - st) * wc + mbx * 8 + x];
    }
    if (lane < 16) {  // chroma column -1
        int c = lane >> 3, y = lane & 7;
        const uint8_t *pl = c == 0 ? dcb : dcr;
        if (CHROMA && av.A()) wi->C[c][y + 1][0] = pl[(uint64_t)(g.cy + y * st) * wc + mbx * 8 - 1];
    }
    wave_sync();
    // ---- luma
    if (!LUMA) {
    } else if (mb.type == H264G_MB_I4x4) {
        // 4x4 blocks in wavefront order t = bx + 2 by, two blocks per step (lanes 0-15 and
        // 16-31): every neighbour a block reads has a smaller t, and a top-right block that
        // the reference's block order has not decoded yet (blocks 3, 11) counts as not
        // available by rule (tile_a), so the result equals the block-index order.  Each
        // step gathers the two neighbour lines X (pred4x4) from the tile at the indices
        // intra4_prep found, then evaluates every pixel with its four taps.
        const int g = lane >> 4, j = lane & 15, x = j & 3, y = j >> 2;
        const uint8_t *Tf = &wi->T[0][0];
        const int16_t *X = wi->X[g];
#pragma unroll 1
        for (int t = 0; t < 10; t++) {
            const int by = (t < 2 ? 0 : (t - 2) >> 1) + g, bx = t - 2 * by;
            const bool has = lane < 32 && bx >= 0 && by < 4;
            const int xO = bx * 4, yO = by * 4;
            const uint32_t e = wi->p4[t][lane];
            const int xa = (int)(int16_t)(e & 0xFFFFu);
            const uint32_t tp = e >> 16;
            if (has && j < 15) wi->X[g][j] = (int16_t)(xa >= 0 ? (int)Tf[xa] : -1);
            wave_sync();
            if (has) {
                int v = (X[tp & 15u] + X[(tp >> 4) & 15u] + X[(tp >> 8) & 15u] + X[tp >> 12] + 2) >> 2;
                if (tp == 0xFFFFu) {  // DC: the top / left samples are available all or none
                    const bool ta = X[6] >= 0, la = X[4] >= 0;
                    const int st = X[6] + X[7] + X[8] + X[9], sl = X[1] + X[2] + X[3] + X[4];
                    v = ta && la ? (st + sl + 4) >> 3 : la ? (sl + 2) >> 2 : ta ? (st + 2) >> 2 : 128;
                }
                if (res) v = clip1(v + wi->res.rl[(yO + y) * 16 + xO + x]);
                wi->T[yO + y + 1][xO + x + 1] = (uint8_t)v;
            }
            wave_sync();
        }
    } else if (mb.type == H264G_MB_I8x8) {
        // each block: gather its 25 reference samples at the indices intra8_prep found,
        // filter them, then one four-tap sum per pixel
        const uint8_t *Tf = &wi->T[0][0];
#pragma unroll 1
        for (int blk = 0; blk < 4; blk++) {
            const int xO = (blk & 1) * 8, yO = (blk >> 1) * 8;
            if (lane < 25) {
                const int a = wi->p8.ua[blk][lane];
                wi->U[lane] = (int16_t)(a >= 0 ? (int)Tf[a] : -1);
            }
            wave_sync();
            // 8.3.2.2.1 reference sample filtering (H264PictureBase.cpp:1535-1599); the left
            // column and the 16 top samples are available all or none
            if (lane < 25) {
                const int16_t *U = wi->U;
                const int pm = U[0];
                int v = -1;
                if (lane == 0) {  // p'[-1, -1]
                    const int pt = U[9], pl = U[1];
                    if (pm >= 0) {
                        if (pt < 0 || pl < 0) v = pt >= 0 ? (3 * pm + pt + 2) >> 2 : (pl >= 0 ? (3 * pm + pl + 2) >> 2 : pm);
                        else v = (pt + 2 * pm + pl + 2) >> 2;
                    }
                } else if (lane < 9) {  // p'[-1, y]
                    const int y = lane - 1;
                    if (U[1] >= 0) {
                        if (y == 0) v = pm >= 0 ? (pm + 2 * U[1] + U[2] + 2) >> 2 : (3 * U[1] + U[2] + 2) >> 2;
                        else if (y == 7) v = (U[7] + 3 * U[8] + 2) >> 2;
                        else v = (U[y] + 2 * U[y + 1] + U[y + 2] + 2) >> 2;
                    }
                } else {  // p'[x, -1]
                    const int x = lane - 9;
                    if (U[9] >= 0 && U[17] >= 0) {
                        if (x == 0) v = pm >= 0 ? (pm + 2 * U[9] + U[10] + 2) >> 2 : (3 * U[9] + U[10] + 2) >> 2;
                        else if (x == 15) v = (U[23] + 3 * U[24] + 2) >> 2;
                        else v = (U[8 + x] + 2 * U[9 + x] + U[10 + x] + 2) >> 2;
                    }
                }
                wi->pf[lane] = (int16_t)v;
            }
            wave_sync();
            const int x = lane & 7, y = lane >> 3;
            const uint32_t tp = wi->p8.tp[blk][lane];
            const int16_t *pf = wi->pf;
            int v = (pf[tp & 31u] + pf[(tp >> 5) & 31u] + pf[(tp >> 10) & 31u] + pf[(tp >> 15) & 31u] + 2) >> 2;
            if (tp == 0xFFFFFFFFu) {  // DC (8.3.2.2.4): the filtered samples are available all or none
                const bool ta = pf[9] >= 0, la = pf[1] >= 0;
                int st = 0, sl = 0;
#pragma unroll
                for (int k = 0; k < 8; k++) { st += pf[9 + k]; sl += pf[1 + k]; }
                v = ta && la ? (st + sl + 8) >> 4 : la ? (sl + 4) >> 3 : ta ? (st + 4) >> 3 : 128;
            }
            if (res) v = clip1(v + wi->res.rl[(yO + y) * 16 + xO + x]);
            wave_sync();
            wi->T[yO + y + 1][xO + x + 1] = (uint8_t)v;
            wave_sync();
        }
    } else {  // Intra_16x16, 8.3.3 (H264PictureBase.cpp:1847-2056)
        int mode = mb.i16;
        int dc = 128, a = 0, bq = 0, cq = 0;
        if (mode == 2) {
            int st = 0, sl = 0;
            for (int k = 0; k < 16; k++) { st += wi->T[0][k + 1]; sl += wi->T[k + 1][0]; }
            if (av.A() && av.B()) dc = (st + sl + 16) >> 5;
            else if (av.A()) dc = (sl + 8) >> 4;
            else if (av.B()) dc = (st + 8) >> 4;
        } else if (mode == 3) {
            int Hs = 0, Vs = 0;
            for (int k = 0; k < 8; k++) {
                Hs += (k + 1) * (wi->T[0][8 + k + 1] - wi->T[0][6 - k + 1]);
                Vs += (k + 1) * (wi->T[8 + k + 1][0] - wi->T[6 - k + 1][0]);
            }
            a = 16 * (wi->T[16][0] + wi->T[0][16]);
            bq = (5 * Hs + 32) >> 6;
            cq = (5 * Vs + 32) >> 6;
        }
        for (int k = 0; k < 4; k++) {
            int i = lane + k * WAVE, x = i & 15, y = i >> 4;
            int v = mode == 0 ? wi->T[0][x + 1] : mode == 1 ? wi->T[y + 1][0] : mode == 2 ? dc : clip1((a + bq * (x - 7) + cq * (y - 7) + 16) >> 5);
            if (res) v = clip1(v + wi->res.rl[y * 16 + x]);
            wi->T[y + 1][x + 1] = (uint8_t)v;  // only this lane reads/writes pixel i
        }
        wave_sync();
    }
    // ---- chroma, 8.3.4 (H264PictureBase.cpp:2076-2381); DC tests "> 0" (quirk Q1)
    if (CHROMA) {
        int mode = mb.chroma;
        for (int k = 0; k < 2; k++) {
            int i = lane + k * WAVE, c = i >> 6, x = i & 7, y = (i >> 3) & 7;
            const uint8_t (*Cp)[9] = wi->C[c];
            int v;
            if (mode == 0) {
                int xO = x & 4, yO = y & 4;
                int t = av.B() && Cp[0][xO + 1] > 0 && Cp[0][xO + 2] > 0 && Cp[0][xO + 3] > 0 && Cp[0][xO + 4] > 0;
                int l = av.A() && Cp[yO + 1][0] > 0 && Cp[yO + 2][0] > 0 && Cp[yO + 3][0] > 0 && Cp[yO + 4][0] > 0;
                int st = Cp[0][xO + 1] + Cp[0][xO + 2] + Cp[0][xO + 3] + Cp[0][xO + 4];
                int sl = Cp[yO + 1][0] + Cp[yO + 2][0] + Cp[yO + 3][0] + Cp[yO + 4][0];
                if ((xO == 0 && yO == 0) || (xO > 0 && yO > 0)) v = (t && l) ? (st + sl + 4) >> 3 : (l ? (sl + 2) >> 2 : (t ? (st + 2) >> 2 : 128));
                else if (xO > 0) v = t ? (st + 2) >> 2 : (l ? (sl + 2) >> 2 : 128);
                else v = l ? (sl + 2) >> 2 : (t ? (st + 2) >> 2 : 128);
            } else if (mode == 1) {
                v = Cp[y + 1][0];
            } else if (mode == 2) {
                v = Cp[0][x + 1];
            } else {
                int Hs = 0, Vs = 0;
                for (int j = 0; j < 4; j++) {
                    Hs += (j + 1) * (Cp[0][4 + j + 1] - Cp[0][2 - j + 1]);
                    Vs += (j + 1) * (Cp[4 + j + 1][0] - Cp[2 - j + 1][0]);
                }
                int aa = 16 * (Cp[8][0] + Cp[0][8]), bb = (34 * Hs + 32) >> 6, cc = (34 * Vs + 32) >> 6;
                v = clip1((aa + bb * (x - 3) + cc * (y - 3) + 16) >> 5);
            }
            if (res) v = clip1(v + wi->res.rc[c][y * 8 + x]);
            uint8_t *pl = c == 0 ? dcb : dcr;
            pl[(uint64_t)(g.cy + y * st) * wc + mbx * 8 + x] = (uint8_t)v;
        }
    }
    // ---- luma tile -> picture
    for (int k = 0; LUMA && k < 4; k++) {
        int i = lane + k * WAVE, x = i & 15, y = i >> 4;
        dy[(uint64_t)(g.ly + y * st) * wl + mbx * 16 + x] = wi->T[y + 1][x + 1];
    }
    (void)H;
}

// ------------------------------------------------------------ deblocking (8.7)
// What the bS derivation reads of an MB.  Scalar fields only, so that selecting between
// views and per-lane field choices stay in registers.
struct MbView {
    int cls, kind, nz4, nz8;
    uint32_t ref0, ref1;  // reference DPB slot per quadrant q (int8 in byte q), lists 0 / 1
    int pf;
};
__device__ __forceinline__ int view_ref(const MbView &v, int l, int q) { return (int8_t)((l ? v.ref1 : v.ref0) >> (8 * q)); }
__device__ __forceinline__ int dbq_qp(uint32_t q, int plane) { return (q >> (8 * plane)) & 255; }
__device__ __forceinline__ bool dbq_t8(uint32_t q) { return (q >> 24) & 1u; }
// the MB's left / top MB edge lies between slices under disable_deblocking_filter_idc 0:
// its p side takes the MB's own qP (see bs_pair_of_mbs)
constexpr uint32_t DBQ_OWN_LEFT = 1u << 25, DBQ_OWN_TOP = 1u << 26;

__device__ __forceinline__ void load_view(const DevPic &P, int addr, MbView &v) {
    const DevAux ax = G(P.aux)[addr];
    v.cls = G(P.mbs)[addr].mb_type;
    v.kind = ax.kind;
    v.nz4 = ax.nz4;
    v.nz8 = ax.nz8;
    v.pf = ax.pf;
    v.ref0 = (uint32_t)(uint8_t)ax.refid[0][0] | ((uint32_t)(uint8_t)ax.refid[0][1] << 8) |
             ((uint32_t)(uint8_t)ax.refid[0][2] << 16) | ((uint32_t)(uint8_t)ax.refid[0][3] << 24);
    v.ref1 = (uint32_t)(uint8_t)ax.refid[1][0] | ((uint32_t)(uint8_t)ax.refid[1][1] << 8) |
             ((uint32_t)(uint8_t)ax.refid[1][2] << 16) | ((uint32_t)(uint8_t)ax.refid[1][3] << 24);
}
// Deblocking word of an MB (G(P.dbq), written by bs_pair_of_mbs): qP of luma, Cb edges, Cr edges in
// bytes 0..2, transform_size_8x8_flag in bit 24, DBQ_OWN_LEFT / DBQ_OWN_TOP in bits 25, 26.

__device__ __forceinline__ bool mv_far(int ax, int ay, int bx, int by) { return iabs(ax - bx) >= 4 || iabs(ay - by) >= 4; }

// 8.7.2.1 (Deblock.cpp:994-1310) with quirk Q3; I_PCM counts as neither intra nor inter.
__device__ __forceinline__ int bs_luma(const DevPic &P, int ap, const MbView &Pv, int aq, const MbView &Qv, int mb_edge, int xp, int yp, int xq, int yq) {
    bool pin = Pv.kind & AUX_INTRA, qin = Qv.kind & AUX_INTRA;
    if (mb_edge && (pin || qin)) return 4;
    if (pin || qin) return 3;
    int bp4 = 8 * (yp >> 3) + 4 * (xp >> 3) + 2 * ((yp & 7) >> 2) + ((xp & 7) >> 2);
    int bq4 = 8 * (yq >> 3) + 4 * (xq >> 3) + 2 * ((yq & 7) >> 2) + ((xq & 7) >> 2);
    int bp8 = 2 * (yp >> 3) + (xp >> 3), bq8 = 2 * (yq >> 3) + (xq >> 3);
    bool pt8 = Pv.kind & AUX_T8, qt8 = Qv.kind & AUX_T8;
    if ((pt8 && ((Pv.nz8 >> bp8) & 1)) || (!pt8 && ((Pv.nz4 >> bp4) & 1)) ||
        (qt8 && ((Qv.nz8 >> bq8) & 1)) || (!qt8 && ((Qv.nz4 >> bq4) & 1)))
        return 2;
    int qp = 2 * (yp >> 3) + (xp >> 3), qq = 2 * (yq >> 3) + (xq >> 3);
    int rp = (yp >> 2) * 4 + (xp >> 2), rq = (yq >> 2) * 4 + (xq >> 2);
    int p0 = view_ref(Pv, 0, qp), p1 = view_ref(Pv, 1, qp), q0 = view_ref(Qv, 0, qq), q1 = view_ref(Qv, 1, qq);
    int fp0 = (Pv.pf >> qp) & 1, fp1 = (Pv.pf >> (4 + qp)) & 1, fq0 = (Qv.pf >> qq) & 1, fq1 = (Qv.pf >> (4 + qq)) & 1;
    if (!(((p0 == q0 && p1 == q1) || (p0 == q1 && p1 == q0)) && fp0 + fp1 == fq0 + fq1)) return 1;
    const h264g_mb *mp = &G(P.mbs)[ap], *mq = &G(P.mbs)[aq];
    int mp0x = mp->mv[0][rp][0], mp0y = mp->mv[0][rp][1], mp1x = mp->mv[1][rp][0], mp1y = mp->mv[1][rp][1];
    int mq0x = mq->mv[0][rq][0], mq0y = mq->mv[0][rq][1], mq1x = mq->mv[1][rq][0], mq1y = mq->mv[1][rq][1];
    if (fp0 && !fp1 && fq0 && !fq1 && mv_far(mp0x, mp0y, mq0x, mq0y)) return 1;
    if (fp0 && !fp1 && !fq0 && fq1 && mv_far(mp0x, mp0y, mq1x, mq1y)) return 1;
    if (!fp0 && fp1 && fq0 && !fq1 && mv_far(mp1x, mp1y, mq0x, mq0y)) return 1;
    if (!fp0 && fp1 && !fq0 && fq1 && mv_far(mp1x, mp1y, mq1x, mq1y)) return 1;
    if (fp0 && fp1 && p0 != p1 && fq0 && fq1 && ((q0 == p0 && q1 == p1) || (q0 == p1 && q1 == p0))) {
        if (q0 == p0 && (mv_far(mp0x, mp0y, mq0x, mq0y) || mv_far(mp1x, mp1y, mq1x, mq1y))) return 1;
        if (q0 == p1 && (mv_far(mp1x, mp1y, mq0x, mq0y) || mv_far(mp0x, mp0y, mq1x, mq1y))) return 1;
    }
    if (fp0 && fp1 && p0 == p1 && fq0 && fq1 && q0 == q1 && q0 == p0) {
        if (mv_far(mp0x, mp0y, mq0x, mq0y) || (mv_far(mp1x, mp1y, mq1x, mq1y) && mv_far(mp0x, mp0y, mq1x, mq1y)) ||
            mv_far(mp1x, mp1y, mq0x, mq0y))
            return 1;
    }
    return 0;
}

// Tables 8-16 (alpha', beta') and 8-17 (tC0), copied into LDS by every deblocking
// workgroup: lookups with lane-varying indices then cost an LDS read, not a vector
// memory access.
struct DbkTables {
    uint8_t alpha[52], beta[52], tc0[3][52];
};
__device__ void dbk_tables_init(DbkTables *t) {
    for (int i = threadIdx.x; i < 52; i += blockDim.x) {
        t->alpha[i] = c_alpha[i];
        t->beta[i] = c_beta[i];
        t->tc0[0][i] = c_tc0[0][i];
        t->tc0[1][i] = c_tc0[1][i];
        t->tc0[2][i] = c_tc0[2][i];
    }
}

// LDS working set of one deblocking wave, in MB-relative coordinates: luma rows [-4, 15]
// x columns [-16, 15] (the MB and the whole MB to its left), chroma rows [-4, 7] x
// columns [-8, 7].  Rows -4..-1 hold the bottom rows of the MB above.
constexpr int DT_LX = 16, DT_CX = 8;  // tile column of MB column 0 (luma, chroma)
struct alignas(16) WaveDbk {
    uint8_t L[20][32];
    uint8_t C[2][12][16];
};

// Plane pointers of the picture being deblocked.
struct DbkPlanes {
    uint8_t *y, *cb, *cr;
    int wl, wc;
};
__device__ __forceinline__ DbkPlanes dbk_planes(const DevPic &P) {
    DbkPlanes d;
    d.wl = P.W * 16;
    d.wc = P.W * 8;
    d.y = slot_base(P, P.dst);
    d.cb = d.y + (uint64_t)d.wl * (P.H * 16);
    d.cr = d.cb + (uint64_t)d.wc * (P.H * 8);
    return d;
}

// Tile loads.  Region bits: 1 = the MB itself (rows / cols >= 0), 2 = the 4 rows above
// it (cols >= 0), 4 = the 4 columns left of it (rows >= 0).  The corner is never used.
__device__ void dbk_load(const DbkPlanes &d, int mbx, int mby, int region, WaveDbk *wd) {
    const int lane = wave_lane();
    for (int i = lane; i < 400; i += WAVE) {
        const int y = i / 20 - 4, x = i % 20 - 4;
        const int r = (y >= 0 && x >= 0) ? 1 : (y < 0 && x >= 0 ? 2 : (x < 0 && y >= 0 ? 4 : 0));
        if (!(r & region)) continue;
        wd->L[y + 4][x + DT_LX] = d.y[(uint64_t)(mby * 16 + y) * d.wl + mbx * 16 + x];
    }
    for (int i = lane; i < 288; i += WAVE) {
        const int c = i / 144, k = i % 144, y = k / 12 - 4, x = k % 12 - 4;
        const int r = (y >= 0 && x >= 0) ? 1 : (y < 0 && x >= 0 ? 2 : (x < 0 && y >= 0 ? 4 : 0));
        if (!(r & region)) continue;
        const uint8_t *pl = c == 0 ? d.cb : d.cr;
        wd->C[c][y + 4][x + DT_CX] = pl[(uint64_t)(mby * 8 + y) * d.wc + mbx * 8 + x];
    }
}

__device__ __forceinline__ int absdiff(int a, int b) { return (int)__builtin_amdgcn_sad_u16((uint32_t)a, (uint32_t)b, 0u); }
// True when the condition holds on any active lane (the compare's lane mask, no VALU).
__device__ __forceinline__ bool any_lane(bool v) { return __builtin_amdgcn_ballot_w64(v) != 0; }

// Packed 16-bit pairs: the p-side value of a line in the low half, the q-side value in
// the high half.  The p and q sides of 8.7.2.3 / 8.7.2.4 are mirror images, so one packed
// integer operation (v_pk_*_i16) computes both.
typedef short s16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ s16x2 as_pair(uint32_t v) { return __builtin_bit_cast(s16x2, v); }
__device__ __forceinline__ uint32_t as_bits(s16x2 v) { return __builtin_bit_cast(uint32_t, v); }
__device__ __forceinline__ s16x2 pair(int lo, int hi) { return (s16x2){(short)lo, (short)hi}; }
__device__ __forceinline__ s16x2 pair_clip(s16x2 v, s16x2 lo, s16x2 hi) {
    return __builtin_elementwise_min(__builtin_elementwise_max(v, lo), hi);
}
__device__ __forceinline__ s16x2 pair_swap(s16x2 v) { return __builtin_shufflevector(v, v, 1, 0); }
// n where the half's condition holds (hp: p half, hq: q half), else o.
__device__ __forceinline__ s16x2 pair_sel(bool hp, bool hq, s16x2 n, s16x2 o) {
    const uint32_t m = (hp ? 0x0000ffffu : 0u) | (hq ? 0xffff0000u : 0u);
    return as_pair((as_bits(n) & m) | (as_bits(o) & ~m));
}

// Edge J of a line held as 20 bytes in w[0..4] (little-endian; the edge lies between
// words J and J + 1); chroma lines hold 12 bytes and use J = 0, 1 (luma edges 0 and 8
// for the bS).  8.7.2.2 - 8.7.2.4 (Deblock.cpp:1314-1522): alpha = alpha'(indexA), beta =
// beta'(indexB), tc0 = tC0'(bS, indexA) (used for bS 1..3), with indexA / indexB =
// Clip3(0, 51, qPav + filterOffsetA / B).  Every lane takes the same path: the wave skips
// a filter that no lane applies (wave-uniform branches); inside, every candidate value is
// computed on all lanes and chosen per lane with selects, so no per-line condition turns
// into a divergent branch and its exec-mask bookkeeping.  The samples travel as (p, q)
// pairs: P0 = (p0, q0) .. P3 = (p3, q3).
template <int J>
__device__ __forceinline__ void dbk_line_edge(uint32_t (&w)[5], bool act, bool luma, int bS, int alpha, int beta, int tc0) {
    const bool on = act && bS != 0;
    if (!any_lane(on)) return;
    const uint32_t a = w[J], b = w[J + 1];  // a: p3 p2 p1 p0 (bytes 0..3), b: q0 q1 q2 q3
    const s16x2 P0 = as_pair(__builtin_amdgcn_perm(b, a, 0x0c040c03u)), P1 = as_pair(__builtin_amdgcn_perm(b, a, 0x0c050c02u));
    const s16x2 P2 = as_pair(__builtin_amdgcn_perm(b, a, 0x0c060c01u)), P3 = as_pair(__builtin_amdgcn_perm(b, a, 0x0c070c00u));
    const int p0 = P0.x, q0 = P0.y, p1 = P1.x, q1 = P1.y, p2 = P2.x, q2 = P2.y;
    const int d0 = absdiff(p0, q0);
    const bool filt = on & (d0 < alpha) & (absdiff(p1, p0) < beta) & (absdiff(q1, q0) < beta);
    if (!any_lane(filt)) return;
    // ap / aq < beta (8-460, 8-461), only ever used for luma lines
    const bool apl = luma & (absdiff(p2, p0) < beta), aql = luma & (absdiff(q2, q0) < beta);
    s16x2 N0 = P0, N1 = P1, N2 = P2;
    const bool fn = filt & (bS < 4), fs = filt & (bS >= 4);
    const s16x2 X0 = pair_swap(P0), X1 = pair_swap(P1);  // (q0, p0), (q1, p1)
    if (any_lane(fn)) {  // bS < 4 (8.7.2.3)
        const int tc = tc0 + (int)apl + (int)aql + (int)!luma;  // luma tC0 + [ap] + [aq], chroma tC0 + 1
        const int delta = clip3(-tc, tc, (((q0 - p0) << 2) + (p1 - q1) + 4) >> 3);
        const short avg = (short)((p0 + q0 + 1) >> 1);
        // p'0 = Clip1(p0 + delta), q'0 = Clip1(q0 - delta)
        const s16x2 f0 = pair_clip(P0 + pair(delta, -delta), pair(0, 0), pair(255, 255));
        // p'1 = p1 + Clip3(-tC0, tC0, (p2 + avg - 2 p1) >> 1), q'1 alike, kept to 8 bits
        const s16x2 t = (P2 + (s16x2){avg, avg} - (P1 << 1)) >> 1;
        const s16x2 f1 = (P1 + pair_clip(t, pair(-tc0, -tc0), pair(tc0, tc0))) & (s16x2){255, 255};
        N0 = pair_sel(fn, fn, f0, N0);
        N1 = pair_sel(fn & apl, fn & aql, f1, N1);
    }
    if (any_lane(fs)) {  // bS == 4 (8.7.2.4)
        const bool strong = d0 < ((alpha >> 2) + 2);
        const bool sp = fs & apl & strong, sq = fs & aql & strong;
        const s16x2 m = P1 + P0 + X0;                                  // p1 + p0 + q0
        const s16x2 S0 = ((m << 1) + P2 + X1 + (s16x2){4, 4}) >> 3;    // p2 + 2p1 + 2p0 + 2q0 + q1 + 4
        const s16x2 W0 = ((P1 << 1) + P0 + X1 + (s16x2){2, 2}) >> 2;   // 2p1 + p0 + q1 + 2
        const s16x2 S1 = (m + P2 + (s16x2){2, 2}) >> 2;                // p2 + p1 + p0 + q0 + 2
        const s16x2 S2 = ((P3 << 1) + P2 * (s16x2){3, 3} + m + (s16x2){4, 4}) >> 3;  // 2p3 + 3p2 + p1 + p0 + q0 + 4
        N0 = pair_sel(sp, sq, S0, pair_sel(fs, fs, W0, N0));
        N1 = pair_sel(sp, sq, S1, N1);
        N2 = pair_sel(sp, sq, S2, N2);
    }
    // back to bytes: t01 = np0 np1 nq0 nq1, u = np0 np1 np2 nq2
    const uint32_t t01 = __builtin_amdgcn_perm(as_bits(N1), as_bits(N0), 0x06020400u);
    const uint32_t u = __builtin_amdgcn_perm(as_bits(N2), t01, 0x06040100u);
    w[J] = __builtin_amdgcn_perm(u, a, 0x04050600u);                                                  // p3 np2 np1 np0
    w[J + 1] = __builtin_amdgcn_perm(b, __builtin_amdgcn_perm(u, t01, 0x0c070302u), 0x07020100u);   // nq0 nq1 nq2 q3
}

// The edges of one direction (DIR 0: vertical edges, 1: horizontal) of the MB in the
// tile.  Lanes 0-15 take luma, 16-23 Cb, 24-31 Cr; lane k of a plane owns line k of the
// MB (a row for vertical edges, a column for horizontal ones) with the 4 samples before
// it, keeps the line in registers and runs its edges in order: left / top MB edge (when
// `edge`), then the internal ones (luma 4 / 12 skipped with the 8x8 transform, chroma
// only 4).  Lines of one direction touch disjoint samples, so this gives the reference's
// edge-by-edge order (8.7, Deblock.cpp:76-635).  qq / eq: deblocking words (see bs_pair_of_mbs) of
// the MB and of the left / top MB.
// cur: tile column of the MB's luma column 0 (16 or 0; chroma cur / 2); the left MB sits
// in the other half of the tile, so a row's columns -4..-1 are at (16 - cur) + 12.
template <int DIR>
__device__ __forceinline__ void dbk_lines(const DevPic &P, uint32_t eq, bool edge, uint32_t qq,
                                          const uint8_t *bsrec, WaveDbk *wd, const DbkTables *tb, int cur) {
    const int lane = wave_lane();
    if (lane >= 32) return;
    const int plane = lane < 16 ? 0 : (lane < 24 ? 1 : 2);
    const bool luma = plane == 0;
    const int k = luma ? lane : (lane & 7);
    // tile row 0 of the plane; the MB's columns start at mc, the left MB's columns -4..-1 at lc
    uint8_t *base = luma ? &wd->L[0][0] : &wd->C[plane - 1][0][0];
    const int stride = luma ? 32 : 16, mc = luma ? cur : cur >> 1, lc = luma ? 28 - cur : 12 - (cur >> 1);
    uint32_t w[5];
    if (DIR == 0) {
        uint8_t *row = base + (k + 4) * stride;
        w[0] = *(const uint32_t *)(row + lc);
        w[1] = *(const uint32_t *)(row + mc);
        w[2] = *(const uint32_t *)(row + mc + 4);
        w[3] = luma ? *(const uint32_t *)(row + mc + 8) : 0u;
        w[4] = luma ? *(const uint32_t *)(row + mc + 12) : 0u;
    } else {
        // the quad of lanes that owns columns 4m..4m+3 reads rows 4i..4i+3 of them as dwords
        // (its lane j row 4i + j) and transposes them into the four columns; quads never
        // mix planes, so a quad agrees on `luma`
        const uint8_t *c = base + mc + (k & ~3) + (k & 3) * stride;
#pragma unroll
        for (int i = 0; i < 5; i++)
            w[i] = quad_transpose_bytes((i < 3 || luma) ? *(const uint32_t *)(c + 4 * i * stride) : 0u, k & 3);
    }
    const bool own = qq & (DIR == 0 ? DBQ_OWN_LEFT : DBQ_OWN_TOP);
    const int qpq = dbq_qp(qq, plane), qpe = edge && !own ? dbq_qp(eq, plane) : qpq;
    const int qav = (qpe + qpq + 1) >> 1;  // internal edges: (qpq + qpq + 1) >> 1 = qpq
    const int iA0 = clip3(0, 51, qav + P.offA), iB0 = clip3(0, 51, qav + P.offB);
    const int iAi = clip3(0, 51, qpq + P.offA), iBi = clip3(0, 51, qpq + P.offB);
    const bool t8 = dbq_t8(qq), on = P.dbk_idc != 1;
    const int seg = luma ? (k >> 2) : (k >> 1);  // 4-line luma segment of the line
    // bS of this segment's edges 0..3 (stored [direction][segment][edge]); chroma
    // edge j lies on luma edge 2j.  All table lookups are issued before the filtering.
    const uint32_t bsv = *(const uint32_t *)&bsrec[DIR * 16 + seg * 4];
    const int bs0 = bsv & 255u, bs1 = luma ? (bsv >> 8) & 255u : (bsv >> 16) & 255u, bs2 = (bsv >> 16) & 255u,
              bs3 = bsv >> 24;
    int a0 = tb->alpha[iA0], b0 = tb->beta[iB0], ai = tb->alpha[iAi], bi = tb->beta[iBi];
    int t0 = tb->tc0[bs0 >= 1 && bs0 <= 3 ? bs0 - 1 : 0][iA0], t1 = tb->tc0[bs1 >= 1 && bs1 <= 3 ? bs1 - 1 : 0][iAi];
    int t2 = tb->tc0[bs2 >= 1 && bs2 <= 3 ? bs2 - 1 : 0][iAi], t3 = tb->tc0[bs3 >= 1 && bs3 <= 3 ? bs3 - 1 : 0][iAi];
    // one LDS round trip for the eight lookups: without this the compiler moves each into
    // the edge that first uses it and waits on it there
    asm volatile("" : "+v"(a0), "+v"(b0), "+v"(ai), "+v"(bi), "+v"(t0), "+v"(t1), "+v"(t2), "+v"(t3));
    dbk_line_edge<0>(w, on && edge, luma, bs0, a0, b0, t0);
    dbk_line_edge<1>(w, on && (luma ? !t8 : true), luma, bs1, ai, bi, t1);
    dbk_line_edge<2>(w, on && luma, luma, bs2, ai, bi, t2);
    dbk_line_edge<3>(w, on && luma && !t8, luma, bs3, ai, bi, t3);
    if (DIR == 0) {
        uint8_t *row = base + (k + 4) * stride;
        *(uint32_t *)(row + lc) = w[0];
        *(uint32_t *)(row + mc) = w[1];
        *(uint32_t *)(row + mc + 4) = w[2];
        if (luma) {
            *(uint32_t *)(row + mc + 8) = w[3];
            *(uint32_t *)(row + mc + 12) = w[4];
        }
    } else {
        // back to rows (the first and last row, p3 / q3 of the outer edges, keep their values)
        uint8_t *c = base + mc + (k & ~3) + (k & 3) * stride;
#pragma unroll
        for (int i = 0; i < 5; i++) {
            const uint32_t v = quad_transpose_bytes(w[i], k & 3);
            if (i < 3 || luma) *(uint32_t *)(c + 4 * i * stride) = v;
        }
    }
}

// The MB's vertical edges, then its horizontal edges, on the tile (8.7, Deblock.cpp:76-635).
// lq / tq are the deblocking words of the left / top MB (read only when present).  bsrec: the MB's 32
// boundary strengths (device memory or an LDS copy).  The caller has synchronised the
// tile; it is complete when this returns.
__device__ __forceinline__ void dbk_filter(const DevPic &P, uint32_t qq, uint32_t lq, uint32_t tq, bool left, bool top,
                           const uint8_t *bsrec, WaveDbk *wd, const DbkTables *tb) {
    dbk_lines<0>(P, lq, left, qq, bsrec, wd, tb, DT_LX);
    wave_sync();
    dbk_lines<1>(P, tq, top, qq, bsrec, wd, tb, DT_LX);
    wave_sync();
}

// Writes back the MB and the strips its MB edges modified (3 columns / rows).
__device__ void dbk_store(const DbkPlanes &d, int mbx, int mby, bool left, bool top, const WaveDbk *wd) {
    const int lane = wave_lane();
    for (int i = lane; i < 400; i += WAVE) {
        int y = i / 20 - 4, x = i % 20 - 4;
        if (x < -3 || y < -3 || (x < 0 && y < 0) || (x < 0 && !left) || (y < 0 && !top)) continue;
        d.y[(uint64_t)(mby * 16 + y) * d.wl + mbx * 16 + x] = wd->L[y + 4][x + DT_LX];
    }
    for (int i = lane; i < 288; i += WAVE) {
        int c = i / 144, k = i % 144, y = k / 12 - 4, x = k % 12 - 4;
        if (x < -3 || y < -3 || (x < 0 && y < 0) || (x < 0 && !left) || (y < 0 && !top)) continue;
        uint8_t *pl = c == 0 ? d.cb : d.cr;
        pl[(uint64_t)(mby * 8 + y) * d.wc + mbx * 8 + x] = wd->C[c][y + 4][x + DT_CX];
    }
}

// One MB with every neighbour sample loaded from the picture (per-MB wavefront).
__device__ void deblock_mb(const DevPic &P, int addr, WaveDbk *wd, const DbkTables *tb) {
    const int W = P.W;
    const int mbx = addr % W, mby = addr / W;
    const DbkPlanes d = dbk_planes(P);
    const bool left = mbx > 0, top = mby > 0;
    dbk_load(d, mbx, mby, 1 | (top ? 2 : 0) | (left ? 4 : 0), wd);
    const uint32_t qq = G(P.dbq)[addr], lq = left ? G(P.dbq)[addr - 1] : 0u, tq = top ? G(P.dbq)[addr - W] : 0u;
    wave_sync();
    dbk_filter(P, qq, lq, tq, left, top, G(P.bs) + (size_t)addr * 32, wd, tb);
    dbk_store(d, mbx, mby, left, top, wd);
}

// After MB x of a row: its columns 12..15 become the left columns of MB x + 1.
__device__ void dbk_carry_left(WaveDbk *wd) {
    const int lane = wave_lane();
    wave_sync();
    for (int i = lane; i < 16 * 4 + 2 * 8 * 4; i += WAVE) {
        if (i < 64) {
            const int y = i >> 2, x = i & 3;
            wd->L[y + 4][DT_LX - 4 + x] = wd->L[y + 4][DT_LX + 12 + x];
        } else {
            const int k = i - 64, c = k >> 5, y = (k >> 2) & 7, x = k & 3;
            wd->C[c][y + 4][DT_CX - 4 + x] = wd->C[c][y + 4][DT_CX + 4 + x];
        }
    }
    wave_sync();
}

__device__ __forceinline__ uint64_t ld_acquire64(const uint64_t *p) {
    return __hip_atomic_load(p, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT);
}

// Waits until row progress word *w >= want (epoch-tagged: epoch << 32 | MBs done).
__device__ void wait_row(const uint64_t *w, uint64_t want, uint32_t *err) {
    for (uint32_t it = 0;; ++it) {
        const uint64_t v = ld_acquire64(w);
        const uint32_t lo = uniform((uint32_t)v), hi = uniform((uint32_t)(v >> 32));
        if ((((uint64_t)hi << 32) | lo) >= want) break;
        if (it >= SPIN_LIMIT) {
            report_timeout(err);
            break;
        }
        if ((it & 255u) == 255u && uniform(__hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) != 0u) break;
        __builtin_amdgcn_s_sleep(1);
    }
    __atomic_thread_fence(__ATOMIC_ACQUIRE);
}

// Row progress across CUs: epoch-tagged 64-bit words in global memory (agent scope).
struct RowSyncGlobal {
    GAS uint64_t *prog;
    uint64_t tag;
    uint32_t *err;
    __device__ void wait(int row, int need) { wait_row(&prog[row], tag | (uint32_t)need, err); }
    __device__ void post(int row, int done) {
        wave_sync();  // every lane's stores before the (wave-wide) release store
        __hip_atomic_store(&prog[row], tag | (uint32_t)done, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
    }
};

constexpr uint32_t LDS_SPIN_LIMIT = 1u << 22;
// One whole MB row, left to right, in raster order.  MB (x, y) needs MB (x + 1, y - 1)
// done (its left-edge filter changed columns 13..15 of (x, y - 1), which (x, y)'s top
// edge reads), i.e. the row above at progress min(x + 2, W).  The left neighbour's
// columns stay in LDS from the previous step.
template <class Sync>
__device__ void deblock_row(const DevPic &P, int mby, Sync &sync, WaveDbk *wd, const DbkTables *tb) {
    const int W = P.W;
    const DbkPlanes d = dbk_planes(P);
    const bool top = mby > 0;
    uint32_t lq = 0u, qq = 0u, tq = 0u;
    for (int mbx = 0; mbx < W; mbx++) {
        const int addr = mby * W + mbx;
        const bool left = mbx > 0;
        dbk_load(d, mbx, mby, 1, wd);  // the MB's own samples: final before this launch
        lq = qq;
        qq = G(P.dbq)[addr];
        if (top) {
            tq = G(P.dbq)[addr - W];
            sync.wait(mby - 1, min(mbx + 2, W));
            dbk_load(d, mbx, mby, 2, wd);
        }
        wave_sync();
        dbk_filter(P, qq, lq, tq, left, top, G(P.bs) + (size_t)addr * 32, wd, tb);
        dbk_store(d, mbx, mby, left, top, wd);
        sync.post(mby, mbx + 1);
        dbk_carry_left(wd);
    }
}

// ------------------------------------------------------------ kernels
// The LDS working sets are per wave and the per-MB code synchronises with wave barriers,
// so a workgroup may hold one wave (most kernels) or several (the band kernels).
// Workgroups are dispatched to the 8 XCDs round-robin (workgroup b on XCD b mod 8), each
// XCD with its own L2.  Item of workgroup b (of n, one item each) such that every XCD
// takes one contiguous run of items: neighbouring MBs then share that XCD's L2 for
// their overlapping reference lines and for the cache lines their rows share.
constexpr uint32_t N_XCD = 8;
__device__ __forceinline__ uint32_t xcd_item(uint32_t b, uint32_t n) {
    const uint32_t x = b % N_XCD, q = n / N_XCD, r = n % N_XCD;
    return x * q + min(x, r) + b / N_XCD;
}

// The MBs of a launch's pictures in runs of MB_CHUNK of one picture: run i starts at MB
// chunks[i] (picture index << 20 | address), or, without a list, at MB i * MB_CHUNK of picture 0.
// Slot s of the launch is MB s mod MB_CHUNK of run s / MB_CHUNK; a picture's last run may go
// past its last MB.
struct MbSlot {
    uint32_t pic;
    int addr;
};
__device__ __forceinline__ MbSlot mb_slot(const uint32_t *chunks, uint32_t s) {
    const uint32_t c = s / MB_CHUNK, it = chunks ? chunks[c] : c * MB_CHUNK;
    return {it >> WI_PIC_SHIFT, (int)((it & WI_MB_MASK) + s % MB_CHUNK)};
}

// One wave per MB: inter (and I_PCM) MBs are reconstructed, intra MBs get their residual and
// their entry built for the intra stage.
// MBAFF: the instance for MBAFF frames (field MBs: geometry, field scans, field references);
// frame pictures run the instance without any of it.
// Blocks from n on derive boundary strengths, which depend on the records alone: in a launch of
// their own they cost a chain of CIF P pictures 3 of 59 us each, one of 1280x720 4 of 164.
__device__ void bs_pair_of_mbs(const DevPic *pics, const uint32_t *chunks, uint32_t b, uint32_t n);
__device__ void bs_mbaff_mb(const DevPic *pics, const uint32_t *chunks, uint32_t b, uint32_t n);
template <bool MBAFF, bool SCALED>
__global__ __launch_bounds__(WAVE) void k_inter(const DevPic *__restrict__ pics, const uint32_t *__restrict__ chunks, uint32_t n) {
    __shared__ WaveRes lds;
    if (blockIdx.x >= n) {
        if (MBAFF) bs_mbaff_mb(pics, chunks, blockIdx.x - n, gridDim.x - n);
        else bs_pair_of_mbs(pics, chunks, blockIdx.x - n, gridDim.x - n);
        return;
    }
    const MbSlot m = mb_slot(chunks, xcd_item(blockIdx.x, n));
    const DevPic &P = pics[m.pic];
    if (m.addr >= P.W * P.H) return;
    if (!(uniform(G(P.aux)[m.addr].kind) & AUX_INTRA)) inter_mb<MBAFF, SCALED>(P, m.addr, &lds);
    else intra_res_build<MBAFF, SCALED>(P, m.addr, &lds);
}

// Neighbour availability of an intra MB for intra prediction (6.4.11, with
// constrained_intra_pred_flag); deps[k] = address of neighbour k (A, B, C, D) when it is
// itself intra-predicted in this picture (its samples come from the intra stage) and its
// samples are read, else -1.
__device__ __forceinline__ Avail intra_avail(const DevPic &P, int addr, int deps[4]) {
    const int W = P.W, mbx = addr % W, mby = addr / W;
    Avail av;
    av.m = (mbx > 0 ? 1u : 0u) | (mby > 0 ? 2u : 0u) | (mby > 0 && mbx < W - 1 ? 4u : 0u) | (mbx > 0 && mby > 0 ? 8u : 0u);
    const int nb[4] = {addr - 1, addr - W, addr - W + 1, addr - W - 1};
#pragma unroll
    for (int k = 0; k < 4; k++) {
        deps[k] = -1;
        if (!(av.m & (1u << k))) continue;
        const int c = G(P.mbs)[nb[k]].mb_type;
        if (P.multi_slice && G(P.mbs)[nb[k]].slice_num != G(P.mbs)[addr].slice_num) {  // another slice (6.4.8)
            av.m &= ~(1u << k);
            continue;
        }
        if (P.cip && cip_hides(G(P.mbs)[nb[k]])) av.m &= ~(1u << k);
        if (cls_intra(c)) deps[k] = nb[k];
    }
    // Samples of C (above right) are read only by Intra_8x8 (the top reference samples
    // p[8..15, -1] of block 1 and their filtering, 8.3.2.2) and by Intra_4x4 block 5 in
    // the modes that use p[4..7, -1] (Diagonal_Down_Left 3, Vertical_Left 7); without
    // them the MB does not wait for C.
    const h264g_mb &m = G(P.mbs)[addr];
    const bool uses_c = m.mb_type == H264G_MB_I8x8 ||
                        (m.mb_type == H264G_MB_I4x4 && (m.intra_pred_modes[5] == 3 || m.intra_pred_modes[5] == 7));
    if (!uses_c) deps[2] = -1;
    return av;
}

// The same for an MB of an MBAFF frame (6.4.10 / Table 6-4; no constrained intra):
// availability of the samples left (A), above (B), above right (C) and above left (D) of
// the MB's view.  A frame MB at the bottom of its pair reads its top MB above it and the
// left pair above left, and has no C; every other MB reads the pairs around its own.
__device__ __forceinline__ Avail intra_avail_mbaff(const DevPic &P, int addr) {
    const int W = P.W, pair = addr >> 1, px = pair % W, py = pair / W, bot = addr & 1;
    const bool field = (G(P.mbs)[addr].flags & H264G_MBF_FIELD) != 0, in_pair = !field && bot;
    const bool A = px > 0, B = py > 0, C = py > 0 && px < W - 1, D = py > 0 && px > 0;
    Avail av;
    av.m = (A ? 1u : 0u) | ((in_pair || B) ? 2u : 0u) | (!in_pair && C ? 4u : 0u) | ((in_pair ? A : D) ? 8u : 0u);
    return av;
}

__global__ __launch_bounds__(WAVE) void k_intra(const DevPic *__restrict__ pics, const uint32_t *__restrict__ items, uint32_t n,
                                                DevCtl *ctl, uint32_t *epoch_p, uint32_t *err) {
    __shared__ WaveIntra lds;
    const uint32_t epoch = launch_epoch(epoch_p);
    for (;;) {
        int t = next_ticket(ctl, n);
        if (t < 0) break;
        const uint32_t it = items[t];
        const DevPic &P = pics[it >> WI_PIC_SHIFT];
        const int addr = (int)(it & WI_MB_MASK);
        int deps[4];
        const Avail av = intra_avail(P, addr, deps);
        const IntraRes r = intra_res_fetch(P, addr);
        if (G(P.mbs)[addr].mb_type == H264G_MB_I4x4) intra4_prep(&G(P.mbs)[addr], av, &lds);
        else if (G(P.mbs)[addr].mb_type == H264G_MB_I8x8) intra8_prep(&G(P.mbs)[addr], av, &lds);
        wait_deps(G(P.flags), deps, 4, epoch, err);
        intra_res_place(r, &lds);
        const GAS h264g_mb &m = G(P.mbs)[addr];
        intra_mb<3>(P, mb_geo<false>(P, addr), {m.mb_type, m.intra16x16_pred_mode, m.intra_chroma_pred_mode}, &lds, av, r.res);
        publish(&G(P.flags)[addr], epoch);
    }
    retire(ctl, gridDim.x, epoch_p, epoch);
}

// ---- bands of MB rows
// A band is consecutive MB rows of one picture, on one workgroup for luma and one for chroma.
// Inside the workgroup the rows hand samples on through LDS.  A band's last row hands what
// the next band's first row reads (in another workgroup, possibly on another XCD) through
// device memory as epoch-tagged 64-bit words, one agent-scope atomic each: the reader polls
// the words themselves, and no agent-scope release / acquire (an L2 write-back or
// invalidation of the whole XCD) is issued.  Work items are (picture, band) in band-major
// order and a workgroup takes its item by ticket when it starts, so the band above always
// belongs to a workgroup that started earlier and never waits on a later one.

// Takes the workgroup's ticket (into *slot) and clears `n` LDS counters.
__device__ __forceinline__ uint32_t band_ticket(DevCtl *ctl, uint32_t *slot, uint32_t *ctr, int n) {
    if (threadIdx.x == 0) *slot = atomicAdd(&ctl->ticket, 1u);
    if ((int)threadIdx.x < n) ctr[threadIdx.x] = 0;
    __syncthreads();
    return uniform(*slot);
}
// Every wave of the workgroup is done: the launch's last workgroup resets the control
// block and advances the epoch (see retire).
__device__ __forceinline__ void band_retire(DevCtl *ctl, uint32_t *epoch, uint32_t cur) {
    __syncthreads();
    if (threadIdx.x == 0) {
        const uint32_t d = atomicAdd(&ctl->done, 1u);
        if (d == gridDim.x - 1) {
            __hip_atomic_store(&ctl->ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(&ctl->done, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(epoch, cur + 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
}
__device__ __forceinline__ uint32_t lds_peek(const uint32_t *w) {
    return __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
// Waits until *w >= need; seen: a value of *w read before.
__device__ __forceinline__ void lds_wait(const uint32_t *w, uint32_t seen, uint32_t need, uint32_t *err) {
    uint32_t v = uniform(seen);
#pragma unroll 1
    for (uint32_t it = 0; v < need; ++it) {
        if (it >= LDS_SPIN_LIMIT) {
            report_timeout(err);
            break;
        }
        if ((it & 1023u) == 1023u && uniform(__hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) != 0u) break;
        if (it) __builtin_amdgcn_s_sleep(1);
        v = uniform(lds_peek(w));
    }
    wave_sync();
}
// Publishes the wave's earlier LDS accesses: one wave's LDS instructions take effect in
// order, so a counter written after them is seen after them, without a wait.
__device__ __forceinline__ void lds_post(uint32_t *w, uint32_t v) {
    wave_sync();
    __hip_atomic_store(w, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// ---- intra prediction over bands: one wave per MB row and plane type
// A band of R MB rows runs on two workgroups, one for luma and one for chroma, whose chains
// never meet: a wave per MB row walks the row's intra MBs, and one wave brings in what the
// band above hands down (istrip_reader).
//
// Bound: the chain through the MBs of an intra picture, W + 1.5 H of them (an MB follows its
// left neighbour and the one above, or above right when it reads it).  What a step of the
// chain costs is LDS round trips and instructions, so everything that does not depend on
// neighbouring samples is off it: the MB's entry (DevPic::imeta), its residual and the
// samples of its inter neighbours (final before this launch) are loaded one MB ahead, the
// tap addresses of every sample come from tables in LDS; samples of intra neighbours never
// travel through device memory inside a band: the MB to the left stays in the tile, the MBs
// above leave their bottom rows in a ring of RING_COLS columns in LDS.  Stores go out one MB
// late, before the next loads, so that no load waits behind them.
// Measured (whole launch, one picture; before: luma and chroma of a row in one wave, which
// took its neighbours from device memory and found its taps inside the chain): I pictures
// 352x288 364 to 72 us, 1920x1088 1866 to 340, 3840x2160 3820 to 682; P pictures (10 % intra
// MBs) 1920x1088 118 to 26 us, 3840x2160 184 to 37.
constexpr int RING_COLS = 64;
constexpr int IT_S = 36, IT_0 = 4;   // luma tile: bytes per row, byte of column 0 (row -1 first)
constexpr int CT_S = 12, CT_0 = 4;   // chroma tile
constexpr uint32_t NO_COL = 0x7FFFFFFFu;

// Byte offset of neighbour-line sample X[i] (i4_taps: L3 L3 L2 L1 L0 TL T0 .. T7 T7) from the
// block's first sample, plus TAP_0 so that it is never negative.
constexpr int TAP_0 = IT_S + 1;
constexpr int x_off(int i, bool tr) {
    if (i < 5) return TAP_0 + (i == 0 ? 3 : 4 - i) * IT_S - 1;
    if (i == 5) return 0;
    const int t = i == 14 ? 7 : i - 6;
    return TAP_0 - IT_S + (t > 3 && !tr ? 3 : t);
}
// Taps of the 16 samples of a 4x4 block as 4 byte offsets; modes 3 and 7 with the top-right
// samples not available (T4..T7 <- T3) are entries 9 and 10; DC reads T0..T3.
struct Tap4Tab {
    uint32_t v[11][16];
};
constexpr Tap4Tab make_tap4() {
    Tap4Tab t{};
    for (int m = 0; m < 11; m++)
        for (int k = 0; k < 16; k++) {
            const int mode = m == 9 ? 3 : m == 10 ? 7 : m;
            uint32_t v = 0;
            for (int i = 0; i < 4; i++) {
                const int x = mode == 2 ? 6 + i : (i4_taps(mode, k & 3, k >> 2) >> (4 * i)) & 15;
                v |= (uint32_t)x_off(x, m < 9) << (8 * i);
            }
            t.v[m][k] = v;
        }
    return t;
}
__constant__ Tap4Tab c_tap4 = make_tap4();
// Intra_8x8: the filtered reference samples stand as L'0..7, T'0..15, TL' in 25 bytes (pf_at:
// from the index of i8_taps); taps as 4 byte indices.
constexpr int pf_at(int i) { return i == 0 ? 24 : i < 9 ? i - 1 : i - 1; }
struct Tap8Tab {
    uint32_t v[9][64];
};
constexpr Tap8Tab make_tap8() {
    Tap8Tab t{};
    for (int m = 0; m < 9; m++)
        for (int k = 0; k < 64; k++) {
            uint32_t v = 0;
            for (int i = 0; i < 4; i++) v |= (uint32_t)(m == 2 ? 0 : pf_at((i8_taps(m, k & 7, k >> 3) >> (5 * i)) & 31)) << (8 * i);
            t.v[m][k] = v;
        }
    return t;
}
__constant__ Tap8Tab c_tap8 = make_tap8();
// 8.3.2.2.1 (H264PictureBase.cpp:1535-1599): every filtered reference sample is (a + 2 b + c + 2)
// >> 2 of three reference samples; at the ends, and beside samples that are not available, a
// sample repeats.  Entry of filtered sample i (bytes as above) in variant tl | tr << 1 (top-left /
// top-right samples available), 10 bits each: byte offsets plus TAP_0.
struct Flt8Tab {
    uint32_t v[4][25];
};
constexpr Flt8Tab make_flt8() {
    Flt8Tab t{};
    for (int q = 0; q < 4; q++) {
        const bool tl = q & 1, tr = q & 2;
        for (int i = 0; i < 25; i++) {
            int a = 0, b = 0, c = 0;  // offsets of L_y: L(y), T_x: T(x), TL: 0
            auto L = [](int y) { return TAP_0 + y * IT_S - 1; };
            auto T = [&](int x) { return TAP_0 - IT_S + (x > 7 && !tr ? 7 : x); };
            if (i < 8) {
                a = i == 0 ? (tl ? 0 : L(0)) : L(i - 1);
                b = L(i);
                c = i == 7 ? L(7) : L(i + 1);
            } else if (i < 24) {
                const int x = i - 8;
                a = x == 0 ? (tl ? 0 : T(0)) : T(x - 1);
                b = T(x);
                c = x == 15 ? T(15) : T(x + 1);
            } else {
                a = T(0); b = 0; c = L(0);
            }
            t.v[q][i] = (uint32_t)(a | b << 10 | c << 20);
        }
    }
    return t;
}
__constant__ Flt8Tab c_flt8 = make_flt8();

struct alignas(16) IntraLumaTile {
    // row -1, then the MB's rows; column -1 at byte IT_0 - 1 (both arrays longer than the MB:
    // lanes without a block in a 4x4 step read past it)
    uint8_t t[21 * IT_S];
    alignas(16) int16_t res[320];
    alignas(16) uint8_t pf[32];
};
struct alignas(16) IntraChromaTile {
    uint8_t t[2][9 * CT_S];
};
struct IntraWgShared {
    union {
        IntraLumaTile l[H264G_INTRA_MAX_ROWS];
        IntraChromaTile c[H264G_INTRA_MAX_ROWS];
    };
    // bottom rows of the intra MBs of the row above row w (luma 16 bytes; chroma Cb 8, Cr 8), MB
    // column x in slot x mod RING_COLS
    alignas(16) uint8_t ring[H264G_INTRA_MAX_ROWS][RING_COLS][16];
    uint32_t prog[H264G_INTRA_MAX_ROWS];   // that row's intra MBs in columns below prog are done
    uint32_t cons[H264G_INTRA_MAX_ROWS];   // row w reads no column below cons any more
    Tap4Tab tap4;
    Tap8Tab tap8;
    Flt8Tab flt8;
};

// The band above's strips (one row of W x 8 words: luma 0..3, chroma 4..7 of each MB) into ring
// 0, for the intra MBs of its last row, whose entries are col[b .. e - 1]; 16 MBs at a time.
__device__ __forceinline__ void istrip_reader(const GAS uint64_t *sw, const GAS uint32_t *col, uint32_t b, uint32_t e, int W,
                                              IntraWgShared &sh, int at, uint32_t epoch, uint32_t *err) {
    constexpr int N = 4, AT_ONCE = WAVE / N;
    const int lane = wave_lane(), mine = lane / N, word = lane % N;
    lds_post(&sh.prog[0], b < e ? uniform(col[b]) & ICOL_X_MASK : (uint32_t)W);
    for (uint32_t i0 = b; i0 < e; i0 += AT_ONCE) {
        const int n = (int)min((uint32_t)AT_ONCE, e - i0);
        const uint32_t x = col[i0 + (uint32_t)min(mine, n - 1)] & ICOL_X_MASK;   // this lane's MB column
        const uint32_t nx = i0 + n < e ? uniform(col[i0 + n]) & ICOL_X_MASK : (uint32_t)W;
        int have = 0;
#pragma unroll 1
        for (uint32_t it = 0; have < n; ++it) {
            const uint64_t r = __hip_atomic_load(&sw[(size_t)x * 8 + at + word], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            // (columns taken together span less than the ring, so that the row below can always
            // get to the point where it frees the last one's slot)
            const uint32_t xf = (uint32_t)__builtin_amdgcn_readlane((int)x, N * have);
            const uint64_t missing = __builtin_amdgcn_ballot_w64((uint32_t)(r >> 32) != epoch || x >= xf + RING_COLS / 2);
            const int got = missing ? min(n, (int)(__builtin_ctzll(missing) / N)) : n;
            if (got > have) {
                // the last column taken now: its slot's previous MB has been read
                const uint32_t xl = (uint32_t)__builtin_amdgcn_readlane((int)x, N * (got - 1));
                if (xl >= (uint32_t)RING_COLS) lds_wait(&sh.cons[0], 0u, xl - RING_COLS + 1, err);
                if (mine >= have && mine < got) *(uint32_t *)&sh.ring[0][x % RING_COLS][4 * word] = (uint32_t)r;
                lds_post(&sh.prog[0], got < n ? (uint32_t)__builtin_amdgcn_readlane((int)x, N * got) : nx);
                have = got;
                continue;
            }
            if (it >= SPIN_LIMIT) {
                report_timeout(err);
                return;
            }
            if ((it & 255u) == 255u && uniform(__hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) != 0u) return;
            __builtin_amdgcn_s_sleep(1);
        }
    }
}

// Sum of v over the wave's 16-lane rows 0 and 1 (lanes 0-31); the result is uniform.
__device__ __forceinline__ int sum32(int v) {
    v += __builtin_amdgcn_mov_dpp(v, 0x128, 0xF, 0xF, true);   // row_ror:8
    v += __builtin_amdgcn_mov_dpp(v, 0x124, 0xF, 0xF, true);   // row_ror:4
    v += __builtin_amdgcn_mov_dpp(v, 0x122, 0xF, 0xF, true);   // row_ror:2
    v += __builtin_amdgcn_mov_dpp(v, 0x121, 0xF, 0xF, true);   // row_ror:1
    return __builtin_amdgcn_readlane(v, 0) + __builtin_amdgcn_readlane(v, 16);
}
__device__ __forceinline__ uint32_t byte_of(uint32_t v, int i) { return (v >> (8 * i)) & 255u; }

// What a row's wave loads ahead for one MB: its entry, then (with the entry) its residual and
// the sample of the lane's neighbour position.
struct IntraAhead {
    uint4 meta;
    uint2 res;
    uint32_t nb;
};
__device__ __forceinline__ uint4 imeta_load(const GAS uint4 *m, uint32_t i, uint32_t e) { return m[min(i, e - 1)]; }

// The luma plane of MB row y = y0 + w of a band; the row is handed down through ring w + 1 (ring_out)
// or, by the band's last row, the strips `gout` (g_out).
__device__ __forceinline__ void intra_luma_row(const DevPic &P, int w, int y, bool ring_out, bool g_out, GAS uint64_t *gout,
                                               IntraWgShared &sh, uint32_t epoch, uint32_t *err) {
    const int W = P.W, lane = wave_lane();
    const GAS uint32_t *const off = G(P.irow);
    const GAS uint4 *const meta = (const GAS uint4 *)G(P.imeta);
    const uint32_t b = uniform(off[y]), e = uniform(off[y + 1]);
    IntraLumaTile *const tile = &sh.l[w];
    uint8_t *const T = tile->t;
    const uint8_t *const rin = &sh.ring[w][0][0];
    if (b == e) {
        if (ring_out) lds_post(&sh.prog[w + 1], (uint32_t)W);
        lds_post(&sh.cons[w], NO_COL);
        return;
    }
    gu8 *const slot = slot_base(P, P.dst);
    const uint32_t pitch = (uint32_t)W * 16u, row0 = (uint32_t)(y * 16) * pitch;
    const GAS int16_t *const ires = G(P.ires);
    // the lane's neighbour position: lanes 0-24 row -1, column lane - 1; lanes 32-47 column -1, row
    // lane - 32; its neighbour's bit (A 1, B 2, C 4, D 8)
    const bool topl = lane < 25, leftl = lane >= 32 && lane < 48;
    const uint32_t nbit = topl ? (lane == 0 ? 8u : lane < 17 ? 2u : 4u) : leftl ? 1u : 0u;
    uint8_t *const nb_at = T + (topl ? IT_0 - 1 + lane : leftl ? (lane - 31) * IT_S + IT_0 - 1 : 0);
    const uint32_t nb_row = (uint32_t)(topl ? max(y * 16 - 1, 0) : y * 16 + (leftl ? lane - 32 : 0)) * pitch;
    const int nb_dx = topl ? lane - 1 : -1;
    auto load_nb = [&](uint32_t ent) -> uint32_t {
        const int x = (int)(ent & ICOL_X_MASK);
        return slot[nb_row + (uint32_t)clip3(0, W * 16 - 1, x * 16 + nb_dx)];
    };
    // lanes of the 4x4 wavefront: block g of a step, sample j
    const int g = (lane >> 4) & 1, j = lane & 15;
    const uint8_t *const src4 = T + g * (4 * IT_S - 8) - TAP_0;
    uint8_t *const dst4 = T + g * (4 * IT_S - 8) + (j >> 2) * IT_S + (j & 3);
    const int16_t *const res4 = tile->res + g * 56 + (j >> 2) * 16 + (j & 3);
    uint8_t *const dst8 = T + (lane >> 3) * IT_S + (lane & 7);
    const int16_t *const res8 = tile->res + (lane >> 3) * 16 + (lane & 7);
    uint8_t *const dstr = T + ((lane >> 2) + 1) * IT_S + IT_0 + 4 * (lane & 3);   // row lane / 4, 4 columns
    uint32_t out = 0u, out_at = 0u;   // the previous MB's row piece and where it goes
    IntraAhead f[2];
    f[0].meta = imeta_load(meta, b, e);
    f[1].meta = imeta_load(meta, b + 1, e);
    {
        const uint32_t ent = uniform(f[0].meta.x);
        f[0].res = *(const GAS uint2 *)(ires + (size_t)b * 384 + lane * 4);
        f[0].nb = load_nb(ent);
        // (the row above may have to pass its slots on before this row's first MB can start)
        lds_post(&sh.cons[w], (ent & ICOL_X_MASK) - min(ent & ICOL_X_MASK, 1u));
        if (ring_out) lds_post(&sh.prog[w + 1], ent & ICOL_X_MASK);
    }
    auto step = [&](uint32_t i, IntraAhead &cur, IntraAhead &nxt) {
        const bool live = i < e;
        const uint32_t ent = uniform(cur.meta.x);
        const uint64_t modes = (uint64_t)uniform(cur.meta.z) << 32 | uniform(cur.meta.y);
        const uint32_t nent = uniform(nxt.meta.x);
        // ---- this MB's residual and its neighbours' samples that were final before this launch
        const uint2 rv = (ent & ICOL_RES) ? cur.res : make_uint2(0u, 0u);
        const uint32_t nb = cur.nb;
        *(uint2 *)&tile->res[lane * 4] = rv;
        // ---- the previous MB goes out, the loads for the next one are issued
        if (i > b) *(GAS uint32_t *)(slot + out_at) = out;
        cur.meta = imeta_load(meta, i + 2, e);
        nxt.res = *(const GAS uint2 *)(ires + (size_t)min(i + 1, e - 1) * 384 + lane * 4);
        nxt.nb = load_nb(nent);
        if (!live) return;
        const int x = (int)(ent & ICOL_X_MASK), type = (int)((ent >> IMETA_TYPE_SHIFT) & 3u);
        const uint32_t av = (ent >> ICOL_AV_SHIFT) & 15u, dep = (ent >> ICOL_DEP_SHIFT) & 15u;
        const bool A = av & 1u, B = av & 2u, C = av & 4u, D = av & 8u;
        // ---- wait for the row above up to C (x + 1), or up to B (x) when only B / D are intra MBs
        const uint32_t need = (dep & 4u) ? (uint32_t)min(x + 2, W) : (dep & 10u) ? (uint32_t)x + 1u : 0u;
        if (need) lds_wait(&sh.prog[w], 0u, need, err);
        // (an intra MB to the left has left its last column in place, see below)
        const uint32_t up = rin[(uint32_t)(x * 16 + nb_dx) % (RING_COLS * 16u)];
        if ((av & nbit) && !(leftl && (dep & 1u))) *nb_at = (uint8_t)((dep & nbit) ? up : nb);
        wave_sync();
        if (type == 0) {
            // Intra_4x4, 8.3.1: blocks in wavefront order t = bx + 2 by, two per step; every
            // neighbour a block reads has a smaller t, and a top-right block that the reference's
            // block order has not decoded yet (blocks 3, 11) counts as not available by rule, so the
            // result equals the block-index order
            uint32_t tp[10];
            int rs[10];
            int m0[10], m1[10];
#pragma unroll
            for (int t = 0; t < 10; t++) {
                const int by = t < 2 ? 0 : (t - 2) >> 1, bx = t - 2 * by;
                auto mode_of = [&](int bx, int by) -> int {
                    if (bx < 0 || bx > 3 || by > 3) return 0;
                    const int blk = 8 * (by >> 1) + 4 * (bx >> 1) + 2 * (by & 1) + (bx & 1);
                    const int m = (int)((modes >> (4 * blk)) & 15u);
                    const bool tr = blk == 5 ? C : !(blk == 3 || blk == 11 || blk == 7 || blk == 13 || blk == 15);
                    return !tr && m == 3 ? 9 : !tr && m == 7 ? 10 : m;
                };
                m0[t] = mode_of(bx, by);
                m1[t] = mode_of(bx - 2, by + 1);
                tp[t] = sh.tap4.v[g ? m1[t] : m0[t]][j];
                rs[t] = res4[by * 64 + bx * 4];
            }
            if (lane < 32) {
#pragma unroll
                for (int t = 0; t < 10; t++) {
                    const int by = t < 2 ? 0 : (t - 2) >> 1, bx = t - 2 * by;
                    const int at = (by * 4 + 1) * IT_S + IT_0 + bx * 4;
                    const uint32_t p = tp[t];
                    int v = (int)src4[at + byte_of(p, 0)] + (int)src4[at + byte_of(p, 1)] + (int)src4[at + byte_of(p, 2)] +
                            (int)src4[at + byte_of(p, 3)];
                    if (m0[t] == 2 || m1[t] == 2) {  // DC: v is the sum of T0..T3
                        const uint8_t *const lp = src4 + TAP_0 + at - 1;
                        const int sl = (int)lp[0] + (int)lp[IT_S] + (int)lp[2 * IT_S] + (int)lp[3 * IT_S];
                        const bool ta = by + g > 0 || B, la = bx - 2 * g > 0 || A;
                        const int dc = ta && la ? (v + sl + 4) >> 3 : la ? (sl + 2) >> 2 : ta ? (v + 2) >> 2 : 128;
                        v = (g ? m1[t] : m0[t]) == 2 ? dc : (v + 2) >> 2;
                    } else {
                        v = (v + 2) >> 2;
                    }
                    v = clip1(v + rs[t]);
                    const bool two = t >= 2 && t < 8;  // steps of two blocks
                    if (two || g == 0) dst4[at] = (uint8_t)v;
                    wave_sync();
                }
            }
        } else if (type == 1) {
            // Intra_8x8, 8.3.2: per block the 25 filtered reference samples, then four taps per sample
#pragma unroll
            for (int blk = 0; blk < 4; blk++) {
                const int xO = (blk & 1) * 8, yO = (blk >> 1) * 8, at = (yO + 1) * IT_S + IT_0 + xO;
                const bool tl = blk == 0 ? D : blk == 1 ? B : blk == 2 ? A : true, tr = blk == 1 ? C : blk != 3;
                const int m = (int)((modes >> (4 * blk)) & 15u);
                const uint32_t tp = sh.tap8.v[m][lane];
                const int rs = res8[yO * 16 + xO];
                if (lane < 25) {
                    const uint32_t fl = sh.flt8.v[(tl ? 1 : 0) | (tr ? 2 : 0)][lane];
                    const uint8_t *const s = T + at - TAP_0;
                    tile->pf[lane] = (uint8_t)(((int)s[fl & 1023u] + 2 * (int)s[(fl >> 10) & 1023u] + (int)s[fl >> 20] + 2) >> 2);
                }
                wave_sync();
                int v;
                if (m == 2) {  // DC (8.3.2.2.4)
                    const uint2 lv = *(const uint2 *)&tile->pf[0], tv = *(const uint2 *)&tile->pf[8];
                    const int sl = (int)__builtin_amdgcn_sad_u8(lv.x, 0u, __builtin_amdgcn_sad_u8(lv.y, 0u, 0u));
                    const int st = (int)__builtin_amdgcn_sad_u8(tv.x, 0u, __builtin_amdgcn_sad_u8(tv.y, 0u, 0u));
                    const bool ta = blk > 1 || B, la = (blk & 1) || A;
                    v = ta && la ? (st + sl + 8) >> 4 : la ? (sl + 4) >> 3 : ta ? (st + 4) >> 3 : 128;
                } else {
                    v = ((int)tile->pf[byte_of(tp, 0)] + (int)tile->pf[byte_of(tp, 1)] + (int)tile->pf[byte_of(tp, 2)] +
                         (int)tile->pf[byte_of(tp, 3)] + 2) >> 2;
                }
                dst8[at] = (uint8_t)clip1(v + rs);
                wave_sync();
            }
        } else {  // Intra_16x16, 8.3.3 (H264PictureBase.cpp:1847-2056): lane = row lane / 4, 4 columns
            const int mode = (int)((ent >> IMETA_I16_SHIFT) & 3u), r = lane >> 2, c4 = 4 * (lane & 3);
            const uint2 rs = rv;
            int v[4];
            if (mode == 0) {
                const uint32_t d = *(const uint32_t *)&T[IT_0 + c4];
#pragma unroll
                for (int k = 0; k < 4; k++) v[k] = (int)byte_of(d, k);
            } else if (mode == 1) {
                const int l = T[(r + 1) * IT_S + IT_0 - 1];
#pragma unroll
                for (int k = 0; k < 4; k++) v[k] = l;
            } else if (mode == 2) {
                // lanes 0-15 the top samples, 16-31 the left ones, those of available neighbours
                const int s = lane < 16 ? (B ? (int)T[IT_0 + j] : 0) : (A ? (int)T[(j + 1) * IT_S + IT_0 - 1] : 0);
                const int sum = sum32(s), dc = A && B ? (sum + 16) >> 5 : A || B ? (sum + 8) >> 4 : 128;
#pragma unroll
                for (int k = 0; k < 4; k++) v[k] = dc;
            } else {
                // lanes 0-7 (k + 1) (T[8 + k] - T[6 - k]), lanes 16-23 the same of the left column
                const int k8 = j & 7;
                const uint8_t *const hi = lane < 16 ? &T[IT_0 + 8 + k8] : &T[(9 + k8) * IT_S + IT_0 - 1];
                const uint8_t *const lo = lane < 16 ? &T[IT_0 + 6 - k8] : &T[(7 - k8) * IT_S + IT_0 - 1];
                const int d = j < 8 ? (k8 + 1) * ((int)*hi - (int)*lo) : 0;
                const int Hs = sum32(lane < 16 ? d : 0), Vs = sum32(lane < 16 ? 0 : d);
                const int a = 16 * ((int)T[16 * IT_S + IT_0 - 1] + (int)T[IT_0 + 15]);
                const int bq = (5 * Hs + 32) >> 6, cq = (5 * Vs + 32) >> 6;
#pragma unroll
                for (int k = 0; k < 4; k++) v[k] = clip1((a + bq * (c4 + k - 7) + cq * (r - 7) + 16) >> 5);
            }
            const int16_t r0 = (int16_t)rs.x, r1 = (int16_t)(rs.x >> 16), r2 = (int16_t)rs.y, r3 = (int16_t)(rs.y >> 16);
            *(uint32_t *)dstr = pack4(clip1(v[0] + r0), clip1(v[1] + r1), clip1(v[2] + r2), clip1(v[3] + r3));
            wave_sync();
        }
        wave_sync();
        // ---- the finished MB: its last column where the next MB's left neighbours stand, its bottom
        // row (lanes 60-63) to the next row
        out = *(const uint32_t *)dstr;
        out_at = row0 + (uint32_t)(lane >> 2) * pitch + (uint32_t)(x * 16 + 4 * (lane & 3));
        wave_sync();
        if ((lane & 3) == 3) T[((lane >> 2) + 1) * IT_S + IT_0 - 1] = (uint8_t)(out >> 24);
        const bool end = i + 1 >= e;
        const uint32_t nx = end ? (uint32_t)W : nent & ICOL_X_MASK;
        if (ring_out) {
            if (x >= RING_COLS) lds_wait(&sh.cons[w + 1], 0u, (uint32_t)(x - RING_COLS + 1), err);
            if (lane >= 60) *(uint32_t *)&sh.ring[w + 1][x % RING_COLS][4 * (lane - 60)] = out;
            lds_post(&sh.prog[w + 1], nx);
        } else if (g_out && lane >= 60) {
            __hip_atomic_store(&gout[(size_t)x * 8 + (lane - 60)], (uint64_t)epoch << 32 | out, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        }
        lds_post(&sh.cons[w], end ? NO_COL : nx - min(nx, 1u));
    };
    for (uint32_t i = b; i < e; i += 2) {
        step(i, f[0], f[1]);
        step(i + 1, f[1], f[0]);
    }
    // an even number of MBs leaves the last one to be stored (else the step past the end did)
    if (((e - b) & 1u) == 0u) *(GAS uint32_t *)(slot + out_at) = out;
}

// The chroma planes of MB row y = y0 + w, alike.  Lane: plane lane / 32, row (lane / 4) mod 8, two
// samples from column 2 (lane mod 4).
__device__ __forceinline__ void intra_chroma_row(const DevPic &P, int w, int y, bool ring_out, bool g_out, GAS uint64_t *gout,
                                                 IntraWgShared &sh, uint32_t epoch, uint32_t *err) {
    const int W = P.W, lane = wave_lane();
    const GAS uint32_t *const off = G(P.irow);
    const GAS uint4 *const meta = (const GAS uint4 *)G(P.imeta);
    const uint32_t b = uniform(off[y]), e = uniform(off[y + 1]);
    IntraChromaTile *const tile = &sh.c[w];
    const uint8_t *const rin = &sh.ring[w][0][0];
    if (b == e) {
        if (ring_out) lds_post(&sh.prog[w + 1], (uint32_t)W);
        lds_post(&sh.cons[w], NO_COL);
        return;
    }
    gu8 *const slot = slot_base(P, P.dst);
    const uint32_t pitch = (uint32_t)W * 8u, np = (uint32_t)(W * P.H), row0 = (uint32_t)(y * 8) * pitch;
    const GAS int16_t *const ires = G(P.ires);
    // neighbour positions: lanes 16 p + i (i < 9) row -1, column i - 1 of plane p; lanes 32 + 8 p + k
    // column -1, row k
    const bool topl = lane < 32 && (lane & 15) < 9, leftl = lane >= 32 && lane < 48;
    const int npl = topl ? lane >> 4 : (lane >> 3) & 1, ni = lane & 15, nk = lane & 7;
    const uint32_t nbit = topl ? (ni == 0 ? 8u : 2u) : leftl ? 1u : 0u;
    uint8_t *const nb_at = tile->t[npl] + (topl ? CT_0 - 1 + ni : leftl ? (nk + 1) * CT_S + CT_0 - 1 : 0);
    const uint32_t nb_row = np * (npl ? 320u : 256u) + (uint32_t)(topl ? max(y * 8 - 1, 0) : y * 8 + (leftl ? nk : 0)) * pitch;
    const int nb_dx = topl ? ni - 1 : -1;
    auto load_nb = [&](uint32_t ent) -> uint32_t {
        const int x = (int)(ent & ICOL_X_MASK);
        return slot[nb_row + (uint32_t)clip3(0, W * 8 - 1, x * 8 + nb_dx)];
    };
    const int c = lane >> 5, r = (lane >> 2) & 7, x2 = 2 * (lane & 3);
    uint8_t *const T = tile->t[c];
    const uint32_t line = np * (c ? 320u : 256u) + row0 + (uint32_t)r * pitch + (uint32_t)x2;
    uint32_t out = 0u, out_at = 0u;
    IntraAhead f[2];
    f[0].meta = imeta_load(meta, b, e);
    f[1].meta = imeta_load(meta, b + 1, e);
    {
        const uint32_t ent = uniform(f[0].meta.x);
        f[0].res.x = *(const GAS uint32_t *)(ires + (size_t)b * 384 + 256 + lane * 2);
        f[0].nb = load_nb(ent);
        // (the row above may have to pass its slots on before this row's first MB can start)
        lds_post(&sh.cons[w], (ent & ICOL_X_MASK) - min(ent & ICOL_X_MASK, 1u));
        if (ring_out) lds_post(&sh.prog[w + 1], ent & ICOL_X_MASK);
    }
    auto step = [&](uint32_t i, IntraAhead &cur, IntraAhead &nxt) {
        const bool live = i < e;
        const uint32_t ent = uniform(cur.meta.x), nent = uniform(nxt.meta.x);
        const uint32_t rv = (ent & ICOL_RES) ? cur.res.x : 0u, nb = cur.nb;
        // (the words are consumed here, before the store and the next loads are issued)
        uint32_t rv_ = rv, nb_ = nb;
        asm volatile("" : "+v"(rv_), "+v"(nb_));
        if (i > b) *(GAS uint16_t *)(slot + out_at) = (uint16_t)out;
        cur.meta = imeta_load(meta, i + 2, e);
        nxt.res.x = *(const GAS uint32_t *)(ires + (size_t)min(i + 1, e - 1) * 384 + 256 + lane * 2);
        nxt.nb = load_nb(nent);
        if (!live) return;
        const int x = (int)(ent & ICOL_X_MASK), mode = (int)((ent >> IMETA_CHROMA_SHIFT) & 3u);
        const uint32_t av = (ent >> ICOL_AV_SHIFT) & 15u, dep = (ent >> ICOL_DEP_SHIFT) & 15u;
        const bool A = av & 1u, B = av & 2u;
        if (dep & 10u) lds_wait(&sh.prog[w], 0u, (uint32_t)x + 1u, err);  // (chroma never reads C)
        const uint32_t cx = (uint32_t)(x * 8 + nb_dx);
        const uint32_t up = rin[((cx >> 3) % RING_COLS) * 16u + (uint32_t)npl * 8u + (cx & 7u)];
        if ((av & nbit) && !(leftl && (dep & 1u))) *nb_at = (uint8_t)((dep & nbit) ? up : nb_);
        wave_sync();
        // ---- 8.3.4 (H264PictureBase.cpp:2076-2381); DC tests "> 0" (quirk Q1)
        int v0, v1;
        if (mode == 0) {
            const int xO = x2 & 4, yO = r & 4;
            const uint32_t t4 = *(const uint32_t *)&T[CT_0 + xO];
            const uint8_t *const lp = &T[(yO + 1) * CT_S + CT_0 - 1];
            const int l0 = lp[0], l1 = lp[CT_S], l2 = lp[2 * CT_S], l3 = lp[3 * CT_S];
            const bool t = B && byte_of(t4, 0) && byte_of(t4, 1) && byte_of(t4, 2) && byte_of(t4, 3);
            const bool l = A && l0 && l1 && l2 && l3;
            const int st = (int)__builtin_amdgcn_sad_u8(t4, 0u, 0u), sl = l0 + l1 + l2 + l3;
            const bool diag = (xO == 0) == (yO == 0);  // the corner blocks average both sides
            const int top = (st + 2) >> 2, left = (sl + 2) >> 2;
            v0 = diag ? (t && l ? (st + sl + 4) >> 3 : l ? left : t ? top : 128) : xO ? (t ? top : l ? left : 128) : (l ? left : t ? top : 128);
            v1 = v0;
        } else if (mode == 1) {
            v0 = v1 = T[(r + 1) * CT_S + CT_0 - 1];
        } else if (mode == 2) {
            const uint32_t d = *(const uint16_t *)&T[CT_0 + x2];
            v0 = (int)(d & 255u);
            v1 = (int)(d >> 8);
        } else {
            int Hs = 0, Vs = 0;
#pragma unroll
            for (int k = 0; k < 4; k++) {
                Hs += (k + 1) * ((int)T[CT_0 + 4 + k] - (int)T[CT_0 + 2 - k]);
                Vs += (k + 1) * ((int)T[(5 + k) * CT_S + CT_0 - 1] - (int)T[(3 - k) * CT_S + CT_0 - 1]);
            }
            const int aa = 16 * ((int)T[8 * CT_S + CT_0 - 1] + (int)T[CT_0 + 7]), bb = (34 * Hs + 32) >> 6, cc = (34 * Vs + 32) >> 6;
            v0 = clip1((aa + bb * (x2 - 3) + cc * (r - 3) + 16) >> 5);
            v1 = clip1((aa + bb * (x2 - 2) + cc * (r - 3) + 16) >> 5);
        }
        v0 = clip1(v0 + (int16_t)rv_);
        v1 = clip1(v1 + (int16_t)(rv_ >> 16));
        out = (uint32_t)v0 | (uint32_t)v1 << 8;
        out_at = line + (uint32_t)x * 8u;
        wave_sync();
        if (x2 == 6) T[(r + 1) * CT_S + CT_0 - 1] = (uint8_t)v1;
        const bool end = i + 1 >= e;
        const uint32_t nx = end ? (uint32_t)W : nent & ICOL_X_MASK;
        if (ring_out) {
            if (x >= RING_COLS) lds_wait(&sh.cons[w + 1], 0u, (uint32_t)(x - RING_COLS + 1), err);
            if (r == 7) *(uint16_t *)&sh.ring[w + 1][x % RING_COLS][c * 8 + x2] = (uint16_t)out;
            lds_post(&sh.prog[w + 1], nx);
        } else if (g_out) {
            const uint32_t d = out | (uint32_t)dpp_xor1((int)out) << 16;  // even lanes: four samples
            if (r == 7 && !(lane & 1))
                __hip_atomic_store(&gout[(size_t)x * 8 + 4 + c * 2 + (x2 >> 2)], (uint64_t)epoch << 32 | d, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
        }
        lds_post(&sh.cons[w], end ? NO_COL : nx - min(nx, 1u));
    };
    for (uint32_t i = b; i < e; i += 2) {
        step(i, f[0], f[1]);
        step(i + 1, f[1], f[0]);
    }
    if (((e - b) & 1u) == 0u) *(GAS uint16_t *)(slot + out_at) = (uint16_t)out;
}

// Two workgroups per band of `rows` MB rows, item 2 i for the luma plane of band i, item 2 i + 1
// for its chroma planes; the workgroup's last wave reads the strips of the band above.
__global__ __launch_bounds__(WAVE *(H264G_INTRA_MAX_ROWS + 1)) void k_intra_band(const DevPic *__restrict__ pics,
                                                                                 const uint32_t *__restrict__ items, uint32_t n,
                                                                                 int rows, DevCtl *ctl, uint32_t *epoch_p,
                                                                                 uint32_t *err) {
    __shared__ IntraWgShared sh;
    __shared__ uint32_t s_ticket;
    const uint32_t epoch = launch_epoch(epoch_p);
    const int w = (int)uniform(threadIdx.x / WAVE);
    if ((int)threadIdx.x < rows) sh.cons[threadIdx.x] = 0;
    const uint32_t t = band_ticket(ctl, &s_ticket, sh.prog, rows);
    const bool chroma = t & 1u;
    if (!chroma) {
        for (int i = threadIdx.x; i < 11 * 16; i += blockDim.x) (&sh.tap4.v[0][0])[i] = (&c_tap4.v[0][0])[i];
        for (int i = threadIdx.x; i < 9 * 64; i += blockDim.x) (&sh.tap8.v[0][0])[i] = (&c_tap8.v[0][0])[i];
        for (int i = threadIdx.x; i < 4 * 25; i += blockDim.x) (&sh.flt8.v[0][0])[i] = (&c_flt8.v[0][0])[i];
        __syncthreads();
    }
    if (t < 2 * n) {
        const uint32_t it = items ? items[t >> 1] : t >> 1;
        const DevPic &P = pics[it >> WI_PIC_SHIFT];
        const int band = (int)(it & WI_MB_MASK), y0 = band * rows, y = y0 + w, y1 = min(P.H, y0 + rows);
        if (P.n_intra != 0) {
            GAS uint64_t *const gout = G(P.istrip) + (size_t)band * P.W * 8;
            if (w < rows) {
                if (y < y1) {
                    const bool ring_out = y + 1 < y1, g_out = !ring_out && y1 < P.H;
                    if (chroma) intra_chroma_row(P, w, y, ring_out, g_out, gout, sh, epoch, err);
                    else intra_luma_row(P, w, y, ring_out, g_out, gout, sh, epoch, err);
                }
            } else if (y0 > 0) {
                const GAS uint32_t *const off = G(P.irow);
                istrip_reader(G(P.istrip) + (size_t)(band - 1) * P.W * 8, off + P.H + 1, uniform(off[y0 - 1]), uniform(off[y0]), P.W,
                              sh, chroma ? 4 : 0, epoch, err);
            }
        }
    }
    band_retire(ctl, epoch_p, epoch);
}

__global__ __launch_bounds__(WAVE) void k_deblock(const DevPic *__restrict__ pics, const uint32_t *__restrict__ items, uint32_t n,
                                                  DevCtl *ctl, uint32_t *epoch_p, uint32_t *err) {
    __shared__ WaveDbk lds;
    __shared__ DbkTables tb;
    dbk_tables_init(&tb);
    __syncthreads();
    const uint32_t epoch = launch_epoch(epoch_p);
    for (;;) {
        int t = next_ticket(ctl, n);
        if (t < 0) break;
        const uint32_t it = items[t];
        const DevPic &P = pics[it >> WI_PIC_SHIFT];
        const int addr = (int)(it & WI_MB_MASK), W = P.W, mbx = addr % W, mby = addr / W;
        int deps[2] = {mbx > 0 ? addr - 1 : -1, mby > 0 ? (mbx < W - 1 ? addr - W + 1 : addr - W) : -1};
        wait_deps(G(P.flags), deps, 2, epoch, err);
        deblock_mb(P, addr, &lds, &tb);
        publish(&G(P.flags)[addr], epoch);
    }
    retire(ctl, gridDim.x, epoch_p, epoch);
}

// ---- deblocking of MBAFF frames
// 8.7.2.1 (Deblock.cpp:994-1310) in an MBAFF frame, for the luma positions (xp, yp) of p0
// in MB ap and (xq, yq) of q0 in MB aq: mixedModeEdgeFlag between a frame and a field MB;
// bS 4 at MB edges between frame MBs and at vertical MB edges, 3 at the other intra edges;
// 2 for levels; 1 at mixed edges; then the motion tests with a vertical limit of 2
// quarter samples when q is a field MB (:1157-1158), comparing RefPicListX[RefIdxLX]
// (G(P.bsref), quirk Q4) with quirk Q3.  I_PCM counts as neither intra nor inter.
__device__ __forceinline__ int bs_mbaff(const DevPic &P, int ap, int aq, int xp, int yp, int xq, int yq, bool vertical) {
    const h264g_mb &mp = G(P.mbs)[ap], &mq = G(P.mbs)[aq];
    const DevAux xa = G(P.aux)[ap], xb = G(P.aux)[aq];
    const bool pf = mp.flags & H264G_MBF_FIELD, qf = mq.flags & H264G_MBF_FIELD;
    const bool intra = ((xa.kind | xb.kind) & AUX_INTRA) != 0, mixed = ap != aq && pf != qf;
    if (ap != aq && intra && ((!pf && !qf) || vertical)) return 4;
    if (intra && (!mixed || !vertical)) return 3;
    const int bp4 = 8 * (yp >> 3) + 4 * (xp >> 3) + 2 * ((yp & 7) >> 2) + ((xp & 7) >> 2);
    const int bq4 = 8 * (yq >> 3) + 4 * (xq >> 3) + 2 * ((yq & 7) >> 2) + ((xq & 7) >> 2);
    const int bp8 = 2 * (yp >> 3) + (xp >> 3), bq8 = 2 * (yq >> 3) + (xq >> 3);
    const bool pt8 = xa.kind & AUX_T8, qt8 = xb.kind & AUX_T8;
    if ((pt8 && ((xa.nz8 >> bp8) & 1)) || (!pt8 && ((xa.nz4 >> bp4) & 1)) || (qt8 && ((xb.nz8 >> bq8) & 1)) ||
        (!qt8 && ((xb.nz4 >> bq4) & 1)))
        return 2;
    if (mixed) return 1;
    const int ylim = qf ? 2 : 4;
    const int qp = bp8, qq = bq8, rp = (yp >> 2) * 4 + (xp >> 2), rq = (yq >> 2) * 4 + (xq >> 2);
    const int p0 = G(P.bsref)[ap * 8 + qp], p1 = G(P.bsref)[ap * 8 + 4 + qp], q0 = G(P.bsref)[aq * 8 + qq], q1 = G(P.bsref)[aq * 8 + 4 + qq];
    const int fp0 = (xa.pf >> qp) & 1, fp1 = (xa.pf >> (4 + qp)) & 1, fq0 = (xb.pf >> qq) & 1, fq1 = (xb.pf >> (4 + qq)) & 1;
    if (!(((p0 == q0 && p1 == q1) || (p0 == q1 && p1 == q0)) && fp0 + fp1 == fq0 + fq1)) return 1;
    auto far = [&](int ax, int ay, int bx, int by) { return iabs(ax - bx) >= 4 || iabs(ay - by) >= ylim; };
    const int mp0x = mp.mv[0][rp][0], mp0y = mp.mv[0][rp][1], mp1x = mp.mv[1][rp][0], mp1y = mp.mv[1][rp][1];
    const int mq0x = mq.mv[0][rq][0], mq0y = mq.mv[0][rq][1], mq1x = mq.mv[1][rq][0], mq1y = mq.mv[1][rq][1];
    if (fp0 && !fp1 && fq0 && !fq1 && far(mp0x, mp0y, mq0x, mq0y)) return 1;
    if (fp0 && !fp1 && !fq0 && fq1 && far(mp0x, mp0y, mq1x, mq1y)) return 1;
    if (!fp0 && fp1 && fq0 && !fq1 && far(mp1x, mp1y, mq0x, mq0y)) return 1;
    if (!fp0 && fp1 && !fq0 && fq1 && far(mp1x, mp1y, mq1x, mq1y)) return 1;
    if (fp0 && fp1 && p0 != p1 && fq0 && fq1 && ((q0 == p0 && q1 == p1) || (q0 == p1 && q1 == p0))) {
        if (q0 == p0 && (far(mp0x, mp0y, mq0x, mq0y) || far(mp1x, mp1y, mq1x, mq1y))) return 1;
        if (q0 == p1 && (far(mp1x, mp1y, mq0x, mq0y) || far(mp0x, mp0y, mq1x, mq1y))) return 1;
    }
    if (fp0 && fp1 && p0 == p1 && fq0 && fq1 && q0 == q1 && q0 == p0) {
        if (far(mp0x, mp0y, mq0x, mq0y) || (far(mp1x, mp1y, mq1x, mq1y) && far(mp0x, mp0y, mq1x, mq1y)) ||
            far(mp1x, mp1y, mq0x, mq0y))
            return 1;
    }
    return 0;
}

// How the MBs of an MBAFF frame around MB addr meet its edges (6.4.11.1 with Table 6-4 at
// (-1, 0) and (0, -1); Deblock.cpp:76-635).
struct MbaffNb {
    int mbA, mbB;              // the MBs holding p0 of the left / top edge, -1: none
    bool left, upper;          // the MB edges that are filtered
    bool leftMix, topMix;      // a frame MB beside / the top frame MB under a field pair
    bool field, t8;
};
// fields of the MB itself, the left pair and the pair above (false where there is none)
__device__ __forceinline__ MbaffNb mbaff_nb(int W, int addr, bool field, bool lfield, bool afield, bool t8) {
    const int pair = addr >> 1, px = pair % W, py = pair / W, bot = addr & 1;
    MbaffNb n;
    n.field = field;
    n.t8 = t8;
    n.mbA = px > 0 ? 2 * (pair - 1) + (field == lfield ? bot : 0) : -1;
    n.mbB = !field && bot ? addr - 1 : (py > 0 ? 2 * (pair - W) + (field && !bot && afield ? 0 : 1) : -1);
    n.left = px > 0;
    n.upper = !(py == 0 && (field || !bot));
    n.leftMix = !field && lfield;
    n.topMix = !bot && py > 0 && !field && afield;
    return n;
}

// Boundary strengths of a MB of an MBAFF frame: 64 nibbles in its 32 bytes of P.bs,
//    0  left edge, luma lines 0..15        16  left edge, chroma lines 0..7
//   24  vertical edges 4, 8, 12, four segments of 4 lines each
//   36  top edge, luma segments (40: chroma); 44, 48: the same of the second pass over the
//       top edge of a frame MB under a field pair (its bottom field lines)
//   52  horizontal edges 4, 8, 12
// (chroma edge 4 lies on luma edge 8), 0 where an edge is not filtered.  Fully parallel: they
// depend on syntax only.  A lane per nibble, a MB per wave.  The MB's deblocking word as in
// bs_pair_of_mbs, with its field flag.
constexpr int MBS_LEFT = 0, MBS_LEFT_C = 16, MBS_V = 24, MBS_TOP = 36, MBS_TOP_C = 40, MBS_TOP2 = 44, MBS_TOP2_C = 48, MBS_H = 52;
constexpr uint32_t DBQ_FIELD = 1u << 27;
__device__ __forceinline__ void bs_mbaff_mb(const DevPic *pics, const uint32_t *chunks, uint32_t b, uint32_t n) {
    const MbSlot m = mb_slot(chunks, xcd_item(b, n));
    const DevPic &P = pics[m.pic];
    const int addr = m.addr, pair = addr >> 1, W = P.W, px = pair % W, py = pair / W;
    if (addr >= W * P.H || P.dbk_idc == 1) return;
    const int l = wave_lane();
    const DevAux &ax = G(P.aux)[addr];
    const MbaffNb nb = mbaff_nb(W, addr, (G(P.mbs)[addr].flags & H264G_MBF_FIELD) != 0,
                                px > 0 && (G(P.mbs)[2 * (pair - 1)].flags & H264G_MBF_FIELD),
                                py > 0 && (G(P.mbs)[2 * (pair - W)].flags & H264G_MBF_FIELD), (ax.kind & AUX_T8) != 0);
    // the lane's edge (position e inside the MB, in chroma samples where s is 2) and line k
    const bool vertical = l < MBS_TOP;
    const bool chroma = vertical ? l >= MBS_LEFT_C && l < MBS_V : (l >= MBS_TOP_C && l < MBS_TOP2) || (l >= MBS_TOP2_C && l < MBS_H);
    const bool second = l >= MBS_TOP2 && l < MBS_H;
    const int s = chroma ? 2 : 1, nE = chroma ? 8 : 16;
    int e, k;
    bool on;
    if (l < MBS_V) {
        e = 0;
        k = chroma ? l - MBS_LEFT_C : l;
        on = nb.left;
    } else if (vertical || l >= MBS_H) {
        const int j = l - (vertical ? MBS_V : MBS_H);
        e = 4 * (1 + (j >> 2));
        k = 4 * (j & 3);
        on = !(nb.t8 && (e & 4));
    } else {
        e = second ? 1 : 0;
        k = (l & 3) * (chroma ? 2 : 4);
        on = second ? nb.topMix : nb.topMix || nb.upper;
    }
    int bS = 0;
    if (on) {
        int ap = addr, xp, yp, xq, yq;
        if (vertical) {
            xp = e - 1;
            if (xp < 0) {
                ap = nb.leftMix ? nb.mbA + (k & 1) : nb.mbA;
                xp += nE;
            }
            yp = yq = k;
            xq = e;
        } else {
            // with a mixed top edge the chroma of both passes takes the bottom MB (quirk Q5)
            yp = (e - 1) - (e & 1);
            if (yp < 0) {
                if (nb.mbB >= 0) ap = nb.topMix && !second && !chroma ? nb.mbB - 1 : nb.mbB;
                yp += nE;
            }
            xp = xq = k;
            yq = e - (e & 1);
        }
        bS = bs_mbaff(P, ap, addr, xp * s, yp * s, xq * s, yq * s, vertical);
    }
    const int hi = dpp_xor1(bS);
    if (!(l & 1)) G(P.bs)[(size_t)addr * 32 + (l >> 1)] = (uint8_t)(bS | hi << 4);
    if (l == 0)
        G(P.dbq)[addr] = (uint32_t)ax.qdb[0] | ((uint32_t)ax.qdb[1] << 8) | ((uint32_t)ax.qdb[2] << 16) | (nb.t8 ? 1u << 24 : 0u) |
                         (nb.field ? DBQ_FIELD : 0u);
}

// ds_read_b64_tr_b8: in each group of 16 lanes, lanes 2j and 2j + 1 name the two 8-byte
// halves of row j (j < 8) of an 8 x 16 byte matrix and lane i gets its column i, byte j
// from row j.  Every lane of the wave takes part.
__device__ __forceinline__ uint2 lds_tr(const uint8_t *p) {
    typedef int v2i __attribute__((ext_vector_type(2)));
    typedef __attribute__((address_space(3))) v2i lds_v2i;
    const v2i r = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_v2i *)p);
    return make_uint2((uint32_t)r.x, (uint32_t)r.y);
}

// ---- deblocking of MBAFF frames over bands of pair rows
// 8.7 (Deblock.cpp:76-635) takes the MBs in address order: a pair's top MB, then its bottom MB,
// each with its vertical edges, left to right, then its horizontal ones, top to bottom.  A band
// is MBAFF_ROWS rows of MB pairs on one workgroup, a wave per row and one more that brings in
// what the band above hands down.
//
// Of one pair, the vertical edges of both MBs go together, half a wave each (luma lines in lanes
// 0-15, Cb 16-23, Cr 24-31): the top MB's horizontal edges touch no row of a bottom frame MB, and
// no line of the other field.  So do the horizontal edges of a field pair; a frame pair's eight
// follow one another on lanes 0-31, and the two passes over the top edge of a frame MB under a
// field pair, each on the lines of one field, go half a wave each before them.  A line is held in
// registers for all its edges.
//
// Pair (x, y) takes the bottom 8 rows of pair (x, y - 1) over from that pair's wave, which has
// left them to it (a field MB's top edge reads four and filters three rows of its parity), once
// pair (x + 1, y - 1) has filtered its right columns; from then on they are its own to store.
// They travel through a ring in LDS, between bands as epoch-tagged words in device memory.
//
// Bound: the chain of W + 2 HP steps of about 3 us, what the lines of one pair take one wave.
// Measured (1920x1088, one launch): 560 us; with one workgroup of 16 waves for the picture, an edge of one MB
// at a time and the samples in device memory between pairs 3300; before that, with a persistent
// wave and a progress word in device memory per pair, 112000.
constexpr int MBAFF_ROWS = H264G_MBAFF_ROWS, MRING_SLOTS = 8, MRING_WORDS = 64;
// One pair's samples: luma rows -8..31 by columns -4..15, chroma rows -8..15 by columns -4..7;
// column -4 at byte 4 of a row, so that column 0 is aligned for ds_read_b64_tr_b8.
constexpr int MR_ROW0 = 8, MR_LP = 24, MR_CP = 16;
struct alignas(16) MbaffRegion {
    uint8_t L[40][MR_LP];
    uint8_t C[2][24][MR_CP];
    uint8_t pad[16];           // (a chroma line is read as if it were as long as a luma line)
};
struct MbaffDbkShared {
    MbaffRegion rg[MBAFF_ROWS];
    uint32_t bs[MBAFF_ROWS][16];                       // the pair's strengths (MBS_*)
    uint32_t ring[MBAFF_ROWS][MRING_SLOTS][MRING_WORDS];  // [w]: what row w takes over
    uint32_t prog[MBAFF_ROWS + 1], cons[MBAFF_ROWS + 1];  // pairs in ring[w], pairs read from it
    DbkTables tb;
};

// Edges of a line: the MB edge with deblocking word qe beyond it, then the internal ones (luma 4,
// 8, 12, chroma 4).  bs: strength nibbles of the MB; be, bi: nibble of the MB edge / of the first
// internal one.
__device__ __forceinline__ void mbaff_line(uint32_t (&w)[5], const DevPic &P, const DbkTables *tb, const uint8_t *bs, int be, int bi,
                                           uint32_t qe, uint32_t qq, int plane, bool act) {
    const bool luma = plane == 0;
    auto bs_at = [&](int n) -> int { return (bs[n >> 1] >> (4 * (n & 1))) & 15; };
    const int b0 = be < 0 ? 0 : bs_at(max(be, 0)), b1 = bs_at(luma ? bi : bi + 4), b2 = bs_at(bi + 4), b3 = bs_at(bi + 8);
    const int q = dbq_qp(qq, plane), qa = (dbq_qp(qe, plane) + q + 1) >> 1;
    const int ia = clip3(0, 51, qa + P.offA), ib = clip3(0, 51, qa + P.offB), ja = clip3(0, 51, q + P.offA), jb = clip3(0, 51, q + P.offB);
    auto tc = [&](int b, int i) -> int { return tb->tc0[clip3(0, 2, b - 1)][i]; };  // (used for bS 1..3)
    const int a0 = tb->alpha[ia], e0 = tb->beta[ib], ai = tb->alpha[ja], ei = tb->beta[jb];
    const int t0 = tc(b0, ia), t1 = tc(b1, ja), t2 = tc(b2, ja), t3 = tc(b3, ja);
    dbk_line_edge<0>(w, act, luma, b0, a0, e0, t0);
    dbk_line_edge<1>(w, act, luma, b1, ai, ei, t1);
    dbk_line_edge<2>(w, act && luma, luma, b2, ai, ei, t2);
    dbk_line_edge<3>(w, act && luma, luma, b3, ai, ei, t3);
}

// One row of pairs, on wave w of the workgroup: rows y0 .. y1 - 1 are the band's.  out: the
// strips to the next band (its last row writes them), W x MRING_WORDS words.
__device__ __forceinline__ void mbaff_dbk_row(const DevPic &P, int w, int y, int y1, GAS uint64_t *out, MbaffDbkShared &sh,
                                              uint32_t epoch, uint32_t *err) {
    const int lane = wave_lane(), W = P.W, HP = P.H >> 1;
    const int h = lane >> 5, l32 = lane & 31, plane = l32 < 16 ? 0 : (l32 < 24 ? 1 : 2), k = plane == 0 ? l32 : l32 & 7;
    const bool luma = plane == 0, last_row = y == HP - 1, ring_out = y + 1 < y1;
    const int seg = luma ? k >> 2 : k >> 1, hs = luma ? 16 : 8;
    const DbkPlanes d = dbk_planes(P);
    MbaffRegion *const rg = &sh.rg[w];
    const uint8_t *const bsb = (const uint8_t *)sh.bs[w];
    const GAS uint32_t *const dq = G(P.dbq);
    // the lane's line as a row / as a column of the region
    uint8_t *const rows = luma ? &rg->L[MR_ROW0][4] : &rg->C[plane - 1][MR_ROW0][4];
    const int pitch = luma ? MR_LP : MR_CP, rmax = luma ? 31 : 15;
    uint8_t *const col = rows + 4 + k;
    // ds_read_b64_tr_b8: the lane's 8-byte half of row tj of its group's 8 x 16 block (chroma: Cb | Cr)
    const int tj = (lane & 15) >> 1;
    const uint8_t *const tr = luma ? &rg->L[MR_ROW0][8 + 8 * (lane & 1)] : &rg->C[lane & 1][MR_ROW0][8];
    // samples of the pair, one pair ahead: luma rows 0..31, chroma rows 0..15 twice, on lanes 0-31
    const int r32 = lane & 31, cp = r32 >> 4, cr = r32 & 15;
    const GAS uint8_t *const gl = G(d.y) + (uint64_t)(y * 32 + r32) * d.wl;
    const GAS uint8_t *const gc = G(cp ? d.cr : d.cb) + (uint64_t)(y * 16 + cr) * d.wc;
    // where it is stored: luma rows -8..31 on lanes 0-39, chroma rows -8..15 twice on lanes 0-47
    const int slr = lane - MR_ROW0, sp = lane >= 24 ? 1 : 0, scr = lane - 24 * sp - MR_ROW0;
    const bool sl = lane < 40 && (slr >= 0 || y > 0) && (slr < 24 || last_row);
    const bool sc = lane < 48 && (scr >= 0 || y > 0) && (scr < 8 || last_row);
    GAS uint8_t *const ol = G(d.y) + (int64_t)(y * 32 + (sl ? slr : 0)) * d.wl;
    GAS uint8_t *const oc = G(sp ? d.cr : d.cb) + (int64_t)(y * 16 + (sc ? scr : 0)) * d.wc;
    // the dword this lane hands down: (luma) row 24 + hr, (chroma) row 8 + hr of the pair
    const int hp = h ? 1 + (l32 >> 4) : 0, hr = h ? (l32 >> 1) & 7 : l32 >> 2, hd = h ? l32 & 1 : l32 & 3;
    const uint8_t *const hrow = h ? &rg->C[hp - 1][16 + hr][4] : &rg->L[32 + hr][4];
    const int hw = h ? 32 + (hp - 1) * 16 + hr * 2 : hr * 4, hn = h ? 2 : 4;  // its row's words in a strip, their number
    uint4 lrow = *(const GAS uint4 *)gl;
    uint2 crow = *(const GAS uint2 *)gc;
    uint32_t bsw = ((const GAS uint32_t *)(G(P.bs) + (size_t)(y * W) * 64))[lane & 15];
    uint32_t n0 = dq[2 * (y * W)], n1 = dq[2 * (y * W) + 1], u0 = y > 0 ? dq[2 * (y * W - W)] : 0u, u1 = y > 0 ? dq[2 * (y * W - W) + 1] : 0u;
    uint32_t left0 = 0u, left1 = 0u;
    uint2 s0, s1, s2;          // the last pair's samples, stored after this pair's have arrived
    uint32_t s3 = 0u, s4 = 0u;
    s0 = s1 = s2 = make_uint2(0u, 0u);
    auto store = [&](int x) {
        if (sl) {
            *(GAS uint4 *)(ol + x * 16) = make_uint4(s0.x, s0.y, s1.x, s1.y);
            if (x > 0 && slr >= 0) *(GAS uint32_t *)(ol + x * 16 - 4) = s3;
        }
        if (sc) {
            *(GAS uint2 *)(oc + x * 8) = s2;
            if (x > 0 && scr >= 0) *(GAS uint32_t *)(oc + x * 8 - 4) = s4;
        }
    };
    for (int x = 0; x < W; x++) {
        const int pair = y * W + x;
        // ---- the pair into the region; the last pair's right columns become the left ones
        {
            uint8_t *const lr = lane < 32 ? &rg->L[MR_ROW0 + r32][4] : &rg->C[cp][MR_ROW0 + cr][4];
            const uint32_t c = *(const uint32_t *)(lr + (lane < 32 ? 16 : 8));
            wave_sync();
            *(uint32_t *)lr = c;
            if (lane < 32) {
                *(uint2 *)&rg->L[MR_ROW0 + r32][8] = make_uint2(lrow.x, lrow.y);
                *(uint2 *)&rg->L[MR_ROW0 + r32][16] = make_uint2(lrow.z, lrow.w);
            }
            wave_sync();
            if (lane < 32) *(uint2 *)&rg->C[cp][MR_ROW0 + cr][8] = crow;
            if (lane < 16) sh.bs[w][lane] = bsw;
        }
        const uint32_t q0 = uniform(n0), q1 = uniform(n1), a0 = uniform(u0), a1 = uniform(u1);
        if (x > 0) store(x - 1);
        if (x + 1 < W) {
            lrow = *(const GAS uint4 *)(gl + (x + 1) * 16);
            crow = *(const GAS uint2 *)(gc + (x + 1) * 8);
            bsw = ((const GAS uint32_t *)(G(P.bs) + (size_t)(pair + 1) * 64))[lane & 15];
            n0 = dq[2 * pair + 2];
            n1 = dq[2 * pair + 3];
            if (y > 0) {
                u0 = dq[2 * (pair - W) + 2];
                u1 = dq[2 * (pair - W) + 3];
            }
        }
        wave_sync();
        const bool field = (q0 & DBQ_FIELD) != 0, lfield = (left0 & DBQ_FIELD) != 0, afield = (a0 & DBQ_FIELD) != 0;
        const uint32_t own = h ? q1 : q0;
        const uint8_t *const bs = bsb + 32 * h;
        uint32_t wv[5];
        // ---- vertical edges.  A frame MB beside a field pair alternates between its MBs, a field
        // MB beside a frame pair takes its top one
        {
            const uint32_t qe = field == lfield ? (h ? left1 : left0) : !field && (k & 1) ? left1 : left0;
            uint8_t *const r = rows + pitch * (field ? h + 2 * k : hs * h + k);
            wv[0] = *(const uint32_t *)r;
            const uint2 m0 = *(const uint2 *)(r + 4), m1 = *(const uint2 *)(r + 12);
            wv[1] = m0.x; wv[2] = m0.y; wv[3] = m1.x; wv[4] = m1.y;
            mbaff_line(wv, P, &sh.tb, bs, luma ? MBS_LEFT + k : MBS_LEFT_C + k, MBS_V + seg, qe, own, plane, true);
            *(uint32_t *)r = wv[0];
            *(uint2 *)(r + 4) = make_uint2(wv[1], wv[2]);
            if (luma) *(uint2 *)(r + 12) = make_uint2(wv[3], wv[4]);
        }
        // ---- the rows above
        if (y > 0) {
            lds_wait(&sh.prog[w], 0u, (uint32_t)x + 1u, err);
            const uint32_t v = sh.ring[w][x % MRING_SLOTS][lane];
            uint8_t *const to = h ? &rg->C[hp - 1][hr][8 + 4 * hd] : &rg->L[hr][8 + 4 * hd];
            *(uint32_t *)to = v;
            lds_post(&sh.cons[w], (uint32_t)x + 1u);
        }
        wave_sync();
        // ---- horizontal edges
        const int top = luma ? MBS_TOP : MBS_TOP_C, hin = MBS_H + seg;
        auto blk = [&](int dy, int r0, int s) -> uint2 { return lds_tr(tr + pitch * min(r0 + dy * (s + tj), rmax)); };
        auto put = [&](uint8_t *c, int dy, uint32_t v) {
            c[0] = (uint8_t)v;
            c[dy * pitch] = (uint8_t)(v >> 8);
            c[2 * dy * pitch] = (uint8_t)(v >> 16);
            c[3 * dy * pitch] = (uint8_t)(v >> 24);
        };
        if (field) {  // each MB on the lines of its field
            const uint2 A = blk(2, h, -4), B = blk(2, h, 4), C = blk(2, h, 12);
            wv[0] = A.x; wv[1] = A.y; wv[2] = B.x; wv[3] = B.y; wv[4] = C.x;
            mbaff_line(wv, P, &sh.tb, bs, top + seg, hin, h || !afield ? a1 : a0, own, plane, true);
            wave_sync();
            uint8_t *const c = col + pitch * h;
            if (y > 0) put(c - 8 * pitch, 2, wv[0]);
            put(c, 2, wv[1]);
            put(c + 8 * pitch, 2, wv[2]);
            if (luma) {
                put(c + 16 * pitch, 2, wv[3]);
                put(c + 24 * pitch, 2, wv[4]);
            }
        } else {
            if (afield) {  // top edge under a field pair: the lines of each field
                const uint2 A = blk(2, h, -4);
                wv[0] = A.x; wv[1] = A.y;
                const int n = (h ? (luma ? MBS_TOP2 : MBS_TOP2_C) : top) + seg;
                const int b = (bsb[n >> 1] >> (4 * (n & 1))) & 15, qa = (dbq_qp(h || !luma ? a1 : a0, plane) + dbq_qp(q0, plane) + 1) >> 1;
                const int ia = clip3(0, 51, qa + P.offA);
                dbk_line_edge<0>(wv, true, luma, b, sh.tb.alpha[ia], sh.tb.beta[clip3(0, 51, qa + P.offB)], sh.tb.tc0[clip3(0, 2, b - 1)][ia]);
                wave_sync();
                put(col + pitch * (h - 8), 2, wv[0]);
                put(col + pitch * h, 2, wv[1]);
                wave_sync();
            }
            const uint2 A = blk(1, 0, -4), B = blk(1, 0, 4), C = blk(1, 0, 12), D = blk(1, 0, 20), E = blk(1, 0, 28);
            wv[0] = A.x; wv[1] = A.y; wv[2] = B.x; wv[3] = B.y; wv[4] = C.x;
            mbaff_line(wv, P, &sh.tb, bsb, afield ? -1 : top + seg, hin, a1, q0, plane, h == 0);
            uint32_t wb[5] = {luma ? wv[4] : wv[2], luma ? C.y : B.y, luma ? D.x : C.x, D.y, E.x};
            mbaff_line(wb, P, &sh.tb, bsb + 32, top + seg, hin, q0, q1, plane, h == 0);
            wave_sync();
            if (h == 0) {
                if (y > 0) put(col - 4 * pitch, 1, wv[0]);
                put(col, 1, wv[1]);
                if (luma) {
                    put(col + 4 * pitch, 1, wv[2]);
                    put(col + 8 * pitch, 1, wv[3]);
                    put(col + 12 * pitch, 1, wb[0]);
                    put(col + 16 * pitch, 1, wb[1]);
                    put(col + 20 * pitch, 1, wb[2]);
                    put(col + 24 * pitch, 1, wb[3]);
                    put(col + 28 * pitch, 1, wb[4]);
                } else {
                    put(col + 4 * pitch, 1, wb[0]);
                    put(col + 8 * pitch, 1, wb[1]);
                    put(col + 12 * pitch, 1, wb[2]);
                }
            }
        }
        wave_sync();
        // ---- the bottom rows to the row below: columns -4..11, the last pair's to the end
        if (!last_row) {
            const uint32_t v = *(const uint32_t *)(hrow + 4 * hd), v2 = *(const uint32_t *)(hrow + 4 * hn);
            const int hx = hd == 0 ? x - 1 : x, hi = hw + (hd == 0 ? hn - 1 : hd - 1);
            if (ring_out) {
                if (x >= MRING_SLOTS) lds_wait(&sh.cons[w + 1], 0u, (uint32_t)(x - MRING_SLOTS + 1), err);
                if (hx >= 0) sh.ring[w + 1][hx % MRING_SLOTS][hi] = v;
                if (x == W - 1 && hd == 0) {
                    wave_sync();
                    sh.ring[w + 1][x % MRING_SLOTS][hw + hn - 1] = v2;
                }
                lds_post(&sh.prog[w + 1], (uint32_t)(x == W - 1 ? W : x));
            } else {
                const uint64_t tag = (uint64_t)epoch << 32;
                if (hx >= 0) __hip_atomic_store(&out[(size_t)hx * MRING_WORDS + hi], tag | v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (x == W - 1 && hd == 0)
                    __hip_atomic_store(&out[(size_t)x * MRING_WORDS + hw + hn - 1], tag | v2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
        // ---- what goes to the picture
        {
            const uint8_t *const l = &rg->L[min(lane, 39)][4], *const c = &rg->C[sp][lane < 48 ? scr + MR_ROW0 : 0][4];
            s3 = *(const uint32_t *)l;
            s0 = *(const uint2 *)(l + 4);
            s1 = *(const uint2 *)(l + 12);
            s4 = *(const uint32_t *)c;
            s2 = *(const uint2 *)(c + 4);
        }
        wave_sync();
        left0 = q0;
        left1 = q1;
    }
    store(W - 1);
}

// Brings the strips of the band above into ring 0, one pair after another.
__device__ __forceinline__ void mbaff_strip_reader(const GAS uint64_t *sw, int W, MbaffDbkShared &sh, uint32_t epoch, uint32_t *err) {
    const int lane = wave_lane();
#pragma unroll 1
    for (int x = 0; x < W; x++) {
        if (x >= MRING_SLOTS) lds_wait(&sh.cons[0], 0u, (uint32_t)(x - MRING_SLOTS + 1), err);
        uint64_t r;
#pragma unroll 1
        for (uint32_t it = 0;; ++it) {
            r = __hip_atomic_load(&sw[(size_t)x * MRING_WORDS + lane], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (__builtin_amdgcn_ballot_w64((uint32_t)(r >> 32) != epoch) == 0) break;
            if (it >= SPIN_LIMIT) {
                report_timeout(err);
                return;
            }
            if ((it & 255u) == 255u && uniform(__hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) != 0u) return;
            __builtin_amdgcn_s_sleep(1);
        }
        sh.ring[0][x % MRING_SLOTS][lane] = (uint32_t)r;
        lds_post(&sh.prog[0], (uint32_t)x + 1u);
    }
}

// Workgroup t is band t / n of picture t mod n, n pictures; those that are no MBAFF frame or
// have no such band have nothing to do.
__global__ __launch_bounds__(WAVE *(MBAFF_ROWS + 1)) void k_deblock_mbaff(const DevPic *__restrict__ pics, uint32_t n, DevCtl *ctl,
                                                                          uint32_t *epoch_p, uint32_t *err) {
    __shared__ MbaffDbkShared sh;
    __shared__ uint32_t s_ticket;
    const uint32_t epoch = launch_epoch(epoch_p);
    const int w = (int)uniform(threadIdx.x / WAVE);
    if ((int)threadIdx.x <= MBAFF_ROWS) sh.cons[threadIdx.x] = 0;
    dbk_tables_init(&sh.tb);
    const uint32_t t = band_ticket(ctl, &s_ticket, sh.prog, MBAFF_ROWS + 1);
    if (t < gridDim.x) {
        const DevPic &P = pics[t % n];
        const int b = (int)(t / n), HP = P.H >> 1, y0 = b * MBAFF_ROWS, y1 = min(HP, y0 + MBAFF_ROWS);
        if (P.mbaff && P.dbk_idc != 1 && y0 < HP) {
            GAS uint64_t *const strips = (GAS uint64_t *)G(P.gstrip);
            const size_t strip = (size_t)P.W * MRING_WORDS;
            if (w < MBAFF_ROWS) {
                if (y0 + w < y1) mbaff_dbk_row(P, w, y0 + w, y1, strips + b * strip, sh, epoch, err);
            } else if (b > 0) {
                mbaff_strip_reader(strips + (b - 1) * strip, P.W, sh, epoch, err);
            }
        }
    }
    band_retire(ctl, epoch_p, epoch);
}

// Intra MBs of MBAFF frames over the same bands, the top MB of a pair before the bottom one.  An
// MB reads MBs of its own and the left pair, earlier in its row, and of the pairs above up to
// x + 1.  A row is three waves: one prepares the row's MBs up to two ahead (residual, tap
// addresses, what the record says) in one of two tiles, one predicts luma and one chroma, whose
// chains never meet.  Inside a band the samples travel through the CU's caches (workgroup scope).
// A band's last row sends the two bottom rows of every pair with an intra MB to the next band as
// epoch-tagged words, and that band's last wave writes them to where they stand already, so that
// its workgroup's reads find them.
// Bound: the chain of W + 2 HP pairs, with two trips through the caches per MB.  1920x1088: an I
// frame 1.44 ms, P and B frames (10 % intra MBs) 0.15; with preparation, luma and chroma on one wave
// 3.06 and 0.33; with one workgroup of 16 such waves per picture 5.4 and 0.6, with persistent
// waves and progress words in device memory 40 and 10.
constexpr int MISTRIP_WORDS = 16;  // luma rows 30, 31 in four dwords each, then two of Cb rows 14, 15 and of Cr
constexpr int MBAFF_INTRA_WAVES = 3 * MBAFF_ROWS + 1;
struct MbaffIntraRow {
    WaveIntra tile[2];
    uint32_t hdr[2][4];        // address, availability, residual flag and modes, field flag
    uint32_t ready, done[2];   // MBs prepared, MBs whose luma / chroma is finished
};
struct MbaffIntraShared {
    MbaffIntraRow row[MBAFF_ROWS];
    uint32_t prog[2][MBAFF_ROWS + 1];  // [c][w]: pairs above row w whose luma / chroma is finished
};
// Whether the pairs x0 .. x0 + 63 of row y have an intra top (bottom) MB.
struct PairMask {
    uint64_t top, bot;
};
__device__ __forceinline__ PairMask mbaff_intra_pairs(const DevPic &P, int y, int x0) {
    const int x = x0 + wave_lane();
    const GAS h264g_mb *const m = G(P.mbs) + 2 * (y * P.W + min(x, P.W - 1));
    return {__builtin_amdgcn_ballot_w64(x < P.W && cls_intra(m[0].mb_type)), __builtin_amdgcn_ballot_w64(x < P.W && cls_intra(m[1].mb_type))};
}
__device__ __forceinline__ void mbaff_intra_prep(const DevPic &P, int y, MbaffIntraRow &row, uint32_t *err) {
    const int W = P.W, lane = wave_lane();
    uint32_t n = 0;
    for (int x0 = 0; x0 < W; x0 += WAVE) {
        const PairMask pm = mbaff_intra_pairs(P, y, x0);
        for (uint64_t todo = pm.top | pm.bot; todo; todo &= todo - 1) {
            const int i = (int)__builtin_ctzll(todo);
            for (int h = 0; h < 2; h++) {
                if (!(((h ? pm.bot : pm.top) >> i) & 1u)) continue;
                const int addr = 2 * (y * W + x0 + i) + h;
                const GAS h264g_mb *const m = &G(P.mbs)[addr];
                WaveIntra *const tile = &row.tile[n & 1u];
                const Avail av = intra_avail_mbaff(P, addr);
                const IntraRes r = intra_res_fetch(P, addr);
                const uint32_t type = m->mb_type, modes = (uint32_t)m->intra16x16_pred_mode << 8 | (uint32_t)m->intra_chroma_pred_mode << 16;
                const uint32_t field = m->flags & H264G_MBF_FIELD ? 1u : 0u;
                if (n >= 2) {  // the tile's last MB is finished
                    lds_wait(&row.done[0], 0u, n - 1, err);
                    lds_wait(&row.done[1], 0u, n - 1, err);
                }
                if (type == H264G_MB_I4x4) intra4_prep((const h264g_mb *)m, av, tile);
                else if (type == H264G_MB_I8x8) intra8_prep((const h264g_mb *)m, av, tile);
                intra_res_place(r, tile);
                if (lane < 4) row.hdr[n & 1u][lane] = lane == 0 ? (uint32_t)addr : lane == 1 ? av.m : lane == 2 ? type | modes | (r.res ? 1u << 31 : 0u) : field;
                lds_post(&row.ready, ++n);
            }
        }
    }
}
// Address of dword i of the two bottom rows of pair (px, py).
__device__ __forceinline__ GAS uint32_t *mbaff_bottom(const DbkPlanes &d, int px, int py, int i) {
    const int j = i & 7;
    GAS uint8_t *const p = i < 8 ? G(d.y) + (uint64_t)(py * 32 + 30 + (j >> 2)) * d.wl + px * 16 + 4 * (j & 3)
                                 : G(j < 4 ? d.cb : d.cr) + (uint64_t)(py * 16 + 14 + ((j >> 1) & 1)) * d.wc + px * 8 + 4 * (j & 1);
    return (GAS uint32_t *)p;
}
// Luma (c = 0) or chroma (1) of the row's MBs.
template <int C>
__device__ __forceinline__ void mbaff_intra_row(const DevPic &P, int w, int y, bool send, GAS uint64_t *out, MbaffIntraShared &sh,
                                                uint32_t epoch, uint32_t *err) {
    const int W = P.W, lane = wave_lane();
    const DbkPlanes d = dbk_planes(P);
    MbaffIntraRow &row = sh.row[w];
    uint32_t n = 0;
    for (int x0 = 0; x0 < W; x0 += WAVE) {
        const PairMask pm = mbaff_intra_pairs(P, y, x0);
        for (uint64_t todo = pm.top | pm.bot; todo; todo &= todo - 1) {
            const int i = (int)__builtin_ctzll(todo), x = x0 + i;
            if (!send) lds_post(&sh.prog[C][w + 1], (uint32_t)x);
            if (y > 0) {
                lds_wait(&sh.prog[C][w], 0u, (uint32_t)min(x + 2, W), err);
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
            }
            for (uint32_t k = (uint32_t)((pm.top >> i) & 1u) + (uint32_t)((pm.bot >> i) & 1u); k; k--) {
                lds_wait(&row.ready, 0u, n + 1, err);
                const uint32_t *const hdr = row.hdr[n & 1u];
                const uint32_t addr = uniform(hdr[0]), m = uniform(hdr[2]), bot = addr & 1u;
                const bool field = uniform(hdr[3]) != 0u;
                const Avail av{uniform(hdr[1])};
                MbGeo g;
                g.mbx = x;
                g.bot = (int)bot;
                g.field = field;
                g.step = field ? 2 : 1;
                g.ly = y * 32 + (int)(field ? bot : 16 * bot);
                g.cy = y * 16 + (int)(field ? bot : 8 * bot);
                g.mcy = 0;
                intra_mb<1 << C>(P, g, {(int)(m & 255u), (int)(m >> 8 & 255u), (int)(m >> 16 & 255u)}, &row.tile[n & 1u], av, (m >> 31) != 0u);
                wave_sync();
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");  // its samples before the next MB reads them
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
                lds_post(&row.done[C], ++n);
            }
            if (send && lane < MISTRIP_WORDS / 2) {
                const uint32_t v = *mbaff_bottom(d, x, y, 8 * C + lane);
                __hip_atomic_store(&out[(size_t)x * MISTRIP_WORDS + 8 * C + lane], (uint64_t)epoch << 32 | v, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
            }
        }
        if (!send) lds_post(&sh.prog[C][w + 1], (uint32_t)min(x0 + WAVE, W));
    }
}
// What pair row y, of the band above, hands down.
__device__ __forceinline__ void mbaff_istrip_reader(const DevPic &P, int y, const GAS uint64_t *sw, MbaffIntraShared &sh, uint32_t epoch,
                                                    uint32_t *err) {
    const int W = P.W, lane = wave_lane();
    const DbkPlanes d = dbk_planes(P);
    auto post = [&](int x) {
        lds_post(&sh.prog[0][0], (uint32_t)x);
        lds_post(&sh.prog[1][0], (uint32_t)x);
    };
    for (int x0 = 0; x0 < W; x0 += WAVE) {
        const PairMask pm = mbaff_intra_pairs(P, y, x0);
        for (uint64_t todo = pm.top | pm.bot; todo; todo &= todo - 1) {
            const int x = x0 + (int)__builtin_ctzll(todo);
            post(x);
            uint64_t r;
#pragma unroll 1
            for (uint32_t it = 0;; ++it) {
                r = __hip_atomic_load(&sw[(size_t)x * MISTRIP_WORDS + (lane & (MISTRIP_WORDS - 1))], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (__builtin_amdgcn_ballot_w64((uint32_t)(r >> 32) != epoch) == 0) break;
                if (it >= SPIN_LIMIT) {
                    report_timeout(err);
                    return;
                }
                if ((it & 255u) == 255u && uniform(__hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) != 0u) return;
                __builtin_amdgcn_s_sleep(1);
            }
            if (lane < MISTRIP_WORDS) *mbaff_bottom(d, x, y, lane) = (uint32_t)r;
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        }
        post(min(x0 + WAVE, W));
    }
}
__global__ __launch_bounds__(WAVE *MBAFF_INTRA_WAVES) void k_intra_mbaff(const DevPic *__restrict__ pics, uint32_t n, DevCtl *ctl,
                                                                         uint32_t *epoch_p, uint32_t *err) {
    __shared__ MbaffIntraShared sh;
    __shared__ uint32_t s_ticket;
    const uint32_t epoch = launch_epoch(epoch_p);
    const int wave = (int)uniform(threadIdx.x / WAVE), w = wave / 3, part = wave % 3;
    if ((int)threadIdx.x < MBAFF_ROWS) sh.row[threadIdx.x].ready = sh.row[threadIdx.x].done[0] = sh.row[threadIdx.x].done[1] = 0;
    const uint32_t t = band_ticket(ctl, &s_ticket, &sh.prog[0][0], 2 * (MBAFF_ROWS + 1));
    if (t < gridDim.x) {
        const DevPic &P = pics[t % n];
        const int b = (int)(t / n), HP = P.H >> 1, y0 = b * MBAFF_ROWS, y1 = min(HP, y0 + MBAFF_ROWS), y = y0 + w;
        if (P.mbaff && P.n_intra != 0 && y0 < HP) {
            GAS uint64_t *const strips = G(P.istrip), *const out = strips + (size_t)b * P.W * MISTRIP_WORDS;
            const bool send = y + 1 == y1 && y1 < HP;
            if (w < MBAFF_ROWS) {
                if (y >= y1) {
                } else if (part == 0) {
                    mbaff_intra_prep(P, y, sh.row[w], err);
                } else if (part == 1) {
                    mbaff_intra_row<0>(P, w, y, send, out, sh, epoch, err);
                } else {
                    mbaff_intra_row<1>(P, w, y, send, out, sh, epoch, err);
                }
            } else if (b > 0) {
                mbaff_istrip_reader(P, y0 - 1, strips + (size_t)(b - 1) * P.W * MISTRIP_WORDS, sh, epoch, err);
            }
        }
    }
    band_retire(ctl, epoch_p, epoch);
}

// Row-pipelined deblocking: a ticket is one MB row of one picture (queue ordered by
// row index across pictures, so the row above always holds an earlier ticket).
__global__ __launch_bounds__(WAVE) void k_deblock_rows(const DevPic *__restrict__ pics, const uint32_t *__restrict__ items,
                                                       uint32_t n, DevCtl *ctl, uint32_t *epoch_p, uint32_t *err) {
    __shared__ WaveDbk lds;
    __shared__ DbkTables tb;
    dbk_tables_init(&tb);
    __syncthreads();
    const uint32_t epoch = launch_epoch(epoch_p);
    const uint64_t tag = (uint64_t)epoch << 32;
    for (;;) {
        int t = next_ticket(ctl, n);
        if (t < 0) break;
        const uint32_t it = items[t];
        const DevPic &P = pics[it >> WI_PIC_SHIFT];
        RowSyncGlobal sync{G(P.rowprog), tag, err};
        deblock_row(P, (int)(it & WI_MB_MASK), sync, &lds, &tb);
    }
    retire(ctl, gridDim.x, epoch_p, epoch);
}

// ---- deblocking over bands: one luma row per wave, its four edges side by side
// A band of R MB rows runs on two workgroups, whose chains never meet: one filters the luma
// plane with a wave per MB row, the other Cb and Cr with a wave per two rows.  A wave walks
// its row from left to right.  Per MB it filters the vertical edges, hands the finished MB
// to its left down to the next row, takes the rows above its MB over from the previous row
// and filters the horizontal edges, so a row runs about one step behind the row above it
// and a picture takes about W + H steps.
//
// Bound: that chain, i.e. the instructions and LDS round trips of one step (about 0.8 us).
// Lane 16 e + k filters edge e (samples 4 e of the direction) on line k: the edges of a line
// do not depend on each other but for one sample (edge_pass), so the four run side by side
// instead of one after the other.  gfx950's transposing LDS read (lds_tr) hands each lane
// the 8 samples around its edge along a column straight from the rows, so ds_read_b64_tr_b8
// is the whole change of direction.  What a step needs from device memory was loaded
// DBK_AHEAD steps before, its thresholds were looked up one step before.  Measured (whole
// launch, one picture; before: two MB rows per wave, a line's edges in order): 352x288 108 to
// 38 us (P), 1920x1088 592 to 159 (P) / 196 us (I), 3840x2160 1152 to 309 / 391 us.  Lines
// kept in registers with the edges in order, four rows per wave, took 330 / 369 us at
// 1920x1088: instructions bound that step too, 8 edges of ~70 each.
//
// Row y hands the bottom 4 rows (chroma: 2) of each MB, the p samples of the next row's top
// edge, to row y + 1 as a strip, as soon as the right neighbour's left edge has taken its
// columns: inside a chroma wave through LDS, from wave to wave through a ring of STRIP_SLOTS
// slots (a slot is written again only once the reader has taken it; every wave of a band is
// resident, so the reader is always running), from a band to the next through tagged words
// in device memory (StripWords), which a wave of its own brings into the next band's first
// ring (strip_reader).  Each sample is written to the picture by one lane: rows 0..12 (chroma
// 0..6) by their own row after the right neighbour's left edge, the others by the row below
// after its top edge.
constexpr int STRIP_SLOTS = 8;
constexpr int DBK_MAX_ROWS = H264G_DBK_MAX_ROWS;  // MB rows of a band, one luma wave each
constexpr int DBK_AHEAD = 3;

struct alignas(16) LumaTile {
    uint8_t img[2][16][16];    // MB x in half x & 1: as loaded, then after its vertical edges
    uint8_t col[16][16];       // its columns after the horizontal edges
};
struct alignas(16) ChromaTile {    // one of a wave's two rows; 16-byte lines: Cb in 0..7, Cr in 8..15
    uint8_t img[2][8][16];
    uint8_t col[8][16];
    uint8_t strip[2][16];      // the rows above the MB
};
// Tables 8-16 / 8-17 as the edges read them: at[indexA][bS] = alpha' | tC0 << 16 (alpha' 0
// for bS 0, so that nothing passes the threshold), beta[indexB] = beta' in both halves.
struct DbkLut {
    uint32_t at[52][8];
    uint32_t beta[52];
};
struct DbkWgShared {
    union {
        LumaTile l[DBK_MAX_ROWS];
        ChromaTile c[DBK_MAX_ROWS];
    };
    // strips on their way: ring 0 from the band above to wave 0, ring w + 1 from wave w to wave
    // w + 1 (chroma: 32 bytes of a slot)
    alignas(16) uint8_t ring[DBK_MAX_ROWS + 1][STRIP_SLOTS][64];
    uint32_t prog[DBK_MAX_ROWS + 1];   // strips 0 .. prog - 1 are in the ring
    uint32_t cons[DBK_MAX_ROWS + 1];   // strips 0 .. cons - 1 have been read
    DbkLut lut;
};

__device__ void dbk_lut_init(DbkLut *t) {
    for (int i = threadIdx.x; i < 52 * 8; i += blockDim.x) {
        const int a = i >> 3, bS = i & 7;
        t->at[a][bS] = bS < 1 || bS > 4 ? 0u : (uint32_t)c_alpha[a] | (bS < 4 ? (uint32_t)c_tc0[bS - 1][a] << 16 : 0u);
    }
    for (int i = threadIdx.x; i < 52; i += blockDim.x) t->beta[i] = (uint32_t)c_beta[i] * 0x10001u;
}

// The value of the lane 16 below (row e of 16 lanes gets row e - 1; row 0 anything).
__device__ __forceinline__ uint32_t row_below(uint32_t v, int e) {
    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
    const u32x2 r = __builtin_amdgcn_permlane16_swap(v, v, false, false);      // rows 0 0 2 2 | 1 1 3 3
    const u32x2 t = __builtin_amdgcn_permlane32_swap(r.y, r.y, false, false);  // rows 1 1 1 1
    return e == 2 ? t.x : r.x;
}

// The edges of one direction of a MB on the lanes' samples: a = p3 p2 p1 p0 (bytes 0..3),
// b = q0 q1 q2 q3 of the lane's line and edge; at: the DbkLut entry of (indexA, bS), beta: of
// indexB; e: the lane's edge (0: the MB edge).  8.7.2.2 - 8.7.2.4 (Deblock.cpp:1314-1522) on
// (p, q) pairs: the two sides are mirror images, so one packed 16-bit operation serves both.
// Conditions are packed sign masks, and the wave skips what no lane needs.
//
// Luma edges side by side: with bS < 4 an edge changes p1 p0 q0 q1 and reads p2 .. q2, so the
// only sample that edge e + 1 sees changed by edge e is its p2 (edge e's q1), and edge e's
// q1 does not depend on its own p2.  So every lane finds its q1, passes it up as the next
// edge's p2 and finishes.  bS 4 (s4, the MB edge only) changes up to q2, which edge 1 reads
// as p1: where a lane needs it, it goes first.  Chroma (LUMA false): p1 .. q1 are read, p0
// and q0 changed, and edges 8 samples apart in luma are 4 apart: nothing is shared.
template <bool LUMA>
__device__ __forceinline__ void edge_pass(uint32_t &a, uint32_t &b, uint32_t at, uint32_t beta, bool s4, int e) {
    const s16x2 zero = {0, 0}, be = as_pair(beta);
    if (any_lane(s4)) {
        const s16x2 t = as_pair(at), al = __builtin_shufflevector(t, t, 0, 0);
        const s16x2 P0 = as_pair(__builtin_amdgcn_perm(b, a, 0x0c040c03u)), P1 = as_pair(__builtin_amdgcn_perm(b, a, 0x0c050c02u));
        const s16x2 X0 = pair_swap(P0), X1 = pair_swap(P1);
        const s16x2 D0 = P0 - X0, A0 = __builtin_elementwise_max(D0, pair_swap(D0));  // |p0 - q0| in both halves
        const s16x2 T = __builtin_elementwise_max(P1 - P0, P0 - P1) - be;
        const s16x2 M = __builtin_elementwise_max(__builtin_elementwise_max(T, pair_swap(T)), A0 - al) >> 15;
        const uint32_t ms = s4 ? as_bits(M) : 0u;
        const uint32_t W0 = as_bits((P1 + P1 + P0 + X1 + (s16x2){2, 2}) >> 2);        // 2p1 + p0 + q1 + 2
        uint32_t n0 = (W0 & ms) | (as_bits(P0) & ~ms);
        if (LUMA) {
            const s16x2 P2 = as_pair(__builtin_amdgcn_perm(b, a, 0x0c060c01u)), P3 = as_pair(__builtin_amdgcn_perm(b, a, 0x0c070c00u));
            const s16x2 MA = (__builtin_elementwise_max(P2 - P0, P0 - P2) - be) >> 15;  // ap, aq < beta
            // strong sides: |p0 - q0| < (alpha >> 2) + 2 as well
            const uint32_t st = as_bits((A0 - ((al >> 2) + (s16x2){2, 2})) >> 15) & as_bits(MA) & ms;
            const s16x2 sum = P1 + P0 + X0;
            const uint32_t S0 = as_bits((sum + sum + P2 + X1 + (s16x2){4, 4}) >> 3);
            const uint32_t S1 = as_bits((sum + P2 + (s16x2){2, 2}) >> 2);
            const uint32_t S2 = as_bits((P3 + P3 + P2 * (s16x2){3, 3} + sum + (s16x2){4, 4}) >> 3);
            n0 = (S0 & st) | (n0 & ~st);
            const uint32_t n1 = (S1 & st) | (as_bits(P1) & ~st), n2 = (S2 & st) | (as_bits(P2) & ~st);
            const uint32_t t01 = __builtin_amdgcn_perm(n1, n0, 0x06020400u);                                // np0 np1 nq0 nq1
            const uint32_t w = __builtin_amdgcn_perm(n2, t01, 0x06040100u);                                 // np0 np1 np2 nq2
            b = __builtin_amdgcn_perm(b, __builtin_amdgcn_perm(w, t01, 0x0c070302u), 0x07020100u);      // nq0 nq1 nq2 q3
            a = __builtin_amdgcn_perm(w, a, 0x04050600u);                                                  // p3 np2 np1 np0
            const uint32_t up = row_below(b, e);
            a = e == 1 ? up : a;                                                                           // edge 1's p side
        } else {
            a = __builtin_amdgcn_perm(n0, a, 0x04020100u);
            b = __builtin_amdgcn_perm(b, n0, 0x07060502u);
        }
    }
    const s16x2 t = as_pair(s4 ? 0u : at), al = __builtin_shufflevector(t, t, 0, 0), tc0 = __builtin_shufflevector(t, t, 1, 1);
    const s16x2 P0 = as_pair(__builtin_amdgcn_perm(b, a, 0x0c040c03u)), P1 = as_pair(__builtin_amdgcn_perm(b, a, 0x0c050c02u));
    const s16x2 D0 = P0 - pair_swap(P0), A0 = __builtin_elementwise_max(D0, pair_swap(D0));
    const s16x2 T = __builtin_elementwise_max(P1 - P0, P0 - P1) - be;
    // all three conditions: negative in both halves
    const s16x2 M = __builtin_elementwise_max(__builtin_elementwise_max(T, pair_swap(T)), A0 - al) >> 15;
    const uint32_t m = as_bits(M);
    if (!any_lane(m != 0u)) return;
    s16x2 tc, N1 = P1;
    if (LUMA) {
        s16x2 P2 = as_pair(__builtin_amdgcn_perm(b, a, 0x0c060c01u));
        // (p0 + q0 + 1) >> 1 in both halves
        const s16x2 avg = as_pair(__builtin_amdgcn_lerp(as_bits(P0), __builtin_amdgcn_alignbit(as_bits(P0), as_bits(P0), 16), 0x01010101u));
        const s16x2 ntc0 = zero - tc0, base = avg - (P1 + P1);
        // p'1 = p1 + Clip3(-tC0, tC0, (p2 + avg - 2 p1) >> 1) where ap < beta, q'1 alike
        auto side1 = [&](s16x2 &ma) {
            ma = (__builtin_elementwise_max(P2 - P0, P0 - P2) - be) >> 15;
            const s16x2 u = pair_clip((P2 + base) >> 1, ntc0, tc0);
            return P1 + as_pair(as_bits(u) & as_bits(ma) & m);
        };
        s16x2 MA;
        const s16x2 Q1 = side1(MA);
        const uint32_t up = row_below(as_bits(Q1) >> 16, e);
        P2 = e ? as_pair((as_bits(P2) & 0xFFFF0000u) | up) : P2;
        N1 = side1(MA);
        tc = tc0 - MA - pair_swap(MA);  // tC0 + [ap < beta] + [aq < beta]
    } else {
        tc = tc0 + (s16x2){1, 1};
    }
    // bS < 4 (8.7.2.3): delta in the low half
    s16x2 dl = (D0 * (s16x2){-4, -4} + (P1 - pair_swap(P1)) + (s16x2){4, 4}) >> 3;
    dl = pair_clip(dl, zero - tc, tc);
    const s16x2 f0 = pair_clip(__builtin_shufflevector(dl, dl, 0, 0) * (s16x2){1, -1} + P0, zero, (s16x2){255, 255});
    const uint32_t n0 = (as_bits(f0) & m) | (as_bits(P0) & ~m);
    if (LUMA) {
        const uint32_t t01 = __builtin_amdgcn_perm(as_bits(N1), n0, 0x06020400u);  // np0 np1 nq0 nq1
        const uint32_t p2 = a;
        a = __builtin_amdgcn_perm(t01, p2, 0x04050100u);                  // p3 p2 np1 np0
        b = __builtin_amdgcn_perm(b, t01, 0x07060302u);                   // nq0 nq1 q2 q3
    } else {
        a = __builtin_amdgcn_perm(n0, a, 0x04020100u);                    // p3 p2 p1 np0
        b = __builtin_amdgcn_perm(b, n0, 0x07060502u);                    // nq0 q1 q2 q3
    }
}

// One lane's edge in one direction: its DbkLut entries and whether its bS is 4.
struct DbkThr {
    uint32_t at, beta;
    bool s4;
};
// mb: the edge is the MB edge to a MB with deblocking word nb (own: or to the MB's own values).
__device__ __forceinline__ DbkThr dbk_threshold(const DbkLut *lut, uint32_t bS, int plane, uint32_t q, uint32_t nb, bool own,
                                                bool mb, int offA, int offB) {
    const int qq = dbq_qp(q, plane), qn = own || !mb ? qq : dbq_qp(nb, plane), qav = (qq + qn + 1) >> 1;
    DbkThr t;
    t.at = lut->at[clip3(0, 51, qav + offA)][bS & 7u];
    t.beta = lut->beta[clip3(0, 51, qav + offB)];
    t.s4 = bS == 4u;
    return t;
}

// Strips that cross from a band to the next (another workgroup, possibly another XCD) go
// through device memory as words of 64 bits: a strip dword in the low half, the launch
// epoch in the high half (luma dwords 0..15, chroma 16..23).  Each word is stored and
// loaded as one agent-scope atomic, so a reader that finds the epoch in a word holds its
// samples; neither side needs a fence, whose L2 write-back / invalidation would also hit
// every other kernel running on those XCDs.
struct StripWords {
    uint64_t w[32];
};
// The reader wave of a band: strips (N words from word AT) of the row `sw` into ring 0, as
// many at a time as the wave has lanes for; the rows then find every strip in LDS, whatever
// the band above lags, and one poll's round trip serves several of them.
template <int N, int AT>
__device__ __forceinline__ void strip_reader(const GAS StripWords *sw, int W, DbkWgShared &sh, uint32_t epoch, uint32_t *err) {
    constexpr int AT_ONCE = WAVE / N;
    static_assert(AT_ONCE <= STRIP_SLOTS, "a round of strips fits the ring");
    const int lane = wave_lane(), mine = lane / N, word = lane % N;
    for (int x0 = 0; x0 < W; x0 += AT_ONCE) {
        const int n = min(AT_ONCE, W - x0);
        int have = 0;  // strips x0 .. x0 + have - 1 are in the ring
#pragma unroll 1
        for (uint32_t it = 0; have < n; ++it) {
            const uint64_t r = __hip_atomic_load(&sw[x0 + min(mine, n - 1)].w[AT + word], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            // the lanes whose words have arrived, up to the first strip that has not
            const uint64_t missing = __builtin_amdgcn_ballot_w64((uint32_t)(r >> 32) != epoch);
            const int got = missing ? min(n, (int)(__builtin_ctzll(missing) / N)) : n;
            if (got > have) {
                const int x = x0 + got - 1;
                if (x >= STRIP_SLOTS) lds_wait(&sh.cons[0], 0u, (uint32_t)(x - STRIP_SLOTS + 1), err);  // slots read?
                if (mine >= have && mine < got) *(uint32_t *)&sh.ring[0][(x0 + mine) % STRIP_SLOTS][4 * word] = (uint32_t)r;
                lds_post(&sh.prog[0], (uint32_t)x + 1);
                have = got;
                continue;
            }
            if (it >= SPIN_LIMIT) {
                report_timeout(err);
                return;
            }
            if ((it & 255u) == 255u && uniform(__hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) != 0u) return;
            __builtin_amdgcn_s_sleep(1);
        }
    }
}

// MB row y = y0 + w of the band of rows y0 .. y1 - 1 (band index b): the luma plane.
__device__ __forceinline__ void deblock_luma_row(const DevPic &P, int w, int y0, int y1, int b, DbkWgShared &sh, uint32_t epoch,
                                                 uint32_t *err) {
    const int W = P.W, H = P.H, y = y0 + w;
    const int lane = wave_lane(), e = lane >> 4, k = lane & 15;
    const bool top = y > 0, last = y == H - 1;
    const bool ring_out = y + 1 < y1, g_out = !ring_out && !last;
    LumaTile *const tile = &sh.l[w];
    GAS StripWords *const gout = (GAS StripWords *)G(P.gstrip) + (size_t)b * W;
    gu8 *const slot = slot_base(P, P.dst);
    const uint32_t pitch = (uint32_t)W * 16u, row0 = (uint32_t)(y * 16) * pitch;
    // as loaded: lane 4 r + d takes dword d of row r; as stored: lanes 0-15 bytes 8..15 of row
    // k, lanes 16-31 bytes 0..7
    const uint32_t ld = row0 + (uint32_t)(lane >> 2) * pitch + (uint32_t)(lane & 3) * 4u;
    const uint32_t so = row0 + (uint32_t)k * pitch + (e == 0 ? 8u : 0u);
    const gu8 *const bsv = G(P.bs) + (uint32_t)((k >> 2) * 4 + e);
    const gu8 *const dq = (const gu8 *)G(P.dbq);
    const uint32_t mb0 = (uint32_t)(y * W), mbt = top ? (uint32_t)W * 4u : 0u;
    const int offA = P.offA, offB = P.offB;
    struct Ahead {
        uint32_t px, bv, bh, q, qt;
    };
    // (no branches, so that the loads stay in flight: past the row's end they read its last MB)
    auto fetch = [&](int x) {
        const uint32_t xc = (uint32_t)min(x, W - 1), a = mb0 + xc;
        Ahead f;
        f.px = *(const GAS uint32_t *)(slot + (ld + xc * 16u));
        f.bv = bsv[a * 32u];
        f.bh = bsv[a * 32u + 16u];
        f.q = *(const GAS uint32_t *)(dq + a * 4u);
        f.qt = *(const GAS uint32_t *)(dq + (a * 4u - mbt));
        return f;
    };
    // LDS addresses: the transposing reads (lane 2j + h of a group names half h of line j)
    const int tj = k >> 1, th = (k & 1) * 8, tr = 4 * (e - 1) + tj;      // row tr around edge e
    const bool tr_strip = tr < 0;
    const uint8_t *const tr_c = &tile->col[(e == 0 ? 8 : 0) + tj][th];  // columns 8..15 for lanes 0-15, else 0..7
    const int sr = k - 12;                                               // the lane's strip row, from row 12 on
    Ahead f[DBK_AHEAD] = {fetch(0), fetch(1), fetch(2)};
    ((uint32_t *)tile->img[0])[lane] = f[0].px;
    wave_sync();
    uint32_t bq = *(const uint32_t *)&tile->img[0][k][4 * e], ap = *(const uint32_t *)&tile->img[0][k][4 * max(e - 1, 0)];
    DbkThr thv = dbk_threshold(&sh.lut, f[0].bv, 0, f[0].q, 0u, false, e == 0, offA, offB);
    DbkThr thh = dbk_threshold(&sh.lut, f[0].bh, 0, f[0].q, f[0].qt, f[0].q & DBQ_OWN_TOP, e == 0, offA, offB);
    uint2 prev = make_uint2(0u, 0u);   // MB x - 1 after its horizontal edges: row k, bytes 8..15 (lanes 0-15) or 0..7
    // MB m = x - 1 once MB x has taken its left edge (seen: sh.cons of the row's ring, read
    // before): final but for rows 13..15, so its strip is handed down and it is stored
    auto finish = [&](int m, uint32_t seen) {
        if (ring_out) {
            if (m >= STRIP_SLOTS) lds_wait(&sh.cons[w + 1], seen, (uint32_t)(m - STRIP_SLOTS + 1), err);  // slot read?
            if (lane < 32 && sr >= 0) *(uint2 *)&sh.ring[w + 1][m % STRIP_SLOTS][sr * 16 + (e == 0 ? 8 : 0)] = prev;
            lds_post(&sh.prog[w + 1], (uint32_t)m + 1);
        } else if (g_out && lane < 32 && sr >= 0) {
            GAS uint64_t *const d = &gout[m].w[sr * 4 + (e == 0 ? 2 : 0)];
            __hip_atomic_store(&d[0], (uint64_t)epoch << 32 | prev.x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(&d[1], (uint64_t)epoch << 32 | prev.y, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        if (lane < 32 && (sr < 1 || last)) *(GAS uint2 *)(slot + (so + (uint32_t)m * 16u)) = prev;
    };
    // MB x; cur: its register set, refilled for MB x + DBK_AHEAD; nxt: that of MB x + 1
    auto step = [&](int x, Ahead &cur, Ahead &nxt) {
        const uint32_t q0 = cur.q;
        cur = fetch(x + DBK_AHEAD);
        uint8_t *const img = &tile->img[x & 1][0][0], *const nimg = &tile->img[(x + 1) & 1][0][0];
        ((uint32_t *)nimg)[lane] = nxt.px;
        const uint32_t seen = lds_peek(&sh.prog[w]), seen_c = lds_peek(&sh.cons[w + 1]);
        // ---- vertical edges: a is row k's dword before the edge, b the one after it
        {
            uint32_t a = e ? ap : prev.y, bb = bq;
            edge_pass<true>(a, bb, thv.at, thv.beta, thv.s4, e);
            *(uint32_t *)&img[k * 16 + 4 * e] = bb;
            wave_sync();  // (the next edge's p side lies in the dword just written)
            if (e) *(uint16_t *)&img[k * 16 + 4 * e - 2] = (uint16_t)(a >> 16);
            else prev.y = a;
        }
        if (x > 0 && x <= W) finish(x - 1, seen_c);
        // ---- the rows above the MB
        if (top && x < W) lds_wait(&sh.prog[w], seen, (uint32_t)x + 1, err);
        const uint8_t *const strip = sh.ring[w][x % STRIP_SLOTS];
        wave_sync();
        // ---- horizontal edges: a and b are rows 4 e - 4 .. 4 e + 3 of column k
        const uint2 c = lds_tr(tr_strip ? strip + (tr + 4) * 16 + th : img + tr * 16 + th);
        bq = *(const uint32_t *)&nimg[k * 16 + 4 * e];
        ap = *(const uint32_t *)&nimg[k * 16 + 4 * max(e - 1, 0)];
        // the next step's thresholds (opaque words: the compiler would narrow them as they
        // arrive and wait for their loads steps ahead of this use)
        asm volatile("" : "+v"(nxt.q), "+v"(nxt.qt), "+v"(nxt.bv), "+v"(nxt.bh));
        const DbkThr nv = dbk_threshold(&sh.lut, x + 1 < W ? nxt.bv : 0u, 0, nxt.q, q0, nxt.q & DBQ_OWN_LEFT, e == 0, offA, offB);
        const DbkThr nh = dbk_threshold(&sh.lut, nxt.bh, 0, nxt.q, nxt.qt, nxt.q & DBQ_OWN_TOP, e == 0, offA, offB);
        lds_post(&sh.cons[w], (uint32_t)x + 1);
        uint32_t a = c.x, bb = c.y;
        edge_pass<true>(a, bb, thh.at, thh.beta, thh.s4, e);
        *(uint32_t *)&tile->col[k][4 * e] = bb;
        wave_sync();
        if (e) {
            *(uint16_t *)&tile->col[k][4 * e - 2] = (uint16_t)(a >> 16);
        } else if (top && x < W) {  // the rows of the MB above that its top edge changes: column k's bytes
            const uint32_t o = row0 - pitch + (uint32_t)(x * 16 + k);
            slot[o] = (uint8_t)(a >> 24);
            slot[o - pitch] = (uint8_t)(a >> 16);
            slot[o - 2u * pitch] = (uint8_t)(a >> 8);
        }
        wave_sync();
        prev = lds_tr(tr_c);
        thv = nv;
        thh = nh;
    };
    // Unrolled over the DBK_AHEAD register sets (moving a set would wait for its loads); steps
    // past the row's end filter nothing (an exit between the steps would make the compiler
    // wait for all stores at the loop's head).
    for (int x = 0; x < W; x += DBK_AHEAD) {
        step(x, f[0], f[1]);
        step(x + 1, f[1], f[2]);
        step(x + 2, f[2], f[0]);
    }
    if (W % DBK_AHEAD == 0) finish(W - 1, 0u);
}

// MB rows y0 + 2 w and y0 + 2 w + 1 (lanes 32-63, one MB behind) of the band of rows
// y0 .. y1 - 1 (band index b): the chroma planes.  Lane 16 e + 8 p + k of a row's 32: edge e
// of line k of plane p.
__device__ __forceinline__ void deblock_chroma_rows(const DevPic &P, int w, int y0, int y1, int b, DbkWgShared &sh, uint32_t epoch,
                                                    uint32_t *err) {
    const int W = P.W, H = P.H, yw = y0 + 2 * w;
    const bool two = yw + 1 < y1;
    const int lane = wave_lane(), g = lane >> 5, e = (lane >> 4) & 1, pk = lane & 15, p = pk >> 3, k = pk & 7;
    const bool rowok = g == 0 || two;
    const int y = yw + (two ? g : 0), gl = two ? 1 : 0, yl = yw + gl;  // (an absent second row reads the first's)
    const bool top = y > 0, last = y == H - 1;
    const bool ring_out = yl + 1 < y1, g_out = !ring_out && yl < H - 1;
    ChromaTile *const tile = &sh.c[2 * w + g];
    uint8_t *const strip_dn = &sh.c[2 * w + 1].strip[0][0];
    GAS StripWords *const gout = (GAS StripWords *)G(P.gstrip) + (size_t)b * W;
    gu8 *const slot = slot_base(P, P.dst);
    const uint32_t pitch = (uint32_t)W * 8u, np = (uint32_t)(W * H), row0 = (uint32_t)(y * 8) * pitch;
    // as loaded: lane 16 p + 2 r + d of the row takes dword d of row r of plane p
    const int lp = (lane >> 4) & 1, lr = (lane >> 1) & 7, ldw = lane & 1;
    const uint32_t ld = np * (lp ? 320u : 256u) + row0 + (uint32_t)lr * pitch + (uint32_t)ldw * 4u;
    const uint32_t pl = np * (p ? 320u : 256u) + row0, so = pl + (uint32_t)k * pitch;
    const gu8 *const bsv = G(P.bs) + (uint32_t)((k >> 1) * 4 + 2 * e);  // chroma edge e lies on luma edge 2 e
    const gu8 *const dq = (const gu8 *)G(P.dbq);
    const uint32_t mb0 = (uint32_t)(y * W), mbt = top ? (uint32_t)W * 4u : 0u;
    const int offA = P.offA, offB = P.offB;
    struct Ahead {
        uint32_t px, bv, bh, q, qt;
    };
    auto fetch = [&](int x) {
        const uint32_t xc = (uint32_t)clip3(0, W - 1, x), a = mb0 + xc;
        Ahead f;
        f.px = *(const GAS uint32_t *)(slot + (ld + xc * 8u));
        f.bv = bsv[a * 32u];
        f.bh = bsv[a * 32u + 16u];
        f.q = *(const GAS uint32_t *)(dq + a * 4u);
        f.qt = *(const GAS uint32_t *)(dq + (a * 4u - mbt));
        return f;
    };
    const int tj = pk >> 1, th = (pk & 1) * 8, tr = 4 * (e - 1) + tj;
    const bool tr_strip = tr < 0;
    const uint8_t *const tr_c = &tile->col[tj][th];
    const int sr = k - 6;
    auto active = [&](int x) { return rowok && (uint32_t)x < (uint32_t)W; };
    Ahead f[DBK_AHEAD] = {fetch(-g), fetch(1 - g), fetch(2 - g)};
    auto place = [&](int x, uint32_t v) {  // MB x as loaded, into its half of the tile
        *(uint32_t *)&tile->img[x & 1][lr][lp * 8 + ldw * 4] = v;
    };
    place(-g, f[0].px);
    wave_sync();
    uint32_t bq = *(const uint32_t *)&tile->img[g & 1][k][p * 8 + 4 * e], ap = *(const uint32_t *)&tile->img[g & 1][k][p * 8];
    DbkThr thv = dbk_threshold(&sh.lut, active(-g) ? f[0].bv : 0u, 1 + p, f[0].q, 0u, false, e == 0, offA, offB);
    DbkThr thh = dbk_threshold(&sh.lut, active(-g) ? f[0].bh : 0u, 1 + p, f[0].q, f[0].qt, f[0].q & DBQ_OWN_TOP, e == 0, offA, offB);
    uint2 prev = make_uint2(0u, 0u);   // MB x - 1 after its horizontal edges: row k of plane p
    // After the vertical edges of step s: MB x - 1 is final but for row 7, so its strip is handed
    // down and it is stored (m: the MB of the wave's last row; seen: sh.cons of its ring)
    auto finish = [&](int s, uint32_t seen) {
        const int x = s - g, m = s - gl - 1;
        const bool had = rowok && x >= 1 && x <= W;
        if (had && e == 0 && sr >= 0 && g < gl) *(uint2 *)(strip_dn + sr * 16 + p * 8) = prev;
        if (m >= 0 && m < W) {
            if (ring_out) {
                if (m >= STRIP_SLOTS) lds_wait(&sh.cons[w + 1], seen, (uint32_t)(m - STRIP_SLOTS + 1), err);  // slot read?
                if (g == gl && e == 0 && sr >= 0) *(uint2 *)&sh.ring[w + 1][m % STRIP_SLOTS][sr * 16 + p * 8] = prev;
                lds_post(&sh.prog[w + 1], (uint32_t)m + 1);
            } else if (g_out && g == gl && e == 0 && sr >= 0) {
                GAS uint64_t *const d = &gout[m].w[16 + sr * 4 + p * 2];
                __hip_atomic_store(&d[0], (uint64_t)epoch << 32 | prev.x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                __hip_atomic_store(&d[1], (uint64_t)epoch << 32 | prev.y, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
        if (had && e == 0 && (sr < 1 || last)) *(GAS uint2 *)(slot + (so + (uint32_t)(x - 1) * 8u)) = prev;
    };
    auto step = [&](int s, Ahead &cur, Ahead &nxt) {
        const int x = s - g;
        const bool act = active(x);
        const uint32_t q0 = cur.q;
        cur = fetch(x + DBK_AHEAD);
        place(x + 1, nxt.px);
        const uint32_t seen = lds_peek(&sh.prog[w]), seen_c = lds_peek(&sh.cons[w + 1]);
        // ---- vertical edges
        uint8_t(*const img)[16] = tile->img[x & 1], (*const nimg)[16] = tile->img[(x + 1) & 1];
        {
            uint32_t a = e ? ap : prev.y, bb = bq;
            edge_pass<false>(a, bb, thv.at, thv.beta, thv.s4, e);
            *(uint32_t *)&img[k][p * 8 + 4 * e] = bb;
            wave_sync();
            if (e) img[k][p * 8 + 3] = (uint8_t)(a >> 24);
            else prev.y = a;
        }
        finish(s, seen_c);
        // ---- the rows above the MBs
        if (y0 + 2 * w > 0 && s < W) lds_wait(&sh.prog[w], seen, (uint32_t)s + 1, err);
        const uint8_t *const strip = g == 0 ? sh.ring[w][s % STRIP_SLOTS] : &tile->strip[0][0];
        wave_sync();
        // ---- horizontal edges (rows -2, -1 are the strip; rows -4, -3 are not read)
        const uint2 c = lds_tr(tr_strip ? strip + max(tr + 2, 0) * 16 + th : &img[max(tr, 0)][th]);
        bq = *(const uint32_t *)&nimg[k][p * 8 + 4 * e];
        ap = *(const uint32_t *)&nimg[k][p * 8];
        asm volatile("" : "+v"(nxt.q), "+v"(nxt.qt), "+v"(nxt.bv), "+v"(nxt.bh));
        const DbkThr nv = dbk_threshold(&sh.lut, active(x + 1) ? nxt.bv : 0u, 1 + p, nxt.q, q0, nxt.q & DBQ_OWN_LEFT, e == 0, offA, offB);
        const DbkThr nh = dbk_threshold(&sh.lut, active(x + 1) ? nxt.bh : 0u, 1 + p, nxt.q, nxt.qt, nxt.q & DBQ_OWN_TOP, e == 0, offA, offB);
        lds_post(&sh.cons[w], (uint32_t)s + 1);
        uint32_t a = c.x, bb = c.y;
        edge_pass<false>(a, bb, thh.at, thh.beta, thh.s4, e);
        *(uint32_t *)&tile->col[k][p * 8 + 4 * e] = bb;
        wave_sync();
        if (e) tile->col[k][p * 8 + 3] = (uint8_t)(a >> 24);
        else if (act && top) slot[pl - pitch + (uint32_t)(x * 8 + k)] = (uint8_t)(a >> 24);  // row 7 of the MB above
        wave_sync();
        prev = lds_tr(tr_c);
        thv = nv;
        thh = nh;
    };
    const int steps = W + gl;
    for (int s = 0; s < steps; s += DBK_AHEAD) {
        step(s, f[0], f[1]);
        step(s + 1, f[1], f[2]);
        step(s + 2, f[2], f[0]);
    }
    if (steps % DBK_AHEAD == 0) finish(steps, 0u);  // the last row's last MB
}

// Two workgroups per band of `rows` MB rows, item 2 i for the luma plane of band i, item
// 2 i + 1 for its chroma planes; the workgroup's last wave reads the strips of the band above.
__global__ __launch_bounds__(WAVE *(DBK_MAX_ROWS + 1)) void k_deblock_band(const DevPic *__restrict__ pics,
                                                                           const uint32_t *__restrict__ items, uint32_t n,
                                                                           int rows, DevCtl *ctl, uint32_t *epoch_p,
                                                                           uint32_t *err) {
    __shared__ DbkWgShared sh;
    __shared__ uint32_t s_ticket;
    const uint32_t epoch = launch_epoch(epoch_p);
    const int w = (int)uniform(threadIdx.x / WAVE);
    if ((int)threadIdx.x <= rows) sh.cons[threadIdx.x] = 0;
    dbk_lut_init(&sh.lut);
    const uint32_t t = band_ticket(ctl, &s_ticket, sh.prog, rows + 1);
    if (t < 2 * n) {
        const uint32_t it = items ? items[t >> 1] : t >> 1;
        const DevPic &P = pics[it >> WI_PIC_SHIFT];
        const int b = (int)(it & WI_MB_MASK), y0 = b * rows, y1 = min(P.H, y0 + rows);
        const GAS StripWords *const above = (const GAS StripWords *)G(P.gstrip) + (size_t)(b > 0 ? b - 1 : 0) * P.W;
        if (P.dbk_idc != 1) {
            if (!(t & 1u)) {
                if (w < rows) {
                    if (y0 + w < y1) deblock_luma_row(P, w, y0, y1, b, sh, epoch, err);
                } else if (b > 0) {
                    strip_reader<16, 0>(above, P.W, sh, epoch, err);
                }
            } else {
                if (w < rows) {
                    if (y0 + 2 * w < y1) deblock_chroma_rows(P, w, y0, y1, b, sh, epoch, err);
                } else if (b > 0) {
                    strip_reader<8, 16>(above, P.W, sh, epoch, err);
                }
            }
        }
    }
    band_retire(ctl, epoch_p, epoch);
}

// Boundary strengths of every edge segment of every MB (8.7.2.1, Deblock.cpp:994-1310),
// stored [direction][4-line segment][edge] so that a deblocking line reads its four edges
// as one dword, and each MB's deblocking word (G(P.dbq): qP of luma / Cb edges / Cr edges in
// bytes 0..2, transform_size_8x8_flag in bit 24, the own-qP flags of its MB edges in bits
// 25 / 26); fully parallel: they depend on syntax
// only, not on samples.  Half a wave per MB (neighbouring MBs, so that an XCD's L2 serves the
// records two MBs share); lane j = 16 * dir + 4 * edge + segment.
__device__ __forceinline__ void bs_pair_of_mbs(const DevPic *pics, const uint32_t *chunks, uint32_t b, uint32_t n) {
    const int lane = wave_lane();
    const MbSlot m = mb_slot(chunks, 2 * xcd_item(b, n));
    const DevPic &P = pics[m.pic];
    const int addr = m.addr + (lane >> 5), W = P.W, mbx = addr % W, mby = addr / W;
    if (addr >= W * P.H || P.dbk_idc == 1) return;
    const int j = lane & 31, dir = j >> 4, e = ((j >> 2) & 3) * 4, k = (j & 3) * 4;
    int bS = 0;
    const bool has_nb = dir == 0 ? mbx > 0 : mby > 0;
    const uint32_t sq = P.multi_slice ? G(P.mbs)[addr].slice_num : 0u;
    const bool other = P.multi_slice && e == 0 && has_nb && G(P.mbs)[dir == 0 ? addr - 1 : addr - W].slice_num != sq;
    // An MB edge at the picture border is not filtered, nor, with disable_deblocking_filter_idc
    // 2, one between two slices (8.7: filterLeftMbEdgeFlag / filterTopMbEdgeFlag); no edge
    // of an MB at or after the deblocking stop is.  With idc 0 the reference filters an
    // edge between slices with the current MB in the neighbour's place (its neighbour
    // derivation reports the other slice's MB as unavailable and the p-MB address stays
    // the current one, Deblock.cpp:747-760, 784-791): the bS of an internal edge between
    // the current MB's blocks at x (or y) 15 and 0, and the current MB's qP on both sides.
    const bool own = e == 0 && other && P.dbk_idc == 0;
    const int ap = (e || own) ? addr : (dir == 0 ? addr - 1 : addr - W);
    // Nor are the internal luma edges 4 and 12 of an MB with the 8x8 transform.
    const bool t8_skip = (e & 4) && (G(P.aux)[addr].kind & AUX_T8);
    const bool edge = (uint32_t)addr < P.dbk_stop && !t8_skip && (e > 0 || (has_nb && !(P.dbk_idc == 2 && other)));
    if (edge) {
        MbView Qv, Pv;
        load_view(P, addr, Qv);
        load_view(P, ap, Pv);
        const int xq = dir == 0 ? e : k, yq = dir == 0 ? k : e;
        const int xp = dir == 0 ? (e ? e - 1 : 15) : k, yp = dir == 0 ? k : (e ? e - 1 : 15);
        bS = bs_luma(P, ap, Pv, addr, Qv, e == 0 && !own, xp, yp, xq, yq);
    }
    G(P.bs)[(size_t)addr * 32 + (j & 16) + ((j & 3) << 2) + ((j >> 2) & 3)] = (uint8_t)bS;  // [dir][segment][edge]
    if (j == 0) {
        const DevAux &ax = G(P.aux)[addr];
        const bool own_t = P.multi_slice && P.dbk_idc == 0 && mby > 0 && G(P.mbs)[addr - W].slice_num != sq;
        G(P.dbq)[addr] = (uint32_t)ax.qdb[0] | ((uint32_t)ax.qdb[1] << 8) | ((uint32_t)ax.qdb[2] << 16) |
                         ((ax.kind & AUX_T8) ? 1u << 24 : 0u) | (own ? DBQ_OWN_LEFT : 0u) | (own_t ? DBQ_OWN_TOP : 0u);
    }
}

// ------------------------------------------------------------ staging
// Validation of a frame picture's syntax records and the per-MB values the other kernels read
// (DevAux, ICOL), a lane per MB, 64 MBs of a row per wave.  The rules are those of the host's
// staging (stage_picture in api.cpp), which decides what an error is called: this kernel only
// names the first MB that breaks one.  Bound: the latency of three dependent rounds of loads
// (record and neighbours, masks, motion), so each round is issued whole: 11 us for a CIF picture,
// 15 for 1920x1088, 29 for 3840x2160, where loads at the checks that use them took 17, 23 and 35.
// The host's pass took 1.6 ms for a 1920x1088 B picture.
__constant__ uint8_t c_cqp[22] = {29, 30, 31, 32, 32, 33, 34, 34, 35, 35, 36, 36, 37, 37, 37, 38, 38, 38, 39, 39, 39, 39};
__device__ __forceinline__ uint32_t stage_chroma_qp(int qp, int off) {  // 8.5.8, Table 8-15
    const int q = clip3(0, 51, qp + off);
    return q < 30 ? (uint32_t)q : c_cqp[q - 30];
}
// Intra4x4 / Intra8x8 mode with neighbouring samples left, above, above left (nxn_mode_ok).
__device__ __forceinline__ bool stage_mode_ok(int mode, bool left, bool top, bool tl) {
    // samples a mode reads (1 left, 2 above, 4 above left), 8 for what is no mode
    const uint32_t need = mode > 8 ? 8u : mode == 2 ? 0u : mode == 0 || mode == 3 || mode == 7 ? 2u : mode == 1 || mode == 8 ? 1u : 7u;
    const uint32_t have = (left ? 1u : 0u) | (top ? 2u : 0u) | (tl ? 4u : 0u);
    return (need & ~have) == 0u;
}
struct StageSums {
    uint32_t inter, intra, lists;
};
// What an MB's record says beside its motion, and the class, shape and slice of its neighbours A,
// B, C and D (of the MB itself where there is none): loaded together, ahead of the checks, whose
// branches would each wait for what they look at.
struct StageRec {
    uint32_t w[9];             // mb_type .. ref_idx
    uint32_t off, sn;
    uint32_t nw[4], nshape[4], nsn[4];
    __device__ __forceinline__ uint32_t byte(int k) const { return (w[k >> 2] >> (8 * (k & 3))) & 255u; }
};
__device__ __forceinline__ StageRec stage_load(const StageIn &S, int a, const int (&nb)[4]) {
    StageRec r;
    const GAS h264g_mb *const mbs = G(S.mbs);
    const GAS uint32_t *const p = (const GAS uint32_t *)&mbs[a];
#pragma unroll
    for (int k = 0; k < 9; k++) r.w[k] = p[k];
    r.off = mbs[a].level_offset;
    r.sn = mbs[a].slice_num;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const GAS h264g_mb &n = mbs[nb[k]];
        r.nw[k] = n.mb_type;
        r.nshape[k] = n.part_shape;
        r.nsn[k] = n.slice_num;
    }
    return r;
}
static_assert(offsetof(h264g_mb, mb_type) == 0 && offsetof(h264g_mb, flags) == 1 && offsetof(h264g_mb, qp_y) == 2 &&
              offsetof(h264g_mb, cbp) == 3 && offsetof(h264g_mb, intra16x16_pred_mode) == 4 && offsetof(h264g_mb, intra_chroma_pred_mode) == 5 &&
              offsetof(h264g_mb, part_shape) == 6 && offsetof(h264g_mb, sub_part_shape) == 8 && offsetof(h264g_mb, intra_pred_modes) == 12 &&
              offsetof(h264g_mb, ref_idx) == 28 && offsetof(h264g_mb, mv) == 36, "StageRec::w");
// A neighbour that constrained intra prediction hides (cip_hides).
__device__ __forceinline__ bool stage_hides(const StageRec &R, int k) {
    return R.nw[k] == H264G_MB_P_SKIP || ((R.nw[k] == H264G_MB_P || R.nw[k] == H264G_MB_B) && R.nshape[k] != H264G_PART_8x8);
}
// One MB; false when it breaks a rule.  ax is complete but for the residual index of an intra MB.
// there: which neighbours are in the picture.
__device__ __forceinline__ bool stage_mb(const StageIn &S, const StageRec &R, int a, uint32_t there, DevAux &ax, StageSums &sum) {
    const GAS h264g_mb &m = G(S.mbs)[a];
    const int cls = (int)R.byte(0), cbp = (int)R.byte(3), qp = (int)R.byte(2), shape = (int)R.byte(6);
    const uint32_t flags = R.byte(1);
    const bool i16 = cls == H264G_MB_I16x16, t8 = flags & H264G_MBF_T8x8;
    const uint64_t off = R.off;
    // the masks: DC of an Intra16x16 MB | luma, four for each 8x8 block of cbp | chroma.  Taken
    // whole (what lies behind the levels is in the picture's block), in pairs.
    const int lm = cbp & 15, cc = cbp >> 4, nl = 4 * __popc((uint32_t)lm), first = i16 ? 1 : 0;
    const GAS uint16_t *const lv = (const GAS uint16_t *)G(S.levels) + min(off, S.n_levels);
    typedef uint32_t __attribute__((aligned(2), may_alias)) u32_a2;
    uint32_t dcm = lv[0], lw[8], cw[5];
#pragma unroll
    for (int k = 0; k < 8; k++) lw[k] = *(const GAS u32_a2 *)(lv + first + 2 * k);
#pragma unroll
    for (int k = 0; k < 5; k++) cw[k] = *(const GAS u32_a2 *)(lv + first + nl + 2 * k);
    if (cls > H264G_MB_B || qp > 51 || off > S.n_levels || (cbp >> 4) > 2) return false;
    if (i16 && (cbp & 15) != 0 && (cbp & 15) != 15) return false;
    if (cls == H264G_MB_P_SKIP && cbp) return false;
    if (cls == H264G_MB_I8x8 && !t8) return false;
    if ((cls == H264G_MB_I4x4 || i16) && t8) return false;
    const uint32_t sub = R.w[2];
    if (cls_inter(cls) && t8 && ((cbp & 15) == 0 || (shape == H264G_PART_8x8 && sub != 0u))) return false;
    if (flags & H264G_MBF_FIELD) return false;
    if (S.slice_type == H264G_SLICE_I && cls_inter(cls)) return false;
    if (S.slice_type != H264G_SLICE_B && cls == H264G_MB_B) return false;
    if (S.slice_type != H264G_SLICE_P && (cls == H264G_MB_P || cls == H264G_MB_P_SKIP)) return false;
    const int qd = cls == H264G_MB_IPCM ? 0 : qp;
    ax.qdb[0] = (uint8_t)qd;
    ax.qdb[1] = (uint8_t)stage_chroma_qp(qd, S.cqo[1]);
    ax.qdb[2] = (uint8_t)stage_chroma_qp(qd, S.cqo[0]);
    ax.qpc[0] = (uint8_t)stage_chroma_qp(qp, S.cqo[0]);
    ax.qpc[1] = (uint8_t)stage_chroma_qp(qp, S.cqo[1]);
    if (cls == H264G_MB_IPCM) {
        if (off + 384 > S.n_levels) return false;
        ax.kind = AUX_PCM;
#pragma unroll
        for (int l = 0; l < 2; l++)
#pragma unroll
            for (int q = 0; q < 4; q++) ax.refid[l][q] = S.nref[l] > 0 ? S.ref_slot[l][0] : (int8_t)-1;
        sum.inter += 384 + 384 * 2 + 16;
        return true;
    }
    const bool intra = cls_intra(cls);
    uint32_t kind = (intra ? AUX_INTRA : AUX_INTER) | (t8 ? AUX_T8 : 0u);
    // ---- levels: masks -> non-zero bits
    const int nmask = first + nl + (cc >= 1 ? 2 : 0) + (cc == 2 ? 8 : 0);
    if (off + (uint64_t)nmask > S.n_levels) return false;
    uint32_t nvals = i16 ? (uint32_t)__popc(dcm) : 0u, nz4 = 0, nz8 = 0, stray = 0;
    const uint32_t lbits = i16 ? 0xFFFEFFFEu : 0xFFFFFFFFu;
    uint32_t left = (uint32_t)lm;
#pragma unroll
    for (int g = 0; g < 4; g++) {  // the masks of the g-th 8x8 block that has any
        const bool on = left != 0u;
        const uint32_t q = on ? (uint32_t)__builtin_ctz(left) : 0u, w0 = on ? lw[2 * g] : 0u, w1 = on ? lw[2 * g + 1] : 0u;
        left &= left - 1u;
        nvals += (uint32_t)__popc(w0) + (uint32_t)__popc(w1);
        stray |= (w0 | w1) & ~lbits;
        const uint32_t nz = ((w0 & 0xFFFFu) ? 1u : 0u) | ((w0 >> 16) ? 2u : 0u) | ((w1 & 0xFFFFu) ? 4u : 0u) | ((w1 >> 16) ? 8u : 0u);
        if (t8) nz8 |= (nz ? 1u : 0u) << q;
        else nz4 |= nz << (4u * q);
    }
    if (cc >= 1) {
        nvals += (uint32_t)__popc(cw[0]);
        stray |= cw[0] & ~0x000F000Fu;
    }
#pragma unroll
    for (int k = 1; k < 5; k++) {
        const uint32_t w = cc == 2 ? cw[k] : 0u;
        nvals += (uint32_t)__popc(w);
        stray |= w & ~0xFFFEFFFEu;
    }
    if (stray) return false;
    if (off + (uint64_t)nmask + nvals > S.n_levels) return false;
    if (nmask) kind |= AUX_RESID;
    ax.kind = (uint8_t)kind;
    ax.nmask = (uint8_t)nmask;
    ax.nz4 = (uint16_t)nz4;
    ax.nz8 = (uint8_t)nz8;
    ax.ires = nvals << AUX_NVALS_SHIFT;
    // ---- intra modes vs neighbour availability
    if (intra) {
        auto avail = [&](int k) -> bool { return ((there >> k) & 1u) && R.nsn[k] == R.sn && !(S.cip && stage_hides(R, k)); };
        const bool A = avail(0), B = avail(1), D = avail(3);
        if (!i16) {
            const int n = cls == H264G_MB_I4x4 ? 4 : 2;
            // byte blk of the modes (shifted out of two registers: words picked from R by a
            // condition would make it an array in scratch memory)
            const uint64_t lo = (uint64_t)R.w[4] << 32 | R.w[3], hi = (uint64_t)R.w[6] << 32 | R.w[5];
            auto mode = [&](int blk) -> uint32_t { return (uint32_t)((blk < 8 ? lo : hi) >> (8 * (blk & 7))) & 255u; };
            for (int by = 0; by < n; by++)
                for (int bx = 0; bx < n; bx++) {
                    const bool left = bx > 0 || A, top = by > 0 || B;
                    const bool tl = bx > 0 ? (by > 0 || B) : (by > 0 ? A : D);
                    const int blk = n == 4 ? 8 * (by >> 1) + 4 * (bx >> 1) + 2 * (by & 1) + (bx & 1) : by * 2 + bx;
                    if (!stage_mode_ok((int)mode(blk), left, top, tl)) return false;
                }
        } else {
            const int md = (int)R.byte(4);
            if (md > 3 || (md == 0 && !B) || (md == 1 && !A) || (md == 3 && !(A && B && D))) return false;
        }
        const int cm = (int)R.byte(5);
        if (cm > 3 || (cm == 1 && !A) || (cm == 2 && !B) || (cm == 3 && !(A && B && D))) return false;
        sum.intra += 384 + 2 * ((uint32_t)nmask + nvals) + 16 * 2 + 48;
        return true;
    }
    // ---- inter: reference slots, prediction flags, weight entries
    if (shape > 3) return false;
    if (shape == H264G_PART_8x8 && (sub & 0xFCFCFCFCu)) return false;
    uint32_t pf = 0, e[4], rejected = 0;
    bool bad = false;
    int8_t slot[2][4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int r0 = (int8_t)(R.w[7] >> (8 * q)), r1 = (int8_t)(R.w[8] >> (8 * q));
        bad |= (r0 < 0 && r1 < 0) || (cls != H264G_MB_B && r1 >= 0) || r0 < -1 || r0 >= S.nref[0] || r1 < -1 || r1 >= S.nref[1];
        pf |= (r0 >= 0 ? 1u : 0u) << q | (r1 >= 0 ? 16u : 0u) << q;
        e[q] = (uint32_t)((r0 + 1) * S.n1 + r1 + 1) & 255u;
        rejected |= S.bad_weight[e[q] >> 5] >> (e[q] & 31u);
        slot[0][q] = S.ref_slot[0][clip3(0, 31, r0)];
        slot[1][q] = S.ref_slot[1][clip3(0, 31, r1)];
    }
    if (bad || (rejected & 1u)) return false;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        ax.refid[0][q] = (pf >> q) & 1u ? slot[0][q] : (int8_t)-1;
        ax.refid[1][q] = (pf >> (4 + q)) & 1u ? slot[1][q] : (int8_t)-1;
        ax.wp[q] = (uint8_t)e[q];
    }
    ax.pf = (uint8_t)pf;
    // ---- algorithmic bytes: per partition and list used (stage_picture)
    const int ps = cls == H264G_MB_P_SKIP ? H264G_PART_16x16 : shape;
    uint32_t bytes = 0, lists = 0;
    uint32_t mv[2][16];
#pragma unroll
    for (int l = 0; l < 2; l++)
#pragma unroll
        for (int b = 0; b < 16; b++) mv[l][b] = ((const GAS uint32_t *)m.mv)[16 * l + b];
#pragma unroll
    for (int b = 0; b < 16; b++) {
        const int bx = b & 3, by = b >> 2, q = (by >> 1) * 2 + (bx >> 1);
        int w, h;
        if (ps != H264G_PART_8x8) {
            w = ps == H264G_PART_8x16 ? 2 : 4;
            h = ps == H264G_PART_16x8 ? 2 : 4;
        } else {
            const uint32_t ss = (sub >> (8 * q)) & 3u;
            w = ss == H264G_SUB_8x8 || ss == H264G_SUB_8x4 ? 2 : 1;
            h = ss == H264G_SUB_8x8 || ss == H264G_SUB_4x8 ? 2 : 1;
        }
        if (bx % w || by % h) continue;
#pragma unroll
        for (int l = 0; l < 2; l++) {
            if (!((pf >> (4 * l + q)) & 1u)) continue;
            const int mx = (int16_t)mv[l][b], my = (int16_t)(mv[l][b] >> 16);
            bytes += (uint32_t)((4 * w + 5 * ((mx & 3) != 0)) * (4 * h + 5 * ((my & 3) != 0)) +
                                2 * (2 * w + ((mx & 7) != 0)) * (2 * h + ((my & 7) != 0)) + 5);
            lists++;
        }
    }
    sum.inter += bytes + 384 + 2 * ((uint32_t)nmask + nvals) + 8;
    sum.lists += lists;
    return true;
}
__global__ __launch_bounds__(WAVE) void k_stage(StageIn S) {
    const int lane = wave_lane(), W = S.W, per = (W + WAVE - 1) / WAVE;
    const int y = (int)(blockIdx.x / (uint32_t)per), x0 = (int)(blockIdx.x % (uint32_t)per) * WAVE, x = x0 + lane;
    const GAS h264g_mb *const mbs = G(S.mbs);
    const bool in = x < W;
    const int xc = in ? x : W - 1, a = y * W + xc;
    const uint32_t there = (xc > 0 ? 1u : 0u) | (y > 0 ? 2u : 0u) | (y > 0 && xc < W - 1 ? 4u : 0u) | (xc > 0 && y > 0 ? 8u : 0u);
    const int nb[4] = {(there & 1u) ? a - 1 : a, (there & 2u) ? a - W : a, (there & 4u) ? a - W + 1 : a, (there & 8u) ? a - W - 1 : a};
    const StageRec R = stage_load(S, a, nb);
    uint32_t before = G(S.irow)[y];
    DevAux ax;
    {
        uint32_t *const w = (uint32_t *)&ax;
#pragma unroll
        for (int k = 0; k < (int)(sizeof(DevAux) / 4); k++) w[k] = k < 2 ? 0xFFFFFFFFu : 0u;  // refid -1, the rest 0
    }
    StageSums sum{0u, 0u, 0u};
    const bool ok = !in || stage_mb(S, R, a, there, ax, sum);
    const uint32_t sn = R.sn, cls = R.byte(0);
    const bool intra = in && cls_intra((int)cls);
    // residual index: the row's intra MBs before this one
    for (int c = 0; c < x0; c += WAVE) before += (uint32_t)__popcll(__builtin_amdgcn_ballot_w64(cls_intra(mbs[y * W + c + lane].mb_type)));
    const uint64_t im = __builtin_amdgcn_ballot_w64(intra);
    const uint32_t idx = before + __builtin_amdgcn_mbcnt_hi((uint32_t)(im >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)im, 0u));
    if (intra) {
        ax.ires |= idx;
        uint32_t av = there, dep = 0;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            if (!(av & (1u << k))) continue;
            if (R.nsn[k] != sn) {
                av &= ~(1u << k);
                continue;
            }
            if (S.cip && stage_hides(R, k)) av &= ~(1u << k);
            if (cls_intra((int)R.nw[k])) dep |= 1u << k;
        }
        const uint32_t m5 = (R.w[4] >> 8) & 255u;  // mode of block 5
        if (!(cls == H264G_MB_I8x8 || (cls == H264G_MB_I4x4 && (m5 == 3u || m5 == 7u)))) dep &= ~4u;
        G(S.icol)[idx] = (uint32_t)x | av << ICOL_AV_SHIFT | dep << ICOL_DEP_SHIFT | ((ax.kind & AUX_RESID) ? ICOL_RES : 0u);
    }
    if (in) {
        GAS uint32_t *const o = (GAS uint32_t *)G(S.aux + a);
        const uint32_t *const w = (const uint32_t *)&ax;
#pragma unroll
        for (int k = 0; k < (int)(sizeof(DevAux) / 4); k++) o[k] = w[k];
    }
    GAS StageResult *const r = G(S.res);
    const uint64_t bad = __builtin_amdgcn_ballot_w64(!ok), none = __builtin_amdgcn_ballot_w64(in && sn == H264G_SLICE_NONE),
                   other = __builtin_amdgcn_ballot_w64(in && sn != H264G_SLICE_NONE && sn != S.first_sn);
#pragma unroll
    for (int d = 1; d < WAVE; d <<= 1) {
        sum.inter += __shfl_xor(sum.inter, d);
        sum.intra += __shfl_xor(sum.intra, d);
        sum.lists += __shfl_xor(sum.lists, d);
    }
    if (lane == 0) {
        const uint32_t base = (uint32_t)(y * W + x0);
        if (bad) atomicMin((uint32_t *)&r->err_mb, base + (uint32_t)__builtin_ctzll(bad));
        if (none) atomicMin((uint32_t *)&r->dbk_stop, base + (uint32_t)__builtin_ctzll(none));
        if (other) atomicOr((uint32_t *)&r->multi_slice, 1u);
        atomicAdd((unsigned long long *)&r->alg[0], (unsigned long long)sum.inter);
        atomicAdd((unsigned long long *)&r->alg[1], (unsigned long long)sum.intra);
        atomicAdd((unsigned long long *)&r->alg[2], (unsigned long long)sum.lists);
    }
}

// Strengths by themselves, for runs that time the stages apart.
template <bool MBAFF>
__global__ __launch_bounds__(WAVE) void k_bs(const DevPic *__restrict__ pics, const uint32_t *__restrict__ chunks) {
    if (MBAFF) bs_mbaff_mb(pics, chunks, blockIdx.x, gridDim.x);
    else bs_pair_of_mbs(pics, chunks, blockIdx.x, gridDim.x);
}

// YUV420P -> BGR24 of one DPB slot (CH264PictureBase::convertYuv420pToBgr24,
// H264PictureBase.cpp:440-495): one thread per 2x2 luma block (one chroma sample);
// BT.601 integer coefficients over 1000 with C division (toward zero), clipped.
__global__ __launch_bounds__(256) void k_bgr24(const uint8_t *__restrict__ yuv, int wl, int hl, uint8_t *__restrict__ bgr,
                                                uint32_t stride, int flip) {
    const int wc = wl >> 1, hc = hl >> 1;
    const int cx = blockIdx.x * blockDim.x + threadIdx.x, cy = blockIdx.y;
    if (cx >= wc || cy >= hc) return;
    const uint8_t *u = yuv + (size_t)wl * hl, *v = u + (size_t)wc * hc;
    const int U = u[(size_t)cy * wc + cx] - 128, V = v[(size_t)cy * wc + cx] - 128;
    const int gb = 2018 * U, gg = -813 * V - 391 * U, gr = 1596 * V;
#pragma unroll
    for (int dy = 0; dy < 2; dy++) {
        const int y = 2 * cy + dy;
        uint8_t *o = bgr + (size_t)(flip ? hl - 1 - y : y) * stride + (size_t)(2 * cx) * 3;
#pragma unroll
        for (int dx = 0; dx < 2; dx++) {
            const int Y = 1164 * (yuv[(size_t)y * wl + 2 * cx + dx] - 16);
            o[3 * dx + 0] = (uint8_t)clip1((Y + gb) / 1000);
            o[3 * dx + 1] = (uint8_t)clip1((Y + gg) / 1000);
            o[3 * dx + 2] = (uint8_t)clip1((Y + gr) / 1000);
        }
    }
}

__global__ void k_copy(const uint4 *src, uint4 *dst, uint64_t n16) {
    for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < n16; i += (uint64_t)gridDim.x * blockDim.x) dst[i] = src[i];
}

}  // namespace

extern "C" {

int h264g_launch_stage(const StageIn *in, void *stream) {
    if (in->W <= 0 || in->H <= 0) return (int)hipErrorInvalidValue;
    hipLaunchKernelGGL(k_stage, dim3((uint32_t)in->H * (uint32_t)((in->W + WAVE - 1) / WAVE)), dim3(WAVE), 0, (hipStream_t)stream, *in);
    return (int)hipGetLastError();
}

int h264g_launch_inter(const DevPic *pics, const uint32_t *chunks, uint32_t n, int mbaff, int scaled, int what, void *stream) {
    const uint32_t most = runs_per_launch(what & INTER_MBS, what & INTER_BS, mbaff);
    if (!chunks && n > most) return (int)hipErrorInvalidValue;  // (one picture never has as many)
    for (uint32_t at = 0; at < n; at += most) {
        const uint32_t runs = n - at < most ? n - at : most;
        const uint32_t n_mb = (what & INTER_MBS) ? runs * MB_CHUNK : 0u;
        const uint32_t *const list = chunks ? chunks + at : nullptr;
        const dim3 grid(runs * blocks_of_run(what & INTER_MBS, what & INTER_BS, mbaff)), block(WAVE);
        if (n_mb == 0 && mbaff)
            hipLaunchKernelGGL((k_bs<true>), grid, block, 0, (hipStream_t)stream, pics, list);
        else if (n_mb == 0)
            hipLaunchKernelGGL((k_bs<false>), grid, block, 0, (hipStream_t)stream, pics, list);
        else if (mbaff)  // (scaling matrices are refused in MBAFF frames)
            hipLaunchKernelGGL((k_inter<true, false>), grid, block, 0, (hipStream_t)stream, pics, list, n_mb);
        else if (scaled)
            hipLaunchKernelGGL((k_inter<false, true>), grid, block, 0, (hipStream_t)stream, pics, list, n_mb);
        else
            hipLaunchKernelGGL((k_inter<false, false>), grid, block, 0, (hipStream_t)stream, pics, list, n_mb);
        if (const hipError_t e = hipGetLastError()) return (int)e;
    }
    return 0;
}

int h264g_launch_intra(const DevPic *pics, const uint32_t *items, uint32_t n, DevCtl *ctl, uint32_t *epoch, uint32_t *err,
                       int waves, void *stream) {
    if (n == 0) return 0;
    uint32_t g = (uint32_t)waves < n ? (uint32_t)waves : n;
    hipLaunchKernelGGL(k_intra, dim3(g), dim3(WAVE), 0, (hipStream_t)stream, pics, items, n, ctl, epoch, err);
    return (int)hipGetLastError();
}

int h264g_launch_intra_mbaff(const DevPic *pics, uint32_t n_pics, uint32_t pair_rows, DevCtl *ctl, uint32_t *epoch, uint32_t *err,
                             void *stream) {
    if (n_pics == 0 || pair_rows == 0) return 0;
    const uint32_t bands = (pair_rows + MBAFF_ROWS - 1) / MBAFF_ROWS;
    hipLaunchKernelGGL(k_intra_mbaff, dim3(n_pics * bands), dim3(WAVE * MBAFF_INTRA_WAVES), 0, (hipStream_t)stream, pics, n_pics, ctl,
                       epoch, err);
    return (int)hipGetLastError();
}

int h264g_launch_deblock(const DevPic *pics, const uint32_t *items, uint32_t n, DevCtl *ctl, uint32_t *epoch, uint32_t *err,
                         int waves, void *stream) {
    if (n == 0) return 0;
    uint32_t g = (uint32_t)waves < n ? (uint32_t)waves : n;
    hipLaunchKernelGGL(k_deblock, dim3(g), dim3(WAVE), 0, (hipStream_t)stream, pics, items, n, ctl, epoch, err);
    return (int)hipGetLastError();
}

int h264g_launch_deblock_rows(const DevPic *pics, const uint32_t *items, uint32_t n, DevCtl *ctl, uint32_t *epoch,
                              uint32_t *err, int waves, void *stream) {
    if (n == 0) return 0;
    uint32_t g = (uint32_t)waves < n ? (uint32_t)waves : n;
    hipLaunchKernelGGL(k_deblock_rows, dim3(g), dim3(WAVE), 0, (hipStream_t)stream, pics, items, n, ctl, epoch, err);
    return (int)hipGetLastError();
}

int h264g_launch_intra_band(const DevPic *pics, const uint32_t *bands, uint32_t n, DevCtl *ctl, uint32_t *epoch,
                            int rows, uint32_t *err, void *stream) {
    if (n == 0) return 0;
    if (rows < 1 || rows > H264G_INTRA_MAX_ROWS) return (int)hipErrorInvalidValue;
    hipLaunchKernelGGL(k_intra_band, dim3(2 * n), dim3(WAVE * (rows + 1)), 0, (hipStream_t)stream, pics, bands, n, rows, ctl,
                       epoch, err);
    return (int)hipGetLastError();
}

int h264g_launch_deblock_band(const DevPic *pics, const uint32_t *bands, uint32_t n, DevCtl *ctl, uint32_t *epoch,
                              int rows, uint32_t *err, void *stream) {
    if (n == 0) return 0;
    if (rows < 1 || rows > DBK_MAX_ROWS) return (int)hipErrorInvalidValue;
    hipLaunchKernelGGL(k_deblock_band, dim3(2 * n), dim3(WAVE * (rows + 1)), 0, (hipStream_t)stream, pics, bands, n, rows, ctl,
                       epoch, err);
    return (int)hipGetLastError();
}

int h264g_launch_deblock_mbaff(const DevPic *pics, uint32_t n_pics, uint32_t pair_rows, DevCtl *ctl, uint32_t *epoch, uint32_t *err,
                               void *stream) {
    if (n_pics == 0 || pair_rows == 0) return 0;
    const uint32_t bands = (pair_rows + MBAFF_ROWS - 1) / MBAFF_ROWS;
    hipLaunchKernelGGL(k_deblock_mbaff, dim3(n_pics * bands), dim3(WAVE * (MBAFF_ROWS + 1)), 0, (hipStream_t)stream, pics, n_pics, ctl,
                       epoch, err);
    return (int)hipGetLastError();
}

int h264g_launch_bgr24(const uint8_t *yuv, int wl, int hl, uint8_t *bgr, uint32_t stride, int flip, void *stream) {
    const int wc = wl / 2, hc = hl / 2;
    hipLaunchKernelGGL(k_bgr24, dim3((wc + 255) / 256, hc), dim3(256), 0, (hipStream_t)stream, yuv, wl, hl, bgr, stride, flip);
    return (int)hipGetLastError();
}

int h264g_launch_copy(const uint8_t *src, uint8_t *dst, uint64_t bytes, void *stream) {
    uint64_t n16 = bytes / 16;
    if (n16 == 0) return 0;
    hipLaunchKernelGGL(k_copy, dim3(1024), dim3(256), 0, (hipStream_t)stream, (const uint4 *)src, (uint4 *)dst, n16);
    return (int)hipGetLastError();
}

}  // extern "C"

// ------------------------------------------------------------ static scratch
// Device memory of the allocation-free entry point (h264g_picture_decode_static): the
// staged syntax of one picture and its stage buffers (records, levels, work lists,
// boundary strengths, intra residuals).  Every device the library runs on holds its own
// copy until the process ends.  In host code `scratch` names a host-side stand-in, so its
// device address is looked up once per device and only that address is used.
namespace {
__device__ __align__(256) uint8_t scratch[H264G_STATIC_SCRATCH_BYTES + H264G_SCRATCH_IMETA];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void *g_scratch_addr[kMaxDevices] = {};
}  // namespace

int h264g_scratch_address(int device, void **out) {
    if (device < 0 || device >= kMaxDevices || !out) return (int)hipErrorInvalidValue;
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_addr[device]) {
        int cur = -1;
        hipError_t e = hipGetDevice(&cur);
        if (e != hipSuccess) return (int)e;
        if (cur != device) return (int)hipErrorInvalidDevice;  // the caller makes `device` current
        void *p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return (int)e;
        if (!p) return (int)hipErrorInvalidSymbol;
        g_scratch_addr[device] = p;
    }
    *out = g_scratch_addr[device];
    return 0;
}
