// h264g_dev.h -- layouts shared by the host side of libh264g and its gfx950 kernels.
#pragma once
#include <stdint.h>
#include "h264g.h"

// Per-MB values derived once while a picture is staged (picture_begin; by k_stage or the
// host): everything the kernels would otherwise recompute per sample.
struct DevAux {
    int8_t   refid[2][4];     // reference picture per list and 8x8 quadrant as a DPB slot,
                              // -1 = none: the MC source when the list is used, and (frame
                              // pictures) the picture identity the bS derivation compares;
                              // field MBs of MBAFF frames: the frame of refIdx / 2
    uint8_t  pf;              // PredFlagLX of quadrant q at bit (4 * X + q)
    uint8_t  kind;            // AUX_* bits below
    uint16_t nz4;             // luma4x4BlkIdx b has non-zero levels (4x4-transform MBs)
    uint8_t  wp[4];           // weight-table entry per quadrant
    uint8_t  nz8;             // 8x8 block has non-zero levels (8x8-transform MBs)
    uint8_t  nmask;           // number of level masks of the MB
    uint8_t  qpc[2];          // QP'C of Cb / Cr for dequantisation
    uint8_t  qdb[3];          // deblocking qP: luma, Cb edges, Cr edges
    uint8_t  fpar;            // field MBs of MBAFF frames: bit (4 * X + q) = the referenced
                              // field is the bottom field (refIdx odd flips the MB's parity)
    uint32_t ires;            // bits 0..21: intra MBs, index of the MB's residual in
                              // DevPic::ires; bits 22..31: number of non-zero level values
};
#define AUX_IRES_MASK    0x3FFFFFu
#define AUX_NVALS_SHIFT  22
static_assert(sizeof(DevAux) == 28, "DevAux layout");

#define AUX_INTRA   0x01u  // Intra_4x4 / Intra_8x8 / Intra_16x16 prediction (bS 3/4)
#define AUX_PCM     0x02u
#define AUX_T8      0x04u  // transform_size_8x8_flag
#define AUX_INTER   0x08u
#define AUX_RESID   0x10u  // has coefficient levels
// Entry of an intra MB in the intra band schedule (DevPic::irow after the row offsets):
// column in bits 0..10, neighbour availability (A, B, C, D) from ICOL_AV_SHIFT, the
// available neighbours that are intra MBs the MB waits for from ICOL_DEP_SHIFT, and
// ICOL_RES when the MB has levels (its residual is at the entry's index in DevPic::ires).
#define ICOL_X_MASK    0x7FFu
#define ICOL_AV_SHIFT  11
#define ICOL_DEP_SHIFT 15
#define ICOL_RES       (1u << 19)
// DevPic::imeta, one uint4 per intra MB at its index in DevPic::ires: its ICOL entry with its
// type (0 I4x4, 1 I8x8, 2 I16x16) and the Intra16x16 / chroma prediction modes, the
// Intra4x4 / Intra8x8 modes as nibbles in the next two words.
#define IMETA_TYPE_SHIFT   20
#define IMETA_I16_SHIFT    22
#define IMETA_CHROMA_SHIFT 24

// Resolved weighted-prediction parameters of one (refIdxL0, refIdxL1) combination.
struct DevWeight {
    int16_t mode;             // 0 default (8.4.2.3.1), 1 weighted (8.4.2.3.2)
    int16_t logWD[3];
    int16_t w0[3], w1[3], o0[3], o1[3];
    // L1-only luma takes (w0, o0) -- handled by the host filling w0/o0 for such entries
};

// One picture as the kernels see it.
struct DevPic {
    const h264g_mb *mbs;
    const DevAux *aux;
    const int16_t *levels;
    const DevWeight *wt;
    uint8_t *dpb;             // slot 0 of the stream's DPB
    uint64_t slot_bytes;      // bytes per DPB slot (Y + Cb + Cr)
    uint32_t *flags;          // per-MB wavefront progress words of the stream
    uint64_t *rowprog;        // per-MB-row progress of row-pipelined deblocking:
                              // epoch << 32 | MBs of the row finished
    uint8_t  *bs;             // boundary strengths, 32 bytes per MB: [dir][4-line segment][edge]
                              // (MBAFF frames: nibbles, see bs_mbaff_mb)
    const uint32_t *irow;     // intra MBs per row: H + 1 offsets, then one ICOL entry per intra MB
    uint32_t n_intra;         // intra-predicted MBs of the picture
    int32_t  dst;             // destination slot
    int32_t  W, H;            // in macroblocks
    int32_t  offA, offB;      // FilterOffsetA / FilterOffsetB
    int32_t  dbk_idc;         // disable_deblocking_filter_idc
    int32_t  cip;             // constrained_intra_pred_flag
    uint8_t  *gstrip;         // deblocking strips between bands of the stream: W x 256 B per band
    uint64_t *istrip;         // intra strips between bands of the stream: W x 8 words per band
    uint32_t *dbq;            // per-MB deblocking word, written with the strengths
    int16_t  *ires;           // residual of each intra MB with levels (DevAux::ires): luma
                              // 16x16 then Cb, Cr 8x8, raster; written by the inter stage
    uint32_t *imeta;          // frame pictures: IMETA entries of the intra MBs, written by the
                              // inter stage, read by the intra band schedule
    int32_t  mbaff;           // MbaffFrameFlag: MB address 2 p + b is the top / bottom MB of
                              // pair p, pairs in raster order
    const int8_t *bsref;      // MBAFF frames: per MB [list][quadrant] the picture identity
                              // the bS derivation compares, RefPicListX[RefIdxLX] (-1: none)
    uint32_t dbk_stop;        // MBs from this address on filter none of their edges (the
                              // first MB of no slice; W * H when every MB has one)
    int32_t  multi_slice;     // the MBs carry more than one slice number (MBs of no slice
                              // aside): bs_pair_of_mbs reads them
    const uint16_t *ls;       // scaling matrices: LevelScale4x4 [intra, inter luma list][qP % 6]
                              // [raster 16] at 0, LevelScale8x8 [list][qP % 6][raster 64] at
                              // LS8_AT; null with flat lists
};
#define LS4_LIST 96           // entries per 4x4 list (6 x 16)
#define LS8_AT   192          // first 8x8 entry
#define LS8_LIST 384          // entries per 8x8 list (6 x 64)
#define LS_ENTRIES 960

// What k_stage finds about a picture besides its DevAux records; initialised by the host.
struct StageResult {
    uint32_t err_mb;          // the first MB that breaks a rule of staging (~0: none)
    uint32_t dbk_stop;        // the first MB of no slice (initially W * H)
    uint32_t multi_slice;     // some MB's slice differs from StageIn::first_sn
    uint32_t pad;
    unsigned long long alg[3];  // algorithmic bytes: inter, intra, (partition, list) pairs
};
// A picture's DevPic and StageResult stand in the 256 bytes that staging counts for it.
constexpr size_t STAGE_RESULT_AT = 200;
static_assert(sizeof(DevPic) <= STAGE_RESULT_AT && STAGE_RESULT_AT + sizeof(StageResult) <= 256, "descriptor and result");

// Arguments of k_stage: a frame picture's records and levels in device memory, and what its
// descriptor says about them.
struct StageIn {
    const h264g_mb *mbs;
    const int16_t *levels;
    uint64_t n_levels;
    DevAux *aux;
    const uint32_t *irow;     // intra MBs before each row
    uint32_t *icol;           // their ICOL entries, from irow[y] on
    StageResult *res;
    int32_t W, H;
    int32_t slice_type, cip;
    int32_t cqo[2];           // chroma_qp_index_offset, second_chroma_qp_index_offset
    int32_t nref[2];          // num_ref_idx_active
    int32_t n1;               // weight entry of (refIdxL0, refIdxL1): (r0 + 1) * n1 + r1 + 1
    uint32_t first_sn;        // slice of the first MB that has one
    int8_t ref_slot[2][32];
    uint32_t bad_weight[8];   // entries whose weights the reference rejects
};

// Work item: picture index in the batch and macroblock address.
#define WI_PIC_SHIFT 20u
#define WI_MB_MASK   ((1u << WI_PIC_SHIFT) - 1u)

// Control block of one persistent launch: ticket dispenser + finished-wave count.
struct DevCtl {
    uint32_t ticket;
    uint32_t done;
    uint32_t pad[14];         // own 64-byte line
};

// Device error bits (ORed into the context's error word).
// The error word of a context, in device memory; kernels take its address as that of `word`.
struct DevErr {
    uint32_t word, pad;
    uint32_t *host;           // its copy in pinned memory
};
#define DEVERR_TIMEOUT  0x1u

#define MB_CHUNK 64u
// Runs of MBs (see h264g_launch_inter) that one launch takes: a grid holds fewer than 2^32 threads,
// 64 of them to a block, and a run takes blocks_of_run blocks: one for each of its MBs, and for the
// boundary strengths one for each two, or each of an MBAFF frame's.
constexpr uint32_t blocks_of_run(bool mbs, bool bs, bool mbaff) {
    return (mbs ? MB_CHUNK : 0u) + (bs ? (mbaff ? MB_CHUNK : MB_CHUNK / 2) : 0u);
}
constexpr uint32_t runs_per_launch(bool mbs, bool bs, bool mbaff) { return (0xFFFFFFFFu / 64u) / blocks_of_run(mbs, bs, mbaff); }

extern "C" {
// Kernel launchers (kernels.hip); all enqueue on `stream` and return a hipError_t.
// Validates a frame picture's records and derives their DevAux and ICOL entries.
int h264g_launch_stage(const StageIn *in, void *stream);
// Launches over MBs take them in runs of MB_CHUNK of one picture: chunks[0 .. n) (picture index
// << 20 | first MB), or null with n runs of picture 0.
// mbaff: every picture of the launch is an MBAFF frame (else none is).
// scaled: some picture of the launch has scaling matrices (DevPic::ls).
// what: INTER_MBS, the inter stage; INTER_BS, the boundary strengths of pictures that are
// deblocked; or both in one launch.
#define INTER_MBS 1
#define INTER_BS  2
// (more runs than a grid has room for take several launches, see runs_per_launch)
int h264g_launch_inter(const DevPic *pics, const uint32_t *chunks, uint32_t n, int mbaff, int scaled, int what, void *stream);
// `epoch` points at the device word shared by all wavefront launches of a context
// (initially 1; each launch's last wave advances it).
int h264g_launch_intra(const DevPic *pics, const uint32_t *items, uint32_t n, DevCtl *ctl, uint32_t *epoch,
                       uint32_t *err, int waves, void *stream);
// Intra MBs of the MBAFF frames among the launch's pictures, in bands of H264G_MBAFF_ROWS of
// their at most pair_rows rows of MB pairs (128 B handed down per pair column and band).
int h264g_launch_intra_mbaff(const DevPic *pics, uint32_t n_pics, uint32_t pair_rows, DevCtl *ctl, uint32_t *epoch, uint32_t *err,
                             void *stream);
int h264g_launch_deblock(const DevPic *pics, const uint32_t *items, uint32_t n, DevCtl *ctl, uint32_t *epoch,
                         uint32_t *err, int waves, void *stream);
int h264g_launch_deblock_rows(const DevPic *pics, const uint32_t *items, uint32_t n, DevCtl *ctl, uint32_t *epoch,
                              uint32_t *err, int waves, void *stream);
// Two workgroups (luma, chroma) of rows + 1 waves per band of `rows` MB rows, rows at most
// H264G_INTRA_MAX_ROWS (one row to a SIMD, as for deblocking).  bands: picture index << 20 |
// band, or null for n bands of picture 0; so for the deblocking bands.
#define H264G_INTRA_MAX_ROWS 4
int h264g_launch_intra_band(const DevPic *pics, const uint32_t *bands, uint32_t n, DevCtl *ctl, uint32_t *epoch,
                            int rows, uint32_t *err, void *stream);
// Two workgroups (luma, chroma) of rows + 1 waves per band of `rows` MB rows, rows at most
// H264G_DBK_MAX_ROWS: with 4 each SIMD of the CU has one luma row to itself, and more rows
// share its issue slots (a 1920x1088 I / P picture: 196 / 159 us with bands of 4 rows, 237 /
// 168 with 8, 348 / 201 with 12, 481 / 249 with 16).
#define H264G_DBK_MAX_ROWS 4
int h264g_launch_deblock_band(const DevPic *pics, const uint32_t *bands, uint32_t n, DevCtl *ctl, uint32_t *epoch,
                              int rows, uint32_t *err, void *stream);
// Deblocking of the MBAFF frames among the launch's pictures, in bands of H264G_MBAFF_ROWS of
// their at most pair_rows rows of MB pairs.  (A band of 4 pair rows hands down 512 B per pair
// column, as much as the two bands of 4 MB rows that a stream's strips have in its place.)
#define H264G_MBAFF_ROWS 4
int h264g_launch_deblock_mbaff(const DevPic *pics, uint32_t n_pics, uint32_t pair_rows, DevCtl *ctl, uint32_t *epoch, uint32_t *err,
                               void *stream);
int h264g_launch_bgr24(const uint8_t *yuv, int wl, int hl, uint8_t *bgr, uint32_t stride, int flip, void *stream);
int h264g_launch_copy(const uint8_t *src, uint8_t *dst, uint64_t bytes, void *stream);
}
// Bytes of the static scratch array beyond H264G_STATIC_SCRATCH_BYTES, for the IMETA entries: an
// intra MB counts at least 768 + 172 + 28 bytes of the array and has 16 here.
#define H264G_SCRATCH_IMETA (2u << 20)
static_assert(H264G_STATIC_SCRATCH_BYTES / 968u * 16u + 256u <= H264G_SCRATCH_IMETA, "every intra MB has its entry");
// Device address of the static scratch array on `device`,
// which must be the current device; looked up on the first call per device.  Returns a
// hipError_t.
int h264g_scratch_address(int device, void **out);
