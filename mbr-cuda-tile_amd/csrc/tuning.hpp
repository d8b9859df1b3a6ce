// Per-kernel launch shapes and cache policies, chosen by measurement on MI355X at the
// MelBandRoformer chunk shapes (T = 801 frames, 60 bands, D = 384, 48060 token rows).
// Every value can be overridden at build time (build.py -D NAME=VALUE) to re-tune.
//
// MBRT_NT_* : non-temporal policy of a kernel's streaming operands, bit 0 = loads,
//             bit 1 = stores.  Operands that are re-read (gamma, bias, gate logits, cos/sin
//             tables) always use ordinary accesses.  Measured with each op's calls back to
//             back (so an op pays for its own write-backs from the 256 MB MALL): uniform
//             policies 0..3 per kernel, the best kept; differences under ~3 % are noise.
#pragma once

// Small inputs are read with ordinary loads, whatever a kernel's policy says: up to MBRT_HOT_BYTES bytes
// by the softmax, the qkv split and the row copy, up to MBRT_HOT_BYTES_GATE of attention values by the
// gate merge, up to MBRT_HOT_BYTES_ACT by the GLU and, of f32, by RMSNorm.  An input that small has
// usually just been written and still sits in the 256 MB MALL (or an L2), which non-temporal
// loads make no use of.  us per call with non-temporal and with ordinary loads, two buffer sets in turn
// (warm), and twelve (cold up to the sizes given last in each row):
//                                            warm           cold
//   split + rotary, 18.6 MB of qkv        8.65   7.04     8.96   7.29
//                   37 MB                14.7   12.6     15.3   15.9
//   gate merge, 6.2 MB of attention       4.03   3.52     4.03   4.18
//               24.6 MB                   9.64   8.95    10.8   11.2
//   softmax f32 [4000, 801], 12.8 MB      5.80   4.99     6.09   5.87
//               [12000, 801], 38 MB      17.2   13.0     17.3   17.7
// The lines lie where the attention layer's three calls stop gaining when its buffers are cold (two
// sets in turn, and six):
//   [60, 110], qkv 20.3 MB, gate 6.8     22.4   20.2     22.6   22.7
//   [60, 120], qkv 22.1 MB (split only)  23.6   21.2     23.4   24.3
//   [60, 150], qkv 27.6 MB, gate 9.2     30.9   27.9     30.2   32.4
//   [200, 60], qkv 36.9 MB, gate 12.3    31.1   29.3     30.9   31.8
// In the token step of T frames (permute, RMSNorm, GELU, GLU; bf16, 384 features) each kernel's share
// goes with what the chain's buffers hold in all.  Step by ordinary loads in one kernel over the step
// without any, one / two / three / six sets in turn:
//                  row copy                  GLU                       RMSNorm
//   T =  50   .98  1.07  .99  .98      .98  1.07 1.00  .99      1.02 1.11 1.05 1.02
//   T =  90  1.01   .98  .98  .99     1.03   .99  .99  .99      1.07  .99  .99 1.01
//   T = 130   .97   .97  .97  .97      .97   .97  .97  .97      1.01 1.00 1.00 1.00
//   T = 201   .96   .99  .98 1.06      .96   .99  .97 1.10       .97  .99  .98 1.10
// RMSNorm of 2-byte inputs has the losses without the gain and keeps its policy; of f32, 192 features,
// it gains (T = 100: 1.02 .95 .95 .95).  12 MB of GLU input are T = 136.
#ifndef MBRT_HOT_BYTES
#define MBRT_HOT_BYTES (20ll << 20)
#endif
#ifndef MBRT_HOT_BYTES_GATE
#define MBRT_HOT_BYTES_GATE (8ll << 20)
#endif
#ifndef MBRT_HOT_BYTES_ACT
#define MBRT_HOT_BYTES_ACT (12ll << 20)
#endif
#ifndef MBRT_NT_RMS
#define MBRT_NT_RMS 3    // residual add + RMSNorm: x, residual, sum, normed
#endif
#ifndef MBRT_NT_ACT
#define MBRT_NT_ACT 2    // bias + activation (GELU)
#endif
#ifndef MBRT_NT_GLU
#define MBRT_NT_GLU 3
#endif
#ifndef MBRT_NT_GATE
#define MBRT_NT_GATE 3   // sigmoid gate x head merge: attention values, merged output
#endif
#ifndef MBRT_NT_SMR
#define MBRT_NT_SMR 0    // register-resident softmax rows (time attention, 801 columns)
#endif
#ifndef MBRT_NT_SMS
#define MBRT_NT_SMS 3    // LDS-staged short softmax rows (freq attention, 60 columns)
#endif
#ifndef MBRT_NT_SML
#define MBRT_NT_SML 3    // LDS-staged long softmax rows (time attention, 801 columns)
#endif
#ifndef MBRT_NT_ROT
#define MBRT_NT_ROT 3    // rotary q/k
#endif
#ifndef MBRT_NT_ROW
#define MBRT_NT_ROW 3    // row copy (permutes that keep the innermost dim)
#endif
#ifndef MBRT_NT_ROWU
#define MBRT_NT_ROWU 2   // row copy of element-aligned rows in 16-byte vectors
#endif
#ifndef MBRT_ROWU_MIN
#define MBRT_ROWU_MIN 64 // shortest such row, in bytes
#endif
#ifndef MBRT_NT_CAT
#define MBRT_NT_CAT 2    // concat of several sources in one launch
#endif
// Concat: sources of this average row and size, and so many bytes in all (beyond the 256 MB MALL with
// the output), are copied one after another.  A launch apiece is little beside them, and a
// thread's rows lie far apart: four f32 sources of 64 MB in rows of 16 MB 94 us one by one and 116 in
// one launch, eight of 32 MB 103 and 109; but four of 32 MB 52 and 40, and two of 64 MB in rows of
// 96 B 101 and 39.
#ifndef MBRT_CAT_ROW
#define MBRT_CAT_ROW (256ll << 10)  // bytes
#endif
#ifndef MBRT_CAT_SRC
#define MBRT_CAT_SRC (24ll << 20)   // bytes
#endif
#ifndef MBRT_CAT_ALL
#define MBRT_CAT_ALL (192ll << 20)  // bytes
#endif
#ifndef MBRT_NT_TR
#define MBRT_NT_TR 0     // LDS tile transpose
#endif
#ifndef MBRT_NT_EW
#define MBRT_NT_EW 0     // convert / unary / scalar / binary vector kernels
#endif
#ifndef MBRT_NT_STFT
#define MBRT_NT_STFT 0   // STFT spectrum stores (bit 1), iSTFT spectrum loads (bit 0)
#endif
#ifndef MBRT_NT_ISTFT
#define MBRT_NT_ISTFT 4  // iSTFT block partials: final-pass loads (bit 0), block stores (bit 1); output stores (bit 2)
#endif
#ifndef MBRT_NT_CHUNK
#define MBRT_NT_CHUNK 3  // chunk accumulate and normalize: chunk and output loads (bit 0), output stores (bit 1)
#endif
#ifndef MBRT_NT_BAND
#define MBRT_NT_BAND 2   // band gather / mask merge: stft, masks, outputs
#endif

#ifndef MBRT_BAND_XCD
#define MBRT_BAND_XCD 8  // band kernels: runs of this many consecutive tiles per XCD (1: launch order)
#endif
#ifndef MBRT_BAND_GATHER_PIPE
#define MBRT_BAND_GATHER_PIPE 1  // band gather: persistent pipelined blocks (1) or one tile per block (0)
#endif
#ifndef MBRT_BAND_GTT
#define MBRT_BAND_GTT 64  // pipelined band gather: frames per tile (32 or 64)
#endif
#ifndef MBRT_BAND_GNW
#define MBRT_BAND_GNW 4  // pipelined band gather: waves per block
#endif
#ifndef MBRT_BAND_GALIGN
#define MBRT_BAND_GALIGN 1  // pipelined band gather: output runs start on 128-byte lines (1) or at the tile (0)
#endif
#ifndef MBRT_BAND_GBPC
#define MBRT_BAND_GBPC 1  // pipelined band gather: persistent blocks per CU
#endif
#ifndef MBRT_BAND_MTF
#define MBRT_BAND_MTF 32  // band merge: freqs per tile (<= 64)
#endif
#ifndef MBRT_BAND_MME
#define MBRT_BAND_MME 64  // band merge: CSR entries staged per chunk (a multiple of 64)
#endif
#ifndef MBRT_BAND_MNW
#define MBRT_BAND_MNW 4  // band merge: waves per block
#endif
#ifndef MBRT_BAND_MERGE_PAIRS
#define MBRT_BAND_MERGE_PAIRS 0  // band merge tile order: pairs of frame tiles within the freq-fastest order (1)
#endif
#ifndef MBRT_BAND_MERGE_TFAST
#define MBRT_BAND_MERGE_TFAST 0  // band merge tile order: frame tiles fastest (1) or freq tiles fastest (0)
#endif
#ifndef MBRT_SM_STAGE_LONG
#define MBRT_SM_STAGE_LONG 1  // softmax rows of 129..1024 elements through LDS when spans align
#endif
#ifndef MBRT_SM_LONG_G
#define MBRT_SM_LONG_G 64  // lanes per staged row of 129..1024 elements when 4-row spans align (64 or 32)
#endif
#ifndef MBRT_SM_STAGE16
#define MBRT_SM_STAGE16 1  // staged softmax: bf16->bf16 / f16->f16 spans kept 2-byte in LDS (1) or as f32 (0)
#endif
#ifndef MBRT_SM_LONG_RPG
#define MBRT_SM_LONG_RPG 1  // staged softmax rows of 129..1024 elements: rows per lane group (block of 4 or 8 rows x this)
#endif
#ifndef MBRT_SM_SHORT_BYTES
#define MBRT_SM_SHORT_BYTES 6144  // staged softmax rows of 33..64: below this many input bytes per 32 rows, 64-row blocks
#endif
#ifndef MBRT_SM_DMA
#define MBRT_SM_DMA 1  // staged softmax: raw spans loaded straight into LDS (direct-to-LDS loads)
#endif
#ifndef MBRT_SM_PAIR_U
#define MBRT_SM_PAIR_U 1  // 2-byte softmax rows of 33..64 (cols % 4 == 0, even row count): row pairs per 16-lane group from registers (0: LDS-staged kernel)
#endif
#ifndef MBRT_NT_SMP
#define MBRT_NT_SMP 3    // softmax row pairs from registers: non-temporal loads (bit 0) and stores (bit 1)
#endif
#ifndef MBRT_SM_PAIR_RCP
#define MBRT_SM_PAIR_RCP 1  // softmax row pairs: 1/sum as v_rcp_f32 (1) or the correctly rounded division (0)
#endif
#ifndef MBRT_SM_PAIR_BPC
#define MBRT_SM_PAIR_BPC 24  // softmax row pairs: blocks per CU of a grid that walks the chunks (0: one chunk per block)
#endif
#ifndef MBRT_SM_SHORT_RPG
#define MBRT_SM_SHORT_RPG 2  // rows per lane group in those blocks
#endif
#ifndef MBRT_ATTN_HEADS_WPC
#define MBRT_ATTN_HEADS_WPC 2  // attention over <= 64 queries and keys: persistent workgroups per CU, each walking heads (0: one head per workgroup)
#endif
#ifndef MBRT_ATTN_NT
#define MBRT_ATTN_NT 0  // attention, one workgroup per query tile: non-temporal q loads (bit 0) and output stores (bit 1); measured: no gain
#endif
#ifndef MBRT_ATTN_HEADS_NT
#define MBRT_ATTN_HEADS_NT 3  // persistent attention over short heads: non-temporal output stores (bit 0) and K/V/Q loads (bit 1)
#endif
#ifndef MBRT_GATE_TPW
#define MBRT_GATE_TPW 4  // gate merge of a head-major [B,H,N,D] input: tokens per run (1: a block step writes whole token rows; measured 4 > 12, 6, 2, 1 by 1 %)
#endif
#ifndef MBRT_ACT_U
#define MBRT_ACT_U 2     // 16-byte groups per thread: bias + activation (GELU)
#endif
#ifndef MBRT_GLU_U
#define MBRT_GLU_U 1     // 16-byte output groups per thread: GLU
#endif
#ifndef MBRT_GATE_U
#define MBRT_GATE_U 2    // 16-byte groups per thread: sigmoid gate x head merge
#endif
#ifndef MBRT_GATE_BPC
#define MBRT_GATE_BPC 16  // sigmoid gate x head merge: blocks per CU of a grid that walks the chunks (0: one chunk per block)
#endif
#ifndef MBRT_CHUNK_CPB
#define MBRT_CHUNK_CPB 4  // chunk accumulate: channels (one wave each) per block over shared positions, 1 to 16 (fewer when there are fewer channels)
#endif
// Bias + activation with an f32 bias beside 2-byte operands: elements from which a thread takes 16 bytes
// of those.  us, 8 bytes against 16: GELU [400, 384] 2.66 and 2.95, [3000, 1536] 5.8 and 6.2, [12000, 384]
// 5.7 and 6.2, [9000, 1024] 8.8 and 9.1; from 17 to 37 million elements within 4 % either way ([12000, 1536]
// 15.5 and 14.9, [24000, 1536] 28.4 and 28.2, [36000, 768] 22.0 and 22.7); [48060, 1536] 61 and 54
// (rocprofv3, out of cache: 64 and 56), [96120, 768] 60 and 54.  Tanh [3000, 1536] 7.0 and 7.7,
// [12000, 1536] 18.3 and 17.1; sigmoid 5.4 and 5.2, 13.6 and 12.3.
#ifndef MBRT_BIAS_WIDE
#define MBRT_BIAS_WIDE (1ll << 23)
#endif
#ifndef MBRT_BIAS_WIDE_GELU
#define MBRT_BIAS_WIDE_GELU (1ll << 24)
#endif
// Pads of 2-byte elements: elements written from which the kernel for whole rows takes them.  Eight of
// them per thread leave few waves below: [64, 100 -> 200] 2.83 us an element per thread, 3.29 by rows;
// [1000, 100 -> 200] 3.15 and 3.27, [2, 100000 -> 100200] 3.15 and 3.0.
#ifndef MBRT_PAD2_MIN
#define MBRT_PAD2_MIN (1ll << 16)
#endif
// Chunk accumulate: samples over all channels from which unaligned chunks go in 16-byte accesses.  us per
// call, one sample per lane against four, buffers warm: [2, 999] 2.53 and 3.10, [2, 44100] 2.90 and
// 3.27, [2, 200002] 3.38 and 3.69, [8, 44100] 3.20 and 3.54; above: [2, 352800] 5.1 and 4.2, [4, 200002]
// 5.3 and 4.3, [8, 352801] 10.5 and 9.0.
#ifndef MBRT_CHUNK_ANY
#define MBRT_CHUNK_ANY (1ll << 19)
#endif
// Chunk normalize: unaligned songs of this length, and of three times as many samples over all channels,
// go in 16-byte accesses.  us per call, one position per thread against four: [2, 352801] 3.5 and 4.0,
// [16, 352801] 11.2 and 15.4, [1, 1000003] 3.7 and 4.0; above: [2, 1000003] 6.1 and 5.5, [2, 2997817]
// 13.0 and 11.8, or 18.8 and 11.9 with buffers out of cache, [8, 1000003] 19.0 and 13.9 out of cache.
// The wide form's non-temporal accesses make no use of a warm cache: [8, 2997817] 35.1 and 38.1 warm, 51.1
// and 39.2 out of cache.
#ifndef MBRT_NORM_ANY
#define MBRT_NORM_ANY (1ll << 19)
#endif
#ifndef MBRT_EW_U
#define MBRT_EW_U 4      // 16-byte groups per thread in the elementwise kernels
#endif
#ifndef MBRT_ROW_U
#define MBRT_ROW_U 1     // row-copy vectors per thread
#endif
#ifndef MBRT_RMS_G
#define MBRT_RMS_G 16    // lanes per row for rows of at most 128 16-byte chunks (16 or 32)
#endif
