// Parameters of prefill_stream_kernel / prefill_merge_kernel (tq_prefill_stream.hip) and their launch.
#pragma once

#include "tq_common.h"

constexpr int kTqPrefillStreamRows = 48;  // rows of a segment
constexpr int kTqPrefillStreamWaves = 8;  // workers per compute unit

// What the merge needs of a cut segment (plan[w]: the one worker w's range begins inside of): its
// sequence's first query row and query count, KV head, row block, the slot of its first piece, the
// workers w0 .. w1 that hold its pieces.  plan[0].rb: the number of workers.
struct TqPrefillCut {
    int q0, nq, kh, rb, slot0, w0, w1;
};

struct TqPrefillStream {
    const void* q;
    int64_t q_st, q_sh;
    int q_dtype;
    const int32_t* cu_q;
    int num_seqs, max_q, hkv, group;
    tq_udiv group_div;
    int step, grow;                     // tokens between row blocks (causal; 0), tokens of a row block
    // keys / values tiles: payload of block 0, head 0, the norms after it in the same tile
    const uint8_t* kptr;
    const uint8_t* vptr;
    int64_t k_sh, v_sh;
    uint32_t k_sb, v_sb, d_kn, d_kr, d_vn;
    const float* k_cent;
    const float* v_cent;
    float k_cs, v_cs, v_cinv;
    int share;                          // K and V use one table
    uint32_t k_row, v_row, s_row, row_bytes;  // LDS addresses of the row tables, their replicas' bytes
    int block_size, tpb;                // tokens and 16-token tiles per block
    tq_udiv tpb_div;
    uint32_t num_blocks;
    const int32_t* bt;
    int64_t bt_stride;
    int max_blocks;
    const int32_t* seq_lens;
    float c1, c2;                       // norms -> log2 units: MSE term (> 0), QJL term
    float c21;                          // c2 / c1
    int causal, rot;
    void* out;
    int out_dtype;
    int64_t out_st, out_sh;
    int n_workers, snap;                // snap: whole segments only (no workspace)
    float* ws_acc;                      // [2 n_workers][48][128]
    float* ws_ml;                       // [2 n_workers][48][2]
    TqPrefillCut* plan;                 // [n_workers]
};

// Launches the kernel on `cus` workgroups (and the merge unless snap).  The tables' addresses, c21,
// group_div, step and grow are set here.
int tq_prefill_stream_launch(TqPrefillStream p, int kb, bool kq, int vb, int cus, hipStream_t stream);
