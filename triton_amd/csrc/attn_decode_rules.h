// Over how many workgroups a head's keys are shared out when at most 32 queries per head read them (attn_decode.hip): plain host
// arithmetic, so that it can be walked over all sizes without a device.
#pragma once
#include <algorithm>
#include <cstdint>

namespace trn {

// Key shares that trn_attn_workspace_bytes has room for, and as many as one launch with score perturbation has, whose workgroup that
// arrives last at a head's counter collects the others' results (4 - 5 us and more for more shares).  Measured with 16 queries per
// head, unsplit / split, us: 32 heads of 128: 2064 keys 13.9 / 22.2, 4112 keys 21.5 / 27.1, 8208 keys 36.7 / 35.8, 16400 keys 69 / 57, 65552
// keys 406 / 198; 8 heads of 128: 4112 keys 20.0 / 18.1, 8208 keys 35 / 22, 65552 keys 232 / 59; 71 heads of 64: 4112 keys 14.1 / 14.5, 8208
// keys 23.9 / 18.9.  Hence: from 4096 keys with at most 16 heads, from 8192 with more, never with 128 heads or more.  The caller provides
// the workspace.
inline int decode_splits(int n_bh, int seq_kv) {
    const int nblk = (seq_kv + 31) / 32;
    if (n_bh >= 128 || seq_kv < (n_bh <= 16 ? 4096 : 8192)) return 1;
    const int ns = std::max(1, std::min(std::min(16, 256 / n_bh), nblk / 4));
    const int bps = (nblk + ns - 1) / ns;                 // blocks per share, as the kernel computes it
    return (nblk + bps - 1) / bps;                        // no empty share: the last one starts inside the keys
}

// Key shares of up to 32 queries in two launches, the second of which adds the shares up (attn_decode_merge_kernel): some 3 us more than a
// launch without shares, against 5 to 7 for arriving and collecting in one, and hardly more for more shares.  Eight of them, or one
// workgroup per CU in all, or some 144 that read keys of their own, which are what the memory takes; sixteen where few heads have many
// keys.  us, 16 queries per head, K and V from beyond the L2s, unsplit / 2 / 4 / 6 / 8 / 16 shares (in brackets: arriving and collecting, as many as
// decode_splits()):
//   128, 8 heads: 1500 keys 11.3 / 14.4 / 12.0 / 11.9 / 11.3, 2200 14.3 / 16.3 / 13.3 / 12.2 / 11.9, 4200 21.5 / 21.7 / 16.3 / 14.7 / 13.6 / 13.6 (18.1), 16000 66 / 53 / 33 / 25.6 / 22.7
//       / 20.4; 32 on 8 KV heads: 1900 12.7 / 15.7 / 13.2 / 12.2 / 12.2, 4200 21.7 / 21.5 / 16.2 / 14.9 / 14.0, 16000 67 / 53 / 33 / 26.3 / 24.5 (26.7); 120 on 8: 2600 18.6 / 18.4,
//       8300 46 / 35 (37.7)
//     24: 1900 12.7 / 16.0 / 13.6 / 13.1, 2200 15.0 / 16.7 / 13.7 / 13.5 / 14.6; 32: 2200 15.2 / 16.6 / 14.5 / 15.3 / 17.3, 4200 22.7 / 22.3 / 18.9 / 19.7 / 21.5, 16000 104 / 86 / 55 / 51 / 52;
//       40: 2600 16.8 / 18.2 / 17.4, 3000 18.9 / 19.6 / 18.2; 38, 15139 101 / 87 / 59.7 / 59.3 (three: 68.9); 64 (three): 3500 24.9 / 25.7, 4200 31.9 / 29.2; 96: 4200 43.4 / 43.7, 5000 52.3 / 50.9
//   64, 16: 1900 8.9 / 11.3 / 9.8 / 9.3 / 9.6, 2200 10.2 / 11.3 / 9.8 / 9.4 / 9.6, 4200 14.8 / 14.5 / 11.7 / 11.0 / 10.8 / 12.6 (15.3), 16000 45 / 34 / 22 / 17.4 / 17.1 / 19.2; 32: 2600
//       11.1 / 12.3 / 11.4 / 11.5, 3000 12.5 / 13.3 / 11.7 / 11.6 / 12.7; 48: 3000 12.9 / 13.5 / 13.2, 3500 14.5 / 14.5 / 14.0; 71 (three): 6000 21.8 / 22.8, 8000 39.4 / 28.4; on
//       one KV head 2600 11.1 / 11.0, 6000 19.8 / 15.3; 100 (two): 5000 25.1 / 26.0, 6000 37.4 / 30.7; 96 on 8: 3000 12.3 / 12.4, 3500 13.8 / 13.2
// Wherever decode_splits() has shares there are some here as well, also where that line lies higher (64, three shares of 76 and more KV heads; unsplit /
// here (arriving and collecting)): 76 heads, 8192 keys 45.1 / 35.4 (40.8), 80, 8500 45.4 / 35.6 (41.2), 85, 8192 45.9 / 40.2 (47.1), 8800 46.6 / 38.5 (44.6).
// Query heads that share keys in a number that the 8 XCDs do not share evenly have a share of these on several XCDs, whose L2s then each read it: fewer
// shares, and later (us, unsplit / 2 / 3 / 4 / 6): 64: 42 on 21 2559 11.0 / 12.2 / 11.7 / 11.8 / 12.5, 72 on 9 4130 16.3 / 14.7 /
// 18.3, 100 on 25 4433 20.5 / 22.9; 128: 36 on 12 4976 25.2 / 23.5 / 19.2 / 17.3 / 15.1, 75 on 25 2340 18.0 / 22.2 / 22.1, 68 on 17 3696 24.0 / 26.7 / 27.5, 75 on 15 4857 34.0 / 30.8 / 34.9, 122 on 61 5958 58.9 / 63.7, 102 on 51 9176
// 73 / 75; but 105 on 15 6262 51 / 37.
inline int pair_shares(int n_bh, int n_bkv, int seq_kv, int head_dim) {
    if (n_bh >= 128) return 1;
    const int nblk = (seq_kv + 31) / 32, most = 256 / n_bh;
    const bool d128 = head_dim == 128;
    int from = d128 ? (most == 2 ? 2500 + 27 * n_bkv + 150 * std::max(0, n_bkv - 96) : (most == 3 ? 2200 : 2000) + 50 * std::max(0, n_bkv - 24))
                    : most == 2 ? 3300 + 24 * n_bkv : most == 3 ? 2600 + 74 * n_bkv : 2200 + 35 * std::max(0, n_bkv - 12);
    const bool many = n_bh <= 8 ? (int64_t)seq_kv * head_dim >= 5000 * 128 : n_bh <= 16 && d128 && seq_kv >= 10000;
    int ns = std::min(std::min(many ? 16 : 8, most), std::max(seq_kv >= 16000 ? 6 : seq_kv >= 8192 ? 4 : 3, 144 / n_bkv));
    if (n_bkv < n_bh && n_bkv > 6 && n_bkv * ns % 8) {
        if (most == 2 && n_bkv > 20) from = std::max(from, d128 && n_bkv % 2 ? 10000 : 6000);
        if (most == 3) {
            if (n_bkv % 2 || (n_bkv % 4 && seq_kv < 10000)) ns = 2;
            from = std::max(from, d128 ? 4300 : n_bkv > 20 ? 6000 : 3600);
        } else if (most > 3 && most < 8) {
            ns = most >= 6 && (n_bkv % 4 == 0 || (n_bkv % 2 == 0 && seq_kv >= 12000)) ? 6 : 4;
            if (n_bkv > 16) from = std::max(from, 2200 + (d128 ? 40 : 35) * n_bkv);
        }
    }
    if (seq_kv < from && decode_splits(n_bh, seq_kv) <= 1) return 1;
    const int bps = (nblk + ns - 1) / ns;      // (blocks per share, as the kernel computes it)
    return (nblk + bps - 1) / bps;
}

// The shares of a call without score perturbation that has its workspace; 1: a single launch that writes the outputs, with nothing for a second
// one to add up.  No more than trn_attn_workspace_bytes has room for, where it has any.
inline int few_query_shares(int n_bh, int n_bkv, int seq_kv, int head_dim) {
    const int room = decode_splits(n_bh, seq_kv), ns = pair_shares(n_bh, n_bkv, seq_kv, head_dim);
    return room > 1 ? std::min(room, ns) : ns;
}

}  // namespace trn
