// Shared by attention.hip (decode / short q) and attention_prefill.hip (long q): launch arguments and geometry.
#pragma once
#include "common.h"

struct AttnArgs {
    const void* q;
    int64_t ld_q;
    const void* kpool;
    const void* vpool;
    const int32_t* bt;
    int64_t max_pages;
    const int32_t* ctx_lens;
    const int32_t* cu_q;
    void* out;
    int out_frag;  // 1: out is [tokens, H * D] in 32-row fragment order (xf_off in common.h), 2: with its columns re-ordered; else row-major
    int H, Hkv, G, Gc, Gp, TQ, HC, NS;
    int Gp_shift;  // Gp is a power of two: column -> (q token, head of the group) by shift and mask, not by division
    int HCB;  // decode kernel: blocks per kv head along the 16-head chunks (HC / chunks per block)
    int xcd_remap;  // decode kernel, HCB > 1: the chunk blocks of a (sequence, split, kv head) group run on one XCD; prefill: its tiles
    float scale_log2;
    float* ws_o;   // [total_q][H][NS][D]        (fused combine: [group][chunk][16 columns][NS][D])
    float* ws_ml;  // [total_q][H][NS][2]        (fused combine: [group][chunk][16 columns][NS][4], {m, l, -, -})
    unsigned* counters;  // fused combine: per-group arrival counters (zero between launches), or nullptr
    int64_t ld_out;  // prefill kernel: elements between two tokens' rows of `out`
    const int32_t* out_cols;  // out_frag 2: output column k is stored as column out_cols[k] (a permutation)
};
// The prefill kernel's.  (Three more fields of its own in AttnArgs cost every launch of the decode kernel 0.05 us: 8 heads of 64 on one at ctx 137 3.94 / 3.99.)
struct AttnPrefillArgs : AttnArgs {
    const void *cosb, *sinb;   // q is rotated as it is read, by these tables [position][D / 2] (or nullptr: it is as it is to be)
    const int32_t* positions;  // of the q tokens
};

constexpr float NEG_BIG = -1.0e30f;

// How the heads of a kv group become MFMA columns: chunks of up to 16 heads, padded to a power of two, TQ q tokens per 16 columns.
struct AttnGeom {
    int G, Gc, Gp, TQ, HC;
};
static inline AttnGeom attn_geom(int H, int Hkv) {
    AttnGeom g;
    g.G = H / Hkv;
    g.Gc = g.G < 16 ? g.G : 16;
    g.HC = (g.G + 15) / 16;
    for (g.Gp = 1; g.Gp < g.Gc;) g.Gp *= 2;
    g.TQ = 16 / g.Gp;
    return g;
}
static inline void attn_set_geom(AttnArgs& a, int H, int Hkv, const AttnGeom& g) {
    a.H = H;
    a.Hkv = Hkv;
    a.G = g.G;
    a.Gc = g.Gc;
    a.Gp = g.Gp;
    a.Gp_shift = 0;
    while ((1 << a.Gp_shift) < g.Gp) ++a.Gp_shift;
    a.TQ = g.TQ;
    a.HC = g.HC;
}

// prefill kernel launcher (attention_prefill.hip): q, pools, tables, out, scale and geometry of `a`; D 64 or 128; rows: the page layout
// of attn_varlen.hip; cos, sin, positions: AttnPrefillArgs
int tgis_launch_attn_prefill(const AttnArgs& a, int64_t B, int Hkv, int D, int64_t max_q_len, int dtype, bool rows, hipStream_t st, const void* cos = nullptr,
                             const void* sin = nullptr, const int32_t* positions = nullptr);
