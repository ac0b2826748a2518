// Prints what the dispatch rules (csrc/plans.h) say of the calls on stdin,
// one JSON object a line:
//   attn n_past0 rows n_heads n_kv_heads head_dim k_fmt v_fmt capacity wlimit
//   gemm rows cols batch
//   span positions
#include <cstdio>
#include <cstring>

#include "../../qt_llama.cpp_amd/csrc/plans.h"

using namespace mrml;

int main()
{
    char op[8];
    while (std::scanf("%7s", op) == 1) {
        if (!std::strcmp(op, "attn")) {
            int a[9];
            for (int &v : a)
                if (std::scanf("%d", &v) != 1) return 1;
            const AttnRowsPlan p = attn_rows_plan(a[0], a[1], a[2], a[3], a[4], a[5], a[6], a[7], a[8]);
            const int nchains = a[1] * (a[2] / a[3]);
            std::printf("{\"span\": %d, \"tiles\": %d, \"score_m\": %d, \"score_reps\": %d, \"score_blocks\": %d, "
                        "\"one_row_scores\": %d, \"short_form\": %d, \"rows_form\": %d, \"softmax_threads\": %d, \"pv\": [%d, %d], \"long\": %d}\n",
                        p.span, p.tiles, p.score_m, p.score_reps, p.score_blocks(nchains), p.one_row_scores, p.short_form, p.rows_form,
                        p.softmax_threads, p.pv_m, p.pv_d, sv_long(p.span));
        } else if (!std::strcmp(op, "gemm")) {
            int rows, cols, batch;
            if (std::scanf("%d %d %d", &rows, &cols, &batch) != 3) return 1;
            std::printf("{\"few\": %d, \"few_fast\": %d, \"few_glu\": %d, \"producers\": %d, \"full_tiles\": %d, "
                        "\"tiles\": %d}\n",
                        gemm_few(rows, cols / 32, batch, false), gemm_few(rows, cols / 32, batch, true),
                        gemm_few_glu(rows, batch), gemm_few_producers(false, rows, batch),
                        gemm_full_tiles(rows, batch), (rows + 31) / 32);
        } else if (!std::strcmp(op, "span")) {
            int span;
            if (std::scanf("%d", &span) != 1) return 1;
            std::printf("{\"long\": %d}\n", sv_long(span));
        } else {
            return 1;
        }
    }
    return 0;
}
