// batch_engine.h -- host side of the batched persistent form.
#pragma once
#include <string>
#include <vector>

#include "batch.h"
#include "scc_amd.h"

namespace sccamd {

class Engine;

class BatchEngine {
  public:
    ~BatchEngine();
    // `checked`: the caller has already validated the graphs (the server's
    // submit does)
    scc_status upload(int device, hipStream_t stream, const scc_batch_host *b, bool checked = false);
    // a batch in device memory in the host layout (row_off/col_off given on
    // the host, d_roff = row_off on the device), valid by construction
    scc_status upload_device(int device, hipStream_t stream, uint32_t ng, const uint32_t *Vs, const uint32_t *Es,
                             const uint64_t *roff, const uint64_t *coff, const uint64_t *d_roff,
                             const uint32_t *dFr, const uint32_t *dBr, const uint32_t *dFc, const uint32_t *dBc);
    scc_status run(const scc_batch_opts &o, scc_batch_stats *out);
    scc_status run_serial(Engine &eng, const scc_opts &o, scc_batch_stats *out);
    scc_status autotune(int sample, std::string *report);
    // lab in the host layout, or graph i's V[i]+1 labels to each[i]
    scc_status labels(uint32_t *lab, uint32_t *nscc, uint32_t *const *each = nullptr);
    // the uploaded batch's sizes and host-layout offsets (arrays may be NULL)
    uint32_t info(uint32_t *Vs, uint32_t *Es, uint64_t *roff, uint64_t *coff) const;

    static constexpr int NBUCKETS = 12;

  private:
    void release();
    scc_status prepare(int device, hipStream_t stream, uint32_t ng, const uint32_t *Vs, const uint32_t *Es,
                       const uint64_t *roff, const uint64_t *coff);
    scc_status upload_host(int device, hipStream_t stream, const scc_batch_host *b, bool checked);
    scc_status install_device(int device, hipStream_t stream, uint32_t ng, const uint32_t *Vs, const uint32_t *Es,
                              const uint64_t *roff, const uint64_t *coff, const uint64_t *d_roff,
                              const uint32_t *dFr, const uint32_t *dBr, const uint32_t *dFc, const uint32_t *dBc);
    scc_status finish_upload(bool check);
    scc_status launch(const std::vector<uint32_t> &idx, const std::vector<uint32_t> &cfg,
                      const std::vector<int> &block, double *ms, std::vector<double> *lat_ms,
                      uint32_t *launches);
    scc_status spread_labels(const uint32_t *packed, uint64_t words, uint32_t *lab);

    int dev = 0;
    hipStream_t s1 = nullptr, stream2 = nullptr;
    BatchDev d;
    uint32_t G = 0;
    std::vector<uint32_t> V, E;
    std::vector<uint64_t> row_off, voff, eoff;
    std::vector<int> bucket;
    std::vector<uint32_t> best_cfg;
    std::vector<int> best_block;
    std::vector<void *> allocs;
    uint64_t capS = 0, capA = 0;
    uint32_t capG = 0;
    uint64_t *m_voff = nullptr, *m_eoff = nullptr;
    uint32_t *m_V = nullptr, *m_Fr = nullptr, *m_Br = nullptr, *m_Fc = nullptr, *m_Bc = nullptr;
    // launch input, one block (one copy per launch): 64 words of work-queue
    // heads, then capG configuration words and capG processing-order entries
    uint32_t *m_meta = nullptr;
    // per-graph results, one block (one copy per run): start and end ticks
    // and SCC counts of capG graphs
    uint64_t *m_res = nullptr;
    // page-locked host side of both blocks
    uint32_t *h_meta = nullptr;
    uint64_t *h_res = nullptr;
    // two page-locked blocks that labels for pageable memory pass through
    // (made on first use, at most kLabelBlock words each: a block's wait costs
    // about 9 us, 190 MB of labels take 14.4 ms in blocks of 2^16 words, 7.9 of
    // 2^18, 7.4 of 2^20)
    static constexpr uint64_t kLabelBlock = 1 << 18;
    uint32_t *h_label = nullptr;
    uint64_t label_words = 0;
    std::vector<uint32_t> label_host;   // the packed labels of a server's batch
    hipEvent_t ev[3] = {nullptr, nullptr, nullptr};   // start, end of each stream
    int occ[3] = {0, 0, 0};                           // workgroups per CU at 1,024, 512 and 256 lanes
    std::vector<uint32_t> stage;        // host staging of the row arrays
    uint64_t nverts = 0, narcs = 0;
    double ticks_per_ms = 100000.0;
    int num_cus = 256;
    bool tuned = false, ran = false;
};

} // namespace sccamd
