// What a step brings to the device beside its products, each in one launch: the block tables' new entries, the states of slots that
// went to a new request, and what changes between two replays of a captured decode step.
//
// All of it is launches, not bytes.  A copy a row and a fill a state took 2.9 to 4.6 us each, and an index made from a list had the
// host wait for the stream.  Whole passes, us: 64 sequences that take over their cached pages and 8 decode steps 9,498 -> 9,030; a prompt
// of 1,999 tokens in 12 layers with 12 states 6,285 -> 5,699.
#include "common.h"

namespace {

// plan: for each row {slot, first entry, how many, where its entries begin in `plan`}, the entries behind them
__global__ void __launch_bounds__(256)
table_rows_kernel(const int* __restrict__ plan, int* __restrict__ table, int width) {
    const int* row = plan + blockIdx.x * 4;
    const int slot = row[0], first = row[1], count = row[2];
    const int* from = plan + row[3];
    int* to = table + static_cast<size_t>(slot) * width + first;
    for (int i = threadIdx.x; i < count; i += 256) to[i] = from[i];
}

// states: for each {address, bytes of a slot's row}
typedef unsigned int words4_t __attribute__((ext_vector_type(4)));

__global__ void __launch_bounds__(256)
clear_rows_kernel(const long* __restrict__ states, const int* __restrict__ slots) {
    const long bytes = states[2 * blockIdx.y + 1];
    char* row = reinterpret_cast<char*>(states[2 * blockIdx.y]) + bytes * slots[blockIdx.z];
    const long first = static_cast<long>(blockIdx.x) * 256 + threadIdx.x, apart = static_cast<long>(gridDim.x) * 256;
    if (bytes % 16 == 0) {  // (the states begin at 16-byte addresses, so every row does)
        for (long i = first; i < bytes / 16; i += apart) reinterpret_cast<words4_t*>(row)[i] = words4_t{0u, 0u, 0u, 0u};
    } else {
        for (long i = first; i < bytes / 2; i += apart) reinterpret_cast<unsigned short*>(row)[i] = 0;
    }
}

constexpr int kStepRows = 128;  // the numbers travel as the kernel's arguments: 2 KB of them

struct StepRows {
    int tokens[kStepRows], positions[kStepRows], slots[kStepRows], feed[kStepRows];
    int n, size, max_context, pad_slot;
    int *token_ids, *positions_at, *seq_start, *seq_slot, *token_feed, *max_context_at;
    void** result_at;  // takes `result`, the address that the replay's last product writes to
    void* result;
};

__global__ void __launch_bounds__(kStepRows) step_rows_kernel(StepRows a) {
    const int i = threadIdx.x;
    if (i == 0) *a.max_context_at = a.max_context;
    if (i == 0 && a.result_at) *a.result_at = a.result;
    if (i >= a.size) return;
    const bool real = i < a.n;
    a.token_ids[i] = real ? a.tokens[i] : 0;
    a.positions_at[i] = real ? a.positions[i] : 0;
    a.seq_start[i] = real ? a.positions[i] : 0;
    a.seq_slot[i] = real ? a.slots[i] : a.pad_slot;
    a.token_feed[i] = real ? a.feed[i] : -1;
}

}  // namespace

// `plan` (on the device) as above for `rows` rows of one table.
CIE_API int cie_table_rows(void* stream, const int* plan, int rows, int* table, int width) {
    if (rows < 1 || width < 1 || !plan || !table) return CIE_BAD_ARGUMENT;
    table_rows_kernel<<<rows, 256, 0, static_cast<hipStream_t>(stream)>>>(plan, table, width);
    return cie_after_launch();
}

// Zeroes row slots[j] (on the device) of each state; `most_bytes`: the largest row.
CIE_API int cie_clear_rows(void* stream, const long* states, int n_states, const int* slots, int n_slots, long most_bytes) {
    if (n_states < 1 || n_states > 65535 || n_slots < 1 || n_slots > 65535 || most_bytes < 2 || !states || !slots) return CIE_BAD_ARGUMENT;
    const long blocks = (most_bytes / 16 + 1023) / 1024;  // (some four pieces a thread of the largest)
    clear_rows_kernel<<<dim3(static_cast<unsigned>(blocks < 1 ? 1 : blocks > 256 ? 256 : blocks), n_states, n_slots), 256, 0,
                        static_cast<hipStream_t>(stream)>>>(states, slots);
    return cie_after_launch();
}

// A captured decode step's numbers: `values` (host memory, read before this returns) holds n tokens, n positions, n slots and, if
// `fed`, n places of the token pool.  Rows n .. size - 1 become padding on pad_slot.  result_at (or null) takes `result`.
CIE_API int cie_step_rows(void* stream, const int* values, int n, int size, int fed, int max_context, int pad_slot, int* token_ids,
                          int* positions, int* seq_start, int* seq_slot, int* token_feed, int* max_context_at, void** result_at,
                          void* result) {
    if (n < 0 || n > size || size < 1 || size > kStepRows || !values || !token_ids || !positions || !seq_start || !seq_slot || !token_feed ||
        !max_context_at)
        return CIE_BAD_ARGUMENT;
    StepRows a;
    for (int i = 0; i < n; ++i) {
        a.tokens[i] = values[i];
        a.positions[i] = values[n + i];
        a.slots[i] = values[2 * n + i];
        a.feed[i] = fed ? values[3 * n + i] : -1;
    }
    for (int i = n; i < kStepRows; ++i) a.tokens[i] = a.positions[i] = a.slots[i] = a.feed[i] = 0;
    a.n = n;
    a.size = size;
    a.max_context = max_context;
    a.pad_slot = pad_slot;
    a.token_ids = token_ids;
    a.positions_at = positions;
    a.seq_start = seq_start;
    a.seq_slot = seq_slot;
    a.token_feed = token_feed;
    a.max_context_at = max_context_at;
    a.result_at = result_at;
    a.result = result;
    step_rows_kernel<<<1, kStepRows, 0, static_cast<hipStream_t>(stream)>>>(a);
    return cie_after_launch();
}
