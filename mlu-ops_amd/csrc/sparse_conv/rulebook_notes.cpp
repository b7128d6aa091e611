// Notes about rulebooks built on a handle: which pair tensors came from
// mluOpGetIndicePairs, and whether their input rows were in cell order.
#include "sparse_conv/rulebook_notes.h"

namespace mluop {
namespace sparse_conv {

RulebookReportTarget openRulebookNote(mluOpContext *handle, const void *pairs, int K, int L) {
  // older notes about this memory describe tensors that are being overwritten
  handle->forgetNotesIn(pairs, (size_t)K * 2 * (size_t)L * sizeof(int32_t));
  const int slot = handle->next_rulebook_note;
  handle->next_rulebook_note = (slot + 1) % mluOpContext::kRulebookNotes;
  mluOpContext::RulebookNote &note = handle->rulebook_notes[slot];
  note.pairs = pairs;
  note.K = K;
  note.L = L;
  note.stamp = handle->next_stamp++;
  note.counts_on_file = false;
  // no word of another rulebook passes for one of this
  unsigned long long *const report = handle->rulebook_reports + slot;
  const unsigned long long empty = stampedWord(~note.stamp, 0);
  __atomic_store_n(report, empty, __ATOMIC_RELAXED);
  RulebookReportTarget t;
  t.stamp = note.stamp;
  // A captured rulebook files no report in host memory: nothing runs now, so no report of
  // this call could arrive, and a replay must not write into a slot that by then belongs to
  // another rulebook (or to a handle that is gone).
  hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(handle->queue, &capturing) != hipSuccess) (void)hipGetLastError();
  if (capturing == hipStreamCaptureStatusNone) {
    t.order_word = report;
    if (K <= mluOpContext::kCountWords) {
      t.count_words = handle->count_words + (size_t)slot * mluOpContext::kCountWords;
      for (int k = 0; k < K; ++k) __atomic_store_n(t.count_words + k, empty, __ATOMIC_RELAXED);
      note.counts_on_file = true;
    }
  }
  return t;
}

RulebookReportTarget rulebookReport(const mluOpContext *handle, const void *pairs, int K) {
  RulebookReportTarget t;
  for (int slot = 0; slot < mluOpContext::kRulebookNotes; ++slot) {
    const mluOpContext::RulebookNote &note = handle->rulebook_notes[slot];
    if (note.pairs != pairs || note.K != K || !note.counts_on_file) continue;
    t.stamp = note.stamp;
    t.order_word = handle->rulebook_reports + slot;
    t.count_words = handle->count_words + (size_t)slot * mluOpContext::kCountWords;
    break;
  }
  return t;
}

void consultRulebookNotes(mluOpContext *handle, int row_column, ConvProblem *p) {
  p->ticket = handle->next_stamp++;
  p->list_trust = ListTrust::kNone;
  if (handle->rulebook_reports == nullptr) return;
  for (int slot = 0; slot < mluOpContext::kRulebookNotes; ++slot) {
    const mluOpContext::RulebookNote &note = handle->rulebook_notes[slot];
    if (note.pairs != p->indice_pairs || note.K != p->K || note.L != p->L) continue;
    const unsigned long long report = __atomic_load_n(handle->rulebook_reports + slot, __ATOMIC_ACQUIRE);
    // (false: not arrived, or never sent: a captured rulebook files none)
    const bool arrived = report >> 32 == (note.stamp & 0xffffffffull), in_order = (uint32_t)report != 0;
    p->scattered = arrived && !in_order;
    if (row_column == 0)
      p->list_trust = ListTrust::kInOrder;
    else if (!arrived)
      p->list_trust = ListTrust::kUnknown;
    else
      p->list_trust = in_order ? ListTrust::kInOrder : ListTrust::kNone;
    return;
  }
}

}  // namespace sparse_conv
}  // namespace mluop
