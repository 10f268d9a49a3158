set -o pipefail
(cp magicdec_amd/ops.py _work/ops_new.py && cp _work/ops_old.py magicdec_amd/ops.py && ! timeout -k 10 200 python -u -m pytest -x -q --timeout 120 --timeout-method thread tests/test_gpu_latent.py -k embed_bigram > gpurun_out/embed_old.log 2>&1; cp _work/ops_new.py magicdec_amd/ops.py) &&
timeout -k 10 200 python -u -m pytest -x -q --timeout 120 --timeout-method thread tests/test_gpu_latent.py tests/test_gpu_step_ops.py > gpurun_out/embed_new.log 2>&1 &&
timeout -k 10 400 python -u _work/m_rule.py > gpurun_out/m_rule.txt 2>&1 &&
timeout -k 10 400 python -u _work/m_stream.py > gpurun_out/m_stream.txt 2>&1
