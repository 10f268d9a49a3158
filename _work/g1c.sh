(bash _work/g1.sh); rc=$?; tail -5 gpurun_out/embed_old.log gpurun_out/embed_new.log gpurun_out/m_stream.txt; exit $rc
